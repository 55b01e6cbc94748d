// MI355X (gfx950) element-wise kernels of the MFT path: GEMM operands (pupil
// phasors or complex data), twiddle tables, detector accumulation, Field
// products and fills.
#include "mftx_device.h"

#include <algorithm>
#include <type_traits>

namespace mftx {

// dtype codes: 0 complex64, 1 float32, 2 complex128, 3 float64
__device__ __forceinline__ float2 load_elem(const void* p, int dtype, long long idx) {
  switch (dtype) {
    case 0: {
      const v2f32 v = ((gptr<const v2f32>)p)[idx];
      return make_float2(v.x, v.y);
    }
    case 1: return make_float2(((gptr<const float>)p)[idx], 0.f);
    case 2: {
      const v2f64 v = ((gptr<const v2f64>)p)[idx];
      return make_float2((float)v.x, (float)v.y);
    }
    default: return make_float2((float)((gptr<const double>)p)[idx], 0.f);
  }
}

// Index of the op that block b0 (its first thread) belongs to: ops start on
// block boundaries, so the search runs on block-uniform values (scalar loads).
template <typename Op>
__device__ __forceinline__ int block_op(const Op* __restrict__ ops, int nops, long long b0) {
  int lo = 0, hi = nops - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (ops[mid].begin <= b0) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

__device__ __forceinline__ double load_real(const void* p, int dtype, long long idx) {
  return dtype == 3 ? ((const double*)p)[idx] : (double)((const float*)p)[idx];
}

// u / d and u % d; the 64-bit division is a long instruction sequence
__device__ __forceinline__ void div_mod(long long u, long long d, long long& q, int& r) {
  if (((u | d) >> 32) == 0) {
    q = (unsigned)u / (unsigned)d;
    r = (int)((unsigned)u - (unsigned)q * (unsigned)d);
  } else {
    q = u / d;
    r = (int)(u - q * d);
  }
}

// Largest value of the block's threads, in every thread (all of them call it).
__device__ __forceinline__ float block_max(float v) {
  __shared__ float w[kGroupBlock / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
  __syncthreads();
  v = w[0];
#pragma unroll
  for (int i = 1; i < kGroupBlock / 64; ++i) v = fmaxf(v, w[i]);
  return v;
}

constexpr float kMaxFloat = 3.4028234663852886e38f;

// Bound over elements [first, m * n) in steps of `step` of an m x n array:
// |re| + |im|, 0 for an element that is not finite (it makes its results
// non-finite whatever the scale), FP32's largest number where the sum of two
// finite parts is past it (at most twice that: scaled operands then reach 2^15
// instead of 2^14, still half of f16's range).  The dtype is tested outside the loop, so
// the loads of 8 elements are in flight together.  SUM: the elements' bounds are
// added up in *sum too.
template <bool SUM, typename Get>
__device__ __forceinline__ float bound_of(long long m, long long n, long long ld, long long first, long long step,
                                          double* sum, Get&& get) {
  float v = 0.f;
  double total_bound = 0.0;
  const long long total = m * n;
  auto one = [&](long long i) {
    const float2 e = get(ld == n ? i : total < (1LL << 31) ? (long long)((unsigned)i / (unsigned)n) * ld + (unsigned)i % (unsigned)n
                                                           : i / n * ld + i % n);
    const float ax = fabsf(e.x), ay = fabsf(e.y);
    return ax <= kMaxFloat && ay <= kMaxFloat ? fminf(ax + ay, kMaxFloat) : 0.f;
  };
  long long i = first;
  for (; i + 7 * step < total; i += 8 * step) {
    float b[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) b[q] = one(i + q * step);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      v = fmaxf(v, b[q]);
      if (SUM) total_bound += (double)b[q];
    }
  }
  for (; i < total; i += step) {
    const float b = one(i);
    v = fmaxf(v, b);
    if (SUM) total_bound += (double)b;
  }
  if (SUM) *sum = total_bound;
  return v;
}
template <bool SUM>
__device__ __forceinline__ float array_bound_sum(const void* src, int dtype, long long m, long long n, long long ld,
                                                 long long first, long long step, double* sum) {
  switch (dtype) {
    case 0:
      return bound_of<SUM>(m, n, ld, first, step, sum, [&](long long i) {
        const v2f32 e = ((gptr<const v2f32>)src)[i];
        return make_float2(e.x, e.y);
      });
    case 1:
      return bound_of<SUM>(m, n, ld, first, step, sum,
                           [&](long long i) { return make_float2(((gptr<const float>)src)[i], 0.f); });
    case 2: return bound_of<SUM>(m, n, ld, first, step, sum, [&](long long i) { return load_elem(src, 2, i); });
    default: return bound_of<SUM>(m, n, ld, first, step, sum, [&](long long i) { return load_elem(src, 3, i); });
  }
}
__device__ __forceinline__ float array_bound(const void* src, int dtype, long long m, long long n, long long ld,
                                             long long first, long long step) {
  return array_bound_sum<false>(src, dtype, m, n, ld, first, step, nullptr);
}

__global__ void absmax_kernel(const MaxOp* __restrict__ ops, int nops) {
  const MaxOp& op = ops[block_op(ops, nops, (long long)blockIdx.x)];
  const int b = (int)((long long)blockIdx.x - op.begin);
  const float v = block_max(array_bound(op.src, op.dtype, op.m, op.n, op.ld, (long long)b * kGroupBlock + threadIdx.x,
                                        (long long)op.nblk * kGroupBlock));
  if (threadIdx.x == 0) op.part[b] = v;
}

hipError_t launch_absmax(const MaxOp* ops, int nops, long long total_blocks, hipStream_t s) {
  if (total_blocks <= 0 || nops <= 0) return hipSuccess;
  hipLaunchKernelGGL(absmax_kernel, dim3((unsigned)total_blocks), dim3(kGroupBlock), 0, s, ops, nops);
  return hipGetLastError();
}

// Exponent of the power of two that takes 4 * bound to at most 2^14 (0 for
// bound 0): -116 to 149, whose inverse is the smallest denormal.  Up to 2^-137
// it is the one wanted; the denormals below have few bits to lose.
__device__ __forceinline__ int operand_exponent(float bound) {
  return bound > 0.f ? min(12 - __builtin_amdgcn_frexp_expf(bound), 149) : 0;  // bound < 2^frexp_exp
}
// x * 2^e, exact (past 2^127 no float holds the factor)
__device__ __forceinline__ float scaled(float x, int e) { return __builtin_amdgcn_ldexpf(x, e); }

// The scale (its exponent) of an operand source (every thread of the block calls it).
__device__ __forceinline__ int block_scale(const ScaleSrc& sc, bool first) {
  if (sc.n == 0) return 0;
  float v = 0.f;
  for (int i = threadIdx.x; i < sc.n; i += kGroupBlock) v = fmaxf(v, sc.part[i]);
  const int e = operand_exponent(block_max(v));
  if (first && threadIdx.x == 0) *sc.inv = scaled(1.0f, -e);
  return e;
}

// --------------------------------------------------------------------------
// GEMM operands: pupil phasors  f = amp * exp(2*pi*i*opd/lambda)  (plane.py:507)
// or complex data, times both stages' folds, paired along both axes
// --------------------------------------------------------------------------

// Sample pair i of an n-sample axis: indices midpoint + x' and midpoint - x'
// (x' = i + 1/2 for even n, i for odd; -1 where there is none: past the end,
// or the middle sample's partner).
__device__ __forceinline__ void pair_index(int n, int i, int& plus, int& minus) {
  const int h = n >> 1;
  plus = h + i < n ? h + i : -1;
  minus = n & 1 ? (i > 0 ? h - i : -1) : h - 1 - i;
  if (minus < 0) minus = -1;
}

__device__ __forceinline__ PhasorWave load_wave(cptr<const PhasorWave> p) {
  PhasorWave w;
  w.inv_wl = p->inv_wl;
  w.fold = p->fold;
  w.x0 = p->x0;
  w.fold2 = p->fold2;
  w.x02 = p->x02;
  return w;
}

// One thread per (op, 16-pair row block, K block of 16 pairs, row pair of the
// block, NP of the K block's pairs, group of sp.waves wavelengths): NP K pairs
// of one row pair, 4 NP source samples, read once; for each wavelength the four
// samples of a (row, K) quad, each with its phase
//     opd * inv_wl + fold * (x0 + k) + fold2 * (x02 + r),
// are combined into the even and odd rows' even and odd parts, split and
// stored as 16 pieces of 2 NP bytes.  Threads run along K within a row's 8
// pairs, then along the rows, so a store covers whole 256-byte runs.
//
// Bound by the arithmetic of the phases (about 40 instructions per sample and
// wavelength, several FP64) beside the stores.  NP = 4 holds 48 registers of
// source and 32 of result, four waves per SIMD; 8 pairs left room for two.
// Where every sample of a wave is outside the aperture (amplitude 0) the
// phases are skipped.
// DT: the dtype of a complex source.
template <int PREC, bool CPLX, int NP, int DT, typename Waves>
__device__ __forceinline__ void operand_thread(const PhasorOp& op, Waves&& wave, int waves, long long u, int scale) {
  auto fit = [&](float x) { return PREC == PREC_FP32 ? scaled(x, scale) : x; };
  static_assert(NP == 2 || NP == 4, "a thread's pairs lie in one half of a K block, its pieces are one or two words");
  constexpr int SUB = 8 / NP;  // threads per (row pair, half K block)
  const int R = op.trans ? op.n : op.m, K = op.trans ? op.m : op.n;
  const int nrb = pair_blocks(R), nkb = pair_blocks(K);
  // a wavelength group spans whole waves, so its descriptors are scalar loads
  const long long per_group = group_threads(R, K, NP);
  long long group;
  int v;
  div_mod(u, per_group, group, v);
  const int g = __builtin_amdgcn_readfirstlane((int)group);
  if (v >= 32 * SUB * nrb * nkb) return;
  const int sub = v & (SUB - 1), lr = (v / SUB) & 15, kh = (v / (16 * SUB)) & 1, blk = v / (32 * SUB);
  const int kb = (unsigned)blk % (unsigned)nkb, rb = (unsigned)blk / (unsigned)nkb;
  int r2[2];
  pair_index(R, rb * 16 + lr, r2[0], r2[1]);
  const int kp0 = kb * 16 + kh * 8 + sub * NP;
  const bool even_k = !(K & 1);
  const int kh2 = K >> 1;
  // K index of pair kp0 + i: plus side kplus0 + i, minus side kminus0 - i
  const int kplus0 = kh2 + kp0, kminus0 = even_k ? kh2 - 1 - kp0 : kh2 - kp0;
  const int w0 = g * waves, nw = min(op.nwave - w0, waves);
  char* out = (char*)op.dst + ((long long)rb * nkb + kb) * A_BLOCK + 16 * (lr + 32 * kh) + 2 * NP * sub;

  // every load is issued before any math and none sits behind a branch: a
  // sample outside the array reads element 0 and is zeroed afterwards
  float a[2][2][NP];                          // amplitude [row side][k side][pair]
  double o[CPLX ? 1 : 2][CPLX ? 1 : 2][CPLX ? 1 : NP];
  float ci[CPLX ? 2 : 1][CPLX ? 2 : 1][CPLX ? NP : 1];
#pragma unroll
  for (int rs = 0; rs < 2; ++rs)
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      long long ia[NP];
      bool in[NP];
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int k = ks ? kminus0 - i : kplus0 + i;
        in[i] = r2[rs] >= 0 && k >= 0 && k < K && !(ks && !even_k && kp0 + i == 0);
        const long long r = r2[rs], kk = k;
        ia[i] = in[i] ? (op.trans ? kk * op.ld_amp + r : r * op.ld_amp + kk) : 0;
      }
      if constexpr (CPLX) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
          const float2 e = load_elem(op.amp, DT, ia[i]);
          a[rs][ks][i] = in[i] ? fit(e.x) : 0.f;
          ci[rs][ks][i] = in[i] ? fit(op.conj ? -e.y : e.y) : 0.f;
        }
      } else {
        if (op.amp_dtype == 3) {
#pragma unroll
          for (int i = 0; i < NP; ++i) a[rs][ks][i] = (float)((gptr<const double>)op.amp)[ia[i]];
        } else {
#pragma unroll
          for (int i = 0; i < NP; ++i) a[rs][ks][i] = ((gptr<const float>)op.amp)[ia[i]];
        }
#pragma unroll
        for (int i = 0; i < NP; ++i) {
          const int k = ks ? kminus0 - i : kplus0 + i;
          const long long r = r2[rs], kk = k;
          ia[i] = in[i] ? (op.trans ? kk * op.ld_opd + r : r * op.ld_opd + kk) : 0;
        }
        if (op.opd_dtype == 3) {
#pragma unroll
          for (int i = 0; i < NP; ++i) o[rs][ks][i] = ((gptr<const double>)op.opd)[ia[i]];
        } else {
#pragma unroll
          for (int i = 0; i < NP; ++i) o[rs][ks][i] = (double)((gptr<const float>)op.opd)[ia[i]];
        }
#pragma unroll
        for (int i = 0; i < NP; ++i) {
          a[rs][ks][i] = in[i] ? fit(a[rs][ks][i]) : 0.f;
          o[rs][ks][i] = in[i] ? o[rs][ks][i] : 0.0;
        }
      }
    }
  bool lit = true;
  if constexpr (!CPLX) {
    // a phase that is not finite makes even a dark sample's phasor NaN
    lit = false;
#pragma unroll
    for (int i = 0; i < 4 * NP; ++i) {
      const float x = a[i / (2 * NP)][i / NP % 2][i % NP];
      const double y = o[i / (2 * NP)][i / NP % 2][i % NP];
      lit = lit || x != 0.f || !(__builtin_fabs(y) < 1e300);
    }
    lit = __any(lit);
  }
#pragma unroll 1
  for (int j = 0; j < nw; ++j) {
    const PhasorWave pw = wave(w0 + j);
    const bool folded = pw.fold != 0.0 || pw.fold2 != 0.0;
    uint32_t w[2][2][4][NP / 2];  // [row parity][part][plane][word]
    if (!lit) {
#pragma unroll
      for (int i = 0; i < 16 * (NP / 2); ++i) w[i / (8 * NP / 2)][i / (4 * NP / 2) % 2][i / (NP / 2) % 4][i % (NP / 2)] = 0u;
    } else {
      // phase of pair 0 of each quadrant; K advances by +-1 per pair
      double base[2][2];
#pragma unroll
      for (int rs = 0; rs < 2; ++rs)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
          base[rs][ks] = __builtin_fma(pw.fold, pw.x0 + (double)(ks ? kminus0 : kplus0),
                                       pw.fold2 * (pw.x02 + (double)r2[rs]));
#pragma unroll
      for (int t = 0; t < NP / 2; ++t) {
        float2 p[2][2][2];  // [row parity][part][pair]
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int i = 2 * t + q;
          float2 e[2][2];
#pragma unroll
          for (int rs = 0; rs < 2; ++rs)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
              const double ph = __builtin_fma(ks ? -pw.fold : pw.fold, (double)i, base[rs][ks]);
              if constexpr (CPLX) {
                const float2 z = make_float2(a[rs][ks][i], ci[rs][ks][i]);
                e[rs][ks] = folded ? cmul(z, cis_quarter(ph)) : z;
              } else {
                const float2 c = cis_quarter(__builtin_fma(o[rs][ks][i], pw.inv_wl, ph));
                e[rs][ks] = make_float2(a[rs][ks][i] * c.x, a[rs][ks][i] * c.y);
              }
            }
#pragma unroll
          for (int par = 0; par < 2; ++par) {
            const float2 kp = par ? make_float2(e[0][0].x - e[1][0].x, e[0][0].y - e[1][0].y)
                                  : make_float2(e[0][0].x + e[1][0].x, e[0][0].y + e[1][0].y);
            const float2 km = par ? make_float2(e[0][1].x - e[1][1].x, e[0][1].y - e[1][1].y)
                                  : make_float2(e[0][1].x + e[1][1].x, e[0][1].y + e[1][1].y);
            p[par][0][q] = make_float2(kp.x + km.x, kp.y + km.y);
            p[par][1][q] = make_float2(kp.x - km.x, kp.y - km.y);
          }
        }
#pragma unroll
        for (int par = 0; par < 2; ++par)
#pragma unroll
          for (int part = 0; part < 2; ++part) {
            split2<PREC>(p[par][part][0].x, p[par][part][1].x, w[par][part][0][t], w[par][part][1][t]);
            split2<PREC>(p[par][part][0].y, p[par][part][1].y, w[par][part][2][t], w[par][part][3][t]);
          }
      }
    }
    char* d = out + (long long)(w0 + j) * op.wave_stride;
#pragma unroll
    for (int par = 0; par < 2; ++par)
#pragma unroll
      for (int part = 0; part < 2; ++part)
#pragma unroll
        for (int pl = 0; pl < 4; ++pl) {
          const uint32_t (&x)[NP / 2] = w[par][part][pl];
          char* dp = d + (part * 4 + pl) * FRAG + par * 256;
          if constexpr (NP == 4) *(gptr<v2u32>)dp = v2u32{x[0], x[1]};
          else *(gptr<uint32_t>)dp = x[0];
        }
  }
}

// operand_thread for the op's source dtype (tested once per thread: a test per
// load would wait for each)
template <int PREC, bool CPLX, int NP, typename Waves>
__device__ __forceinline__ void operand_source(const PhasorOp& op, Waves&& wave, int waves, long long u, int scale) {
  if constexpr (!CPLX) {
    operand_thread<PREC, false, NP, 0>(op, wave, waves, u, scale);
  } else {
    switch (op.amp_dtype) {
      case 0: operand_thread<PREC, true, NP, 0>(op, wave, waves, u, scale); break;
      case 1: operand_thread<PREC, true, NP, 1>(op, wave, waves, u, scale); break;
      case 2: operand_thread<PREC, true, NP, 2>(op, wave, waves, u, scale); break;
      default: operand_thread<PREC, true, NP, 3>(op, wave, waves, u, scale);
    }
  }
}

// Every operand source of a plan in one launch (the op is found by a
// block-uniform search).
template <int PREC, bool CPLX, int NP>
__global__ __launch_bounds__(kGroupBlock, 4) void operand_group_kernel(const PhasorOp* __restrict__ ops, int nops,
                                                                       int waves) {
  const long long b0 = (long long)blockIdx.x * kGroupBlock;
  const PhasorOp& op = ops[block_op(ops, nops, b0)];
  const int scale = block_scale(op.sc, b0 == op.begin);
  const long long u = b0 + threadIdx.x - op.begin;
  if (u >= operand_threads(op.trans ? op.n : op.m, op.trans ? op.m : op.n, op.nwave, OperandSplit{NP, waves})) return;
  operand_source<PREC, CPLX, NP>(op, [&](int w) { return load_wave((cptr<const PhasorWave>)op.waves + w); }, waves, u,
                                 scale);
}

template <int PREC, bool CPLX>
static void launch_operands_of(OperandSplit sp, dim3 grid, const PhasorOp* ops, int nops, hipStream_t s) {
  if (sp.np == 2)
    hipLaunchKernelGGL((operand_group_kernel<PREC, CPLX, 2>), grid, dim3(kGroupBlock), 0, s, ops, nops, sp.waves);
  else
    hipLaunchKernelGGL((operand_group_kernel<PREC, CPLX, 4>), grid, dim3(kGroupBlock), 0, s, ops, nops, sp.waves);
}

hipError_t launch_operands(int prec, bool cplx, OperandSplit sp, const PhasorOp* ops, int nops, long long total,
                           hipStream_t s) {
  if (total <= 0 || nops <= 0) return hipSuccess;
  const dim3 grid((unsigned)((total + kGroupBlock - 1) / kGroupBlock));
  if (prec == PREC_BF16X3) {
    if (cplx) launch_operands_of<PREC_BF16X3, true>(sp, grid, ops, nops, s);
    else launch_operands_of<PREC_BF16X3, false>(sp, grid, ops, nops, s);
  } else {
    if (cplx) launch_operands_of<PREC_FP32, true>(sp, grid, ops, nops, s);
    else launch_operands_of<PREC_FP32, false>(sp, grid, ops, nops, s);
  }
  return hipGetLastError();
}

// --------------------------------------------------------------------------
// twiddle tables
// --------------------------------------------------------------------------

// (cos, sin)(2 pi t) in FP64 for t in turns: t is reduced to a quarter-turn
// index and a remainder |a| <= pi/4, whose Taylor series to degree 13 (sin)
// and 14 (cos) are below 1e-13 off there.
__device__ __forceinline__ double2 cis_turns64(double t) {
  const double q = t * 4.0;
  const double n = __builtin_rint(q);
  const int quad = (int)n;  // |q| below 2^31, as for cis_quarter
  const double a = (q - n) * 1.57079632679489661923, a2 = a * a;
  double s = 1.0 / 6227020800.0;
  s = __builtin_fma(s, a2, -1.0 / 39916800.0);
  s = __builtin_fma(s, a2, 1.0 / 362880.0);
  s = __builtin_fma(s, a2, -1.0 / 5040.0);
  s = __builtin_fma(s, a2, 1.0 / 120.0);
  s = __builtin_fma(s, a2, -1.0 / 6.0);
  s = __builtin_fma(a * a2, s, a);
  double c = -1.0 / 87178291200.0;
  c = __builtin_fma(c, a2, 1.0 / 479001600.0);
  c = __builtin_fma(c, a2, -1.0 / 3628800.0);
  c = __builtin_fma(c, a2, 1.0 / 40320.0);
  c = __builtin_fma(c, a2, -1.0 / 720.0);
  c = __builtin_fma(c, a2, 1.0 / 24.0);
  c = __builtin_fma(c, a2, -0.5);
  c = __builtin_fma(c, a2, 1.0);
  const double re = quad & 1 ? s : c, im = quad & 1 ? c : s;
  return make_double2((quad + 1) & 2 ? -re : re, quad & 2 ? -im : im);
}

// One thread per (slot, 2 k').  The values are correctly rounded to the
// format's hi + lo but for 1e-13, tighter than FP32 twiddles.
template <int PREC>
__device__ __forceinline__ void table_thread(const TableOp& op, long long u) {
  const int t = (int)(u & 3), l = (int)(u >> 2) & 63;
  long long sb;
  int kb;
  div_mod(u >> 8, op.nkb, sb, kb);
  const double y = op.y0 + (double)((op.sb0 + (int)sb) * 32 + (l & 31));
  const double x0 = op.x0 + (double)(kb * 16 + 8 * (l >> 5) + 2 * t);
  const float ts = tw_scale(PREC);
  double2 v[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    v[q] = cis_turns64(op.alpha * ((x0 + (double)q) * y));
    v[q].x *= ts;
    v[q].y *= ts;
  }
  auto pk = [](float x, float z) { return PREC == PREC_BF16X3 ? pack_bf16(x, z) : pack_f16(x, z); };
  auto widen = [](uint32_t h, int q) -> double {
    if constexpr (PREC == PREC_BF16X3) return q ? bf16_hi_to_f32(h) : bf16_lo_to_f32(h);
    else return (double)(float)(__builtin_bit_cast(f16x2_t, h)[q]);
  };
  const uint32_t ch = pk((float)v[0].x, (float)v[1].x), sh = pk((float)v[0].y, (float)v[1].y);
  const uint32_t cl = pk((float)(v[0].x - widen(ch, 0)), (float)(v[1].x - widen(ch, 1)));
  const uint32_t sl = pk((float)(v[0].y - widen(sh, 0)), (float)(v[1].y - widen(sh, 1)));
  char* d = (char*)op.dst + (sb * op.nkb + kb) * B_BLOCK + 16 * l + 4 * t;
  *(gptr<uint32_t>)d = ch;
  *(gptr<uint32_t>)(d + FRAG) = cl;
  *(gptr<uint32_t>)(d + 2 * FRAG) = sh;
  *(gptr<uint32_t>)(d + 3 * FRAG) = sl;
}

template <int PREC>
__global__ void table_group_kernel(const TableOp* __restrict__ ops, int nops, long long first) {
  const long long b0 = first + (long long)blockIdx.x * kGroupBlock;
  const TableOp& op = ops[block_op(ops, nops, b0)];
  const long long u = b0 + threadIdx.x - op.begin;
  if (u < table_threads(op.nsb, op.nkb)) table_thread<PREC>(op, u);
}

hipError_t launch_tables(int prec, const TableOp* ops, int nops, long long total, hipStream_t s) {
  if (nops <= 0) return hipSuccess;
  // a launch holds fewer than 2^32 threads: 64 GiB of tables (more were cut off without an error)
  constexpr long long kMost = 1LL << 31;
  for (long long first = 0; first < total; first += kMost) {
    const dim3 grid((unsigned)((std::min(total - first, kMost) + kGroupBlock - 1) / kGroupBlock)), block(kGroupBlock);
    if (prec == PREC_BF16X3) hipLaunchKernelGGL((table_group_kernel<PREC_BF16X3>), grid, block, 0, s, ops, nops, first);
    else hipLaunchKernelGGL((table_group_kernel<PREC_FP32>), grid, block, 0, s, ops, nops, first);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

__global__ void row_phase_kernel(const RowPhase* __restrict__ ops) {
  const RowPhase op = ops[blockIdx.y];
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= op.rows) return;
  const double2 v = cis_turns64(op.rate * ((double)t - op.centre));
  op.table[t] = make_float2((float)v.x, (float)v.y);
}

hipError_t launch_row_phases(const RowPhase* ops, int nops, int most_rows, hipStream_t s) {
  for (int b = 0; b < nops && most_rows > 0; b += 65535)
    hipLaunchKernelGGL(row_phase_kernel, dim3((unsigned)((most_rows + 255) / 256), std::min(nops - b, 65535)), dim3(256),
                       0, s, ops + b);
  return hipGetLastError();
}

// --------------------------------------------------------------------------
// one transform: absolute maximum, then operand, both tables and the GEMMs'
// descriptors in one launch, everything passed by value
// --------------------------------------------------------------------------
template <int PREC>
__global__ __launch_bounds__(kGroupBlock, 4) void prepare_one_kernel(PhasorOp op, PhasorWave wave, TableOp tab0,
                                                                     TableOp tab1, OneDesc desc, OneDesc* out,
                                                                     int op_blocks, int tab_blocks) {
  const int b = (int)blockIdx.x;
  if (b < op_blocks) {
    int scale = 0;
    if (PREC == PREC_FP32) {
      if (op.sc.n == 0) {  // a small source: every block takes its maximum
        scale = operand_exponent(block_max(array_bound(op.amp, op.amp_dtype, op.m, op.n, op.ld_amp, threadIdx.x,
                                                       kGroupBlock)));
        if (b == 0 && threadIdx.x == 0) *op.sc.inv = scaled(1.0f, -scale);
      } else {
        scale = block_scale(op.sc, b == 0);
      }
    }
    if (b == 0 && threadIdx.x == 0) *out = desc;
    const long long u = (long long)b * kGroupBlock + threadIdx.x;
    if (u < operand_threads(op.trans ? op.n : op.m, op.trans ? op.m : op.n, 1, OperandSplit{2, 1}))
      operand_source<PREC, true, 2>(op, [=](int) { return wave; }, 1, u, scale);
    return;
  }
  long long u = (long long)(b - op_blocks) * kGroupBlock + threadIdx.x;
  if (b - op_blocks < tab_blocks) {
    if (u < table_threads(tab0.nsb, tab0.nkb)) table_thread<PREC>(tab0, u);
    return;
  }
  u -= (long long)tab_blocks * kGroupBlock;
  if (u < table_threads(tab1.nsb, tab1.nkb)) table_thread<PREC>(tab1, u);
}

template <int PREC>
__global__ void table_one_kernel(TableOp op) {
  const long long u = (long long)blockIdx.x * kGroupBlock + threadIdx.x;
  if (u < table_threads(op.nsb, op.nkb)) table_thread<PREC>(op, u);
}

// Sum of v over the block (every thread calls it once).
__device__ double block_sum(double v) {
  __shared__ double w[kGroupBlock / 64];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
  __syncthreads();
  v = 0.0;
  for (int i = 0; i < kGroupBlock / 64; ++i) v += w[i];
  return v;
}

// SUM: also sums[b], the sum of block b's element bounds.
template <bool SUM>
__global__ void absmax_one_kernel(MaxOp op, double* __restrict__ sums) {
  double sum = 0.0;
  const float v = block_max(array_bound_sum<SUM>(op.src, op.dtype, op.m, op.n, op.ld,
                                                 (long long)blockIdx.x * kGroupBlock + threadIdx.x,
                                                 (long long)op.nblk * kGroupBlock, &sum));
  if (threadIdx.x == 0) op.part[blockIdx.x] = v;
  if (SUM) {
    sum = block_sum(sum);
    if (threadIdx.x == 0) sums[blockIdx.x] = sum;
  }
}

// Raises the source's bound to 2^-16 of the sum S of its samples: the operand's
// scale 2^e then keeps S 2^e, and so stage 1's sums over any number of pairs,
// below 2^28, 2^14 after the store's 2^-14 (one block, n <= kGroupBlock).
__global__ void long_bound_kernel(float* __restrict__ part, const double* __restrict__ sums, int n) {
  const double s = block_sum((int)threadIdx.x < n ? sums[threadIdx.x] : 0.0);
  if (threadIdx.x == 0) part[0] = fmaxf(part[0], (float)fmin(s * 0x1p-16, (double)kMaxFloat));
}
static_assert(kMaxBlocks <= kGroupBlock, "one block adds every sum");

hipError_t launch_prepare_one(int prec, const OneMft& one, const MaxOp& mx, hipStream_t s) {
  if (prec == PREC_FP32 && one.op.sc.n > 0) {
    if (one.sums) {
      hipLaunchKernelGGL((absmax_one_kernel<true>), dim3(mx.nblk), dim3(kGroupBlock), 0, s, mx, one.sums);
      hipLaunchKernelGGL(long_bound_kernel, dim3(1), dim3(kGroupBlock), 0, s, mx.part, one.sums, mx.nblk);
    } else {
      hipLaunchKernelGGL((absmax_one_kernel<false>), dim3(mx.nblk), dim3(kGroupBlock), 0, s, mx, nullptr);
    }
  }
  const PhasorOp& op = one.op;
  const int op_blocks =
      (int)((operand_threads(op.trans ? op.n : op.m, op.trans ? op.m : op.n, 1, OperandSplit{2, 1}) + kGroupBlock - 1) /
            kGroupBlock);
  int blocks[2];
  for (int t = 0; t < 2; ++t)
    blocks[t] = (int)((table_threads(one.tab[t].nsb, one.tab[t].nkb) + kGroupBlock - 1) / kGroupBlock);
  const dim3 grid(op_blocks + blocks[0] + blocks[1]), block(kGroupBlock);
  if (prec == PREC_BF16X3)
    hipLaunchKernelGGL((prepare_one_kernel<PREC_BF16X3>), grid, block, 0, s, op, one.wave, one.tab[0], one.tab[1],
                       one.desc, one.desc_dev, op_blocks, blocks[0]);
  else
    hipLaunchKernelGGL((prepare_one_kernel<PREC_FP32>), grid, block, 0, s, op, one.wave, one.tab[0], one.tab[1],
                       one.desc, one.desc_dev, op_blocks, blocks[0]);
  return hipGetLastError();
}

hipError_t launch_table_one(int prec, const TableOp& op, hipStream_t s) {
  const dim3 grid((unsigned)((table_threads(op.nsb, op.nkb) + kGroupBlock - 1) / kGroupBlock)), block(kGroupBlock);
  if (prec == PREC_BF16X3) hipLaunchKernelGGL((table_one_kernel<PREC_BF16X3>), grid, block, 0, s, op);
  else hipLaunchKernelGGL((table_one_kernel<PREC_FP32>), grid, block, 0, s, op);
  return hipGetLastError();
}

// Plain complex64 phasor Fields (one wavelength), row-major m x n each, item
// blockIdx.y of the list in the kernel arguments.  A segment's phasor is a few
// thousand samples, so a launch (2.6 us on the device, 6 us of the host) costs
// more than its work: one launch makes up to 32 of them.
template <int N>
struct PhasorFields {
  PhasorField it[N];
};
template <int N>
__global__ void phasor_field_kernel(PhasorFields<N> list, double inv_wl) {
  const PhasorField& q = list.it[N == 1 ? 0 : blockIdx.y];
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)q.m * q.n) return;
  const long long row = t / q.n, k = t % q.n;
  const float a = (float)load_real(q.amp, q.amp_dtype, row * q.ld_amp + k);
  const float2 c = cis_turns(load_real(q.opd, q.opd_dtype, row * q.ld_opd + k) * inv_wl);
  q.dst[t] = make_float2(a * c.x, a * c.y);
}

template <int N>
static void phasor_fields(const PhasorField* items, int n, long long most, double inv_wl, hipStream_t s) {
  PhasorFields<N> list = {};
  for (int i = 0; i < n; ++i) list.it[i] = items[i];
  hipLaunchKernelGGL((phasor_field_kernel<N>), dim3((unsigned)((most + 255) / 256), (unsigned)n), dim3(256), 0, s, list,
                     inv_wl);
}

hipError_t launch_phasor_fields(const PhasorField* items, int count, double inv_wl, hipStream_t s) {
  for (int b = 0; b < count; b += 32) {
    const int n = count - b < 32 ? count - b : 32;
    long long most = 0;
    for (int i = b; i < b + n; ++i) most = std::max(most, (long long)items[i].m * items[i].n);
    if (n == 1) phasor_fields<1>(items + b, n, most, inv_wl, s);
    else if (n <= 8) phasor_fields<8>(items + b, n, most, inv_wl, s);
    else phasor_fields<32>(items + b, n, most, inv_wl, s);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// --------------------------------------------------------------------------
// detector accumulation
// --------------------------------------------------------------------------

// Rows of an image that one launch of a thread per pixel covers: a launch of
// 2^32 threads or more is cut off without an error.
static int image_rows(int rows, int cols) {
  const int per_row = (cols + 255) / 256;
  return std::min(rows, std::max(1, (1 << 23) / per_row));
}

// One thread per image pixel: the partial images of every region that covers
// it are summed in FP64 and the pixel is written (or added to) once, regions
// or not, so nothing is cleared first.  Bound by reading the partial images;
// one launch for all regions: 4 side by side (512^2, 8 partials each) took a
// clear and 4 launches of 4.7 us, 24 us in all.
__global__ void reduce_kernel(const ReduceOp* __restrict__ ops, int nops, void* __restrict__ image, int dtype,
                              long long ldi, int row0, int cols, int accumulate, double unit) {
  const unsigned per_row = (unsigned)(cols + 255) / 256;
  const int r = row0 + (int)(blockIdx.x / per_row), c = (int)(blockIdx.x % per_row) * 256 + (int)threadIdx.x;
  if (c >= cols) return;
  double acc = 0.0;
  for (int i = 0; i < nops; ++i) {
    const int pr = r - ops[i].r0, pc = c - ops[i].c0;
    if (pr < 0 || pr >= ops[i].rows || pc < 0 || pc >= ops[i].cols) continue;
    gptr<const float> p = (gptr<const float>)ops[i].partial + ((long long)pr * ops[i].ldp + pc);
    const long long step = ops[i].gstride;
    const int n = ops[i].ngroups;
#pragma unroll 8
    for (int g = 0; g < n; ++g) acc += (double)p[(long long)g * step];
  }
  acc *= unit;
  const long long o = (long long)r * ldi + c;
  if (dtype == 3) {
    double* d = (double*)image;
    d[o] = accumulate ? d[o] + acc : acc;
  } else {
    float* d = (float*)image;
    d[o] = accumulate ? (float)((double)d[o] + acc) : (float)acc;
  }
}

hipError_t launch_reduce(const ReduceOp* ops, int nops, void* image, int dtype, long long ldi, int rows, int cols,
                         int accumulate, double unit, hipStream_t s) {
  if (rows <= 0 || cols <= 0 || (nops == 0 && accumulate)) return hipSuccess;
  const int step = image_rows(rows, cols);
  for (int r = 0; r < rows; r += step)
    hipLaunchKernelGGL(reduce_kernel, dim3((unsigned)std::min(step, rows - r) * (unsigned)((cols + 255) / 256)), dim3(256),
                       0, s, ops, nops, image, dtype, ldi, r, cols, accumulate, unit);
  return hipGetLastError();
}

// One thread per image pixel: every coherent group's Fields are summed where
// they cover the pixel (in the group's order, FP32 as _merge sums them), the
// squares weighted and added in FP64, the image written once.  Bound by reading
// the Fields, whose rows consecutive threads read contiguously: 144 Fields of
// 384^2 (18 segments, 8 wavelengths) took 152 launches and 425 us when every
// Field was added to an accumulator and every accumulator to the image.
__global__ void coherent_kernel(const CoherentGroup* __restrict__ groups, int ngroups,
                                const CoherentAdd* __restrict__ adds, void* __restrict__ image, int dtype,
                                long long ldi, int row0, int cols, int accumulate) {
  const unsigned per_row = (unsigned)(cols + 255) / 256;
  const int r = row0 + (int)(blockIdx.x / per_row), c = (int)(blockIdx.x % per_row) * 256 + (int)threadIdx.x;
  if (c >= cols) return;
  double acc = 0.0;
  for (int g = 0; g < ngroups; ++g) {
    float re = 0.f, im = 0.f;
    const int first = groups[g].first, end = first + groups[g].count;
#pragma unroll 8
    for (int a = first; a < end; ++a) {
      const int fr = r - adds[a].r0, fc = c - adds[a].c0;
      const bool in = fr >= 0 && fr < adds[a].M && fc >= 0 && fc < adds[a].N;
      const v2f32 e = ((gptr<const v2f32>)adds[a].F)[in ? (long long)fr * adds[a].N + fc : 0];
      re += in ? e.x : 0.f;
      im += in ? e.y : 0.f;
    }
    acc += ((double)re * re + (double)im * im) * groups[g].weight;
  }
  const long long o = (long long)r * ldi + c;
  if (dtype == 3) {
    double* d = (double*)image;
    d[o] = accumulate ? d[o] + acc : acc;
  } else {
    float* d = (float*)image;
    d[o] = accumulate ? (float)((double)d[o] + acc) : (float)acc;
  }
}

hipError_t launch_coherent(const CoherentGroup* groups, int ngroups, const CoherentAdd* adds, void* image, int dtype,
                           long long ldi, int rows, int cols, int accumulate, hipStream_t s) {
  if (rows <= 0 || cols <= 0) return hipSuccess;
  const int step = image_rows(rows, cols);
  for (int r = 0; r < rows; r += step)
    hipLaunchKernelGGL(coherent_kernel, dim3((unsigned)std::min(step, rows - r) * (unsigned)((cols + 255) / 256)), dim3(256),
                       0, s, groups, ngroups, adds, image, dtype, ldi, r, cols, accumulate);
  return hipGetLastError();
}

// out[or0 + r][oc0 + c] += weight * |E|^2  or  weight * E   (field.py:301-304)
// for E = field[fr0 + r][fc0 + c], r < h, c < w (already clipped by the host).
__global__ void insert_kernel(const float2* __restrict__ field, long long ldf, int fr0, int fc0, int h, int w,
                              void* __restrict__ out, int out_dtype, long long ldo, int or0, int oc0,
                              int intensity, double weight) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)h * w) return;
  const int r = (int)(t / w), c = (int)(t % w);
  const float2 e = field[(long long)(fr0 + r) * ldf + (fc0 + c)];
  const long long o = (long long)(or0 + r) * ldo + (oc0 + c);
  if (intensity) {
    const double i2 = ((double)e.x * e.x + (double)e.y * e.y) * weight;
    if (out_dtype == 3) ((double*)out)[o] += i2;
    else ((float*)out)[o] += (float)i2;
  } else {
    if (out_dtype == 2) {
      double2* d = (double2*)out;
      d[o].x += (double)e.x * weight;
      d[o].y += (double)e.y * weight;
    } else {
      float2* d = (float2*)out;
      d[o].x += (float)(e.x * weight);
      d[o].y += (float)(e.y * weight);
    }
  }
}

hipError_t launch_insert(const void* field, long long ldf, int fr0, int fc0, int h, int w, void* out,
                         int out_dtype, long long ldo, int or0, int oc0, int intensity, double weight,
                         hipStream_t s) {
  const long long total = (long long)h * w;
  if (total <= 0) return hipSuccess;
  const int bs = 256;
  hipLaunchKernelGGL(insert_kernel, dim3((unsigned)((total + bs - 1) / bs)), dim3(bs), 0, s,
                     (const float2*)field, ldf, fr0, fc0, h, w, out, out_dtype, ldo, or0, oc0, intensity, weight);
  return hipGetLastError();
}

// out[r][c] += weight * |sum of the Fields at the pixel|^2 over the box (r0, c0)
// of h x w output pixels that holds them all (field.py:331-346, 301-304): the
// Fields are summed in FP32 in list order, as merging them one by one into a
// union array sums them.  One launch and one pass over the Fields, where the
// merge took a clear, a launch per Field that read and wrote the union, and the
// insertion: 8 launches, 21 us, for six Fields of 303^2.
template <int N>
struct FieldItems {
  FieldItem it[N];
};
template <int N>
__global__ void insert_group_kernel(FieldItems<N> list, int count, int r0, int c0, int h, int w,
                                    void* __restrict__ out, int out_dtype, long long ldo, double weight) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)h * w) return;
  const int r = r0 + (int)(t / w), c = c0 + (int)(t % w);
  float re = 0.f, im = 0.f;
#pragma unroll 4
  for (int i = 0; i < count; ++i) {
    const FieldItem& f = list.it[i];
    const int fr = r - f.r0, fc = c - f.c0;
    const bool in = fr >= 0 && fr < f.h && fc >= 0 && fc < f.w;
    const v2f32 e = ((gptr<const v2f32>)f.F)[in ? (long long)fr * f.ld + fc : 0];
    re += in ? e.x : 0.f;
    im += in ? e.y : 0.f;
  }
  const long long o = (long long)r * ldo + c;
  const double i2 = ((double)re * re + (double)im * im) * weight;
  if (out_dtype == 3) ((double*)out)[o] += i2;
  else ((float*)out)[o] += (float)i2;
}

template <int N>
static void insert_group(const FieldItem* items, int count, int r0, int c0, int h, int w, void* out, int out_dtype,
                         long long ldo, double weight, hipStream_t s) {
  FieldItems<N> list = {};
  for (int i = 0; i < count; ++i) list.it[i] = items[i];
  hipLaunchKernelGGL((insert_group_kernel<N>), dim3((unsigned)(((long long)h * w + 255) / 256)), dim3(256), 0, s, list,
                     count, r0, c0, h, w, out, out_dtype, ldo, weight);
}

hipError_t launch_insert_group(const FieldItem* items, int count, int r0, int c0, int h, int w, void* out,
                               int out_dtype, long long ldo, double weight, hipStream_t s) {
  if (h <= 0 || w <= 0 || count <= 0) return hipSuccess;
  if (count > kGroupFields) return hipErrorInvalidValue;
  if (count <= 8) insert_group<8>(items, count, r0, c0, h, w, out, out_dtype, ldo, weight, s);
  else insert_group<kGroupFields>(items, count, r0, c0, h, w, out, out_dtype, ldo, weight, s);
  return hipGetLastError();
}

// --------------------------------------------------------------------------
// phase-retrieval backward pass (no counterpart in the reference)
// --------------------------------------------------------------------------

// out[r][c] = scale * w[r][c] * F[r][c]: the cotangent w * dL/dI * F of a
// weighted intensity image (d|F|^2 / d conj(F) = F).
__global__ void weight_field_kernel(const float2* __restrict__ F, long long ldF, const void* __restrict__ w,
                                    int w_dtype, long long ldw, double scale, float2* __restrict__ out,
                                    long long ldo, int h, int wd) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)h * wd) return;
  const long long r = t / wd, c = t % wd;
  const double g = (w_dtype == 3 ? ((const double*)w)[r * ldw + c] : (double)((const float*)w)[r * ldw + c]) * scale;
  const float2 v = F[r * ldF + c];
  out[r * ldo + c] = make_float2((float)(g * v.x), (float)(g * v.y));
}

hipError_t launch_weight_field(const void* F, long long ldF, const void* w, int w_dtype, long long ldw, double scale,
                               void* out, long long ldo, int h, int wd, hipStream_t s) {
  const long long total = (long long)h * wd;
  if (total <= 0) return hipSuccess;
  const int bs = 256;
  hipLaunchKernelGGL(weight_field_kernel, dim3((unsigned)((total + bs - 1) / bs)), dim3(bs), 0, s, (const float2*)F,
                     ldF, w, w_dtype, ldw, scale, (float2*)out, ldo, h, wd);
  return hipGetLastError();
}

__device__ __forceinline__ double get_real(const void* p, int dtype, long long i) {
  return dtype == 3 ? ((gptr<const double>)p)[i] : (double)((gptr<const float>)p)[i];
}
__device__ __forceinline__ void put_grad(void* g, int dtype, long long i, double v) {
  if (dtype == 3) ((gptr<double>)g)[i] = v;
  else ((gptr<float>)g)[i] = (float)v;
}

// Given D_dw = dL/d conj(f_dw) for f_dw = amp * exp(2 pi i opd_d / lambda_w),
// d = 0 .. nopd-1, w = 0 .. nwave-1 (D_dw at D + (d nwave + w) * strideD):
//   grad_opd (+)= sum_dw (2 pi / lambda_w) * (-2) Im(conj(D_dw) f_dw)
//   grad_amp (+)= sum_dw 2 Re(conj(D_dw) exp(2 pi i opd_d / lambda_w))   (if grad_amp)
// f is recomputed from amp and opd (opd already includes any diversity); the
// 1/lambda values are inv_wls[w] on the device, or inv_wl0 when inv_wls is null.
// Bound by reading D (8 bytes each): a thread per sample keeps 8 loads in
// flight and sums in FP64 over every OPD, so the gradient is written once.
// 4 OPDs x 16 wavelengths of 512^2 (134 MB): one launch per OPD, each with its
// wavelengths uploaded first and the gradient read back and added to, took 88 us.
// BATCH: wavelengths whose loads are in flight together.  8 of them take registers
// and loads that a gradient of fewer lacks, and a loop waits for what was loaded
// before it, so one OPD (ONE) and one wavelength (BATCH 0) have none: one of 8000^2
// took 566 us in the general form, 326 in its own.
template <int BATCH, bool ONE>
__global__ void phase_grad_kernel(PhaseGrad q) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)q.m * q.n) return;
  const long long r = t / q.n, c = t % q.n;
  const long long ia = r * q.ld_amp + c, io = r * q.ld_opd + c;
  const double a = get_real(q.amp, q.amp_dtype, ia);
  // what the sums are added to, loaded with the rest
  const long long jo = r * q.ld_go + c, ja = r * q.ld_ga + c;
  double go0 = 0.0, ga0 = 0.0;
  if (q.accumulate) {
    go0 = get_real(q.g_opd, q.go_dtype, jo);
    if (q.g_amp) ga0 = get_real(q.g_amp, q.ga_dtype, ja);
  }
  double go = 0.0, ga = 0.0;
  gptr<const v2f32> D = (gptr<const v2f32>)q.D + (r * q.ldD + c);
  for (int d = 0; d < (ONE ? 1 : q.nopd); ++d, D += q.nwave * q.strideD) {
    const long long id = io + d * q.strideO;
    const double o = get_real(q.opd, q.opd_dtype, id);
    int w = 0;
    // the next N wavelengths, their loads in flight together
    auto batch = [&](auto count) {
      constexpr int N = decltype(count)::value;
      v2f32 v[N];
#pragma unroll
      for (int i = 0; i < N; ++i) v[i] = D[(w + i) * q.strideD];
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const double inv_wl = q.inv_wls ? q.inv_wls[w + i] : q.inv_wl0;
        const float2 e = cis_turns(o * inv_wl);
        // conj(D) * e = (x - i y)(e.x + i e.y)
        const double re = (double)v[i].x * e.x + (double)v[i].y * e.y;
        const double im = (double)v[i].x * e.y - (double)v[i].y * e.x;
        go += -4.0 * 3.14159265358979323846 * inv_wl * a * im;
        ga += 2.0 * re;
      }
      w += N;
    };
    if constexpr (BATCH == 8)
      while (w + 8 <= q.nwave) batch(std::integral_constant<int, 8>());
    if constexpr (BATCH >= 4)
      while (w + 4 <= q.nwave) batch(std::integral_constant<int, 4>());
    if constexpr (BATCH == 0) batch(std::integral_constant<int, 1>());
    else
      while (w < q.nwave) batch(std::integral_constant<int, 1>());
  }
  put_grad(q.g_opd, q.go_dtype, jo, q.accumulate ? go0 + go : go);
  if (q.g_amp) put_grad(q.g_amp, q.ga_dtype, ja, q.accumulate ? ga0 + ga : ga);
}

hipError_t launch_phase_grad(const PhaseGrad& q, hipStream_t s) {
  const long long total = (long long)q.m * q.n;
  if (total <= 0 || q.nwave <= 0 || q.nopd <= 0) return hipSuccess;
  const int bs = 256;
  const auto one = q.nwave >= 8 ? phase_grad_kernel<8, true> : q.nwave >= 4 ? phase_grad_kernel<4, true>
                   : q.nwave > 1 ? phase_grad_kernel<1, true> : phase_grad_kernel<0, true>;
  const auto several = q.nwave >= 8 ? phase_grad_kernel<8, false> : q.nwave >= 4 ? phase_grad_kernel<4, false>
                                                                                 : phase_grad_kernel<1, false>;
  const auto kernel = q.nopd == 1 ? one : several;
  hipLaunchKernelGGL(kernel, dim3((unsigned)((total + bs - 1) / bs)), dim3(bs), 0, s, q);
  return hipGetLastError();
}

// out[r][c] = a[r][c] * b[r][c] (complex64), the Field product of field.py:142.
__global__ void multiply_kernel(const float2* __restrict__ a, long long lda, const float2* __restrict__ b,
                                long long ldb, float2* __restrict__ out, long long ldo, int h, int w) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)h * w) return;
  const long long r = t / w, c = t % w;
  out[r * ldo + c] = cmul(a[r * lda + c], b[r * ldb + c]);
}

hipError_t launch_multiply(const void* a, long long lda, const void* b, long long ldb, void* out, long long ldo,
                           int h, int w, hipStream_t s) {
  const long long total = (long long)h * w;
  if (total <= 0) return hipSuccess;
  const int bs = 256;
  hipLaunchKernelGGL(multiply_kernel, dim3((unsigned)((total + bs - 1) / bs)), dim3(bs), 0, s, (const float2*)a, lda,
                     (const float2*)b, ldb, (float2*)out, ldo, h, w);
  return hipGetLastError();
}

__global__ void zero_kernel(uint4* __restrict__ p, long long n16, unsigned char* __restrict__ tail, int ntail) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n16) p[t] = make_uint4(0, 0, 0, 0);
  if (t < ntail) tail[t] = 0;
}

// Zero rows x cols elements of esz bytes (4 or 8) at row stride ld elements;
// the bytes between rows and after the last row are left alone.
__global__ void zero_rows_kernel(void* __restrict__ p, int esz, long long rows, long long cols, long long ld) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= rows * cols) return;
  const long long o = (t / cols) * ld + t % cols;
  if (esz == 8) ((unsigned long long*)p)[o] = 0ull;
  else ((unsigned int*)p)[o] = 0u;
}

hipError_t launch_zero_rows(void* p, int esz, long long rows, long long cols, long long ld, hipStream_t s) {
  if (rows <= 0 || cols <= 0) return hipSuccess;
  if (esz != 4 && esz != 8) return hipErrorInvalidValue;
  if (ld == cols && ((uintptr_t)p & 15) == 0) return launch_zero(p, (size_t)esz * rows * cols, s);
  const long long total = rows * cols;
  const int bs = 256;
  hipLaunchKernelGGL(zero_rows_kernel, dim3((unsigned)((total + bs - 1) / bs)), dim3(bs), 0, s, p, esz, rows, cols,
                     ld);
  return hipGetLastError();
}

hipError_t launch_zero(void* p, size_t bytes, hipStream_t s) {
  if (bytes == 0) return hipSuccess;
  const long long n16 = (long long)(bytes / 16);
  const int ntail = (int)(bytes % 16);
  const long long total = n16 > ntail ? n16 : ntail;
  const int bs = 256;
  hipLaunchKernelGGL(zero_kernel, dim3((unsigned)((total + bs - 1) / bs)), dim3(bs), 0, s, (uint4*)p, n16,
                     (unsigned char*)p + n16 * 16, ntail);
  return hipGetLastError();
}

}  // namespace mftx
