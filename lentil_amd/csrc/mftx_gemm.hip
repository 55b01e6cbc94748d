// Complex x twiddle GEMM of the two MFT stages on gfx950 MFMA.
//
//     stage 1:  G   = f   . E2      (stored as the operand of stage 2, G^T)
//     stage 2:  F^T = G^T . E1^T    (|F|^2 accumulated, or F stored)
// which is the triple product of lentil fourier.py:97 with the twiddles of
// fourier.py:108-109, both coordinates paired (Problem in mftx_internal.h):
// P = Ae cos, Q = Ao sin over K/2 pairs and N/2 slots, a quarter of the real
// products of the direct complex product.  Ae and Ao (the operand's two
// parts) and the cos and sin tables are split into hi and lo 16-bit planes and
// stored as MFMA fragments; a real product is hi*hi + hi*lo + lo*hi on
// v_mfma_f32_32x32x16 with FP32 accumulation.
//
// One 32-row x 32-slot block of C and 16 pairs of K are 12 MFMAs: accumulators
// P_re, P_im += (re, im of Ae) cos and Q_re, Q_im += (re, im of Ao) sin.
//
// TILE_BIG and TILE_MID (gemm_tile_kernel): workgroups of WR x WC waves, each
// wave one 32-row block by S 32-slot blocks.  Operand and twiddle blocks of a
// K block ("chunk") go straight from global memory into one of three LDS
// stages (global_load_lds_dwordx4), two chunks ahead, one barrier per chunk:
//   BIG: 4 x 2 waves, S = 2: 128 rows x 128 slots (256 output columns), 48 KiB
//        per stage, one workgroup (two waves per SIMD) per CU;
//   MID: 2 x 2 waves, S = 1: 64 rows x 64 slots, 24 KiB per stage, two
//        workgroups per CU (TILE_MULTI: the same, for problems of several
//        K segments).
// What bounds them: the matrix pipe at the clock the power management allows
// (a BIG chunk is 1536 MFMA cycles per SIMD against 128 KiB of fragment reads
// and 48 KiB of LDS writes, 115 B per cycle of a 256 B/cycle read path).  S = 2
// because a wave's operand fragments then feed two slot blocks: 16 fragment
// reads per 24 MFMAs and 48 KiB of loads, where S = 1 takes 12 per 12 and 40.
//
// Measured on the 512^2 -> 1024^2 sweep of 64 wavelengths (bf16 pairs): stage 1
// 128 us, stage 2 157 us = 1.31 PFLOP/s of executed products, the rate of a
// large library GEMM on this card (1.28); 187 and 318 us when the sums ran over
// all K samples with twiddles generated in the kernel.  Two workgroups per CU
// of 64 rows x 128 slots were slower (157 and 176 us): the operand is then
// loaded 1.33 times as often per product.
//
// TILE_SMALL (gemm_small_kernel): four waves split the K blocks of one 32 x 32
// block between them, load fragments straight into registers and add their
// sums through LDS.  For single transforms, whose few tiles would leave most
// of the chip idle: the time is latency, and it is a quarter of the K loop.
#include "mftx_device.h"

namespace mftx {

template <int PREC> struct Num;
template <> struct Num<PREC_BF16X3> {
  typedef bf16x8_t frag;
  static __device__ __forceinline__ f32x16 mfma(frag a, frag b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct Num<PREC_FP32> {
  typedef f16x8_t frag;
  static __device__ __forceinline__ f32x16 mfma(frag a, frag b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

typedef __attribute__((address_space(3))) void lds_void;
typedef float v4f32a8 __attribute__((ext_vector_type(4), aligned(8)));  // two complex64 at any element offset

// Weight-map values at map offsets idx[0..n-1] (1 without a map).  No load
// sits behind a branch, so they are in flight together.
template <int NW>
__device__ __forceinline__ void load_weights(const Problem& P, const long long (&idx)[NW], float (&wv)[NW]) {
  if (!P.wmap) {
#pragma unroll
    for (int t = 0; t < NW; ++t) wv[t] = 1.0f;
  } else if (P.wdtype == 3) {
#pragma unroll
    for (int t = 0; t < NW; ++t) wv[t] = (float)((gptr<const double>)P.wmap)[idx[t]];
  } else {
#pragma unroll
    for (int t = 0; t < NW; ++t) wv[t] = ((gptr<const float>)P.wmap)[idx[t]];
  }
}

// Index i of the map's n rows or columns, i < 2 n.
__device__ __forceinline__ int wrapped(int i, int n) { return i >= n ? i - n : i; }

// Map offset of F's element (u, v).
__device__ __forceinline__ long long weight_index(const Problem& P, int u, int v) {
  return (long long)wrapped(u + P.wrow, P.wrows) * P.ldw + wrapped(v + P.wcol, P.wcols);
}

// A lane's (cos, sin) of the store's output phase for its slot: column cp + s
// turns by (c, s), column cm - s by (c, -s).
__device__ __forceinline__ float2 slot_phase(const Problem& P, int slot) {
  return P.xrot != 0.0 ? cis_turns(P.xrot * (P.y0 + (double)slot)) : make_float2(1.0f, 0.0f);
}
// What undoes the operand's scaling, 1 without one.
// (a scalar load: a vector load's wait would drain the operand loads in flight)
__device__ __forceinline__ float unscale(const Problem& P) { return P.inv ? *(cptr<const float>)P.inv : 1.0f; }

// Sum of intensities plus weight * |scale * (re, im)|^2, given w =
// intensity_weight(weight, scale).  The f16 form's scale undoes the operand's
// scaling: for an amplitude near 1e-16 it is about 2^-66, and its square would
// leave FP32's range although the intensity does not.  So one factor of it
// meets the large sums before the other meets the weight; a power of two, it
// rounds nothing.  (The bf16 form's scale is 1.)
template <int PREC>
__device__ __forceinline__ float intensity_weight(float weight, float scale) {
  return PREC == PREC_FP32 ? weight * scale : weight * scale * scale;
}
template <int PREC>
__device__ __forceinline__ float add_intensity(float sum, float w, float scale, float re, float im) {
  const float i2 = __builtin_fmaf(re, re, im * im);
  return __builtin_fmaf(w, PREC == PREC_FP32 ? i2 * scale : i2, sum);
}

// Four 16-byte pieces per lane, transposed within each quad of lanes: piece t
// of lane q becomes piece q of lane t.
__device__ __forceinline__ void quad_transpose(float (&v)[16]) {
  const int lane = threadIdx.x;
  const bool b0 = lane & 1, b1 = lane & 2;
  auto flip1 = [](float x) {  // the value of lane ^ 1
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xb1, 0xf, 0xf, true));
  };
  auto flip2 = [](float x) {  // of lane ^ 2
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x4e, 0xf, 0xf, true));
  };
#pragma unroll
  for (int t = 0; t < 4; t += 2)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x = v[4 * t + e], y = v[4 * t + 4 + e], fx = flip1(x), fy = flip1(y);
      v[4 * t + e] = b0 ? fy : x;
      v[4 * t + 4 + e] = b0 ? y : fx;
    }
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x = v[4 * t + e], y = v[4 * t + 8 + e], fx = flip2(x), fy = flip2(y);
      v[4 * t + e] = b1 ? fy : x;
      v[4 * t + 8 + e] = b1 ? y : fx;
    }
}

// Store one side (0: column cp + s from P + iQ, 1: cm - s from P - iQ) of half
// h of a 32 x 32 block: this lane's slot and the 8 rows 16 h + 8 g + 4 (lane /
// 32) + e, g = 0, 1, e = 0 .. 3 of row block rb; re, im hold them unscaled.
//
// Lane l holds rows 0-3 and 8-11 of the 16, lane l + 32 rows 4-7 and 12-15.
// One lane swap per word (v_permlane32_swap: the high half of the first
// operand trades places with the low half of the second) gives lane l rows 0-7
// and lane l + 32 rows 8-15, so a lane stores 16-byte pieces.  The operand's
// pieces of 32 lanes are contiguous.  Those of a transposed field lie a row
// stride apart, so quads of lanes trade theirs first: a store instruction then
// writes 128 contiguous bytes of 8 rows instead of 32 of 32, and its loads of a
// weight map touch 8 rows instead of 32 (64 adjoint fields of 512^2 91 -> 83 us,
// a 1024^2 -> 2048^2 transform 64 -> 60.5).
template <int PREC, int EPI>
__device__ __forceinline__ void store_half(const Problem& P, int rb, int h, int side, int slot, int lane, float sc,
                                           float inv, float2 ph, float (&re)[8], float (&im)[8]) {
  const int j = side ? P.cm - slot : P.cp + slot;
  const bool has = j >= (EPI == EPI_STORE_CPLX ? P.j0 : 0) && j < (EPI == EPI_STORE_CPLX ? P.j1 : P.ncols) &&
                   !(side && j == P.cp + slot);
  if (P.xrot != 0.0) {
    const float ps = side ? -ph.y : ph.y;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float2 v = cmul(make_float2(re[q], im[q]), make_float2(ph.x, ps));
      re[q] = v.x;
      im[q] = v.y;
    }
  }
  // the block's first C row, opaque to the compiler: the row indices below
  // stay in the epilogue instead of being hoisted out of the K loop and spilled
  int row0 = rb * 32 + 16 * h;
  asm volatile("" : "+v"(row0));
  if (EPI == EPI_STORE_CPLX) {
    if (P.rowph) {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int row = row0 + 8 * (q >> 2) + 4 * (lane >> 5) + (q & 3);
        const v2f32 r = ((gptr<const v2f32>)P.rowph)[row < P.i1 ? row : 0];
        const float2 v = cmul(make_float2(re[q], im[q]), make_float2(r.x, r.y));
        re[q] = v.x;
        im[q] = v.y;
      }
    }
    // one after the other: their product may be below the smallest denormal
    // where the results are not (sources near 1e-38)
    auto out = [&](float x) { return PREC == PREC_FP32 ? x * sc * inv : x * sc; };
    float2* dst = (float2*)P.dst;
    if (!P.trans) {
      long long wi[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int row = row0 + 8 * (q >> 2) + 4 * (lane >> 5) + (q & 3);
        wi[q] = has && row >= P.i0 && row < P.i1 ? weight_index(P, row - P.i0, j - P.j0) : 0;
      }
      float wv[8];
      load_weights(P, wi, wv);
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int row = row0 + 8 * (q >> 2) + 4 * (lane >> 5) + (q & 3);
        if (has && row >= P.i0 && row < P.i1)
          ((gptr<v2f32>)dst)[(long long)(row - P.i0) * P.ldd + (j - P.j0)] = v2f32{out(re[q]) * wv[q], out(im[q]) * wv[q]};
      }
      return;
    }
    float o[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(out(re[q])), __float_as_uint(out(re[4 + q])),
                                                      false, false);
      const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(out(im[q])), __float_as_uint(out(im[4 + q])),
                                                      false, false);
      o[2 * q] = __uint_as_float(a[0]);
      o[2 * q + 1] = __uint_as_float(b[0]);
      o[8 + 2 * q] = __uint_as_float(a[1]);
      o[9 + 2 * q] = __uint_as_float(b[1]);
    }
    // lane q of a quad: rows 2 q, 2 q + 1 of the 8, of the quad's four columns in turn
    quad_transpose(o);
    const int r = row0 + 8 * (lane >> 5) + 2 * (lane & 3) - P.i0, nr = P.i1 - P.i0;  // first of the two, in the window
    const bool in0 = r >= 0 && r < nr, in1 = r + 1 >= 0 && r + 1 < nr;
    int jt[4];  // the columns; -1: not stored
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int st = (slot & ~3) + t, j = side ? P.cm - st : P.cp + st;
      jt[t] = j >= P.j0 && j < P.j1 && !(side && j == P.cp + st) ? j - P.j0 : -1;
    }
    if (P.wmap) {
      // rows and columns that are not stored read the map's first ones
      const int v0 = in0 ? wrapped(r + P.wcol, P.wcols) : 0, v1 = in1 ? wrapped(r + 1 + P.wcol, P.wcols) : 0;
      long long wi[8];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const long long u = jt[t] >= 0 ? (long long)wrapped(jt[t] + P.wrow, P.wrows) * P.ldw : 0;
        wi[2 * t] = u + v0;
        wi[2 * t + 1] = u + v1;
      }
      float wv[8];
      load_weights(P, wi, wv);
#pragma unroll
      for (int q = 0; q < 16; ++q) o[q] *= wv[q >> 1];
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (jt[t] < 0) continue;
      float2* d = dst + (long long)jt[t] * P.ldd + r;
      if (in0 && in1) {
        *(gptr<v4f32a8>)d = v4f32a8{o[4 * t], o[4 * t + 1], o[4 * t + 2], o[4 * t + 3]};
      } else {
        if (in0) ((gptr<v2f32>)d)[0] = v2f32{o[4 * t], o[4 * t + 1]};
        if (in1) ((gptr<v2f32>)d)[1] = v2f32{o[4 * t + 2], o[4 * t + 3]};
      }
    }
    return;
  }
  // EPI_STORE_PACKED: row j of the next operand, K block rb, part h (the
  // operand's rows come as 16 even and 16 odd rows per block)
  uint32_t w[4][4];  // [plane][word]
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    uint32_t rh0, rl0, rh1, rl1, ih0, il0, ih1, il1;
    split2<PREC>(re[2 * q] * sc, re[2 * q + 1] * sc, rh0, rl0);
    split2<PREC>(re[4 + 2 * q] * sc, re[5 + 2 * q] * sc, rh1, rl1);
    split2<PREC>(im[2 * q] * sc, im[2 * q + 1] * sc, ih0, il0);
    split2<PREC>(im[4 + 2 * q] * sc, im[5 + 2 * q] * sc, ih1, il1);
    const auto a = __builtin_amdgcn_permlane32_swap(rh0, rh1, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(rl0, rl1, false, false);
    const auto c = __builtin_amdgcn_permlane32_swap(ih0, ih1, false, false);
    const auto d = __builtin_amdgcn_permlane32_swap(il0, il1, false, false);
    w[0][q] = a[0];
    w[0][2 + q] = a[1];
    w[1][q] = b[0];
    w[1][2 + q] = b[1];
    w[2][q] = c[0];
    w[2][2 + q] = c[1];
    w[3][q] = d[0];
    w[3][2 + q] = d[1];
  }
  if (!has) return;
  char* d = (char*)P.dst + ((long long)(j >> 5) * P.ldd + (row0 >> 5)) * A_BLOCK + h * 4 * FRAG +
            16 * ((j & 31) + 32 * (lane >> 5));
#pragma unroll
  for (int pl = 0; pl < 4; ++pl)
    *(gptr<v4u32>)(d + pl * FRAG) = v4u32{w[pl][0], w[pl][1], w[pl][2], w[pl][3]};
}

// The summed intensity of one 32 x 32 block into the work item's partial image
// (transposed like the problems' trans flag), clipped to the partial extent:
// this lane's slot and C rows row0 + 8 g + 4 (lane / 32) + e for its NG groups.
template <int NG>
__device__ __forceinline__ void store_partial(const Work& wk, const Problem& P, int row0, int side, int slot, int lane,
                                              const float (&v)[4 * NG]) {
  const int j = side ? P.cm - slot : P.cp + slot;
  const bool has = side ? (j >= 0 && j < P.ncols && j != P.cp + slot) : j < P.ncols;
  if (!has) return;
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const int row = row0 + 8 * g + 4 * (lane >> 5);
    if (P.trans) {
      // C rows run along the partial's rows, so a lane's 4 consecutive C rows
      // are one aligned 16-byte store (the partial and its row stride are
      // multiples of 128 floats).  Rows past pcols land in the partial's
      // padding columns, inside its allocation, which the reduction never reads.
      if (j < wk.prows)
        *(gptr<v4f32>)&((gptr<float>)wk.partial)[(long long)j * wk.ldp + row] =
            v4f32{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
    } else if (j < wk.pcols) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (row + e < wk.prows) ((gptr<float>)wk.partial)[(long long)(row + e) * wk.ldp + j] = v[4 * g + e];
    }
  }
}

// Work item of a launch without a work list: tile (t / ntc, tc0 + t % ntc) of
// problem 0, t < ntiles.  Workgroups go to the 8 XCDs in turn, so workgroup b
// takes t = (b % 8) ceil(ntiles / 8) + b / 8: an XCD's tiles are neighbouring
// rows, and its L2 fetches an eighth of the operand (and the table) instead of
// all of it (a 1024^2 filter, four such launches: 60 instead of 70 us).
// The twiddle table holds the slot blocks from sb0 on.
struct OneWork {
  int ntc, tc0, nch, sb0, ntiles;
};
__device__ __forceinline__ Work get_work(const Work* __restrict__ works, const OneWork& one) {
  if (works) return works[blockIdx.x];
  Work wk = {};
  const int t = (int)(blockIdx.x & 7) * ((one.ntiles + 7) >> 3) + (int)(blockIdx.x >> 3);
  if (t >= one.ntiles) return wk;  // an empty item
  wk.pend = 1;
  wk.tr = t / one.ntc;
  wk.tc = one.tc0 + t % one.ntc;
  wk.nch = one.nch;
  return wk;
}

// ---------------------------------------------------------------------------
// LDS-staged tiles
// ---------------------------------------------------------------------------
template <int WR, int WC, int S> struct Cfg {
  static constexpr int NW = WR * WC;            // waves
  static constexpr int NT = 64 * NW;            // threads
  static constexpr int RB = WR, SB = WC * S;    // row and slot blocks per workgroup
  static constexpr int ABYTES = RB * A_BLOCK, STAGE = ABYTES + SB * B_BLOCK;
  static constexpr int NSTAGE = 3;
  static constexpr int WG_PER_CU = 163840 / (NSTAGE * STAGE);
  // every wave loads one part (4 fragments) of an operand block and one half
  // (2 fragments: cos or sin) of a twiddle block per chunk
  static_assert(2 * RB == NW && 2 * SB == NW, "loads divide evenly over the waves");
};

// A wave's load cursor: the chunk its next six direct-to-LDS loads fetch.
// Everything is wave-uniform and lives in SGPRs; a lane adds 16 bytes times
// its index plus the fragment's offset.
struct Cursor {
  int seg, kb, nkb;
  const char *a, *b;
};

// One direct-to-LDS load: lane l's 16 bytes at src + voff land at LDS byte dst
// + 16 l.  Written out rather than through the builtin: the compiler counts a
// builtin LDS DMA on the LDS/scalar counter too, and then waits for every
// fragment read at once (lgkmcnt(0)) where a count would do; the load has no
// register result, and the waits for it (vmcnt) are explicit.  SALU writes of
// M0 need one wait state before an LDS DMA reads it.  The compiler reserves M0
// and warns that it will not restore it across the statement; these loads are
// the only M0 readers and writers here, so nothing needs it restored.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_load(const char* src, int voff, unsigned dst) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(voff), "s"(src), "s"(dst) : "memory", "m0");
}
#pragma clang diagnostic pop

__device__ __forceinline__ const char* uniform_ptr(const char* p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (const char*)(((uint64_t)hi << 32) | lo);
}

// MULTI: problems may have several segments (the turn between them costs the
// registers of a second set of accumulators, so only MID is built with it).
template <int PREC, int EPI, int WR, int WC, int S, bool MULTI>
__global__ __launch_bounds__((Cfg<WR, WC, S>::NT), (Cfg<WR, WC, S>::WG_PER_CU)) void gemm_tile_kernel(
    const Work* __restrict__ works, const Problem* __restrict__ probs, const Seg* __restrict__ segs, OneWork one) {
  using C = Cfg<WR, WC, S>;
  using N = Num<PREC>;
  typedef typename N::frag frag;
  __shared__ alignas(16) char lds[C::NSTAGE * C::STAGE];
  const Work wk = get_work(works, one);
  if (wk.pbeg >= wk.pend) return;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wr = wid / WC, wc = wid % WC;

  // ---- loads ----
  const int lrow = wid >> 1, lhalf = wid & 1;  // the block this wave loads, and its part / half
  int voff[4];
#pragma unroll
  for (int f = 0; f < 4; ++f) voff[f] = 16 * lane + f * FRAG;
  const unsigned lds0 = (unsigned)(size_t)(lds_void*)&lds[0];
  const unsigned dst_a = lds0 + lrow * A_BLOCK + lhalf * 4 * FRAG;
  const unsigned dst_b = lds0 + C::ABYTES + lrow * B_BLOCK + lhalf * 2 * FRAG;
  const int seg_end = probs[wk.pend - 1].send;
  // blocks past the operand's or table's last one reload it: valid memory
  // whose results nobody stores
  const int lrb = min(wk.tr * C::RB + lrow, probs[wk.pbeg].rblocks - 1);
  const int lsb = min(wk.tc * C::SB + lrow, probs[wk.pbeg].sblocks - 1) - one.sb0;
  Cursor cur;
  auto cursor_set = [&](int seg) {
    const Seg& sg = segs[seg];
    cur.seg = seg;
    cur.kb = 0;
    cur.nkb = sg.nkb;
    cur.a = uniform_ptr((const char*)sg.a + (long long)lrb * sg.a_nkb * A_BLOCK + lhalf * 4 * FRAG);
    cur.b = uniform_ptr((const char*)sg.b + (long long)lsb * sg.b_nkb * B_BLOCK + lhalf * 2 * FRAG);
  };
  // past the work's last chunk the cursor stays on it: the loads stay valid and nobody reads them
  auto cursor_next = [&]() {
    if (cur.kb + 1 < cur.nkb) {
      ++cur.kb;
      cur.a += A_BLOCK;
      cur.b += B_BLOCK;
    } else if (cur.seg + 1 < seg_end) {
      cursor_set(cur.seg + 1);
    }
  };
  auto load = [&](int stage, int i) {  // i = 0..3: operand fragments, 4, 5: twiddle fragments
    const unsigned st = (unsigned)(stage * C::STAGE);
    if (i < 4) lds_load(cur.a, voff[i], dst_a + st + i * FRAG);
    else lds_load(cur.b, voff[i - 4], dst_b + st + (i - 4) * FRAG);
  };
  cursor_set(probs[wk.pbeg].sbeg);
#pragma unroll
  for (int st = 0; st < 2; ++st) {
#pragma unroll
    for (int i = 0; i < 6; ++i) load(st, i);
    cursor_next();
  }
  asm volatile("s_waitcnt vmcnt(6)\n\ts_barrier" ::: "memory");

  // ---- accumulators ----
  f32x16 acc[S][4];  // P_re, P_im, Q_re, Q_im of each slot block
  float ip[EPI == EPI_INTENSITY ? S : 1][16] = {}, im[EPI == EPI_INTENSITY ? S : 1][16] = {};
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[s][i] = f32x16{};
  const int rb = wk.tr * C::RB + wr;  // this wave's row block
  const bool mf = rb < probs[wk.pbeg].rblocks;  // wave-uniform: past the last row block a wave issues no MFMAs

  // fragment reads: operand part p fragment f (re hi, re lo, im hi, im lo),
  // twiddle slot block s, half p (cos, sin), fragment f (hi, lo)
  const char* la = lds + wr * A_BLOCK + 16 * lane;
  const char* lb = lds + C::ABYTES + wc * S * B_BLOCK + 16 * lane;
  auto rd_a = [&](int stage, int p, int f) { return *(const frag*)(la + stage * C::STAGE + (4 * p + f) * FRAG); };
  auto rd_b = [&](int stage, int s, int p, int f) {
    return *(const frag*)(lb + stage * C::STAGE + s * B_BLOCK + (2 * p + f) * FRAG);
  };
  auto group = [&](int p, const frag (&x)[2], const frag (&y)[S]) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      acc[s][2 * p] = N::mfma(x[0], y[s], acc[s][2 * p]);
      acc[s][2 * p + 1] = N::mfma(x[1], y[s], acc[s][2 * p + 1]);
    }
  };
  auto fence = [&]() { __builtin_amdgcn_sched_barrier(0); };
  auto loads = [&](int stage, int i0, int i1) {
    fence();
#pragma unroll
    for (int i = i0; i < i1; ++i) load(stage, i);
    fence();
  };
  // Nothing is outstanding on the LDS/scalar counter after this wait; the
  // compiler sees it (the barrier's own waits are in asm it cannot read), so
  // it waits for each fragment read below by count, not for all at once.
  auto drained = [&]() { __builtin_amdgcn_s_waitcnt(0xc07f); };  // lgkmcnt(0); vmcnt, expcnt unrestricted
  auto barrier = [&]() {
    // Wait for this wave's chunk s + 1 loads (the 6 just issued for chunk
    // s + 2 may stay in flight: loads complete in issue order, so epilogue
    // stores in between do not weaken this) and its fragment reads.
    asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    drained();
  };
  frag ah[2] = {}, bl[S] = {};
  auto first_reads = [&](int stage) {
    ah[0] = rd_a(stage, 0, 0);
    ah[1] = rd_a(stage, 0, 2);
#pragma unroll
    for (int s = 0; s < S; ++s) bl[s] = rd_b(stage, s, 0, 1);
  };

  int pc = wk.pbeg, sc = probs[pc].sbeg, left = segs[sc].nkb;  // compute cursor: problem, segment, chunks left in it
  int st = 0, ld = 2;                                          // LDS stages of chunks s and s + 2
  drained();
  if (mf) first_reads(0);
  for (int n = 0; n < wk.nch; ++n) {
    const int nx = st == 2 ? 0 : st + 1;
    if (mf) {
      // The three products run in the order hi*lo, hi*hi, lo*hi, so each
      // operand pair is dead as early as possible and the next fragments are
      // read into its registers while the current group multiplies.  The
      // chunk's barrier comes before its last group: by then every fragment
      // read of chunk s and every load of chunk s + 2 is issued, and after it
      // chunk s + 1 is complete in LDS and its first fragments are read under
      // that group.  Scheduling barriers pin this order.
      frag al[2] = {rd_a(st, 0, 1), rd_a(st, 0, 3)};
      frag bh[S];
#pragma unroll
      for (int s = 0; s < S; ++s) bh[s] = rd_b(st, s, 0, 0);
      group(0, ah, bl);
      loads(ld, 0, 1);
#pragma unroll
      for (int s = 0; s < S; ++s) bl[s] = rd_b(st, s, 1, 1);
      group(0, ah, bh);
      loads(ld, 1, 2);
      ah[0] = rd_a(st, 1, 0);
      ah[1] = rd_a(st, 1, 2);
      group(0, al, bh);
      loads(ld, 2, 3);
#pragma unroll
      for (int s = 0; s < S; ++s) bh[s] = rd_b(st, s, 1, 0);
      al[0] = rd_a(st, 1, 1);
      al[1] = rd_a(st, 1, 3);
      fence();
      group(1, ah, bl);
      loads(ld, 3, 5);
      group(1, ah, bh);
      loads(ld, 5, 6);
      barrier();
      fence();
      first_reads(nx);  // past the last chunk: a stage nobody writes any more, read and unused
      fence();
      group(1, al, bh);
    } else {
      loads(ld, 0, 6);
      barrier();
    }
    cursor_next();
    st = nx;
    ld = ld == 2 ? 0 : ld + 1;
    if (--left > 0) continue;
    const Problem& P = probs[pc];
    ++sc;
    if (MULTI && sc < P.send) {
      // the next segment's midpoint: turn (P, Q) by its rotation
      const Seg& sg = segs[sc];
      left = sg.nkb;
      if (mf) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
          const float2 r = cis_turns(sg.rot * (P.y0 + (double)((wk.tc * C::SB + wc * S + s) * 32 + (lane & 31))));
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              const float p = acc[s][i][e], q = acc[s][2 + i][e];
              acc[s][i][e] = r.x * p - r.y * q;
              acc[s][2 + i][e] = r.y * p + r.x * q;
            }
        }
      }
      continue;
    }
    if (mf) {
      const float inv = unscale(P), sc0 = P.scale, scale = sc0 * inv;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const int slot = (wk.tc * C::SB + wc * S + s) * 32 + (lane & 31);
        if (EPI == EPI_INTENSITY) {
          const float w = intensity_weight<PREC>(P.weight, scale);
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const float pr = acc[s][0][e], pi = acc[s][1][e], qr = acc[s][2][e], qi = acc[s][3][e];
            const float ar = pr - qi, ai = pi + qr;   // P + iQ
            const float br = pr + qi, bi = pi - qr;   // P - iQ
            ip[s][e] = add_intensity<PREC>(ip[s][e], w, scale, ar, ai);
            im[s][e] = add_intensity<PREC>(im[s][e], w, scale, br, bi);
          }
        } else {
          const float2 ph = slot_phase(P, slot);
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int side = 0; side < 2; ++side) {
              float re[8], imv[8];
#pragma unroll
              for (int q = 0; q < 8; ++q) {
                const int e = 8 * h + q;
                const float pr = acc[s][0][e], pi = acc[s][1][e], qr = acc[s][2][e], qi = acc[s][3][e];
                re[q] = side ? pr + qi : pr - qi;
                imv[q] = side ? pi - qr : pi + qr;
              }
              store_half<PREC, EPI>(P, rb, h, side, slot, lane, sc0, inv, ph, re, imv);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[s][i] = f32x16{};
      }
    }
    if (++pc < wk.pend) left = segs[sc].nkb;  // its first segment follows the last one
  }
  // no load may still be writing LDS when the workgroup ends
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (EPI == EPI_INTENSITY && mf) {
    const Problem& P = probs[wk.pbeg];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int slot = (wk.tc * C::SB + wc * S + s) * 32 + (lane & 31);
      store_partial<4>(wk, P, rb * 32, 0, slot, lane, ip[s]);
      store_partial<4>(wk, P, rb * 32, 1, slot, lane, im[s]);
    }
  }
}

// ---------------------------------------------------------------------------
// One 32 x 32 block per workgroup, K split over its four waves
// ---------------------------------------------------------------------------
template <int PREC, int EPI>
__global__ __launch_bounds__(256, 2) void gemm_small_kernel(const Work* __restrict__ works,
                                                            const Problem* __restrict__ probs,
                                                            const Seg* __restrict__ segs, OneWork one) {
  using N = Num<PREC>;
  typedef typename N::frag frag;
  __shared__ alignas(16) float red[4][4][4][64][4];  // [wave][accumulator][row group][lane][element]
  const Work wk = get_work(works, one);
  if (wk.pbeg >= wk.pend) return;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int h = wid & 1, side = wid >> 1;  // the rows and columns this wave stores
  const int slot = wk.tc * 32 + (lane & 31);
  float isum[8] = {};
  for (int pc = wk.pbeg; pc < wk.pend; ++pc) {
    const Problem& P = probs[pc];
    f32x16 acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = f32x16{};
    for (int sg = P.sbeg; sg < P.send; ++sg) {
      const Seg& sgm = segs[sg];
      if (sg > P.sbeg) {
        const float2 r = cis_turns(sgm.rot * (P.y0 + (double)slot));
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const float p = acc[i][e], q = acc[2 + i][e];
            acc[i][e] = r.x * p - r.y * q;
            acc[2 + i][e] = r.y * p + r.x * q;
          }
      }
      gptr<const char> a = (gptr<const char>)sgm.a + (long long)wk.tr * sgm.a_nkb * A_BLOCK + 16 * lane;
      gptr<const char> b = (gptr<const char>)sgm.b + (long long)(wk.tc - one.sb0) * sgm.b_nkb * B_BLOCK + 16 * lane;
      frag af[2][8], bf[2][4];
      auto get = [&](int buf, int kb) {
#pragma unroll
        for (int f = 0; f < 8; ++f) af[buf][f] = *(gptr<const frag>)(a + (long long)kb * A_BLOCK + f * FRAG);
#pragma unroll
        for (int f = 0; f < 4; ++f) bf[buf][f] = *(gptr<const frag>)(b + (long long)kb * B_BLOCK + f * FRAG);
      };
      auto mul = [&](int buf) {
#pragma unroll
        for (int t = 0; t < 3; ++t) {
          const int ia = t == 2 ? 1 : 0, ib = t == 0 ? 1 : 0;  // hi*lo, hi*hi, lo*hi
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            acc[2 * p] = N::mfma(af[buf][4 * p + ia], bf[buf][2 * p + ib], acc[2 * p]);
            acc[2 * p + 1] = N::mfma(af[buf][4 * p + 2 + ia], bf[buf][2 * p + ib], acc[2 * p + 1]);
          }
        }
      };
      // the next block's fragments are loaded while the current one multiplies
      int kb = wid;
      if (kb < sgm.nkb) get(0, kb);
      while (kb < sgm.nkb) {
        if (kb + 4 < sgm.nkb) get(1, kb + 4);
        mul(0);
        kb += 4;
        if (kb >= sgm.nkb) break;
        if (kb + 4 < sgm.nkb) get(0, kb + 4);
        mul(1);
        kb += 4;
      }
    }
    if (pc > wk.pbeg) __syncthreads();  // the last problem's sums have been read
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *(v4f32*)red[wid][i][g][lane] = v4f32{acc[i][4 * g], acc[i][4 * g + 1], acc[i][4 * g + 2], acc[i][4 * g + 3]};
    __syncthreads();
    float t[4][8];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        v4f32 v = *(const v4f32*)red[0][i][2 * h + g][lane];
#pragma unroll
        for (int w = 1; w < 4; ++w) v += *(const v4f32*)red[w][i][2 * h + g][lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) t[i][4 * g + e] = v[e];
      }
    float re[8], imv[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      re[q] = side ? t[0][q] + t[3][q] : t[0][q] - t[3][q];
      imv[q] = side ? t[1][q] - t[2][q] : t[1][q] + t[2][q];
    }
    const float inv = unscale(P), sc0 = P.scale, scale = sc0 * inv;
    if (EPI == EPI_INTENSITY) {
      const float w = intensity_weight<PREC>(P.weight, scale);
#pragma unroll
      for (int q = 0; q < 8; ++q) isum[q] = add_intensity<PREC>(isum[q], w, scale, re[q], imv[q]);
    } else {
      store_half<PREC, EPI>(P, wk.tr, h, side, slot, lane, sc0, inv, slot_phase(P, slot), re, imv);
    }
  }
  if (EPI == EPI_INTENSITY) store_partial<2>(wk, probs[wk.pbeg], wk.tr * 32 + 16 * h, side, slot, lane, isum);
}

// ---------------------------------------------------------------------------
// Coherent groups whose Fields have their own windows of one output grid
// ---------------------------------------------------------------------------
// Work item: the 32 x 32 block (tr, tc) of the grid and the problems of one
// group (a Field each, its windows in i0 .. j1).  The four waves take the
// Fields in turn; a wave adds each Field's (P + iQ, P - iQ), turned by its
// phase and cut to its window, to its complex sum in LDS (in registers it would
// spill), and the weighted |sum|^2 of the four goes into the group's partial
// image.
// No Field is stored.  Bound by the fragments' way from L2 (12 KiB per K block
// and wave, double-buffered).  A Field has few K blocks (a segment's box) and
// its window few blocks, so more of them per work item leave the chip idle:
// 18 segments, 8 wavelengths of 384^2 take 38 us, with 32 x 64 per item (one
// wave per SIMD) 69, and 121 when the Fields were stored and summed.
template <int PREC>
__global__ __launch_bounds__(256, 2) void gemm_coherent_kernel(const Work* __restrict__ works,
                                                               const Problem* __restrict__ probs,
                                                               const Seg* __restrict__ segs) {
  using N = Num<PREC>;
  typedef typename N::frag frag;
  // the waves' sums so far: [wave][side, re / im, row group][lane][element]
  __shared__ alignas(16) float sum[4][16][64][4];
  const Work wk = works[blockIdx.x];
  if (wk.pbeg >= wk.pend) return;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
#pragma unroll
  for (int i = 0; i < 16; ++i) *(v4f32*)sum[wid][i][lane] = v4f32{};

  // Load cursor: the K block the next fragments come from.  Uniform, in SGPRs.
  struct Cursor {
    int pc, sg, send, kb, nkb;
    const char *a, *b;
  } ld;
  auto open = [&](Cursor& c) {
    const Seg& sg = segs[c.sg];
    c.kb = 0;
    c.nkb = sg.nkb;
    c.a = (const char*)sg.a + (long long)wk.tr * sg.a_nkb * A_BLOCK;
    c.b = (const char*)sg.b + (long long)wk.tc * sg.b_nkb * B_BLOCK;
  };
  auto begin = [&](Cursor& c, int pc) {
    c.pc = pc;
    c.sg = probs[pc].sbeg;
    c.send = probs[pc].send;
    open(c);
  };
  const unsigned voff = 16u * lane;
  frag af[2][8], bf[2][4];
  // the fragments of the wave's next K block: of the segment, the problem's
  // next segment, the wave's next problem
  auto get = [&](int buf) {
#pragma unroll
    for (int f = 0; f < 8; ++f) af[buf][f] = *(gptr<const frag>)((gptr<const char>)ld.a + f * FRAG + voff);
#pragma unroll
    for (int f = 0; f < 4; ++f) bf[buf][f] = *(gptr<const frag>)((gptr<const char>)ld.b + f * FRAG + voff);
    if (++ld.kb < ld.nkb) {
      ld.a += A_BLOCK;
      ld.b += B_BLOCK;
    } else if (++ld.sg < ld.send) {
      open(ld);
    } else if (ld.pc + 4 < wk.pend) {
      begin(ld, ld.pc + 4);
    }  // past the wave's last block the cursor stays: valid memory, read and unused
  };
  f32x16 acc[4];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = f32x16{};
  };
  auto mul = [&](int buf) {
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const int ia = t == 2 ? 1 : 0, ib = t == 0 ? 1 : 0;  // hi*lo, hi*hi, lo*hi
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        acc[2 * p] = N::mfma(af[buf][4 * p + ia], bf[buf][2 * p + ib], acc[2 * p]);
        acc[2 * p + 1] = N::mfma(af[buf][4 * p + 2 + ia], bf[buf][2 * p + ib], acc[2 * p + 1]);
      }
    }
  };
  auto finish = [&](const Problem& P) {
    const float scale = P.scale * unscale(P);
    const int slot = wk.tc * 32 + (lane & 31);
    float2 ph = slot_phase(P, slot);
    ph.x *= scale;
    ph.y *= scale;
    const int jp = P.cp + slot, jm = P.cm - slot;
    const bool hp = jp >= P.j0 && jp < P.j1, hm = jm >= P.j0 && jm < P.j1 && jm != jp;
    int row0 = wk.tr * 32 + 4 * (lane >> 5);
    asm volatile("" : "+v"(row0));
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      v4f32* f = (v4f32*)sum[wid][g][lane];  // plus side re, then im, minus side re, im, 256 vectors apart
      v4f32 ar = f[0], ai = f[256], br = f[512], bi = f[768];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int e = 4 * g + q, row = row0 + 8 * g + q;
        const bool in = row >= P.i0 && row < P.i1;
        const float pr = acc[0][e], pi = acc[1][e], qr = acc[2][e], qi = acc[3][e];
        const float2 a = cmul(make_float2(pr - qi, pi + qr), ph);                       // P + iQ
        const float2 b = cmul(make_float2(pr + qi, pi - qr), make_float2(ph.x, -ph.y));  // P - iQ
        ar[q] += in && hp ? a.x : 0.f;
        ai[q] += in && hp ? a.y : 0.f;
        br[q] += in && hm ? b.x : 0.f;
        bi[q] += in && hm ? b.y : 0.f;
      }
      f[0] = ar;
      f[256] = ai;
      f[512] = br;
      f[768] = bi;
    }
  };
  // one segment after the other; the next K block's fragments, whichever
  // segment they belong to, load while one multiplies
  int pc = wk.pbeg + wid, sg = 0, left = 0;
  clear();
  if (pc < wk.pend) {
    begin(ld, pc);
    sg = ld.sg;
    left = ld.nkb;
    get(0);
  }
  while (pc < wk.pend) {
    for (;;) {
      get(1);
      mul(0);
      if (--left == 0) {  // the next block is in the second buffer
#pragma unroll
        for (int f = 0; f < 8; ++f) af[0][f] = af[1][f];
#pragma unroll
        for (int f = 0; f < 4; ++f) bf[0][f] = bf[1][f];
        break;
      }
      get(0);
      mul(1);
      if (--left == 0) break;
    }
    const Problem& P = probs[pc];
    if (++sg < P.send) {  // the next segment's midpoint: turn (P, Q) by its rotation
      left = segs[sg].nkb;
      const float2 r = cis_turns(segs[sg].rot * (P.y0 + (double)(wk.tc * 32 + (lane & 31))));
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const float p = acc[i][e], q = acc[2 + i][e];
          acc[i][e] = r.x * p - r.y * q;
          acc[2 + i][e] = r.y * p + r.x * q;
        }
    } else {
      finish(P);
      clear();
      pc += 4;
      if (pc < wk.pend) {
        sg = probs[pc].sbeg;
        left = segs[sg].nkb;
      }
    }
  }
  // ---- the four sums, this wave's quarter of the block: rows 16 h .. 16 h + 15 of one side ----
  __syncthreads();
  const int h = wid & 1, side = wid >> 1;
  const Problem& P = probs[wk.pbeg];
  float v[8];
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const int i = 8 * side + 2 * h + g;
    v4f32 re = *(const v4f32*)sum[0][i][lane], im = *(const v4f32*)sum[0][i + 4][lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      re += *(const v4f32*)sum[w][i][lane];
      im += *(const v4f32*)sum[w][i + 4][lane];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[4 * g + e] = (float)(((double)re[e] * re[e] + (double)im[e] * im[e]) * (double)P.weight);
  }
  store_partial<2>(wk, P, wk.tr * 32 + 16 * h, side, wk.tc * 32 + (lane & 31), lane, v);
}

hipError_t launch_gemm_coherent(int prec, const Work* work, int nwork, const Problem* probs, const Seg* segs,
                                hipStream_t s) {
  if (nwork <= 0) return hipSuccess;
  if (prec == PREC_BF16X3)
    hipLaunchKernelGGL((gemm_coherent_kernel<PREC_BF16X3>), dim3(nwork), dim3(256), 0, s, work, probs, segs);
  else
    hipLaunchKernelGGL((gemm_coherent_kernel<PREC_FP32>), dim3(nwork), dim3(256), 0, s, work, probs, segs);
  return hipGetLastError();
}

template <int PREC, int EPI>
static hipError_t launch_epi(int tile, const Work* work, int nwork, const Problem* probs, const Seg* segs,
                             const OneWork& one, hipStream_t s) {
  if (tile == TILE_BIG)
    hipLaunchKernelGGL((gemm_tile_kernel<PREC, EPI, 4, 2, 2, false>), dim3(nwork), dim3(Cfg<4, 2, 2>::NT), 0, s, work, probs,
                       segs, one);
  else if (tile == TILE_MID)
    hipLaunchKernelGGL((gemm_tile_kernel<PREC, EPI, 2, 2, 1, false>), dim3(nwork), dim3(Cfg<2, 2, 1>::NT), 0, s, work,
                       probs, segs, one);
  else if (tile == TILE_MULTI)
    hipLaunchKernelGGL((gemm_tile_kernel<PREC, EPI, 2, 2, 1, true>), dim3(nwork), dim3(Cfg<2, 2, 1>::NT), 0, s, work,
                       probs, segs, one);
  else
    hipLaunchKernelGGL((gemm_small_kernel<PREC, EPI>), dim3(nwork), dim3(256), 0, s, work, probs, segs, one);
  return hipGetLastError();
}

template <int PREC>
static hipError_t launch_prec(int epi, int tile, const Work* work, int nwork, const Problem* probs, const Seg* segs,
                              const OneWork& one, hipStream_t s) {
  if (epi == EPI_STORE_CPLX) return launch_epi<PREC, EPI_STORE_CPLX>(tile, work, nwork, probs, segs, one, s);
  if (epi == EPI_STORE_PACKED) return launch_epi<PREC, EPI_STORE_PACKED>(tile, work, nwork, probs, segs, one, s);
  return launch_epi<PREC, EPI_INTENSITY>(tile, work, nwork, probs, segs, one, s);
}

static hipError_t launch_any(int prec, int epi, int tile, const Work* work, int nwork, const Problem* probs,
                             const Seg* segs, const OneWork& one, hipStream_t s) {
  if (nwork <= 0) return hipSuccess;
  return prec == PREC_BF16X3 ? launch_prec<PREC_BF16X3>(epi, tile, work, nwork, probs, segs, one, s)
                             : launch_prec<PREC_FP32>(epi, tile, work, nwork, probs, segs, one, s);
}

hipError_t launch_gemm(int prec, int epi, int tile, const Work* work, int nwork, const Problem* probs, const Seg* segs,
                       hipStream_t s) {
  return launch_any(prec, epi, tile, work, nwork, probs, segs, OneWork{}, s);
}

hipError_t launch_gemm_one(int prec, int epi, int tile, int rblocks, int sb0, int sb1, int nch, const Problem* prob,
                           const Seg* seg, hipStream_t s) {
  const int tr = (rblocks + tile_rows(tile) - 1) / tile_rows(tile);
  const int tc0 = sb0 / tile_slots(tile), ntc = (sb1 + tile_slots(tile) - 1) / tile_slots(tile) - tc0;
  const int ntiles = tr * ntc;
  return launch_any(prec, epi, tile, nullptr, (ntiles + 7) / 8 * 8, prob, seg, OneWork{ntc, tc0, nch, sb0, ntiles}, s);
}

}  // namespace mftx
