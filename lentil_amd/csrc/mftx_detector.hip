// MI355X (gfx950) kernels of the detector-grid post-processing: integer
// rebinning (util.py:221-259), the magnitude / weight-preserving passes of
// the FFT filters (detector.py:167-225, convolvable.py:4-169) and the cubic
// B-spline resampling of rescale (util.py:262-349).  All HBM-bound; the
// arithmetic is FP64 so results follow the reference's float64 numpy/scipy
// to rounding.
#include "../../include/mftx.h"
#include "mftx_device.h"

#include <algorithm>
#include <cmath>
#include <vector>

namespace mftx {

namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ double load_real(const void* p, int dtype, long long i) {
  return dtype == 3 ? ((const double*)p)[i] : (double)((const float*)p)[i];
}

// component `comp` (0 real, 1 imaginary) of element i of a real or complex array
__device__ __forceinline__ double load_component(const void* p, int dtype, long long i, int comp) {
  switch (dtype) {
    case 0: return comp ? ((const float2*)p)[i].y : ((const float2*)p)[i].x;
    case 2: return comp ? ((const double2*)p)[i].y : ((const double2*)p)[i].x;
    default: return comp ? 0.0 : load_real(p, dtype, i);
  }
}

__device__ __forceinline__ void store_real(void* p, int dtype, long long i, double v) {
  if (dtype == 3) ((double*)p)[i] = v;
  else ((float*)p)[i] = (float)v;
}

// Sum of v over the block, in every thread (fixed order: deterministic).
__device__ double block_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  __shared__ double w[kBlock / 64];
  __syncthreads();  // an earlier sum's readers are done
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  for (int i = 0; i < kBlock / 64; ++i) s += w[i];
  return s;
}

// Reductions leave one partial sum per block, at most kMaxPart of them, and
// whoever needs the total adds them itself: a launch to finish the sum took
// longer (5 us) than reading 1024 doubles in every block of the consumer.
__device__ double total(const double* __restrict__ part, int n) {
  double v = 0.0;
  for (int i = threadIdx.x; i < n; i += kBlock) v += part[i];
  return block_sum(v);
}
int part_blocks(long long n) {
  const long long b = (n + kBlock - 1) / kBlock;
  return (int)(b < 1 ? 1 : b > kMaxPart ? kMaxPart : b);
}

unsigned blocks_for(long long n) { return (unsigned)((n + kBlock - 1) / kBlock); }

}  // namespace

// --------------------------------------------------------------------------
// rebin: out[i][r][c] = sum of the factor x factor block (util.py:251-257)
// --------------------------------------------------------------------------
__global__ void rebin_kernel(const void* __restrict__ src, int dtype, long long nimg, long long rows, long long cols,
                             long long ld, int factor, void* __restrict__ dst, int odt) {
  const long long orows = rows / factor, ocols = cols / factor;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nimg * orows * ocols) return;
  const long long img = t / (orows * ocols), rem = t % (orows * ocols);
  const long long r = rem / ocols, c = rem % ocols;
  const long long base = img * rows * ld;
  double s = 0.0;
  for (int i = 0; i < factor; ++i)
    for (int j = 0; j < factor; ++j) s += load_real(src, dtype, base + (r * factor + i) * ld + c * factor + j);
  store_real(dst, odt, t, s);
}

hipError_t launch_rebin(const void* src, int dtype, long long nimg, long long rows, long long cols, long long ld,
                        int factor, void* dst, int odt, hipStream_t s) {
  const long long n = nimg * (rows / factor) * (cols / factor);
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(rebin_kernel, dim3(blocks_for(n)), dim3(kBlock), 0, s, src, dtype, nimg, rows, cols, ld, factor,
                     dst, odt);
  return hipGetLastError();
}

// --------------------------------------------------------------------------
// reductions and the weight-preserving rescale of the filters
// --------------------------------------------------------------------------

// part[b] = sum of component comp (0 real, 1 imaginary) of a rows x cols array
// over block b's elements (every gridDim-th run of 256)
__global__ void sum_kernel(const void* __restrict__ x, int dtype, int comp, long long rows, long long cols,
                           long long ld, double* __restrict__ part) {
  const long long n = rows * cols, step = (long long)gridDim.x * kBlock;
  double v = 0.0;
#pragma unroll 4
  for (long long t = (long long)blockIdx.x * kBlock + threadIdx.x; t < n; t += step)
    v += load_component(x, dtype, ld == cols ? t : t / cols * ld + t % cols, comp);
  v = block_sum(v);
  if (threadIdx.x == 0) part[blockIdx.x] = v;
}

// out[r][c] = |F[(r + r0) % rows][(c + c0) % cols]| (F complex64, 0 <= r0 < rows,
// 0 <= c0 < cols), part[b] = block sums of out
__global__ void magnitude_kernel(const float2* __restrict__ F, long long ldF, long long rows, long long cols,
                                 long long r0, long long c0, void* __restrict__ out, int odt, long long ldo,
                                 double* __restrict__ part) {
  const long long n = rows * cols, step = (long long)gridDim.x * kBlock;
  double sum = 0.0;
#pragma unroll 4
  for (long long t = (long long)blockIdx.x * kBlock + threadIdx.x; t < n; t += step) {
    const long long r = t / cols, c = t % cols;
    const long long fr = r + r0 < rows ? r + r0 : r + r0 - rows, fc = c + c0 < cols ? c + c0 : c + c0 - cols;
    const float2 f = F[fr * ldF + fc];
    const double v = sqrt((double)f.x * f.x + (double)f.y * f.y);
    store_real(out, odt, r * ldo + c, v);
    sum += odt != 3 ? (double)(float)v : v;  // sum what was stored
  }
  sum = block_sum(sum);
  if (threadIdx.x == 0) part[blockIdx.x] = sum;
}

// x *= sum(num) / sum(den)  (partial sums)
__global__ void scale_ratio_kernel(void* __restrict__ x, int dtype, long long rows, long long cols, long long ld,
                                   const double* __restrict__ num, const double* __restrict__ den, int nparts) {
  const double ratio = total(num, nparts) / total(den, nparts);
  const long long n = rows * cols, step = (long long)gridDim.x * kBlock;
  for (long long t = (long long)blockIdx.x * kBlock + threadIdx.x; t < n; t += step) {
    const long long i = (t / cols) * ld + t % cols;
    store_real(x, dtype, i, load_real(x, dtype, i) * ratio);
  }
}

static hipError_t launch_component_sum(const void* x, int dtype, int comp, long long rows, long long cols,
                                       long long ld, double* part, hipStream_t s) {
  hipLaunchKernelGGL(sum_kernel, dim3(part_blocks(rows * cols)), dim3(kBlock), 0, s, x, dtype, comp, rows, cols, ld,
                     part);
  return hipGetLastError();
}

hipError_t launch_sum(const void* x, int dtype, long long rows, long long cols, long long ld, double* part,
                      hipStream_t s) {
  return launch_component_sum(x, dtype, 0, rows, cols, ld, part, s);
}

hipError_t launch_magnitude(const void* F, long long ldF, long long rows, long long cols, long long r0, long long c0,
                            void* out, int odt, long long ldo, double* part, hipStream_t s) {
  hipLaunchKernelGGL(magnitude_kernel, dim3(part_blocks(rows * cols)), dim3(kBlock), 0, s, (const float2*)F, ldF, rows,
                     cols, r0, c0, out, odt, ldo, part);
  return hipGetLastError();
}

hipError_t launch_scale_ratio(void* x, int dtype, long long rows, long long cols, long long ld, const double* num,
                              const double* den, hipStream_t s) {
  if (rows * cols <= 0) return hipSuccess;
  const int nb = part_blocks(rows * cols);
  hipLaunchKernelGGL(scale_ratio_kernel, dim3(nb), dim3(kBlock), 0, s, x, dtype, rows, cols, ld, num, den, nb);
  return hipGetLastError();
}

// --------------------------------------------------------------------------
// rescale: map_coordinates(order 0..5, any boundary mode) on the device
// --------------------------------------------------------------------------
// The algorithm of scipy.ndimage.map_coordinates as util.rescale calls it:
// orders >= 2 prefilter the input with the inverse B-spline filter (after
// 12 samples of padding in modes 'nearest' and 'grid-constant'), with the
// mode's boundary rule; the spline of order p is then sampled with p + 1
// taps per axis, taps past the line extended by the mode's rule; 'constant'
// gives 0 outside [0, n - 1], and unpadded modes move an outside coordinate
// inside by their symmetry first.  cval is 0 (rescale never passes one).

namespace {

// index extension rules
enum { EX_CLAMP = 0, EX_REFLECT = 1, EX_MIRROR = 2, EX_PERIODIC = 3, EX_ZERO = 4 };

__host__ __device__ inline int filter_rule(int mode) {
  return mode == MFTX_MODE_GRID_WRAP ? EX_PERIODIC
         : (mode == MFTX_MODE_NEAREST || mode == MFTX_MODE_REFLECT || mode == MFTX_MODE_GRID_MIRROR) ? EX_REFLECT
                                                                                                    : EX_MIRROR;
}
__device__ inline int tap_rule(int mode) {
  switch (mode) {
    case MFTX_MODE_NEAREST: return EX_CLAMP;
    case MFTX_MODE_REFLECT:
    case MFTX_MODE_GRID_MIRROR: return EX_REFLECT;
    case MFTX_MODE_GRID_WRAP: return EX_PERIODIC;
    case MFTX_MODE_GRID_CONSTANT: return EX_ZERO;
    default: return EX_MIRROR;  // mirror, wrap (after its coordinate map), constant
  }
}

// Index of sample i of an n-sample line under a rule; -1 reads 0 (EX_ZERO).
__device__ __forceinline__ long long extend_index(long long i, long long n, int rule) {
  if (i >= 0 && i < n) return i;
  switch (rule) {
    case EX_CLAMP: return i < 0 ? 0 : n - 1;
    case EX_REFLECT: {  // half-sample symmetric, period 2n
      const long long p = 2 * n;
      long long k = i % p;
      if (k < 0) k += p;
      return k >= n ? p - 1 - k : k;
    }
    case EX_MIRROR: {  // whole-sample symmetric, period 2n - 2
      if (n == 1) return 0;
      const long long p = 2 * n - 2;
      long long k = i % p;
      if (k < 0) k += p;
      return k >= n ? p - k : k;
    }
    case EX_PERIODIC: {
      long long k = i % n;
      return k < 0 ? k + n : k;
    }
    default: return -1;
  }
}

// A coordinate outside [0, n - 1] moved inside by the mode's symmetry (only
// for unpadded lines; the other modes keep it).  For orders >= 1 this is
// the same as extending the taps; for order 0 it decides where a
// half-integer coordinate rounds to.
__device__ __forceinline__ double map_coordinate(double x, long long n, int mode) {
  const double last = (double)(n - 1);
  if (x >= 0.0 && x <= last) return x;
  const bool sym = mode == MFTX_MODE_MIRROR || mode == MFTX_MODE_REFLECT || mode == MFTX_MODE_GRID_MIRROR ||
                   mode == MFTX_MODE_WRAP || mode == MFTX_MODE_GRID_WRAP || mode == MFTX_MODE_NEAREST;
  if (!sym) return x;
  if (n <= 1) return 0.0;
  switch (mode) {
    case MFTX_MODE_MIRROR: {
      const double p = 2.0 * n - 2.0;
      if (x < 0) {
        x += p * trunc(-x / p);
        return x <= 1.0 - n ? x + p : -x;
      }
      x -= p * trunc(x / p);
      return x >= n ? p - x : x;
    }
    case MFTX_MODE_REFLECT:
    case MFTX_MODE_GRID_MIRROR: {
      const double p = 2.0 * n;
      if (x < 0) {
        if (x < -p) x += p * trunc(-x / p);
        return x < -n ? x + p : (x > -1e-15 ? 1e-15 : -x) - 1.0;
      }
      x -= p * trunc(x / p);
      return x >= n ? p - x - 1.0 : x;
    }
    case MFTX_MODE_WRAP: {
      const double p = (double)(n - 1);
      return x < 0 ? x + p * (trunc(-x / p) + 1.0) : x - p * trunc(x / p);
    }
    case MFTX_MODE_GRID_WRAP:
      return x < 0 ? x + n * (trunc(-x / n) + 1.0) : x - n * trunc(x / n);
    default:  // nearest
      return x < 0 ? 0.0 : last;
  }
}

// The centred B-spline of degree `order` at t.
__device__ __forceinline__ double bspline(int order, double t) {
  t = fabs(t);
  switch (order) {
    case 0: return t <= 0.5 ? 1.0 : 0.0;
    case 1: return t < 1.0 ? 1.0 - t : 0.0;
    case 2: return t < 0.5 ? 0.75 - t * t : (t < 1.5 ? 0.5 * (1.5 - t) * (1.5 - t) : 0.0);
    case 3: return t < 1.0 ? 2.0 / 3.0 - t * t + 0.5 * t * t * t : (t < 2.0 ? (2.0 - t) * (2.0 - t) * (2.0 - t) / 6.0 : 0.0);
    case 4: {
      const double t2 = t * t;
      if (t < 0.5) return 115.0 / 192.0 - 5.0 * t2 / 8.0 + t2 * t2 / 4.0;
      if (t < 1.5) return 55.0 / 96.0 + 5.0 * t / 24.0 - 5.0 * t2 / 4.0 + 5.0 * t2 * t / 6.0 - t2 * t2 / 6.0;
      if (t < 2.5) { const double u = 2.5 - t; return u * u * u * u / 24.0; }
      return 0.0;
    }
    default: {
      const double t2 = t * t;
      if (t < 1.0) return 11.0 / 20.0 - t2 / 2.0 + t2 * t2 / 4.0 - t2 * t2 * t / 12.0;
      if (t < 2.0)
        return 17.0 / 40.0 + 5.0 * t / 8.0 - 7.0 * t2 / 4.0 + 5.0 * t2 * t / 4.0 - 3.0 * t2 * t2 / 8.0 +
               t2 * t2 * t / 24.0;
      if (t < 3.0) { const double u = 3.0 - t; return u * u * u * u * u / 120.0; }
      return 0.0;
    }
  }
}

__device__ __forceinline__ long long first_tap(double c, int order) {
  return order & 1 ? (long long)floor(c) - (order - 1) / 2 : (long long)floor(c + 0.5) - order / 2;
}

__device__ __forceinline__ bool nonzero(const void* p, int dtype, long long i) {
  return load_component(p, dtype, i, 0) != 0.0 || ((dtype == 0 || dtype == 2) && load_component(p, dtype, i, 1) != 0.0);
}

}  // namespace

// P (P0 x P1, double) = component comp of img (rows x cols) with npad samples
// of padding on every side: edge values (numpy.pad mode='edge') or zeros.
__global__ void rescale_load_kernel(const void* __restrict__ img, int dtype, int comp, long long rows, long long cols,
                                    long long ld, int npad, int pad_zero, double* __restrict__ P) {
  const long long P0 = rows + 2 * npad, P1 = cols + 2 * npad;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= P0 * P1) return;
  const long long i = t / P1 - npad, j = t % P1 - npad;
  if (pad_zero && (i < 0 || i >= rows || j < 0 || j >= cols)) {
    P[t] = 0.0;
    return;
  }
  const long long r = min(max(i, 0LL), rows - 1), c = min(max(j, 0LL), cols - 1);
  P[t] = load_component(img, dtype, r * ld + c, comp);
}

// The B-spline prefilter, one axis at a time, as its two-sided impulse response
//     dst[i] = sum_{|k| <= taps} h[|k|] src[extend(i + k)].
// h is the product over the order's poles z of (1 - z) / (1 + z) z^|k|,
// truncated where it falls below double rounding (launch_rescale says where);
// the boundary rule is the mode's.  Each block stages its samples and their halo in LDS once, the
// extension rule applied there (the loads in batches, so their latency is paid
// a few times); a thread computes NQ consecutive outputs from two windows that
// slide by one sample per tap, two LDS reads per tap for all of them.  The sum
// runs in the order k = 0, 1, ...  Every output reading its neighbours through
// the caches and extending every index itself took 95 us per axis for 1048^2.
//
// window(d): this thread's sample at distance d from its first output.
template <int NQ, typename Window>
__device__ __forceinline__ void fir_outputs(const PrefilterTaps& taps, Window&& window, double (&s)[NQ]) {
  double l[NQ], r[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    l[q] = r[q] = window(q);
    s[q] = taps.h[0] * l[q];
  }
  auto step = [&](int k) {
    const double h = taps.h[k];
#pragma unroll
    for (int q = NQ - 1; q > 0; --q) l[q] = l[q - 1];
    l[0] = window(-k);
#pragma unroll
    for (int q = 0; q < NQ - 1; ++q) r[q] = r[q + 1];
    r[NQ - 1] = window(NQ - 1 + k);
#pragma unroll
    for (int q = 0; q < NQ; ++q) s[q] += h * (l[q] + r[q]);
  };
  int k = 1;
  for (; k + NQ - 1 <= taps.n; k += NQ)  // whole turns of the windows: the shifts are renames
#pragma unroll
    for (int u = 0; u < NQ; ++u) step(k + u);
  for (; k <= taps.n; ++k) step(k);
}

// Columns (axis 0), straight from the image: component comp with npad samples
// of edge values (or zeros) around it.  256 threads: 32 columns x 64 rows, 8
// rows per thread.  The dtype is a template parameter (a test per load would
// wait for each); HALO is the LDS reserved for the taps, at most that many:
// orders 2 and 3 fit 32, so five blocks fit a CU.
constexpr int kFirRows = 64, kFirCols = 32;
template <int DT, int HALO>
__global__ __launch_bounds__(256) void fir_columns_kernel(const void* __restrict__ img, int comp,
                                                          long long rows, long long cols, long long ld, int npad,
                                                          int pad_zero, int rule, PrefilterTaps taps,
                                                          double* __restrict__ dst) {
  __shared__ double L[kFirRows + 2 * HALO][kFirCols];
  const long long P0 = rows + 2 * npad, P1 = cols + 2 * npad;
  const unsigned nbc = (unsigned)((P1 + kFirCols - 1) / kFirCols);
  const int lc = threadIdx.x & 31, group = threadIdx.x >> 5;
  const long long c = (long long)(blockIdx.x % nbc) * kFirCols + lc, r0 = (long long)(blockIdx.x / nbc) * kFirRows;
  const long long ic = min(max(c - npad, 0LL), cols - 1);
  const bool zc = pad_zero && (c - npad < 0 || c - npad >= cols);
  const int nload = (int)min((long long)kFirRows, P0 - r0) + 2 * taps.n;
  for (int i0 = group; i0 < nload; i0 += 64) {
    double v[8];
    bool z[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const long long r = extend_index(r0 + min(i0 + 8 * b, nload - 1) - taps.n, P0, rule) - npad;
      z[b] = zc || (pad_zero && (r < 0 || r >= rows));
      v[b] = load_component(img, DT, min(max(r, 0LL), rows - 1) * ld + ic, comp);
    }
#pragma unroll
    for (int b = 0; b < 8; ++b)
      if (i0 + 8 * b < nload) L[i0 + 8 * b][lc] = z[b] ? 0.0 : v[b];
  }
  __syncthreads();
  double s[8];
  // rows past the last are computed from whatever LDS holds and not stored
  fir_outputs<8>(taps, [&](int d) { return L[group * 8 + taps.n + d][lc]; }, s);
  if (c >= P1) return;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const long long r = r0 + group * 8 + q;
    if (r < P0) dst[r * P1 + c] = s[q];
  }
}

// Rows (axis 1) of a P0 x P1 array.  256 threads: 4 rows x 256 columns, a
// thread 4 adjacent columns; column c of a row lies at [c & 3][c >> 2], so
// lanes 4 columns apart read neighbouring LDS words.
constexpr int kFirSpan = 256;
__global__ __launch_bounds__(256) void fir_rows_kernel(const double* __restrict__ src, long long P0, long long P1,
                                                       int rule, PrefilterTaps taps, double* __restrict__ dst) {
  constexpr int W = (kFirSpan + 2 * kPrefilterTaps) / 4;
  __shared__ double L[4][4][W];
  const long long nbc = (P1 + kFirSpan - 1) / kFirSpan;
  const long long c0 = blockIdx.x % nbc * kFirSpan, r0 = blockIdx.x / nbc * 4;
  const int nrow = (int)min(4LL, P0 - r0);
  const int nload = (int)min((long long)kFirSpan, P1 - c0) + 2 * taps.n;
  for (int i = threadIdx.x; i < nload; i += 256) {
    const long long c = extend_index(c0 + i - taps.n, P1, rule);
    double v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = src[(r0 + min(q, nrow - 1)) * P1 + c];
#pragma unroll
    for (int q = 0; q < 4; ++q) L[q][i & 3][i >> 2] = v[q];
  }
  __syncthreads();
  const int row = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double s[4];
  fir_outputs<4>(taps, [&](int d) { return L[row][(taps.n + d) & 3][lane + ((taps.n + d) >> 2)]; }, s);
  if (row >= nrow) return;
  const long long c = c0 + 4 * (threadIdx.x & 63);
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (c + q < P1) dst[(r0 + row) * P1 + c + q] = s[q];
}

// Resample at the coordinates of util.py:333-336,
//   y = (r - orows / 2) / scale + rows / 2,  x = (c - ocols / 2) / scale + cols / 2,
// from the coefficients C (P0 x P1, npad samples of padding) with spline
// order 0..5 and the mode's tap and coordinate rules.  With mval, the mask
// (mask_mode 1: img != 0; 2: a real mask array) is sampled with order 1,
// mode 'nearest', on the unpadded grid and zeroed below eps
// (util.py:338-339).  raw = interpolated value, part = block sums of raw.
// The order is a template parameter, so a low one loads no taps that it has not: a
// rescale from 2000^2 to 3200^2 at order 0 takes 171.8 us, 267 with six taps for every
// order (and every block of the last launch adding the partial sums for 256 pixels).
template <int order>
__global__ void resample_kernel(const double* __restrict__ C, long long P0, long long P1, int npad,
                                int mode, long long rows, long long cols, double scale, long long orows,
                                long long ocols, const void* __restrict__ msrc, int mask_mode, int mdt, long long ldm,
                                double eps, double* __restrict__ raw, double* __restrict__ mval,
                                double* __restrict__ part) {
  double sum = 0.0;
  const long long n = orows * ocols, step = (long long)gridDim.x * kBlock;
  for (long long t = (long long)blockIdx.x * kBlock + threadIdx.x; t < n; t += step) {
    double v = 0.0;
    const long long r = t / ocols, c = t % ocols;
    const double y = ((double)r - (double)orows / 2.0) / scale + (double)rows / 2.0;
    const double x = ((double)c - (double)ocols / 2.0) / scale + (double)cols / 2.0;
    const bool outside = mode == MFTX_MODE_CONSTANT && (y < 0.0 || y > (double)(rows - 1) || x < 0.0 ||
                                                       x > (double)(cols - 1));
    if (!outside) {
      const double cy = (npad ? y : map_coordinate(y, rows, mode)) + npad;
      const double cx = (npad ? x : map_coordinate(x, cols, mode)) + npad;
      const int rule = tap_rule(mode);
      const long long sy = first_tap(cy, order), sx = first_tap(cx, order);
      // the columns' taps and weights once, every load of a row before its sum
      long long cc[order + 1];
      double wx[order + 1];
      unsigned past = 0;  // taps outside the line (EX_ZERO): they read column 0, which may not be finite
#pragma unroll
      for (int b = 0; b <= order; ++b) {
        cc[b] = extend_index(sx + b, P1, rule);
        wx[b] = cc[b] >= 0 ? bspline(order, cx - (double)(sx + b)) : 0.0;
        if (cc[b] < 0) past |= 1u << b;
        cc[b] = max(cc[b], 0LL);
      }
      for (int a = 0; a <= order; ++a) {
        const long long rr = extend_index(sy + a, P0, rule);
        if (rr < 0) continue;
        double e[order + 1], row = 0.0;
#pragma unroll
        for (int b = 0; b <= order; ++b) e[b] = C[rr * P1 + cc[b]];
        if (past) {
#pragma unroll
          for (int b = 0; b <= order; ++b) e[b] = past >> b & 1 ? 0.0 : e[b];
        }
#pragma unroll
        for (int b = 0; b <= order; ++b) row += wx[b] * e[b];
        v += bspline(order, cy - (double)(sy + a)) * row;
      }
    }
    raw[t] = v;
    sum += v;
    if (mval) {
      const double my = fmin(fmax(y, 0.0), (double)(rows - 1)), mx = fmin(fmax(x, 0.0), (double)(cols - 1));
      const long long fy = (long long)floor(my), fx = (long long)floor(mx);
      const double ty = my - fy, tx = mx - fx;
      const long long r1 = min(fy + 1, rows - 1), c1 = min(fx + 1, cols - 1);
      auto m = [&](long long rr, long long cc) -> double {
        return mask_mode == 1 ? (nonzero(msrc, mdt, rr * ldm + cc) ? 1.0 : 0.0) : load_real(msrc, mdt, rr * ldm + cc);
      };
      double mv =
          (1 - ty) * ((1 - tx) * m(fy, fx) + tx * m(fy, c1)) + ty * ((1 - tx) * m(r1, fx) + tx * m(r1, c1));
      if (mv < eps) mv = 0.0;
      mval[t] = mv;
    }
  }
  sum = block_sum(sum);
  if (threadIdx.x == 0) part[blockIdx.x] = sum;
}

// out = raw * (unitary ? sum(img) / sum(raw) : 1) * mval   (util.py:340-347);
// with raw_im, complex: the ratio of the complex sums, out complex64 (odt 0)
// or complex128 (odt 2).  The partial sums of (img_re, img_im, raw_re, raw_im)
// lie kMaxPart apart, ni of each image sum and nr of each resampled one.
__global__ void rescale_finish_kernel(const double* __restrict__ raw, const double* __restrict__ raw_im,
                                      const double* __restrict__ mval, long long orows, long long ocols, int unitary,
                                      const double* __restrict__ part, int ni, int nr, void* __restrict__ out,
                                      int odt, long long ldo) {
  double sums[4] = {};
  if (unitary)
    for (int q = 0; q < 4; ++q)
      if (raw_im || !(q & 1)) sums[q] = total(part + q * kMaxPart, q < 2 ? ni : nr);
  const double ratio = sums[0] / sums[2];
  const long long n = orows * ocols, step = (long long)gridDim.x * kBlock;
  for (long long t = (long long)blockIdx.x * kBlock + threadIdx.x; t < n; t += step) {
    const long long o = (t / ocols) * ldo + t % ocols;
    if (!raw_im) {
      double v = raw[t];
      if (unitary) v *= ratio;
      store_real(out, odt, o, v * mval[t]);
      continue;
    }
    double re = raw[t], im = raw_im[t];
    if (unitary) {
      // (a + ib) / (c + id) with a, b = sum(img), c, d = sum(raw)
      const double a = sums[0], b = sums[1], c = sums[2], d = sums[3];
      const double den = c * c + d * d;
      const double qr = (a * c + b * d) / den, qi = (b * c - a * d) / den;
      const double nr = re * qr - im * qi;
      im = re * qi + im * qr;
      re = nr;
    }
    re *= mval[t];
    im *= mval[t];
    if (odt == 2) ((double2*)out)[o] = make_double2(re, im);
    else ((float2*)out)[o] = make_float2((float)re, (float)im);
  }
}

// The order's prefilter response h[|k|], k <= kPrefilterTaps, computed once
// per order on the host: the product over the B-spline's poles z (Unser's
// values) of (1 - z) / (1 + z) z^|k|, formed on a support four times wider
// than kept so the truncation drops only terms below double rounding
// (|z|^48 < 3e-18 for the largest pole, order 5).
static PrefilterTaps make_prefilter_taps(int order) {
  PrefilterTaps h = {};
  h.h[0] = 1.0;
  if (order < 2) return h;
  std::vector<double> z;
  if (order == 2) z = {std::sqrt(8.0) - 3.0};
  if (order == 3) z = {std::sqrt(3.0) - 2.0};
  if (order == 4)
    z = {std::sqrt(664.0 - std::sqrt(438976.0)) + std::sqrt(304.0) - 19.0,
         std::sqrt(664.0 + std::sqrt(438976.0)) - std::sqrt(304.0) - 19.0};
  if (order == 5)
    z = {std::sqrt(67.5 - std::sqrt(4436.25)) + std::sqrt(26.25) - 6.5,
         std::sqrt(67.5 + std::sqrt(4436.25)) - std::sqrt(26.25) - 6.5};
  constexpr int W = 4 * kPrefilterTaps;
  std::vector<double> cur(2 * W + 1, 0.0), nxt(2 * W + 1), g(2 * W + 1);
  cur[W] = 1.0;
  for (double zp : z) {
    double zk = (1.0 - zp) / (1.0 + zp);
    for (int k = 0; k <= W; ++k, zk *= zp) g[W + k] = g[W - k] = zk;
    for (int i = 0; i <= 2 * W; ++i) {
      double acc = 0.0;
      for (int j = std::max(0, i - W); j <= std::min(2 * W, i + W); ++j) acc += g[W + i - j] * cur[j];
      nxt[i] = acc;
    }
    cur.swap(nxt);
  }
  for (int k = 0; k <= kPrefilterTaps; ++k) h.h[k] = cur[W + k];
  // the last tap that is not lost in the rounding of the first (2^-56 of it:
  // 23 taps for order 2, 30, 39 and 46 for orders 3 to 5)
  while (h.n < kPrefilterTaps && std::fabs(h.h[h.n + 1]) > std::ldexp(h.h[0], -56)) ++h.n;
  return h;
}

PrefilterTaps prefilter_taps(int order) {
  static const PrefilterTaps table[6] = {make_prefilter_taps(0), make_prefilter_taps(1), make_prefilter_taps(2),
                                         make_prefilter_taps(3), make_prefilter_taps(4), make_prefilter_taps(5)};
  return table[order < 0 || order > 5 ? 0 : order];
}

hipError_t launch_rescale(const void* img, int dtype, long long rows, long long cols, long long ld, const void* msrc,
                          int mask_mode, int mdt, long long ldm, double eps, double scale, long long orows,
                          long long ocols, int order, int mode, int unitary, void* out, int odt, long long ldo,
                          double* P, double* T, double* raw, double* raw_im, double* mval, double* part,
                          hipStream_t s) {
  const bool cplx = dtype == 0 || dtype == 2;
  const int npad = order > 1 && (mode == MFTX_MODE_NEAREST || mode == MFTX_MODE_GRID_CONSTANT) ? 12 : 0;
  const int zero = mode == MFTX_MODE_GRID_CONSTANT ? 1 : 0;
  const long long P0 = rows + 2 * npad, P1 = cols + 2 * npad;
  const int ni = part_blocks(rows * cols), nr = part_blocks(orows * ocols);
  // Taps lost in rounding still carry a sample that is not finite to 48 outputs
  // on either side; after the unitary ratio nothing of such an image is finite,
  // so they are left out there (1024^2 by 4, order 3: a call takes 43 us with them, 36 without)
  PrefilterTaps taps = prefilter_taps(order);
  if (!unitary) taps.n = kPrefilterTaps;
  for (int comp = 0; comp < (cplx ? 2 : 1); ++comp) {
    if (unitary) {
      const hipError_t e = launch_component_sum(img, dtype, comp, rows, cols, ld, part + comp * kMaxPart, s);
      if (e != hipSuccess) return e;
    }
    if (order > 1) {
      const auto columns = taps.n <= 32 ? (dtype == 0 ? fir_columns_kernel<0, 32> : dtype == 1 ? fir_columns_kernel<1, 32>
                                           : dtype == 2 ? fir_columns_kernel<2, 32> : fir_columns_kernel<3, 32>)
                                        : (dtype == 0 ? fir_columns_kernel<0, kPrefilterTaps>
                                           : dtype == 1 ? fir_columns_kernel<1, kPrefilterTaps>
                                           : dtype == 2 ? fir_columns_kernel<2, kPrefilterTaps>
                                                        : fir_columns_kernel<3, kPrefilterTaps>);
      hipLaunchKernelGGL(columns, dim3((unsigned)((P1 + kFirCols - 1) / kFirCols * ((P0 + kFirRows - 1) / kFirRows))),
                         dim3(256), 0, s, img, comp, rows, cols, ld, npad, zero, filter_rule(mode), taps, T);
      hipLaunchKernelGGL(fir_rows_kernel, dim3((unsigned)((P1 + 255) / 256 * ((P0 + 3) / 4))), dim3(256), 0, s,
                         (const double*)T, P0, P1, filter_rule(mode), taps, P);
    } else {
      hipLaunchKernelGGL(rescale_load_kernel, dim3(blocks_for(P0 * P1)), dim3(kBlock), 0, s, img, dtype, comp, rows,
                         cols, ld, npad, zero, P);
    }
    const auto resample = order == 0 ? resample_kernel<0> : order == 1 ? resample_kernel<1> : order == 2 ? resample_kernel<2>
                          : order == 3 ? resample_kernel<3> : order == 4 ? resample_kernel<4> : resample_kernel<5>;
    hipLaunchKernelGGL(resample, dim3(nr), dim3(kBlock), 0, s, (const double*)P, P0, P1, npad, mode,
                       rows, cols, scale, orows, ocols, msrc, mask_mode, mdt, ldm, eps, comp ? raw_im : raw,
                       comp ? (double*)nullptr : mval, part + (2 + comp) * kMaxPart);
  }
  // every block adds the partial sums, so there are no more blocks than fill the chip
  hipLaunchKernelGGL(rescale_finish_kernel, dim3(std::min(blocks_for(orows * ocols), 2048u)), dim3(kBlock), 0, s, (const double*)raw,
                     cplx ? (const double*)raw_im : nullptr, (const double*)mval, orows, ocols, unitary,
                     (const double*)part, ni, nr, out, odt, ldo);
  return hipGetLastError();
}

}  // namespace mftx
