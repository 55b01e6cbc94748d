// Internal declarations shared by the MFT kernels and the C-ABI host code.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

struct mftx_ctx;

namespace mftx {

// Every GEMM operand lives in HBM as MFMA fragments: 1 KiB blocks, one per
// 32 rows (or slots) x 16 K values of one 16-bit plane, holding lane l's eight
// K values 8 (l / 32) .. + 7 of row l % 32 at byte 16 l.  A block is loaded
// into LDS or registers by one 16-byte-per-lane access, whole cache lines,
// and read from LDS without bank conflicts.
constexpr int BK = 16;                 // K values per block
constexpr int FRAG = 1024;             // bytes of one fragment
constexpr int A_BLOCK = 8 * FRAG;      // operand bytes per (32 rows, K block): two parts x four planes
constexpr int B_BLOCK = 4 * FRAG;      // twiddle bytes per (32 slots, K block): cos hi, cos lo, sin hi, sin lo

// Number formats of the split operands: every value is hi + lo of one 16-bit
// type, a real product is hi*hi + hi*lo + lo*hi with FP32 accumulation.
//   PREC_FP32   : f16 pairs (22 bits).  The operand is scaled by a power of two
//                 per launch so its largest value fits f16 (see ScaleSrc).  From
//                 about 24 samples an axis on, the result's error is below that
//                 of FP32 MFMAs, whose rounding grows with the K / 2 accumulations
//                 of a K = 2 instruction; a handful of samples or of bright ones
//                 adds few roundings, and there the 22 bits show (1.4e-7, not 8e-8).
//   PREC_BF16X3 : bf16 pairs (16 bits), no scaling.
enum Precision { PREC_FP32 = 0, PREC_BF16X3 = 1 };

// Epilogues of the GEMM.
enum Epilogue {
  EPI_STORE_CPLX = 0,    // dst complex64, (r, j) -> dst[j*ld + r] if trans else dst[r*ld + j]; * scale; bounds
  EPI_STORE_PACKED = 1,  // dst is the next stage's operand: rows = output columns j, K = C rows
  EPI_INTENSITY = 2,     // accumulate w*|C|^2 over the work item's problems into a partial image
};

// Workgroup tiles of the GEMM (see mftx_gemm.hip).
enum Tile { TILE_SMALL = 0, TILE_MID = 1, TILE_BIG = 2, TILE_MULTI = 3 };
inline int tile_rows(int t) { return t == TILE_BIG ? 4 : t == TILE_SMALL ? 1 : 2; }  // 32-row blocks
inline int tile_slots(int t) { return tile_rows(t); }                               // 32-slot blocks

// One K segment of a GEMM problem.
struct Seg {
  const void* a;        // operand: [row block][a_nkb][A_BLOCK]
  const void* b;        // twiddles: [slot block][b_nkb][B_BLOCK]
  double rot;           // turns per unit Y the accumulators turn by before this segment (0: none)
  int nkb;              // K blocks
  int a_nkb, b_nkb;     // K blocks per row block of a / per slot block of b
  int pad_;
};

// One complex GEMM problem: one MFT stage,
//   C[i][j] = sum_k A[i][k] cis(alpha x_k (j - N/2 - shift)),   0 <= j < N = ncols,
// with cis(t) = exp(2 pi i t) and N/2 the integer half, computed about a
// pairing centre c (integer or half-integer; the host picks it at the PSF core
// j = N/2 + shift or at the grid centre next to it).  The producer of A has
// multiplied A[i][k] by the fold cis(-alpha (shift + N/2 - c) x_k), so that
// with Y = j - c
//   C[i][j] = sum_k A'[i][k] cis(alpha x_k Y).
// Both coordinates are paired.  x runs symmetrically about its midpoint xc,
// x = xc +- x' with x' = k' + 1/2 (even length) or k' (odd), and the operand
// holds the even and odd parts Ae = A'(+x') + A'(-x'), Ao = A'(+x') - A'(-x'):
//   C[i][j] = cis(alpha xc Y) (P + iQ),  P = sum_k' Ae cos(2 pi alpha x' Y),
//                                        Q = sum_k' Ao sin(2 pi alpha x' Y),
// half the K of the plain product.  P is even and Q odd in Y, so the GEMM runs
// over slots s = 0 .. cols-1 with Y_s = y0 + s only (y0 = 0 for integer c, 1/2
// otherwise) and gives both output columns cp + s (P + iQ) and cm - s (P - iQ)
// (cp = ceil(c), cm = floor(c); outputs outside [0, N) are dropped, and the
// second where it equals the first).  c = 0 is the direct product (one output
// per slot).  The phase cis(alpha xc Y) is left out where only |C|^2 of one
// segment matters, and applied by the store otherwise (xrot).  Segments with
// their own xc follow each other along K: turning (P, Q) by alpha (xc - xc')
// re-expresses the sum so far about the next segment's midpoint.
struct Problem {
  int sbeg, send;       // K segments
  int rblocks, sblocks; // 32-row blocks of the operand, 32-slot blocks of the twiddle table
  int cols;             // slots
  int ncols;            // N: output columns
  int i0, i1, j0, j1;   // EPI_STORE_CPLX and coherent sums: the C rows and columns that count (a window
                        //   of C; the stored array starts at (i0, j0))
  int cp, cm;           // output columns of slot 0 (P + iQ, P - iQ)
  int trans;            // EPI_STORE_CPLX / EPI_INTENSITY: write C transposed
  double y0;            // Y of slot 0
  double xrot;          // stores: turns per unit Y of the phase applied to the output (0: none)
  const float* inv;     // optional device factor of the scale (undoes the operand's scaling)
  float scale;          // store: C *= scale; intensity: C *= scale before |C|^2
  float weight;         // intensity: weight of |C|^2
  void* dst;            // store destination (EPI_STORE_*)
  long long ldd;        // EPI_STORE_CPLX: row stride; EPI_STORE_PACKED: K blocks per row block of dst
  const void* wmap;     // EPI_STORE_CPLX: optional real map multiplied into each stored value,
  long long ldw;        //   indexed like the destination (row stride ldw)
  int wdtype;           //   1 float32, 3 float64
  int wrow, wcol;       //   added to F's row and column index, modulo wrows and wcols
  int wrows, wcols;
  int pad2_;
  const float2* rowph;  // EPI_STORE_CPLX: optional phase per C row
};

// A workgroup's unit of work: problems [pbeg, pend) on tile (tr, tc) of C.
// For EPI_INTENSITY the problems' |C|^2 are summed into partial[r][c]
// (row-major, stride ldp, transposed like the problems' trans flag).  nch is
// the K blocks of all its problems together.
struct Work {
  int pbeg, pend;
  int tr, tc;
  float* partial;
  long long ldp;
  int prows, pcols;     // partial image extent (bounds for the store)
  int nch, pad_;
};

// Extents of a paired operand axis of n samples: pairs, and 16-pair blocks.
__host__ __device__ inline long long pairs(long long n) { return (n + 1) / 2; }
__host__ __device__ inline int pair_blocks(long long n) { return (int)((pairs(n) + BK - 1) / BK); }
// Bytes of the operand of an r x k array (row pairs in blocks of 16: the 16
// even rows, then the 16 odd rows, of each block), and of a plain-row operand
// (stage 2: rows are output columns) with nkb K blocks.
inline size_t folded_bytes(long long r, long long k) { return (size_t)pair_blocks(r) * pair_blocks(k) * A_BLOCK; }
inline size_t plain_bytes(long long rows, int nkb) { return (size_t)((rows + 31) / 32) * nkb * A_BLOCK; }

// Scaling of a PREC_FP32 operand: `part` holds absolute maxima of the source
// (written by launch_absmax); the consumers scale by the power of two that
// takes four times their maximum (the sum of a pixel and its three mirror
// images) to at most 2^14, and *inv receives its reciprocal.  n = 0: no scaling.
struct ScaleSrc {
  const float* part;
  float* inv;
  int n, pad_;
};
// One absolute-maximum job: blocks [begin, begin + nblk) of the launch write
// part[0 .. nblk).
struct MaxOp {
  const void* src;
  int dtype;            // 0..3 (see load_elem)
  int nblk;
  long long m, n, ld;
  float* part;
  long long begin;
};
constexpr int kMaxBlocks = 256;  // blocks (and part entries) of one absolute-maximum job, at most
inline int max_blocks(long long m, long long n) {
  const long long b = (m * n + 1023) / 1024;
  return (int)(b < 1 ? 1 : b > kMaxBlocks ? kMaxBlocks : b);
}

// One twiddle table: cos and sin of 2 pi alpha x' (y0 + s), x' = k' + x0,
// times tw_scale(prec), for nsb blocks of 32 slots from slot block sb0 and nkb
// blocks of 16 k'.
struct TableOp {
  double alpha, x0, y0;
  int nsb, nkb, sb0, pad_;
  void* dst;
  long long begin;      // first thread: one per (slot, 2 k')
};
__host__ __device__ inline long long table_threads(int nsb, int nkb) { return 256LL * nsb * nkb; }
inline size_t table_bytes(int nsb, int nkb) { return (size_t)nsb * nkb * B_BLOCK; }
// Twiddles of the f16 form are scaled so the lo parts of small ones stay normal.
__host__ __device__ inline float tw_scale(int prec) { return prec == PREC_FP32 ? 256.0f : 1.0f; }

// Per-wavelength parameters of a phasor launch, in quarter turns (rates times
// 4, so the kernels reduce the phase without a product): the phase opd * inv_wl, the
// stage-1 fold cis(fold * (x0 + k)) along the operand's K index k, and the
// stage-2 fold cis(fold2 * (x02 + r)) along its row index r (stage 1's C row r
// is the operand's row r times the row's phase, so the stage-1 output comes
// out folded for stage 2).  k and r index the source before pairing.
struct PhasorWave {
  double inv_wl;
  double fold;
  double x0;
  double fold2;
  double x02;
};

// One operand source (a pupil phasor at nwave wavelengths, or complex data:
// nwave = 1): the folded, paired operand of the m x n source (rows are the
// source's columns when trans) for every wavelength, written wave_stride bytes
// apart.  `begin` is the op's first thread in the grouped launch.
struct PhasorOp {
  const void* amp;      // amplitude, or the complex source
  const void* opd;      // OPD; null for a complex source
  int amp_dtype, opd_dtype;
  long long ld_amp, ld_opd;
  int m, n, trans, nwave;
  int conj, pad_;       // complex source: conjugate it
  const PhasorWave* waves;
  void* dst;
  long long wave_stride;
  ScaleSrc sc;
  long long begin;
};
// How an operand launch splits its work: K pairs (2 or 4) and wavelengths
// per thread.
struct OperandSplit {
  int np, waves;
};
// threads of one wavelength group of an r x k operand (whole waves)
__host__ __device__ inline long long group_threads(long long r, long long k, int np) {
  return ((long long)pair_blocks(r) * pair_blocks(k) * (256 / np) + 63) / 64 * 64;
}
__host__ __device__ inline long long operand_threads(long long r, long long k, int nwave, OperandSplit sp) {
  return group_threads(r, k, sp.np) * ((nwave + sp.waves - 1) / sp.waves);
}
// The split of a launch of `quads` (row pair, K pair) quads over all its
// sources and wavelengths.  Large launches: 4 pairs and 4 wavelengths per
// thread, so a source is read once per 4 wavelengths.  Where that would leave
// fewer than two waves per SIMD (131072 threads), one wavelength and 2 pairs:
// the launch then takes the latency of 8 samples instead of 64.
inline OperandSplit operand_split(long long quads) {
  return quads / 16 >= 131072 ? OperandSplit{4, 4} : OperandSplit{2, 1};
}
inline long long operand_quads(long long r, long long k, int nwave) {
  return 256LL * pair_blocks(r) * pair_blocks(k) * nwave;
}

// Grouped launches (phasor, table, maximum ops): blocks of kGroupBlock threads, and
// every op's first thread is a multiple of kGroupBlock, so a block belongs to
// one op and finds it with a block-uniform search.
constexpr int kGroupBlock = 256;
inline long long group_begin(long long total) { return (total + kGroupBlock - 1) / kGroupBlock * kGroupBlock; }

// launchers (mftx_gemm.hip, mftx_kernels.hip)
hipError_t launch_gemm(int prec, int epi, int tile, const Work* work, int nwork, const Problem* probs,
                       const Seg* segs, hipStream_t s);
// groups of windows of one grid (gemm_coherent_kernel)
hipError_t launch_gemm_coherent(int prec, const Work* work, int nwork, const Problem* probs, const Seg* segs,
                                hipStream_t s);
// one problem (on the device, with its one segment of nch K blocks) over row
// blocks [0, rblocks) and slot blocks [sb0, sb1), sb0 on a tile boundary
hipError_t launch_gemm_one(int prec, int epi, int tile, int rblocks, int sb0, int sb1, int nch, const Problem* prob,
                           const Seg* seg, hipStream_t s);
// every operand source of a plan in one launch (ops_dev on the device, sorted
// by begin): pupil phasors, or (cplx) complex arrays
hipError_t launch_operands(int prec, bool cplx, OperandSplit sp, const PhasorOp* ops_dev, int nops,
                           long long total_threads, hipStream_t s);
// every twiddle table / absolute maximum in one launch (sorted by begin)
hipError_t launch_tables(int prec, const TableOp* ops_dev, int nops, long long total_threads, hipStream_t s);
hipError_t launch_absmax(const MaxOp* ops_dev, int nops, long long total_blocks, hipStream_t s);
// One transform's operand, twiddle tables and descriptors (prepare_one_kernel),
// passed by value: nothing is uploaded.  With op.sc.n == 0 the f16 form's
// maximum is taken inside the launch; tables with nsb = 0 are there already.
struct OneDesc {
  Problem prob[2];
  Seg seg[2];
};
struct OneMft {
  PhasorOp op;
  PhasorWave wave;
  TableOp tab[2];
  OneDesc desc;
  OneDesc* desc_dev;    // device copy for the GEMM launches
  double* sums;         // f16 form of a long transform: space for the source's block sums, else null
};
hipError_t launch_prepare_one(int prec, const OneMft& one, const MaxOp& mx, hipStream_t s);
hipError_t launch_table_one(int prec, const TableOp& op, hipStream_t s);
// table[r] = cis(rate * (r - centre)) for every op (rows 0: none)
struct RowPhase {
  double rate, centre;
  float2* table;
  int rows, pad_;
};
hipError_t launch_row_phases(const RowPhase* ops_dev, int nops, int most_rows, hipStream_t s);
// A phasor Field of a list: dst = amp exp(2 pi i opd inv_wl), m x n, dense.
struct PhasorField {
  const void *amp, *opd;
  float2* dst;
  long long ld_amp, ld_opd;
  int m, n, amp_dtype, opd_dtype;
};
hipError_t launch_phasor_fields(const PhasorField* items, int count, double inv_wl, hipStream_t s);
// One region of the image: ngroups partial images of rows x cols (row stride
// ldp, gstride floats apart) whose first pixel lies at (r0, c0).
struct ReduceOp {
  const float* partial;
  long long gstride, ldp;
  int ngroups, rows, cols, r0, c0, pad_;
};
// image (+)= unit times the sum of the regions
hipError_t launch_reduce(const ReduceOp* ops, int nops, void* image, int dtype, long long ldi, int rows, int cols,
                         int accumulate, double unit, hipStream_t s);
// Coherent groups of a plan whose Fields have several output grids: group g's
// Fields are adds[first .. first + count) of the launch.
struct CoherentAdd {
  const float2* F;      // M x N, row stride N
  int M, N;
  int r0, c0;           // image pixel of F[0][0] (may lie outside the image)
};
struct CoherentGroup {
  int first, count;
  double weight;
};
// image (+)= sum_g weight_g |sum of the group's Fields|^2
hipError_t launch_coherent(const CoherentGroup* groups_dev, int ngroups, const CoherentAdd* adds_dev, void* image,
                           int dtype, long long ldi, int rows, int cols, int accumulate, hipStream_t s);
hipError_t launch_insert(const void* field, long long ldf, int fr0, int fc0, int h, int w,
                         void* out, int out_dtype, long long ldo, int or0, int oc0,
                         int intensity, double weight, hipStream_t s);
// A Field of a coherent group: h x w samples at F (row stride ld) whose first
// lies at output pixel (r0, c0).
struct FieldItem {
  const void* F;
  long long ld;
  int h, w, r0, c0;
};
constexpr int kGroupFields = 64;  // per launch (2 KiB of kernel arguments)
hipError_t launch_insert_group(const FieldItem* items, int count, int r0, int c0, int h, int w, void* out,
                               int out_dtype, long long ldo, double weight, hipStream_t s);
hipError_t launch_multiply(const void* a, long long lda, const void* b, long long ldb, void* out,
                           long long ldo, int h, int w, hipStream_t s);
hipError_t launch_zero(void* p, size_t bytes, hipStream_t s);
// rows x cols elements of esz (4 or 8) bytes at row stride ld elements
hipError_t launch_zero_rows(void* p, int esz, long long rows, long long cols, long long ld, hipStream_t s);
hipError_t launch_weight_field(const void* F, long long ldF, const void* w, int w_dtype, long long ldw,
                               double scale, void* out, long long ldo, int h, int wd, hipStream_t s);
// nwave wavelengths (inv_wls on the device, or inv_wl0 alone when null), D_w at D + w * strideD
struct PhaseGrad {
  const void *amp, *opd;
  int amp_dtype, opd_dtype;        // 1 = f32, 3 = f64, also of the gradients
  long long ld_amp, ld_opd, strideO;
  int nopd, m, n, nwave;
  const double* inv_wls;           // device, or null: inv_wl0 and one wavelength
  double inv_wl0;
  const void* D;
  long long ldD, strideD;
  void *g_opd, *g_amp;             // g_amp may be null
  int go_dtype, ga_dtype;
  long long ld_go, ld_ga;
  int accumulate;
};
hipError_t launch_phase_grad(const PhaseGrad& q, hipStream_t s);

// detector-grid post-processing (mftx_detector.hip)
hipError_t launch_rebin(const void* src, int dtype, long long nimg, long long rows, long long cols, long long ld,
                        int factor, void* dst, int odt, hipStream_t s);
// Reductions leave at most kMaxPart partial sums, the same number for arrays of
// one size; their users add them up.
constexpr int kMaxPart = 1024;
// part = partial sums of a real array
hipError_t launch_sum(const void* x, int dtype, long long rows, long long cols, long long ld, double* part,
                      hipStream_t s);
// out[r][c] = |F[(r + r0) % rows][(c + c0) % cols]| (F complex64), part = partial sums of out
hipError_t launch_magnitude(const void* F, long long ldF, long long rows, long long cols, long long r0, long long c0,
                            void* out, int odt, long long ldo, double* part, hipStream_t s);
// x *= sum(num) / sum(den), partial sums of arrays of its size
hipError_t launch_scale_ratio(void* x, int dtype, long long rows, long long cols, long long ld, const double* num,
                              const double* den, hipStream_t s);
// The B-spline prefilter of a spline order as its two-sided impulse response
// h[|k|], |k| <= n (n = 0 for orders 0 and 1).
constexpr int kPrefilterTaps = 48;
struct PrefilterTaps {
  int n;
  double h[kPrefilterTaps + 1];
};
PrefilterTaps prefilter_taps(int order);
// rescale (util.py:262-349): map_coordinates(order 0..5, mode MFTX_MODE_*)
// of a real or complex (dtype 0 / 2) image, mask, unitary ratio; P and T hold
// the padded image (rows + 24) x (cols + 24) doubles each, raw / raw_im / mval
// the output size, part 4 kMaxPart doubles.
hipError_t launch_rescale(const void* img, int dtype, long long rows, long long cols, long long ld, const void* msrc,
                          int mask_mode, int mdt, long long ldm, double eps, double scale, long long orows,
                          long long ocols, int order, int mode, int unitary, void* out, int odt, long long ldo,
                          double* P, double* T, double* raw, double* raw_im, double* mval, double* part,
                          hipStream_t s);

// modal OPD operations (mftx_modal.hip)
// out[seg][9] = normal equations of the piston/tip/tilt fit; part: nseg * ceil(rows*cols/256) * 9 doubles
hipError_t launch_ptt_normal(const void* opd, int odt, long long ld_opd, const void* masks, int mdt, long long ld_mask,
                             long long mask_stride, int nseg, long long rows, long long cols, double dx_r, double dx_c,
                             double* part, double* out, hipStream_t s);
hipError_t launch_remove_tilt(const void* opd, int odt, long long ld_opd, const void* masks, int mdt,
                              long long ld_mask, long long mask_stride, int nseg, int multi, long long rows,
                              long long cols, double dx_r, double dx_c, const double* tilt, double* out,
                              long long ldo, hipStream_t s);
hipError_t launch_zernike(const double* rho, const double* theta, const void* mask, int mdt, long long npix,
                          int nmodes, const int* desc, const double* coef, const int* pw, const double* norm,
                          double* out, hipStream_t s);

// host side of the C ABI (mftx_api.cpp)
// mftx_dft2 on the caller's workspace ws of ws_bytes (for transforms of up to
// cap bytes, see the definition), or on the context's own growable workspace when
// ws is null
int dft2_on_workspace(mftx_ctx* ctx, const void* f, int f_dtype, int64_t m, int64_t n, int64_t ldf, void* F,
                      int64_t M, int64_t N, int64_t ldF, double alpha_r, double alpha_c, double shift_r,
                      double shift_c, double offset_r, double offset_c, double scale, int conj, int precision,
                      void* ws, size_t ws_bytes, size_t cap);
// record msg as the context's last error and return code
int set_error(mftx_ctx* ctx, int code, const char* msg);
// the device a context was created on
int context_device(const mftx_ctx* ctx);
// device address of the no-allocation entry point's scratch array on `device`
// (current), looked up once per device (mftx_noalloc.hip)
hipError_t scratch_address(int device, void** out);

}  // namespace mftx
