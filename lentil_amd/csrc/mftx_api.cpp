// C-ABI of the mftx library (declared in include/mftx.h).
//
// An MFT F = c * E1 . f . E2 (lentil fourier.py:97) runs as two launches of
// the complex GEMM C = A . B (A an operand of paired samples, B twiddle tables):
//   order B (row-first):    G   = f . E2        -> stored as G^T
//                           F^T = G^T . E1^T    -> F or |F|^2
//   order A (column-first): T^T = f^T . E1^T    -> stored as T
//                           F   = T . E2        -> F or |F|^2
// Order B costs m*n*N + M*m*N complex MACs, order A M*m*n + M*n*N; the
// cheaper one is used.  Several Fields summed coherently share one output
// grid, so their stage-2 GEMMs concatenate along K (one GEMM per coherent
// group, each K segment with its own midpoint), or run as windows of one grid
// that are summed on chip (sum_windows).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <new>
#include <stdexcept>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/mftx.h"
#include "mftx_internal.h"

using namespace mftx;

namespace {

constexpr int kRingSlots = 16;
// Twiddle table bytes per stage of one mftx_dft2: a larger table is used in
// pieces.  Pieces of kTableCap where those give every CU two tiles; of up to
// kTableMost where they do not (long, thin transforms: with pieces of 64 MiB
// 1 x 40000 -> 1 x 40000 took 25 launches of 25 workgroups, 9.3 ms, now 3.1,
// and 1 x 500000 -> 1 x 3001 47 launches of one, 82 ms, now 10.7).
constexpr size_t kTableCap = 64u << 20, kTableMost = 1u << 30;
constexpr size_t kSlotBytes = 512 * 1024;
constexpr size_t kListTables = 1u << 30;  // twiddle table bytes of one launch of a list

int64_t round_up(int64_t v, int64_t m) { return (v + m - 1) / m * m; }
double centre(int64_t k) { return (double)(k / 2); }  // floor(k/2), k >= 0 (fourier.py:117-120)

// MACs of the two contraction orders for an m x n -> M x N transform
double cost_row_first(double m, double n, double M, double N) { return m * n * N + M * m * N; }
double cost_col_first(double m, double n, double M, double N) { return M * m * n + M * n * N; }

Work empty_work() { return Work{}; }

// XCD-aware order: the works, listed so that neighbours share operand rows and
// twiddle tables, are cut into 8 equal runs, one per XCD; workgroup i of a
// launch runs on XCD i % 8, so each XCD walks its own run and its L2 serves
// what neighbours share.
std::vector<Work> xcd_order(const std::vector<Work>& works) {
  const size_t n = works.size();
  std::vector<Work> out;
  size_t most = 0;
  for (size_t x = 0; x < 8; ++x) most = std::max(most, (x + 1) * n / 8 - x * n / 8);
  out.reserve(most * 8);
  for (size_t i = 0; i < most; ++i)
    for (size_t x = 0; x < 8; ++x) {
      const size_t b = x * n / 8, e = (x + 1) * n / 8;
      out.push_back(b + i < e ? works[b + i] : empty_work());
    }
  while (!out.empty() && out.back().pend == 0) out.pop_back();
  return out;
}

// Works covering rblocks x sblocks 32 x 32 blocks of C for problems [pb, pe)
// (nch K blocks in all): panels of 8 tile columns, so that 32 neighbouring
// works are 4 tile rows by 8 tile columns and read few distinct blocks.
void add_tiles(std::vector<Work>& works, int tile, int pb, int pe, int nch, int rblocks, int sblocks,
               float* partial = nullptr, long long ldp = 0, int prows = 0, int pcols = 0) {
  const int tr = (rblocks + tile_rows(tile) - 1) / tile_rows(tile);
  const int tc = (sblocks + tile_slots(tile) - 1) / tile_slots(tile);
  for (int c0 = 0; c0 < tc; c0 += 8)
    for (int r = 0; r < tr; ++r)
      for (int c = c0; c < std::min(tc, c0 + 8); ++c)
        works.push_back(Work{pb, pe, r, c, partial, ldp, prows, pcols, nch, 0});
}

int64_t blocks32(int64_t n) { return (n + 31) / 32; }

constexpr int kCUs = 256;

// Estimated time (us) of a launch whose work items each run `run` problems of
// nkb K blocks on one tile of rblocks x sblocks blocks, `sets` such runs.
// Fitted to kernel traces of single transforms (64^2 to 2048^2 -> 4096^2, every
// tile forced) and of the broadband and segmented sweeps (every tile and run
// length forced), within 20% of them; per K block a workgroup takes
//   BIG    1.38 us, one per CU on a full chip (1.0 on up to half of the CUs),
//   MID    0.95 us with two on the CU, 0.48 alone,
//   SMALL  0.33 us with two on the CU, 0.27 alone (a wave runs a quarter),
// and each problem adds its epilogue, each round of work items its start.
double tile_cost(int tile, int64_t rblocks, int64_t sblocks, int64_t nkb, int64_t run, int64_t sets) {
  struct Rate { double start, full, light, epilogue; };
  const Rate r = tile == TILE_BIG ? Rate{6.0, 1.38, 1.0, 2.0}
               : tile == TILE_SMALL ? Rate{1.0, 0.33, 0.27, 1.0} : Rate{1.5, 0.95, 0.48, 1.5};
  const int64_t w = ((rblocks + tile_rows(tile) - 1) / tile_rows(tile)) *
                    ((sblocks + tile_slots(tile) - 1) / tile_slots(tile)) * sets;
  const int64_t per = tile == TILE_BIG ? kCUs : 2 * kCUs;
  const int64_t rounds = w / per, rest = w % per;
  const double full = r.start + run * (r.full * nkb + r.epilogue);
  const double light = r.start + run * (r.light * nkb + r.epilogue);
  return rounds * full + (rest == 0 ? 0.0 : 2 * rest > per ? full : light);
}

// Tile and run length (problems per work item, at most `most`) of a launch of
// `count` problems of one shape that estimates fastest; a fixed tile is kept.
// Ties go to the longer run (fewer partial images, a longer pipeline).
struct Schedule {
  int tile, run;
};
Schedule pick_schedule(int fixed, bool multi, int64_t rblocks, int64_t sblocks, int64_t nkb, int64_t count,
                       int64_t most) {
  Schedule best{TILE_MID, 1};
  double cost = -1;
  const int cand[3] = {TILE_BIG, multi ? TILE_MULTI : TILE_MID, TILE_SMALL};
  for (int t : cand) {
    if (multi && t == TILE_BIG) continue;
    if (fixed >= 0 && t != fixed) continue;
    for (int64_t g = std::min(most, count); g >= 1; --g) {
      const double c = tile_cost(t, rblocks, sblocks, nkb, g, (count + g - 1) / g);
      if (cost < 0 || c < 0.999 * cost) {
        cost = c;
        best = Schedule{t, (int)g};
      }
    }
  }
  return best;
}

// Powers of two of the f16 form: the operand is scaled to at most 2^14 per
// paired element (ScaleSrc), the tables by tw_scale, so stage 1's sums over K
// pairs stay below K 2^14 tw_scale; stage 1 stores them times
// 1 / (tw_scale 2^ceil(log2 K)), again at most 2^14, and stage 2 undoes all of it.
double stage1_scale(int prec, int64_t k_pairs) {
  if (prec != PREC_FP32) return 1.0;
  int b = 0;
  while ((1LL << b) < k_pairs) ++b;
  return std::ldexp(1.0 / tw_scale(prec), -b);
}
double stage2_scale(int prec, int64_t k_pairs) {
  return prec != PREC_FP32 ? 1.0 : 1.0 / (tw_scale(prec) * tw_scale(prec)) / stage1_scale(prec, k_pairs);
}

// Beyond kLongPairs that worst case, every pair as bright as the brightest,
// leaves too little of f16's range: stage 1's output for a few bright samples
// would be below 2^-2, where the pair's lo part runs out (one sample among
// 500000: results 3.1e-6 off).  Such a transform takes the sum of its samples'
// magnitudes too, and scales the operand so that stage 1 stays below 2^14 with
// the factor of kLongPairs (OneMft::sums): 7e-8, as for short ones.
constexpr int64_t kLongPairs = 1 << 14;
bool is_long(int prec, int64_t k_pairs) { return prec == PREC_FP32 && k_pairs > kLongPairs; }

// Output grid of one MFT stage with N columns, signed twiddle scale alpha and
// output shift: the slots and pairing centre the GEMM runs on (see Problem)
// and the fold of its A operand.  Outputs are paired about the PSF core
// j = N/2 + shift, snapped to the half-pixel grid, so the two outputs of a
// slot have comparable magnitude and neither inherits the rounding of a much
// brighter partner; when the core sits within a pixel of the grid centre the
// centre itself is used (fewest slots), and when pairing would save less than
// a quarter of the work (core far from the centre or outside the grid) every
// slot computes one column directly (c = 0).
struct OutGrid {
  int slots, cp, cm;
  double y0, fold;
};

// (`about`: the shift of the core to pair about, where grids of several
// shifts have to share their slots.)
OutGrid make_grid(double alpha, double shift, int N, double about) {
  const int h = N / 2;
  const double core = h + about;
  const double mid = 0.5 * (N - 1);
  double c;
  if (std::fabs(core - mid) <= 1.0) {
    c = mid;
  } else {
    c = std::nearbyint(2.0 * core) / 2.0;
    if (!(c >= 0.0 && c <= N - 1) || std::max(N - std::ceil(c), std::floor(c) + 1) > 0.75 * N) c = 0.0;
  }
  OutGrid g;
  g.cm = (int)std::floor(c);
  g.cp = (int)std::ceil(c);
  g.y0 = c - g.cm;
  g.slots = std::max(N - g.cp, g.cm + 1);
  g.fold = -alpha * (shift + h - c);
  return g;
}

OutGrid make_grid(double alpha, double shift, int N) { return make_grid(alpha, shift, N, shift); }

// Twiddle tables of a launch, shared by every problem with the same rate, slot
// origin and sample parity (x' = k' + 1/2 for an even number of samples, k'
// for an odd one).
class Tables {
 public:
  // index of the table for `samples` input samples and `slots` output slots
  int get(double alpha, double y0, int64_t samples, int64_t slots) {
    if (2 * ops.size() >= index_.size()) grow();
    int& at = index_[find(alpha, y0, samples & 1 ? 0.0 : 0.5)];
    if (at < 0) {
      at = (int)ops.size();
      TableOp op = {};
      op.alpha = alpha;
      op.x0 = samples & 1 ? 0.0 : 0.5;
      op.y0 = y0;
      ops.push_back(op);
    }
    TableOp& op = ops[at];
    op.nsb = std::max(op.nsb, (int)blocks32(slots));
    op.nkb = std::max(op.nkb, pair_blocks(samples));
    return at;
  }
  // thread ranges of the launch and offsets of the tables from `base`; the total bytes
  size_t place(size_t base) {
    off.clear();
    threads = 0;
    size_t at = base;
    for (auto& op : ops) {
      off.push_back(at);
      at += table_bytes(op.nsb, op.nkb);
      op.begin = group_begin(threads);
      threads = op.begin + table_threads(op.nsb, op.nkb);
    }
    return at - base;
  }
  std::vector<TableOp> ops;
  std::vector<size_t> off;
  long long threads = 0;

 private:
  // Open hashing over indices of ops (-1: free).  Rates are compared by their
  // bits: a NaN rate is unequal to itself, and in an ordered container equal to
  // every other one.
  static uint64_t bits(double v) {
    uint64_t u;
    std::memcpy(&u, &v, sizeof u);
    return u;
  }
  size_t find(double alpha, double y0, double x0) const {
    uint64_t h = (bits(alpha) ^ bits(y0) * 3 ^ bits(x0) * 5) * 0x9E3779B97F4A7C15ull;
    for (h ^= h >> 32;; ++h) {
      const size_t i = h & (index_.size() - 1);
      if (index_[i] < 0) return i;
      const TableOp& op = ops[index_[i]];
      if (bits(op.alpha) == bits(alpha) && bits(op.y0) == bits(y0) && bits(op.x0) == bits(x0)) return i;
    }
  }
  void grow() {
    index_.assign(std::max<size_t>(16, 4 * index_.size()), -1);
    for (size_t k = 0; k < ops.size(); ++k) index_[find(ops[k].alpha, ops[k].y0, ops[k].x0)] = (int)k;
  }
  std::vector<int> index_;  // a power of two, at most half of it used
};

}  // namespace

struct mftx_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  void* ws = nullptr;
  size_t ws_bytes = 0;
  void* aux = nullptr;  // intermediates of the detector operators (ws holds their MFT operands)
  size_t aux_bytes = 0;
  // descriptor ring: pinned host staging + device slots, reused round-robin
  char* ring_host = nullptr;
  char* ring_dev = nullptr;
  hipEvent_t ring_ev[kRingSlots] = {};
  bool ring_used[kRingSlots] = {};
  int ring_next = 0;
};

struct mftx_plan {
  mftx_ctx* ctx = nullptr;
  int prec = 0;
  int tile1 = 0, tile2 = 0, tile2c = 0, tile_f = 0;  // GEMM tiles of the launches below
  int64_t img_rows = 0, img_cols = 0;
  void* ws = nullptr;  // workspace: operands, intermediates, partial images, descriptors
  Work* works1 = nullptr;
  Work* works2 = nullptr;
  Problem* probs1 = nullptr;
  Problem* probs2 = nullptr;
  Seg* segs = nullptr;          // K segments of every problem list
  PhasorWave* waves = nullptr;  // per phasor wavelength slot: 1/λ and both stages' folds
  MaxOp* max_ops = nullptr;     // f16 form: the tiles' amplitude maxima
  int n_max_ops = 0;
  long long max_blocks = 0;
  int nwork1 = 0, nwork2 = 0;
  // stage 2 of the classes whose coherent group has several output grids:
  // their complex fields, summed by the coherent launch (every other class
  // runs the intensity launch above)
  Work* works2w = nullptr;  // groups whose Fields are windows of one grid
  Problem* probs2w = nullptr;
  int nwork2w = 0;
  Work* works2c = nullptr;
  Problem* probs2c = nullptr;
  int nwork2c = 0;
  PhasorOp* phasor_ops = nullptr;  // device descriptors of the grouped phasor launch
  int n_phasor_ops = 0;
  OperandSplit split{2, 1};
  long long phasor_threads = 0;
  std::vector<ReduceOp> reduces;   // regions of the image written from partial images
  ReduceOp* reduce_ops = nullptr;  // ... on the device
  double unit = 1.0;               // what one unit of the partial images is worth
  // coherent groups whose Fields have several output grids: complex outputs,
  // summed and squared into the image by one launch (field.py:331-346)
  CoherentGroup* cgroups = nullptr;
  CoherentAdd* cadds = nullptr;
  int n_cgroups = 0;
  mftx_plan_info info = {};
  int use_graph = 0;  // mftx_plan_profile times prefix graphs
  // complex fields of every class from the stage-1 operands already in the
  // workspace (mftx_plan_set_fields / mftx_plan_execute_fields)
  Work* works_f = nullptr;
  Problem* probs_f = nullptr;
  int nwork_f = 0;
  std::vector<Problem> pf;       // host copy, pointers filled by set_fields
  RowPhase* row_phases = nullptr;  // device: per class, the phase stage 1 left out
  int max_rows = 0;                // the longest of them
  std::vector<double> field_scale;  // what undoes the f16 form's scaling, per class
  std::vector<int> class_first;  // first member (problem index) of each class
  int fields_ready = 0;
};

static int fail(mftx_ctx* ctx, int code, const std::string& msg) {
  if (ctx) ctx->err = msg;
  return code;
}

int mftx::set_error(mftx_ctx* ctx, int code, const char* msg) { return fail(ctx, code, msg); }
int mftx::context_device(const mftx_ctx* ctx) { return ctx->device; }

static int hipfail(mftx_ctx* ctx, hipError_t e, const char* what) {
  return fail(ctx, MFTX_EDEVICE, std::string(what) + ": " + hipGetErrorString(e));
}

// Host-side exceptions (allocation failures of the plan builders' containers)
// end at the C boundary as status codes.
template <class F> static int guarded(mftx_ctx* ctx, F&& body) {
  try {
    return body();
  } catch (const std::bad_alloc&) {
    return fail(ctx, MFTX_ENOMEM, "host allocation failed");
  } catch (const std::exception& e) {
    return fail(ctx, MFTX_EDEVICE, e.what());
  } catch (...) {
    return fail(ctx, MFTX_EDEVICE, "unexpected host exception");
  }
}

// Device allocation whose failure is an ordinary status: the runtime's
// pending error is cleared, so the next launch check (hipGetLastError after a
// kernel launch) does not report this allocation's failure as its own.
static bool try_malloc(void** p, size_t bytes) {
  if (hipMalloc(p, bytes) == hipSuccess) return true;
  *p = nullptr;
  (void)hipGetLastError();
  return false;
}

#define HIPCHK(ctx, expr)                                   \
  do {                                                      \
    hipError_t e_ = (expr);                                 \
    if (e_ != hipSuccess) return hipfail((ctx), e_, #expr); \
  } while (0)

// Grow the context workspace to at least `bytes`, by at least half its old
// size, so a run of slowly growing calls reallocates (and synchronises) only
// a few times.
static int ensure_ws(mftx_ctx* ctx, size_t bytes) {
  if (bytes <= ctx->ws_bytes) return MFTX_OK;
  const size_t old = ctx->ws_bytes;
  if (ctx->ws) {
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    HIPCHK(ctx, hipFree(ctx->ws));
    ctx->ws = nullptr;
    ctx->ws_bytes = 0;
  }
  const size_t nb = std::max(bytes, old + old / 2);
  if (!try_malloc(&ctx->ws, nb)) {
    ctx->ws = nullptr;
    return fail(ctx, MFTX_ENOMEM, "workspace allocation of " + std::to_string(nb) + " bytes failed");
  }
  ctx->ws_bytes = nb;
  return MFTX_OK;
}

// Take the next ring slot (waiting until its previous upload has been
// consumed); *host is its pinned staging area, *dev its device address.
static int reserve_desc(mftx_ctx* ctx, int* slot, char** host, char** dev) {
  const int s = ctx->ring_next;
  ctx->ring_next = (s + 1) % kRingSlots;
  if (ctx->ring_used[s]) HIPCHK(ctx, hipEventSynchronize(ctx->ring_ev[s]));
  ctx->ring_used[s] = false;
  *slot = s;
  *host = ctx->ring_host + (size_t)s * kSlotBytes;
  *dev = ctx->ring_dev + (size_t)s * kSlotBytes;
  return MFTX_OK;
}

// Queue the upload of the first `bytes` of a reserved slot on the context stream.
static int commit_desc(mftx_ctx* ctx, int s, size_t bytes) {
  char* h = ctx->ring_host + (size_t)s * kSlotBytes;
  char* d = ctx->ring_dev + (size_t)s * kSlotBytes;
  HIPCHK(ctx, hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(ctx, hipEventRecord(ctx->ring_ev[s], ctx->stream));
  ctx->ring_used[s] = true;
  return MFTX_OK;
}

static int ensure_aux(mftx_ctx* ctx, size_t bytes) {
  if (bytes <= ctx->aux_bytes) return MFTX_OK;
  if (ctx->aux) {
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    HIPCHK(ctx, hipFree(ctx->aux));
    ctx->aux = nullptr;
    ctx->aux_bytes = 0;
  }
  if (!try_malloc(&ctx->aux, bytes)) {
    ctx->aux = nullptr;
    return fail(ctx, MFTX_ENOMEM, "workspace allocation of " + std::to_string(bytes) + " bytes failed");
  }
  ctx->aux_bytes = bytes;
  return MFTX_OK;
}

// Stage `bytes` of descriptors into a ring slot and queue the upload on the
// context stream; returns the device address of the slot.
static int upload_desc(mftx_ctx* ctx, const void* src, size_t bytes, void** dev) {
  if (bytes > kSlotBytes) return fail(ctx, MFTX_EINVAL, "descriptor block too large (output too big for one call)");
  int s;
  char *h, *d;
  int rc = reserve_desc(ctx, &s, &h, &d);
  if (rc) return rc;
  std::memcpy(h, src, bytes);
  rc = commit_desc(ctx, s, bytes);
  if (rc) return rc;
  *dev = d;
  return MFTX_OK;
}

// Problem ranges [b, e) for work items: runs of g consecutive problems with
// one tiling and K length share a work item, so the GEMM's load pipeline runs
// across their K loops.  Grouping is used only when every run has the same
// length g: a launch that mixed long and short work items would finish on its
// long tail.
static std::vector<std::pair<int, int>> group_runs(const std::vector<Problem>& ps, const std::vector<int>& nkb, int g) {
  const int n = (int)ps.size();
  std::vector<std::pair<int, int>> runs;
  bool uniform = true;
  for (int i = 0; i < n;) {
    int e = i + 1;
    while (e < n && e - i < g && ps[e].rblocks == ps[i].rblocks && ps[e].cols == ps[i].cols && nkb[e] == nkb[i]) ++e;
    uniform = uniform && e - i == g;
    runs.emplace_back(i, e);
    i = e;
  }
  if (!uniform) {
    runs.clear();
    for (int i = 0; i < n; ++i) runs.emplace_back(i, i + 1);
  }
  return runs;
}

// Schedule and works of a list of independent problems (of one segment each
// unless multi, nkb[i] K blocks): the tile is chosen for the whole launch by
// the summed estimate of its shapes; runs of equal problems share work items.
static int list_works(std::vector<Work>& works, const std::vector<Problem>& ps, const std::vector<int>& nkb, int fixed,
                      int64_t most, bool multi = false) {
  struct Shape { int rb, sb, nkb; };
  std::map<std::tuple<int, int, int>, int64_t> shapes;
  for (size_t i = 0; i < ps.size(); ++i) ++shapes[{ps[i].rblocks, (int)blocks32(ps[i].cols), nkb[i]}];
  // the shape with most work decides
  std::tuple<int, int, int> top{};
  double big = -1;
  int64_t total = 0;
  for (auto& kv : shapes) {
    const double w = (double)std::get<0>(kv.first) * std::get<1>(kv.first) * std::get<2>(kv.first) * kv.second;
    if (w > big) {
      big = w;
      top = kv.first;
    }
    total += kv.second;
  }
  const Schedule sch = pick_schedule(fixed, multi, std::get<0>(top), std::get<1>(top), std::get<2>(top), total, most);
  for (const auto& r : group_runs(ps, nkb, sch.run)) {
    int nch = 0;
    for (int i = r.first; i < r.second; ++i) nch += nkb[i];
    add_tiles(works, sch.tile, r.first, r.second, nch, ps[r.first].rblocks, (int)blocks32(ps[r.first].cols));
  }
  return sch.tile;
}

// Geometry of one entry of mftx_dft2_many (the quantities mftx_dft2 derives).
namespace {
struct MftGeo {
  bool col_first;
  int64_t r1, k1, c1, c2;  // stage-1 operand rows and K, stage-1 and stage-2 output columns
  double alpha1, alpha2, x01, x02;
  OutGrid g1, g2;
  double xc1() const { return x01 + 0.5 * (double)(k1 - 1); }  // midpoints of the two input axes
  double xc2() const { return x02 + 0.5 * (double)(r1 - 1); }
  size_t off1 = 0, off2 = 0;  // workspace offsets of the stage-1 and stage-2 operands
  size_t off_max = 0;         // ... of the source's maxima, then its inverse scale (f16 form)
};

MftGeo mft_geometry(int64_t m, int64_t n, int64_t M, int64_t N, double alpha_r, double alpha_c, double shift_r,
                    double shift_c, double offset_r, double offset_c, int conj) {
  MftGeo g;
  g.col_first = cost_col_first(m, n, M, N) < cost_row_first(m, n, M, N);
  g.r1 = g.col_first ? n : m;
  g.k1 = g.col_first ? m : n;
  g.c1 = g.col_first ? M : N;
  g.c2 = g.col_first ? N : M;
  const double sgn = conj ? 1.0 : -1.0;
  g.alpha1 = sgn * (g.col_first ? alpha_r : alpha_c);
  g.alpha2 = sgn * (g.col_first ? alpha_c : alpha_r);
  g.g1 = make_grid(g.alpha1, g.col_first ? shift_r : shift_c, (int)g.c1);
  g.g2 = make_grid(g.alpha2, g.col_first ? shift_c : shift_r, (int)g.c2);
  // twiddle coordinates: rows x = R + or against U - sr; columns x = S + oc
  // against V - sc; each stage's output shift is folded into its A operand
  const double xr0 = -centre(m) + offset_r, xc0 = -centre(n) + offset_c;
  g.x01 = g.col_first ? xr0 : xc0;
  g.x02 = g.col_first ? xc0 : xr0;
  return g;
}

// The two GEMM problems of one transform (addresses filled by the caller);
// k_pairs: how many pairs of the operand's largest value stage 1's sums reach.
void mft_problems(const MftGeo& g, int prec, double scale, int64_t k_pairs, Problem& a, Problem& b) {
  a = Problem{};
  a.rblocks = pair_blocks(g.r1);
  a.sblocks = (int)blocks32(g.g1.slots);
  a.cols = g.g1.slots;
  a.ncols = (int)g.c1;
  a.cp = g.g1.cp;
  a.cm = g.g1.cm;
  a.y0 = g.g1.y0;
  a.xrot = g.alpha1 * g.xc1();
  a.scale = (float)stage1_scale(prec, k_pairs);
  a.ldd = pair_blocks(g.r1);
  b = Problem{};
  b.rblocks = (int)blocks32(g.c1);
  b.sblocks = (int)blocks32(g.g2.slots);
  b.i1 = (int)g.c1;
  b.j1 = (int)g.c2;
  b.cols = g.g2.slots;
  b.ncols = (int)g.c2;
  b.cp = g.g2.cp;
  b.cm = g.g2.cm;
  b.y0 = g.g2.y0;
  b.xrot = g.alpha2 * g.xc2();
  b.scale = (float)(scale * stage2_scale(prec, k_pairs));
  b.trans = g.col_first ? 0 : 1;  // C is F (column-first) or F^T (row-first)
  b.wrows = (int)(g.col_first ? g.c1 : g.c2);
  b.wcols = (int)(g.col_first ? g.c2 : g.c1);
}

// A transform whose output takes more tiles of 128 rows by 64 or 128 columns
// than a descriptor block of kSlotBytes once held (40 bytes each behind 112
// bytes and 8 per 16 K values; a list entry's two stages together, with 104
// bytes of source) is refused, as it always was.
bool too_large(const MftGeo& g, bool list_entry) {
  auto up = [](int64_t v, int64_t q) { return (v + q - 1) / q * q; };
  const int64_t t1 = up(g.r1, 128) / 128, t2 = up(g.c1, 128) / 128;
  const int64_t wide = std::max(t1 * ((g.g1.slots + 63) / 64), t2 * ((g.g2.slots + 63) / 64));
  const int64_t bs = wide >= 256 ? 64 : 32, kg = wide >= 256 ? 32 : 16;
  auto bytes = [&](int64_t tr, int64_t slots, int64_t k) {
    const int64_t tc = (slots + bs - 1) / bs, mx = (tr + 7) / 8 * tc;
    const int64_t works = (mx - 1) * 8 + (tr % 8 ? tr % 8 : 8);
    return up(112 + up(k, kg) / 16 * 8, 16) + 40 * works;
  };
  const int64_t b1 = bytes(t1, g.g1.slots, g.k1), b2 = bytes(t2, g.g2.slots, g.r1);
  return list_entry ? 112 + b1 + b2 > (int64_t)kSlotBytes : std::max(b1, b2) > (int64_t)kSlotBytes;
}
}  // namespace

// The launches of a list of MFTs: all entries in one operand launch per input
// kind and one GEMM launch per stage.  many_build derives the geometry and the
// descriptors (workspace and descriptor addresses as offsets); many_place
// rebases them onto a workspace and a device descriptor block and writes the
// host copy of that block; many_tables and many_launch issue the launches.
struct ManyBatch {
  int tile1 = 0, tile2 = 0;
  size_t ws = 0, bytes = 0;  // workspace and descriptor block sizes
  size_t table_bytes = 0;    // the workspace's part for twiddle tables
  size_t o_wv = 0, o_ph = 0, o_pk = 0, o_mx = 0, o_tb = 0, o_p1 = 0, o_p2 = 0, o_s1 = 0, o_s2 = 0, o_w1 = 0, o_w2 = 0;
  std::vector<MftGeo> geo;
  std::vector<PhasorWave> waves;
  std::vector<PhasorOp> phops, packs;  // phasor and complex sources
  std::vector<MaxOp> maxes;
  std::vector<int> op_of;  // phasor op of entry i, or -(pack index + 1)
  Tables tables;
  std::vector<int> tab1, tab2;
  std::vector<Problem> p1, p2;
  std::vector<Seg> s1, s2;
  std::vector<Work> w1, w2;
  OperandSplit ph_split{2, 1}, pk_split{2, 1};
  long long ph_total = 0, pk_total = 0, mx_total = 0;
};

// `fixed`: the GEMM tile, or -1 to choose it.
static void many_build(const mftx_mft* mfts, int32_t count, int prec, int fixed, ManyBatch& mb) {
  std::vector<MftGeo>& geo = mb.geo;
  geo.clear();
  for (auto* v : {&mb.op_of, &mb.tab1, &mb.tab2}) v->reserve(count);
  geo.reserve(count);
  mb.waves.reserve(count);
  mb.s1.reserve(count);
  mb.s2.reserve(count);
  const int nsource = (int)std::count_if(mfts, mfts + count, [](const mftx_mft& q) { return q.f != nullptr; });
  mb.packs.reserve(nsource);
  mb.phops.reserve(count - nsource);
  if (prec == PREC_FP32) mb.maxes.reserve(count);
  size_t ws = 0;
  for (int32_t i = 0; i < count; ++i) {
    const mftx_mft& q = mfts[i];
    geo.push_back(mft_geometry(q.m, q.n, q.M, q.N, q.alpha_r, q.alpha_c, q.shift_r, q.shift_c, q.offset_r, q.offset_c,
                               q.conj));
    geo[i].off1 = ws;
    ws += folded_bytes(geo[i].r1, geo[i].k1);
  }
  for (auto& g : geo) {
    g.off2 = ws;
    ws += plain_bytes(g.c1, pair_blocks(g.r1));
  }
  for (auto& g : geo) {
    mb.tab1.push_back(mb.tables.get(g.alpha1, g.g1.y0, g.k1, g.g1.slots));
    mb.tab2.push_back(mb.tables.get(g.alpha2, g.g2.y0, g.r1, g.g2.slots));
  }
  mb.table_bytes = mb.tables.place(ws);
  ws += mb.table_bytes;

  // ---- sources -----------------------------------------------------------------
  long long ph_quads = 0, pk_quads = 0;
  for (int32_t i = 0; i < count; ++i) (mfts[i].f ? pk_quads : ph_quads) += operand_quads(geo[i].r1, geo[i].k1, 1);
  mb.ph_split = operand_split(ph_quads);
  mb.pk_split = operand_split(pk_quads);
  auto source = [&](std::vector<PhasorOp>& ops, long long& total, const MftGeo& g, const mftx_mft& q) -> PhasorOp& {
    PhasorOp op = {};
    op.m = (int)q.m;
    op.n = (int)q.n;
    op.trans = g.col_first ? 1 : 0;
    op.waves = (const PhasorWave*)(uintptr_t)mb.waves.size();  // index, rebased by many_place
    op.dst = (void*)(uintptr_t)g.off1;                          // offset, rebased by many_place
    op.wave_stride = (long long)folded_bytes(g.r1, g.k1);
    op.begin = group_begin(total);
    ops.push_back(op);
    return ops.back();
  };
  for (int32_t i = 0; i < count; ++i) {
    const mftx_mft& q = mfts[i];
    const MftGeo& g = geo[i];
    // consecutive phasor entries of one pupil and geometry share an op
    // (their operands are one fixed stride apart in the workspace)
    bool joined = false;
    if (!q.f && i > 0 && !mfts[i - 1].f) {
      const mftx_mft& p = mfts[i - 1];
      const MftGeo& h = geo[i - 1];
      joined = p.amp == q.amp && p.opd == q.opd && p.amp_dtype == q.amp_dtype && p.opd_dtype == q.opd_dtype &&
               p.ld_amp == q.ld_amp && p.ld_opd == q.ld_opd && p.m == q.m && p.n == q.n && h.col_first == g.col_first;
    }
    if (!joined) {
      PhasorOp& op = q.f ? source(mb.packs, mb.pk_total, g, q) : source(mb.phops, mb.ph_total, g, q);
      op.amp = q.f ? q.f : q.amp;
      op.amp_dtype = q.f ? q.f_dtype : q.amp_dtype;
      op.ld_amp = q.f ? q.ldf : q.ld_amp;
      op.opd = q.f ? nullptr : q.opd;
      op.opd_dtype = q.f ? 0 : q.opd_dtype;
      op.ld_opd = q.f ? 0 : q.ld_opd;
      if (prec == PREC_FP32) {
        MaxOp mx = {};
        mx.src = op.amp;
        mx.dtype = op.amp_dtype;
        mx.m = q.m;
        mx.n = q.n;
        mx.ld = op.ld_amp;
        mx.nblk = max_blocks(q.m, q.n);
        mx.part = (float*)(uintptr_t)ws;
        mx.begin = mb.mx_total;
        mb.mx_total += mx.nblk;
        op.sc = ScaleSrc{mx.part, (float*)(uintptr_t)(ws + sizeof(float) * mx.nblk), mx.nblk, 0};
        ws += round_up((int64_t)(sizeof(float) * (mx.nblk + 1)), 256);
        mb.maxes.push_back(mx);
      }
    }
    PhasorOp& op = q.f ? mb.packs.back() : mb.phops.back();
    op.nwave += 1;
    mb.waves.push_back(PhasorWave{q.f ? 0.0 : 4.0 * q.inv_wl, 4.0 * g.g1.fold, g.x01, 4.0 * g.g2.fold, g.x02});
    mb.op_of.push_back(q.f ? -(int)mb.packs.size() : (int)mb.phops.size() - 1);
    (q.f ? mb.pk_total : mb.ph_total) = op.begin + operand_threads(g.r1, g.k1, op.nwave, q.f ? mb.pk_split : mb.ph_split);
  }
  mb.ws = ws;

  // ---- problems and works ------------------------------------------------------
  std::vector<int> nkb1, nkb2;
  nkb1.reserve(count);
  nkb2.reserve(count);
  mb.p1.resize(count);
  mb.p2.resize(count);
  for (int32_t i = 0; i < count; ++i) {
    const mftx_mft& q = mfts[i];
    const MftGeo& g = geo[i];
    Problem& a = mb.p1[i];
    Problem& b = mb.p2[i];
    mft_problems(g, prec, q.scale, pairs(g.k1), a, b);
    a.sbeg = b.sbeg = i;
    a.send = b.send = i + 1;
    b.dst = q.F;
    b.ldd = q.ldF;
    b.wmap = q.w;
    b.ldw = q.ldw;
    b.wdtype = q.w_dtype;
    const int n1 = pair_blocks(g.k1), n2 = pair_blocks(g.r1);
    mb.s1.push_back(Seg{nullptr, nullptr, 0.0, n1, n1, mb.tables.ops[mb.tab1[i]].nkb, 0});
    mb.s2.push_back(Seg{nullptr, nullptr, 0.0, n2, n2, mb.tables.ops[mb.tab2[i]].nkb, 0});
    nkb1.push_back(n1);
    nkb2.push_back(n2);
  }
  std::vector<Work> w1, w2;
  mb.tile1 = list_works(w1, mb.p1, nkb1, fixed, 8);
  mb.tile2 = list_works(w2, mb.p2, nkb2, fixed, 8);
  mb.w1 = xcd_order(w1);
  mb.w2 = xcd_order(w2);

  // one descriptor block: waves, source ops, tables, problems, segments, works
  size_t off = 0;
  auto take = [&](size_t b) { const size_t o = off; off = round_up((int64_t)(off + b), 16); return o; };
  mb.o_wv = take(sizeof(PhasorWave) * mb.waves.size());
  mb.o_ph = take(sizeof(PhasorOp) * mb.phops.size());
  mb.o_pk = take(sizeof(PhasorOp) * mb.packs.size());
  mb.o_mx = take(sizeof(MaxOp) * mb.maxes.size());
  mb.o_tb = take(sizeof(TableOp) * mb.tables.ops.size());
  mb.o_p1 = take(sizeof(Problem) * mb.p1.size());
  mb.o_p2 = take(sizeof(Problem) * mb.p2.size());
  mb.o_s1 = take(sizeof(Seg) * mb.s1.size());
  mb.o_s2 = take(sizeof(Seg) * mb.s2.size());
  mb.o_w1 = take(sizeof(Work) * mb.w1.size());
  mb.o_w2 = take(sizeof(Work) * mb.w2.size());
  mb.bytes = off;
}

// Rebase the batch's descriptors onto workspace `base` and the device
// descriptor block `d`, and write the block's contents to host memory `h`.
static void many_place(ManyBatch& mb, char* base, char* d, char* h) {
  for (auto* ops : {&mb.phops, &mb.packs})
    for (auto& op : *ops) {
      op.waves = (const PhasorWave*)(d + mb.o_wv) + (uintptr_t)op.waves;
      op.dst = base + (uintptr_t)op.dst;
      if (op.sc.n) {
        op.sc.part = (const float*)(base + (uintptr_t)op.sc.part);
        op.sc.inv = (float*)(base + (uintptr_t)op.sc.inv);
      }
    }
  for (auto& mx : mb.maxes) mx.part = (float*)(base + (uintptr_t)mx.part);
  for (size_t t = 0; t < mb.tables.ops.size(); ++t) mb.tables.ops[t].dst = base + mb.tables.off[t];
  for (size_t i = 0; i < mb.geo.size(); ++i) {
    mb.s1[i].a = base + mb.geo[i].off1;
    mb.s1[i].b = base + mb.tables.off[mb.tab1[i]];
    mb.s2[i].a = base + mb.geo[i].off2;
    mb.s2[i].b = base + mb.tables.off[mb.tab2[i]];
    mb.p1[i].dst = base + mb.geo[i].off2;
    const PhasorOp& op = mb.op_of[i] < 0 ? mb.packs[-mb.op_of[i] - 1] : mb.phops[mb.op_of[i]];
    mb.p2[i].inv = op.sc.n ? op.sc.inv : nullptr;
  }
  auto put = [&](size_t o, const auto& v) {
    if (!v.empty()) std::memcpy(h + o, v.data(), sizeof(v[0]) * v.size());
  };
  put(mb.o_wv, mb.waves);
  put(mb.o_ph, mb.phops);
  put(mb.o_pk, mb.packs);
  put(mb.o_mx, mb.maxes);
  put(mb.o_tb, mb.tables.ops);
  put(mb.o_p1, mb.p1);
  put(mb.o_p2, mb.p2);
  put(mb.o_s1, mb.s1);
  put(mb.o_s2, mb.s2);
  put(mb.o_w1, mb.w1);
  put(mb.o_w2, mb.w2);
}

// The twiddle tables of a placed batch (descriptors at device address d).
static hipError_t many_tables(const ManyBatch& mb, int prec, const char* d, hipStream_t s) {
  return launch_tables(prec, (const TableOp*)(d + mb.o_tb), (int)mb.tables.ops.size(), mb.tables.threads, s);
}

// The launches of a placed batch, its tables already made.
static hipError_t many_launch(const ManyBatch& mb, int prec, const char* d, hipStream_t s) {
  hipError_t e = launch_absmax((const MaxOp*)(d + mb.o_mx), (int)mb.maxes.size(), mb.mx_total, s);
  if (e == hipSuccess)
    e = launch_operands(prec, false, mb.ph_split, (const PhasorOp*)(d + mb.o_ph), (int)mb.phops.size(), mb.ph_total, s);
  if (e == hipSuccess)
    e = launch_operands(prec, true, mb.pk_split, (const PhasorOp*)(d + mb.o_pk), (int)mb.packs.size(), mb.pk_total, s);
  if (e == hipSuccess)
    e = launch_gemm(prec, EPI_STORE_PACKED, mb.tile1, (const Work*)(d + mb.o_w1), (int)mb.w1.size(),
                    (const Problem*)(d + mb.o_p1), (const Seg*)(d + mb.o_s1), s);
  if (e == hipSuccess)
    e = launch_gemm(prec, EPI_STORE_CPLX, mb.tile2, (const Work*)(d + mb.o_w2), (int)mb.w2.size(),
                    (const Problem*)(d + mb.o_p2), (const Seg*)(d + mb.o_s2), s);
  return e;
}

// One entry of a list by itself (below, beside mftx_dft2's code).
static int run_entry(mftx_ctx* ctx, const mftx_mft& q, int prec);

// All entries [0, count) on the context stream with the context workspace and
// one descriptor ring slot; a batch whose descriptors exceed a slot is split,
// and so is one whose tables exceed kListTables: they hold 2 bytes per input
// sample and output pixel of an axis (1 x 100000 -> 1 x 100000: 20 GB, for
// arrays of 1.6 MB), where an entry alone makes its own in pieces.  So is one
// with an entry that needs a sum of its samples (is_long).
static int dft2_many_run(mftx_ctx* ctx, const mftx_mft* mfts, int32_t count, int prec) {
  std::unique_ptr<ManyBatch> mb(new ManyBatch());
  many_build(mfts, count, prec, -1, *mb);
  auto halves = [&]() {
    const int32_t h = count / 2;
    const int rc = dft2_many_run(ctx, mfts, h, prec);
    return rc ? rc : dft2_many_run(ctx, mfts + h, count - h, prec);
  };
  if (mb->bytes > kSlotBytes || (count == 1 && too_large(mb->geo[0], true))) {
    if (count > 1) return halves();
    // the widest tiles need the fewest descriptors
    mb.reset(new ManyBatch());
    many_build(mfts, count, prec, TILE_BIG, *mb);
    if (mb->bytes > kSlotBytes || too_large(mb->geo[0], true))
      return fail(ctx, MFTX_EINVAL, "descriptor block too large (output too big for one call)");
  }
  bool alone = mb->table_bytes > kListTables;
  for (const MftGeo& g : mb->geo) alone = alone || is_long(prec, pairs(g.k1));
  if (alone) return count > 1 ? halves() : run_entry(ctx, mfts[0], prec);
  int rc = ensure_ws(ctx, mb->ws);
  if (rc) return rc;
  // the slot is reserved first: the descriptors hold device addresses inside it
  int slot;
  char *h, *d;
  rc = reserve_desc(ctx, &slot, &h, &d);
  if (rc) return rc;
  many_place(*mb, (char*)ctx->ws, d, h);
  rc = commit_desc(ctx, slot, mb->bytes);
  if (rc) return rc;
  HIPCHK(ctx, many_tables(*mb, prec, d, ctx->stream));
  HIPCHK(ctx, many_launch(*mb, prec, d, ctx->stream));
  return MFTX_OK;
}

// A persistent list of MFTs (mftx_mft_plan_*): plan-owned workspace and
// descriptors, built once, the twiddle tables with them.
struct mftx_mft_plan {
  mftx_ctx* ctx = nullptr;
  int prec = 0;
  ManyBatch mb;
  void* mem = nullptr;   // operand workspace, then the descriptor block
  char* desc = nullptr;
  ~mftx_mft_plan() {
    if (mem) (void)hipFree(mem);
  }
};

// Argument checks shared by mftx_dft2_many and mftx_mft_plan_create.
static int check_mfts(mftx_ctx* ctx, const mftx_mft* mfts, int32_t count, int32_t precision) {
  if (count < 0 || (count > 0 && !mfts)) return fail(ctx, MFTX_EINVAL, "bad MFT list");
  if (precision != MFTX_PREC_FP32 && precision != MFTX_PREC_BF16X3) return fail(ctx, MFTX_EINVAL, "unknown precision");
  for (int32_t i = 0; i < count; ++i) {
    const mftx_mft& q = mfts[i];
    auto bad = [&](const char* what) { return fail(ctx, MFTX_EINVAL, "MFT " + std::to_string(i) + ": " + what); };
    if (!q.F) return bad("null output pointer");
    if (q.m <= 0 || q.n <= 0 || q.M <= 0 || q.N <= 0) return bad("shapes must be positive");
    if (q.m > (1 << 20) || q.n > (1 << 20) || q.M > (1 << 20) || q.N > (1 << 20))
      return bad("dimension too large");
    if (q.ldF < q.N) return bad("output row stride smaller than row length");
    if (q.f) {
      if (q.f_dtype < 0 || q.f_dtype > 3) return bad("unknown input dtype");
      if (q.ldf < q.n) return bad("input row stride smaller than row length");
    } else {
      if (!q.amp || !q.opd) return bad("phasor input needs amp and opd");
      if ((q.amp_dtype != 1 && q.amp_dtype != 3) || (q.opd_dtype != 1 && q.opd_dtype != 3))
        return bad("amp/opd must be float32 or float64");
      if (q.ld_amp < q.n || q.ld_opd < q.n) return bad("phasor row stride too small");
      if (!(q.inv_wl > 0) || !std::isfinite(q.inv_wl)) return bad("inv_wl must be positive");
    }
    if (q.w) {
      if (q.w_dtype != 1 && q.w_dtype != 3) return bad("weight must be float32 or float64");
      if (q.ldw < q.N) return bad("weight row stride smaller than row length");
    }
  }
  return MFTX_OK;
}

extern "C" {

int mftx_version(void) { return 10100; }

int mftx_create(int device, mftx_ctx** out) {
  return guarded(nullptr, [&]() -> int {
  if (!out) return MFTX_EINVAL;
  *out = nullptr;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return MFTX_EDEVICE;
  if (device < 0 || device >= n) return MFTX_EINVAL;
  mftx_ctx* ctx = new mftx_ctx();
  ctx->device = device;
  if (hipSetDevice(device) != hipSuccess ||
      hipHostMalloc((void**)&ctx->ring_host, kRingSlots * kSlotBytes, hipHostMallocDefault) != hipSuccess ||
      !try_malloc((void**)&ctx->ring_dev, kRingSlots * kSlotBytes)) {
    mftx_destroy(ctx);
    return MFTX_ENOMEM;
  }
  for (int i = 0; i < kRingSlots; ++i) {
    if (hipEventCreateWithFlags(&ctx->ring_ev[i], hipEventDisableTiming) != hipSuccess) {
      mftx_destroy(ctx);
      return MFTX_EDEVICE;
    }
  }
  // the no-allocation entry point's scratch address on this device
  void* scratch = nullptr;
  if (scratch_address(device, &scratch) != hipSuccess) {
    mftx_destroy(ctx);
    return MFTX_EDEVICE;
  }

  *out = ctx;
  return MFTX_OK;
  });
}

int mftx_destroy(mftx_ctx* ctx) {
  if (!ctx) return MFTX_EHANDLE;
  (void)hipSetDevice(ctx->device);
  (void)hipStreamSynchronize(ctx->stream);
  for (int i = 0; i < kRingSlots; ++i)
    if (ctx->ring_ev[i]) (void)hipEventDestroy(ctx->ring_ev[i]);
  if (ctx->ring_host) (void)hipHostFree(ctx->ring_host);
  if (ctx->ring_dev) (void)hipFree(ctx->ring_dev);
  if (ctx->ws) (void)hipFree(ctx->ws);
  if (ctx->aux) (void)hipFree(ctx->aux);
  delete ctx;
  return MFTX_OK;
}

const char* mftx_last_error(const mftx_ctx* ctx) { return ctx ? ctx->err.c_str() : "null context"; }

int mftx_set_stream(mftx_ctx* ctx, void* stream) {
  if (!ctx) return MFTX_EHANDLE;
  if ((hipStream_t)stream != ctx->stream) HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  ctx->stream = (hipStream_t)stream;
  return MFTX_OK;
}

int mftx_synchronize(mftx_ctx* ctx) {
  if (!ctx) return MFTX_EHANDLE;
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  return MFTX_OK;
}

int mftx_dft2(mftx_ctx* ctx, const void* f, int f_dtype, int64_t m, int64_t n, int64_t ldf, void* F, int64_t M,
              int64_t N, int64_t ldF, double alpha_r, double alpha_c, double shift_r, double shift_c,
              double offset_r, double offset_c, double scale, int conj, int precision) {
  return mftx::dft2_on_workspace(ctx, f, f_dtype, m, n, ldf, F, M, N, ldF, alpha_r, alpha_c, shift_r, shift_c,
                                 offset_r, offset_c, scale, conj, precision, nullptr, 0, 0);
}

}  // extern "C"

// One transform (the arguments of mftx_dft2, checked) with a real weight map on
// the output, wrapped by (wrow, wcol), or a conjugated input.  reuse_tables:
// the last transform on this workspace had the same geometry but for offsets,
// and its twiddle tables are still there.
namespace {
struct OneSpec {
  const void* f;
  int f_dtype;
  int64_t m, n, ldf;
  void* F;
  int64_t M, N, ldF;
  double alpha_r, alpha_c, shift_r, shift_c, offset_r, offset_c, scale;
  int conj, precision;
  const void* w = nullptr;
  int w_dtype = 0;
  int64_t ldw = 0;
  int wrow = 0, wcol = 0;
  bool conj_input = false, reuse_tables = false;
};
}  // namespace

// One transform on the caller's workspace `ws` of ws_bytes, or on the context's
// growable workspace when ws is null.  Nothing is uploaded: the source's maximum
// (f16 form, larger sources only; one launch more for a long one), then operand,
// twiddle tables and descriptors (launch_prepare_one), then the two GEMMs.  A
// table larger than its space is made and used in pieces of whole tile columns.
//
// `cap` bounds the transform as the no-allocation entry point documents it:
// complex64-sized operands with rows padded to 128 and K to 16 or 32.  The
// workspace then holds operands of up to twice that (K is padded to 32 and
// paired), the descriptors, and tables in the rest.  The operands are fully
// written before they are read (the source's operand with its zero padding,
// then stage 1's output for every K the second stage reads), so the workspace
// needs no clearing; padding rows beyond the output only feed output rows that
// are never stored.
static int run_one(mftx_ctx* ctx, const OneSpec& q, void* ws, size_t ws_bytes, size_t cap) {
  HIPCHK(ctx, hipSetDevice(ctx->device));
  const int prec = q.precision;
  const int64_t m = q.m, n = q.n;
  const MftGeo g = mft_geometry(m, n, q.M, q.N, q.alpha_r, q.alpha_c, q.shift_r, q.shift_c, q.offset_r, q.offset_c,
                                q.conj);
  if (ws) {
    const int64_t rows1 = round_up(g.r1, 128), rows2 = round_up(g.c1, 128);
    const int64_t wide = std::max(rows1 / 128 * ((g.g1.slots + 63) / 64), rows2 / 128 * ((g.g2.slots + 63) / 64));
    const int64_t kg = wide >= 256 ? 32 : 16;
    const int64_t need = round_up(rows1 * round_up(g.k1, kg) * 8, 256) + rows2 * round_up(g.r1, kg) * 8;
    if (need > (int64_t)cap)
      return fail(ctx, MFTX_EINVAL, "transform needs " + std::to_string(need) + " bytes of workspace, more than the " +
                                        std::to_string(cap) + " available");
  }
  const int nkb1 = pair_blocks(g.k1), nkb2 = pair_blocks(g.r1);
  OneMft one = {};
  Problem& p1 = one.desc.prob[0];
  Problem& p2 = one.desc.prob[1];
  const bool long_k = is_long(prec, pairs(g.k1));
  mft_problems(g, prec, q.scale, long_k ? kLongPairs : pairs(g.k1), p1, p2);
  const int tile[2] = {pick_schedule(-1, false, p1.rblocks, p1.sblocks, nkb1, 1, 1).tile,
                       pick_schedule(-1, false, p2.rblocks, p2.sblocks, nkb2, 1, 1).tile};
  // workspace: descriptors, maxima and inverse scale (and sums), operands, tables
  const size_t o_max = round_up(sizeof(OneDesc), 256), o_sum = o_max + 2048;
  const size_t o_a1 = o_sum + (long_k ? sizeof(double) * kMaxBlocks : 0);
  const size_t o_a2 = o_a1 + folded_bytes(g.r1, g.k1), o_t1 = o_a2 + plain_bytes(g.c1, nkb2);
  // slot blocks of a stage whose table fits its space (whole tiles): kTableCap,
  // more where that gives a CU less than two tiles, half of what the operands
  // leave of a caller's workspace at most
  const size_t room = !ws ? kTableMost : o_t1 < ws_bytes ? (ws_bytes - o_t1) / 2 : 0;
  auto piece = [&](const Problem& p, int nkb, int t) {
    const int64_t tr = (p.rblocks + tile_rows(t) - 1) / tile_rows(t);
    const size_t fill = table_bytes((int)((2 * kCUs + tr - 1) / tr) * tile_slots(t), nkb);
    const int64_t fit = (int64_t)(std::min(room, std::max(kTableCap, fill)) / table_bytes(1, nkb)) / tile_slots(t) * tile_slots(t);
    return (int)std::min<int64_t>(p.sblocks, std::max<int64_t>(fit, tile_slots(t)));
  };
  const int piece1 = piece(p1, nkb1, tile[0]), piece2 = piece(p2, nkb2, tile[1]);
  const size_t o_t2 = o_t1 + table_bytes(piece1, nkb1), need = o_t2 + table_bytes(piece2, nkb2);
  static_assert((kMaxBlocks + 1) * sizeof(float) <= 2048, "maxima and inverse scale fit their space");
  int rc = MFTX_OK;
  if (!ws) {
    rc = ensure_ws(ctx, need);
    if (rc) return rc;
    ws = ctx->ws;
  } else if (need > ws_bytes) {
    // the array is made so that a transform within the cap fits; this keeps the kernels inside it whatever changes
    return fail(ctx, MFTX_EINVAL, "transform needs " + std::to_string(need) + " bytes of workspace, more than the " +
                                      std::to_string(ws_bytes) + " available");
  }
  if (too_large(g, false)) return fail(ctx, MFTX_EINVAL, "descriptor block too large (output too big for one call)");
  char* base = (char*)ws;
  float* part = (float*)(base + o_max);
  float* inv = part + kMaxBlocks;

  one.op.amp = q.f;
  one.op.amp_dtype = q.f_dtype;
  one.op.ld_amp = q.ldf;
  one.op.conj = q.conj_input ? 1 : 0;
  one.op.m = (int)m;
  one.op.n = (int)n;
  one.op.trans = g.col_first ? 1 : 0;
  one.op.nwave = 1;
  one.op.dst = base + o_a1;
  MaxOp mx = {};
  if (prec == PREC_FP32) {
    mx.src = q.f;
    mx.dtype = q.f_dtype;
    mx.m = m;
    mx.n = n;
    mx.ld = q.ldf;
    mx.nblk = max_blocks(m, n);
    mx.part = part;
    // a source of up to 8192 elements is read whole by every operand block
    // instead: cheaper than a launch of its own
    one.op.sc = ScaleSrc{part, inv, m * n <= 8192 ? 0 : mx.nblk, 0};
    if (long_k) one.sums = (double*)(base + o_sum);
    p2.inv = inv;
  }
  one.wave = PhasorWave{0.0, 4.0 * g.g1.fold, g.x01, 4.0 * g.g2.fold, g.x02};
  one.tab[0] = TableOp{g.alpha1, g.k1 & 1 ? 0.0 : 0.5, g.g1.y0, piece1, nkb1, 0, 0, base + o_t1, 0};
  one.tab[1] = TableOp{g.alpha2, g.r1 & 1 ? 0.0 : 0.5, g.g2.y0, piece2, nkb2, 0, 0, base + o_t2, 0};
  one.desc.seg[0] = Seg{base + o_a1, base + o_t1, 0.0, nkb1, nkb1, nkb1, 0};
  one.desc.seg[1] = Seg{base + o_a2, base + o_t2, 0.0, nkb2, nkb2, nkb2, 0};
  p1.sbeg = p2.sbeg = 0;
  p1.send = p2.send = 1;
  p1.dst = base + o_a2;
  p2.dst = q.F;
  p2.ldd = q.ldF;
  p2.wmap = q.w;
  p2.wdtype = q.w_dtype;
  p2.ldw = q.ldw;
  p2.wrow = q.wrow;
  p2.wcol = q.wcol;
  one.desc_dev = (OneDesc*)base;
  {
    OneMft first = one;
    // a table used in pieces is always made again
    if (q.reuse_tables && piece1 == p1.sblocks) first.tab[0].nsb = 0;
    if (q.reuse_tables && piece2 == p2.sblocks) first.tab[1].nsb = 0;
    HIPCHK(ctx, launch_prepare_one(prec, first, mx, ctx->stream));
  }
  for (int st = 0; st < 2; ++st) {
    const int sblocks = st ? p2.sblocks : p1.sblocks, step = st ? piece2 : piece1;
    const int rblocks = st ? p2.rblocks : p1.rblocks, nkb = st ? nkb2 : nkb1;
    for (int sb = 0; sb < sblocks; sb += step) {
      TableOp t = one.tab[st];
      t.sb0 = sb;
      t.nsb = std::min(step, sblocks - sb);
      if (sb) HIPCHK(ctx, launch_table_one(prec, t, ctx->stream));
      HIPCHK(ctx, launch_gemm_one(prec, st ? EPI_STORE_CPLX : EPI_STORE_PACKED, tile[st], rblocks, sb, sb + t.nsb, nkb,
                                  &one.desc_dev->prob[st], &one.desc_dev->seg[st], ctx->stream));
    }
  }
  return MFTX_OK;
}

// A phasor source is made as a complex64 array first.
static int run_entry(mftx_ctx* ctx, const mftx_mft& q, int prec) {
  OneSpec one{q.f, q.f_dtype, q.m, q.n, q.ldf, q.F, q.M, q.N, q.ldF, q.alpha_r, q.alpha_c, q.shift_r, q.shift_c,
              q.offset_r, q.offset_c, q.scale, q.conj, prec};
  one.w = q.w;
  one.w_dtype = q.w_dtype;
  one.ldw = q.ldw;
  if (!q.f) {
    const int rc = ensure_aux(ctx, sizeof(float2) * (size_t)q.m * q.n);
    if (rc) return rc;
    const PhasorField ph{q.amp, q.opd, (float2*)ctx->aux, q.ld_amp, q.ld_opd, (int)q.m, (int)q.n, q.amp_dtype, q.opd_dtype};
    HIPCHK(ctx, launch_phasor_fields(&ph, 1, q.inv_wl, ctx->stream));
    one.f = ctx->aux;
    one.f_dtype = MFTX_DTYPE_C64;
    one.ldf = q.n;
  }
  return run_one(ctx, one, nullptr, 0, 0);
}

int mftx::dft2_on_workspace(mftx_ctx* ctx, const void* f, int f_dtype, int64_t m, int64_t n, int64_t ldf, void* F,
                            int64_t M, int64_t N, int64_t ldF, double alpha_r, double alpha_c, double shift_r,
                            double shift_c, double offset_r, double offset_c, double scale, int conj, int precision,
                            void* ws, size_t ws_bytes, size_t cap) {
  if (!ctx) return MFTX_EHANDLE;
  if (!f || !F) return fail(ctx, MFTX_EINVAL, "null array pointer");
  if (m <= 0 || n <= 0 || M <= 0 || N <= 0) return fail(ctx, MFTX_EINVAL, "shapes must be positive");
  if (ldf < n || ldF < N) return fail(ctx, MFTX_EINVAL, "row stride smaller than row length");
  if (f_dtype < 0 || f_dtype > 3) return fail(ctx, MFTX_EINVAL, "unknown input dtype");
  if (precision != MFTX_PREC_FP32 && precision != MFTX_PREC_BF16X3) return fail(ctx, MFTX_EINVAL, "unknown precision");
  if (m > (1 << 20) || n > (1 << 20) || M > (1 << 20) || N > (1 << 20))
    return fail(ctx, MFTX_EINVAL, "dimension too large");
  OneSpec q{f, f_dtype, m, n, ldf, F, M, N, ldF, alpha_r, alpha_c, shift_r, shift_c, offset_r, offset_c, scale, conj,
            precision};
  return run_one(ctx, q, ws, ws_bytes, cap);
}

extern "C" {

int mftx_phasor(mftx_ctx* ctx, const void* amp, int amp_dtype, int64_t ld_amp, const void* opd, int opd_dtype,
                int64_t ld_opd, int64_t m, int64_t n, double wavelength, void* out) {
  if (!ctx) return MFTX_EHANDLE;
  if (!amp || !opd || !out) return fail(ctx, MFTX_EINVAL, "null array pointer");
  if ((amp_dtype != 1 && amp_dtype != 3) || (opd_dtype != 1 && opd_dtype != 3))
    return fail(ctx, MFTX_EINVAL, "amp/opd must be float32 or float64");
  if (m <= 0 || n <= 0 || ld_amp < n || ld_opd < n || m > (1 << 20) || n > (1 << 20))
    return fail(ctx, MFTX_EINVAL, "bad phasor shape");
  if (!(wavelength > 0)) return fail(ctx, MFTX_EINVAL, "wavelength must be positive");
  HIPCHK(ctx, hipSetDevice(ctx->device));
  const PhasorField q{amp, opd, (float2*)out, ld_amp, ld_opd, (int)m, (int)n, amp_dtype, opd_dtype};
  HIPCHK(ctx, launch_phasor_fields(&q, 1, 1.0 / wavelength, ctx->stream));
  return MFTX_OK;
}

int mftx_phasor_many(mftx_ctx* ctx, const mftx_tile* tiles, int32_t count, double wavelength, void* const* out) {
  if (!ctx) return MFTX_EHANDLE;
  return guarded(ctx, [&]() -> int {
    if (count < 0 || (count > 0 && (!tiles || !out))) return fail(ctx, MFTX_EINVAL, "null array pointer");
    if (!(wavelength > 0)) return fail(ctx, MFTX_EINVAL, "wavelength must be positive");
    std::vector<PhasorField> items;
    items.reserve(count);
    for (int32_t i = 0; i < count; ++i) {
      const mftx_tile& T = tiles[i];
      if (!T.amp || !T.opd || !out[i]) return fail(ctx, MFTX_EINVAL, "null array pointer");
      if ((T.amp_dtype != 1 && T.amp_dtype != 3) || (T.opd_dtype != 1 && T.opd_dtype != 3))
        return fail(ctx, MFTX_EINVAL, "amp/opd must be float32 or float64");
      if (T.m <= 0 || T.n <= 0 || T.ld_amp < T.n || T.ld_opd < T.n || T.m > (1 << 20) || T.n > (1 << 20))
        return fail(ctx, MFTX_EINVAL, "bad phasor shape");
      items.push_back(PhasorField{T.amp, T.opd, (float2*)out[i], T.ld_amp, T.ld_opd, (int)T.m, (int)T.n, T.amp_dtype,
                                  T.opd_dtype});
    }
    HIPCHK(ctx, hipSetDevice(ctx->device));
    HIPCHK(ctx, launch_phasor_fields(items.data(), count, 1.0 / wavelength, ctx->stream));
    return MFTX_OK;
  });
}

int mftx_insert(mftx_ctx* ctx, const void* field, int64_t ldf, int64_t fr0, int64_t fc0, int64_t h, int64_t w,
                void* out, int out_dtype, int64_t ldo, int64_t or0, int64_t oc0, int intensity, double weight) {
  if (!ctx) return MFTX_EHANDLE;
  if (!field || !out) return fail(ctx, MFTX_EINVAL, "null array pointer");
  if (h < 0 || w < 0 || fr0 < 0 || fc0 < 0 || or0 < 0 || oc0 < 0) return fail(ctx, MFTX_EINVAL, "negative slice");
  if (h > (1 << 20) || w > (1 << 20) || fr0 > (1 << 30) || fc0 > (1 << 30) || or0 > (1 << 30) || oc0 > (1 << 30))
    return fail(ctx, MFTX_EINVAL, "slice too large");
  if (h > 0 && w > 0 && (ldf < fc0 + w || ldo < oc0 + w))
    return fail(ctx, MFTX_EINVAL, "slice wider than its row stride");
  if (intensity && out_dtype != 1 && out_dtype != 3) return fail(ctx, MFTX_EINVAL, "intensity output must be real");
  if (!intensity && out_dtype != 0 && out_dtype != 2) return fail(ctx, MFTX_EINVAL, "field output must be complex");
  HIPCHK(ctx, hipSetDevice(ctx->device));
  HIPCHK(ctx, launch_insert(field, ldf, (int)fr0, (int)fc0, (int)h, (int)w, out, out_dtype, ldo, (int)or0,
                            (int)oc0, intensity, weight, ctx->stream));
  return MFTX_OK;
}

int mftx_insert_group(mftx_ctx* ctx, const mftx_field* fields, int32_t count, void* out, int out_dtype, int64_t rows,
                      int64_t cols, int64_t ldo, double weight) {
  if (!ctx) return MFTX_EHANDLE;
  return guarded(ctx, [&]() -> int {
    if (!out || count < 0 || (count > 0 && !fields)) return fail(ctx, MFTX_EINVAL, "null array pointer");
    if (count > kGroupFields) return fail(ctx, MFTX_EINVAL, "too many Fields in one group");
    if (out_dtype != 1 && out_dtype != 3) return fail(ctx, MFTX_EINVAL, "intensity output must be real");
    if (rows < 0 || cols < 0 || rows > (1 << 20) || cols > (1 << 20) || ldo < cols)
      return fail(ctx, MFTX_EINVAL, "bad output shape");
    std::vector<FieldItem> items;
    int64_t r0 = rows, r1 = 0, c0 = cols, c1 = 0;
    for (int32_t i = 0; i < count; ++i) {
      const mftx_field& f = fields[i];
      if (!f.F) return fail(ctx, MFTX_EINVAL, "null array pointer");
      if (f.h <= 0 || f.w <= 0 || f.h > (1 << 20) || f.w > (1 << 20) || f.ld < f.w)
        return fail(ctx, MFTX_EINVAL, "bad Field shape");
      // a Field beside the output adds nothing
      if (f.r0 >= rows || f.c0 >= cols || f.r0 + f.h <= 0 || f.c0 + f.w <= 0) continue;
      items.push_back(FieldItem{f.F, f.ld, (int)f.h, (int)f.w, (int)f.r0, (int)f.c0});
      r0 = std::min(r0, std::max<int64_t>(f.r0, 0));
      c0 = std::min(c0, std::max<int64_t>(f.c0, 0));
      r1 = std::max(r1, std::min(f.r0 + f.h, rows));
      c1 = std::max(c1, std::min(f.c0 + f.w, cols));
    }
    if (items.empty()) return MFTX_OK;
    HIPCHK(ctx, hipSetDevice(ctx->device));
    HIPCHK(ctx, launch_insert_group(items.data(), (int)items.size(), (int)r0, (int)c0, (int)(r1 - r0), (int)(c1 - c0),
                                    out, out_dtype, ldo, weight, ctx->stream));
    return MFTX_OK;
  });
}

int mftx_multiply(mftx_ctx* ctx, const void* a, int64_t lda, const void* b, int64_t ldb, void* out, int64_t ldo,
                  int64_t h, int64_t w) {
  if (!ctx) return MFTX_EHANDLE;
  if (!a || !b || !out) return fail(ctx, MFTX_EINVAL, "null array pointer");
  if (h < 0 || w < 0 || lda < w || ldb < w || ldo < w || h > (1 << 20) || w > (1 << 20))
    return fail(ctx, MFTX_EINVAL, "bad multiply shape");
  HIPCHK(ctx, hipSetDevice(ctx->device));
  HIPCHK(ctx, launch_multiply(a, lda, b, ldb, out, ldo, (int)h, (int)w, ctx->stream));
  return MFTX_OK;
}

int mftx_weight_field(mftx_ctx* ctx, const void* F, int64_t ldF, const void* w, int w_dtype, int64_t ldw,
                      double scale, void* out, int64_t ldo, int64_t h, int64_t wd) {
  if (!ctx) return MFTX_EHANDLE;
  if (!F || !w || !out) return fail(ctx, MFTX_EINVAL, "null array pointer");
  if (w_dtype != 1 && w_dtype != 3) return fail(ctx, MFTX_EINVAL, "weight must be float32 or float64");
  if (h < 0 || wd < 0 || ldF < wd || ldw < wd || ldo < wd || h > (1 << 20) || wd > (1 << 20))
    return fail(ctx, MFTX_EINVAL, "bad weight shape");
  HIPCHK(ctx, hipSetDevice(ctx->device));
  HIPCHK(ctx, launch_weight_field(F, ldF, w, w_dtype, ldw, scale, out, ldo, (int)h, (int)wd, ctx->stream));
  return MFTX_OK;
}

int mftx_phase_grad(mftx_ctx* ctx, const void* amp, int amp_dtype, int64_t ld_amp, const void* opd, int opd_dtype,
                    int64_t ld_opd, int64_t m, int64_t n, double wavelength, const void* D, int64_t ldD,
                    double* grad_opd, int64_t ld_gopd, double* grad_amp, int64_t ld_gamp) {
  if (!ctx) return MFTX_EHANDLE;
  if (!amp || !opd || !D || !grad_opd) return fail(ctx, MFTX_EINVAL, "null array pointer");
  if ((amp_dtype != 1 && amp_dtype != 3) || (opd_dtype != 1 && opd_dtype != 3))
    return fail(ctx, MFTX_EINVAL, "amp/opd must be float32 or float64");
  if (m <= 0 || n <= 0 || ld_amp < n || ld_opd < n || ldD < n || ld_gopd < n || (grad_amp && ld_gamp < n) ||
      m > (1 << 20) || n > (1 << 20))
    return fail(ctx, MFTX_EINVAL, "bad gradient shape");
  if (!(wavelength > 0)) return fail(ctx, MFTX_EINVAL, "wavelength must be positive");
  HIPCHK(ctx, hipSetDevice(ctx->device));
  HIPCHK(ctx, launch_phase_grad(PhaseGrad{amp, opd, amp_dtype, opd_dtype, ld_amp, ld_opd, 0, 1, (int)m, (int)n, 1, nullptr,
                                          1.0 / wavelength, D, ldD, 0, grad_opd, grad_amp, 3, 3, ld_gopd, ld_gamp, 1},
                                ctx->stream));
  return MFTX_OK;
}

int mftx_phase_grad_many(mftx_ctx* ctx, const void* amp, int amp_dtype, int64_t ld_amp, const void* opd,
                         int opd_dtype, int64_t ld_opd, int64_t m, int64_t n, const double* wavelengths,
                         int32_t nwave, const void* D, int64_t ldD, int64_t strideD, double* grad_opd,
                         int64_t ld_gopd, double* grad_amp, int64_t ld_gamp) {
  if (!ctx) return MFTX_EHANDLE;
  if (!amp || !opd || !D || !grad_opd || (nwave > 0 && !wavelengths))
    return fail(ctx, MFTX_EINVAL, "null array pointer");
  if ((amp_dtype != 1 && amp_dtype != 3) || (opd_dtype != 1 && opd_dtype != 3))
    return fail(ctx, MFTX_EINVAL, "amp/opd must be float32 or float64");
  if (m <= 0 || n <= 0 || ld_amp < n || ld_opd < n || ldD < n || ld_gopd < n || (grad_amp && ld_gamp < n) ||
      m > (1 << 20) || n > (1 << 20))
    return fail(ctx, MFTX_EINVAL, "bad gradient shape");
  if (nwave < 0 || (nwave > 1 && strideD < m * ldD)) return fail(ctx, MFTX_EINVAL, "bad wavelength count or stride");
  if ((size_t)nwave * sizeof(double) > kSlotBytes) return fail(ctx, MFTX_EINVAL, "too many wavelengths");
  std::vector<double> inv(nwave);
  for (int32_t w = 0; w < nwave; ++w) {
    if (!(wavelengths[w] > 0) || !std::isfinite(wavelengths[w]))
      return fail(ctx, MFTX_EINVAL, "wavelengths must be positive");
    inv[w] = 1.0 / wavelengths[w];
  }
  if (nwave == 0) return MFTX_OK;
  HIPCHK(ctx, hipSetDevice(ctx->device));
  void* dev = nullptr;
  const int rc = upload_desc(ctx, inv.data(), sizeof(double) * inv.size(), &dev);
  if (rc) return rc;
  HIPCHK(ctx, launch_phase_grad(PhaseGrad{amp, opd, amp_dtype, opd_dtype, ld_amp, ld_opd, 0, 1, (int)m, (int)n, nwave,
                                          (const double*)dev, 0.0, D, ldD, strideD, grad_opd, grad_amp, 3, 3, ld_gopd,
                                          ld_gamp, 1},
                                ctx->stream));
  return MFTX_OK;
}

int mftx_phase_grad_stack(mftx_ctx* ctx, const void* amp, int amp_dtype, int64_t ld_amp, const void* opd,
                          int opd_dtype, int64_t ld_opd, int64_t strideO, int32_t nopd, int64_t m, int64_t n,
                          const double* inv_wavelengths, int32_t nwave, const void* D, int64_t ldD, int64_t strideD,
                          void* grad_opd, int gopd_dtype, int64_t ld_gopd, void* grad_amp, int gamp_dtype,
                          int64_t ld_gamp) {
  if (!ctx) return MFTX_EHANDLE;
  if (!amp || !opd || !D || !grad_opd || !inv_wavelengths) return fail(ctx, MFTX_EINVAL, "null array pointer");
  if ((amp_dtype != 1 && amp_dtype != 3) || (opd_dtype != 1 && opd_dtype != 3) ||
      (gopd_dtype != 1 && gopd_dtype != 3) || (grad_amp && gamp_dtype != 1 && gamp_dtype != 3))
    return fail(ctx, MFTX_EINVAL, "amp, opd and gradients must be float32 or float64");
  if (m <= 0 || n <= 0 || ld_amp < n || ld_opd < n || ldD < n || ld_gopd < n || (grad_amp && ld_gamp < n) ||
      m > (1 << 20) || n > (1 << 20))
    return fail(ctx, MFTX_EINVAL, "bad gradient shape");
  if (nwave < 1 || nopd < 1 || ((int64_t)nwave * nopd > 1 && strideD < m * ldD) || (nopd > 1 && strideO < m * ld_opd))
    return fail(ctx, MFTX_EINVAL, "bad wavelength or OPD count or stride");
  HIPCHK(ctx, hipSetDevice(ctx->device));
  HIPCHK(ctx, launch_phase_grad(PhaseGrad{amp, opd, amp_dtype, opd_dtype, ld_amp, ld_opd, strideO, nopd, (int)m, (int)n,
                                          nwave, inv_wavelengths, 0.0, D, ldD, strideD, grad_opd, grad_amp, gopd_dtype,
                                          gamp_dtype, ld_gopd, ld_gamp, 0},
                                ctx->stream));
  return MFTX_OK;
}

int mftx_dft2_many(mftx_ctx* ctx, const mftx_mft* mfts, int32_t count, int32_t precision) {
  return guarded(ctx, [&]() -> int {
  if (!ctx) return MFTX_EHANDLE;
  const int rc = check_mfts(ctx, mfts, count, precision);
  if (rc) return rc;
  if (count == 0) return MFTX_OK;
  HIPCHK(ctx, hipSetDevice(ctx->device));
  return dft2_many_run(ctx, mfts, count, precision);
  });
}

int mftx_mft_plan_create(mftx_ctx* ctx, const mftx_mft* mfts, int32_t count, int32_t precision,
                         mftx_mft_plan** out) {
  return guarded(ctx, [&]() -> int {
  if (!ctx) return MFTX_EHANDLE;
  if (!out) return fail(ctx, MFTX_EINVAL, "null argument");
  *out = nullptr;
  if (count <= 0) return fail(ctx, MFTX_EINVAL, "empty MFT list");
  int rc = check_mfts(ctx, mfts, count, precision);
  if (rc) return rc;
  HIPCHK(ctx, hipSetDevice(ctx->device));
  std::unique_ptr<mftx_mft_plan> plan(new mftx_mft_plan());  // frees its device block on every exit
  plan->ctx = ctx;
  plan->prec = precision;
  many_build(mfts, count, precision, -1, plan->mb);
  const size_t wsb = (size_t)round_up((int64_t)plan->mb.ws, 256);
  if (!try_malloc(&plan->mem, wsb + plan->mb.bytes)) {
    plan->mem = nullptr;
    return fail(ctx, MFTX_ENOMEM, "MFT plan allocation failed");
  }
  plan->desc = (char*)plan->mem + wsb;
  std::vector<char> host(plan->mb.bytes);
  many_place(plan->mb, (char*)plan->mem, plan->desc, host.data());
  if (hipMemcpy(plan->desc, host.data(), host.size(), hipMemcpyHostToDevice) != hipSuccess)
    return fail(ctx, MFTX_EDEVICE, "MFT plan upload failed");
  HIPCHK(ctx, many_tables(plan->mb, precision, plan->desc, ctx->stream));
  *out = plan.release();
  return MFTX_OK;
  });
}

int mftx_mft_plan_execute(mftx_mft_plan* plan) {
  if (!plan) return MFTX_EHANDLE;
  mftx_ctx* ctx = plan->ctx;
  HIPCHK(ctx, hipSetDevice(ctx->device));
  HIPCHK(ctx, many_launch(plan->mb, plan->prec, plan->desc, ctx->stream));
  return MFTX_OK;
}

int mftx_mft_plan_destroy(mftx_mft_plan* plan) {
  if (!plan) return MFTX_EHANDLE;
  (void)hipSetDevice(plan->ctx->device);
  (void)hipStreamSynchronize(plan->ctx->stream);
  delete plan;
  return MFTX_OK;
}

// ---------------------------------------------------------------------------
// detector-grid post-processing
// ---------------------------------------------------------------------------

int mftx_rebin(mftx_ctx* ctx, const void* img, int dtype, int64_t nimg, int64_t rows, int64_t cols, int64_t ld,
               int64_t factor, void* out, int out_dtype) {
  if (!ctx) return MFTX_EHANDLE;
  if (!img || !out) return fail(ctx, MFTX_EINVAL, "null array pointer");
  if ((dtype != 1 && dtype != 3) || (out_dtype != 1 && out_dtype != 3))
    return fail(ctx, MFTX_EINVAL, "rebin is defined for float32/float64 data");
  if (nimg <= 0 || rows <= 0 || cols <= 0 || ld < cols || factor <= 0 || factor > (1 << 16))
    return fail(ctx, MFTX_EINVAL, "bad rebin shape");
  // util.rebin reshapes into factor x factor blocks, which needs whole blocks
  if (rows % factor || cols % factor) return fail(ctx, MFTX_EINVAL, "rebin factor must divide the image shape");
  HIPCHK(ctx, hipSetDevice(ctx->device));
  HIPCHK(ctx, launch_rebin(img, dtype, nimg, rows, cols, ld, (int)factor, out, out_dtype, ctx->stream));
  return MFTX_OK;
}

// wrap v modulo n into (-n/2, n/2]
static double wrap_coord(int64_t v, int64_t n) {
  int64_t w = ((v % n) + n) % n;
  if (2 * w > n) w -= n;
  return (double)w;
}

int mftx_fft_filter(mftx_ctx* ctx, const void* img, int dtype, int64_t rows, int64_t cols, int64_t ld,
                    const void* kernel, int kernel_dtype, int64_t ldk, int normalize, void* out, int out_dtype,
                    int64_t ldo, int precision) {
  if (!ctx) return MFTX_EHANDLE;
  if (!img || !kernel || !out) return fail(ctx, MFTX_EINVAL, "null array pointer");
  if ((dtype != 1 && dtype != 3) || (kernel_dtype != 1 && kernel_dtype != 3) || (out_dtype != 1 && out_dtype != 3))
    return fail(ctx, MFTX_EINVAL, "image, kernel and output must be float32 or float64");
  if (rows <= 0 || cols <= 0 || ld < cols || ldk < cols || ldo < cols || rows > (1 << 20) || cols > (1 << 20))
    return fail(ctx, MFTX_EINVAL, "bad filter shape");
  if (precision != MFTX_PREC_FP32 && precision != MFTX_PREC_BF16X3) return fail(ctx, MFTX_EINVAL, "unknown precision");
  HIPCHK(ctx, hipSetDevice(ctx->device));
  const size_t fbytes = (size_t)round_up(rows * cols * (int64_t)sizeof(float2), 256);
  int rc = ensure_aux(ctx, 2 * fbytes + sizeof(double) * 2 * kMaxPart);
  if (rc) return rc;
  char* a = (char*)ctx->aux;
  float2* F = (float2*)a;
  float2* Y = (float2*)(a + fbytes);
  double* part = (double*)(a + 2 * fbytes);
  // fft2, the MTF, then |ifft2|, as two MFTs with alpha = 1/N.  Both outputs
  // are computed about their centre, where columns pair (the coordinates are
  // integers modulo N, so the order of the outputs is free): the spectrum is
  // held centred, with the MTF (in numpy's fftfreq order) read wrapped, and
  // the magnitude is taken from the wrapped result.  |ifft2(G)| is |fft2(conj
  // G)| / n, so the second transform uses the first one's twiddle tables.
  const int64_t hr = rows / 2, hc = cols / 2;
  // the size limit is that of the uncentred transform
  if (too_large(mft_geometry(rows, cols, rows, cols, 1.0 / (double)rows, 1.0 / (double)cols, wrap_coord(-hr, rows),
                             wrap_coord(-hc, cols), wrap_coord(hr, rows), wrap_coord(hc, cols), 0), true))
    return fail(ctx, MFTX_EINVAL, "descriptor block too large (output too big for one call)");
  OneSpec q{img, dtype, rows, cols, ld, F, rows, cols, cols, 1.0 / (double)rows, 1.0 / (double)cols, 0.0, 0.0,
            wrap_coord(hr, rows), wrap_coord(hc, cols), 1.0, 0, precision};
  q.w = kernel;
  q.w_dtype = kernel_dtype;
  q.ldw = ldk;
  q.wrow = (int)((rows - hr) % rows);
  q.wcol = (int)((cols - hc) % cols);
  rc = run_one(ctx, q, nullptr, 0, 0);
  if (rc) return rc;
  OneSpec b = q;
  b.f = F;
  b.f_dtype = 0;
  b.ldf = cols;
  b.F = Y;
  b.offset_r = b.offset_c = 0.0;
  b.scale = 1.0 / ((double)rows * (double)cols);
  b.w = nullptr;
  b.conj_input = true;
  b.reuse_tables = true;
  rc = run_one(ctx, b, nullptr, 0, 0);
  if (rc) return rc;
  HIPCHK(ctx, launch_magnitude(Y, cols, rows, cols, hr, hc, out, out_dtype, ldo, part, ctx->stream));
  if (normalize) {
    HIPCHK(ctx, launch_sum(img, dtype, rows, cols, ld, part + kMaxPart, ctx->stream));
    HIPCHK(ctx, launch_scale_ratio(out, out_dtype, rows, cols, ldo, part + kMaxPart, part, ctx->stream));
  }
  return MFTX_OK;
}

int mftx_rescale(mftx_ctx* ctx, const void* img, int dtype, int64_t rows, int64_t cols, int64_t ld, const void* mask,
                 int mask_dtype, int64_t ldm, double scale, int64_t out_rows, int64_t out_cols, int order, int mode,
                 int unitary, void* out, int out_dtype, int64_t ldo) {
  if (!ctx) return MFTX_EHANDLE;
  if (!img || !out) return fail(ctx, MFTX_EINVAL, "null array pointer");
  const bool cplx = dtype == 0 || dtype == 2;
  if (dtype < 0 || dtype > 3 || (mask && mask_dtype != 1 && mask_dtype != 3))
    return fail(ctx, MFTX_EINVAL, "image must be float32, float64, complex64 or complex128 and a mask real");
  if (cplx ? (out_dtype != 0 && out_dtype != 2) : (out_dtype != 1 && out_dtype != 3))
    return fail(ctx, MFTX_EINVAL, "the output must be real for a real image and complex for a complex one");
  if (order < 0 || order > 5) return fail(ctx, MFTX_EINVAL, "spline order must be in 0..5");
  if (mode < MFTX_MODE_NEAREST || mode > MFTX_MODE_GRID_CONSTANT) return fail(ctx, MFTX_EINVAL, "unknown boundary mode");
  if (rows <= 0 || cols <= 0 || ld < cols || out_rows <= 0 || out_cols <= 0 || ldo < out_cols ||
      (mask && ldm < cols) || rows > (1 << 20) || cols > (1 << 20) || out_rows > (1 << 20) || out_cols > (1 << 20))
    return fail(ctx, MFTX_EINVAL, "bad rescale shape");
  if (!(scale > 0) || !std::isfinite(scale)) return fail(ctx, MFTX_EINVAL, "scale must be positive");
  HIPCHK(ctx, hipSetDevice(ctx->device));
  const int npad = 12;  // the most any mode pads
  const int64_t np_ = (rows + 2 * npad) * (cols + 2 * npad), no = out_rows * out_cols;
  const size_t b_pad = (size_t)round_up(np_ * 8, 256), b_out = (size_t)round_up(no * 8, 256);
  int rc = ensure_aux(ctx, 2 * b_pad + 3 * b_out + sizeof(double) * 4 * kMaxPart);
  if (rc) return rc;
  char* a = (char*)ctx->aux;
  double* P = (double*)a;
  double* T = (double*)(a + b_pad);
  double* raw = (double*)(a + 2 * b_pad);
  double* raw_im = (double*)(a + 2 * b_pad + b_out);
  double* mval = (double*)(a + 2 * b_pad + 2 * b_out);
  double* part = (double*)(a + 2 * b_pad + 3 * b_out);
  // the mask's dtype sets the threshold (util.py:338-339, numpy finfo eps of
  // the mask, or of the image's real dtype when the mask is derived from it)
  const int mdt = mask ? mask_dtype : dtype;
  const bool single = mdt == 0 || mdt == 1;
  const double eps = single ? 1.1920928955078125e-07 : 2.220446049250313e-16;
  HIPCHK(ctx, launch_rescale(img, dtype, rows, cols, ld, mask ? mask : img, mask ? 2 : 1, mdt, mask ? ldm : ld, eps,
                             scale, out_rows, out_cols, order, mode, unitary, out, out_dtype, ldo, P, T, raw, raw_im,
                             mval, part, ctx->stream));
  return MFTX_OK;
}

// ---------------------------------------------------------------------------
// modal OPD operations
// ---------------------------------------------------------------------------

int mftx_ptt_fit(mftx_ctx* ctx, const void* opd, int opd_dtype, int64_t ld_opd, const void* masks, int mask_dtype,
                 int64_t ld_mask, int64_t mask_stride, int32_t nseg, int64_t rows, int64_t cols, double dx_r,
                 double dx_c, double* normal) {
  if (!ctx) return MFTX_EHANDLE;
  if (!opd || !masks || !normal) return fail(ctx, MFTX_EINVAL, "null array pointer");
  if ((opd_dtype != 1 && opd_dtype != 3) || (mask_dtype != 1 && mask_dtype != 3))
    return fail(ctx, MFTX_EINVAL, "opd and masks must be float32 or float64");
  if (rows <= 0 || cols <= 0 || ld_opd < cols || ld_mask < cols || nseg <= 0 || nseg > 65535 ||
      (nseg > 1 && mask_stride < rows * ld_mask))
    return fail(ctx, MFTX_EINVAL, "bad tilt-fit shape");
  HIPCHK(ctx, hipSetDevice(ctx->device));
  const int64_t nblk = (rows * cols + 255) / 256;
  int rc = ensure_aux(ctx, sizeof(double) * (size_t)(nseg * nblk * 9 + nseg * 9));
  if (rc) return rc;
  double* part = (double*)ctx->aux;
  double* out = part + nseg * nblk * 9;
  HIPCHK(ctx, launch_ptt_normal(opd, opd_dtype, ld_opd, masks, mask_dtype, ld_mask, mask_stride, nseg, rows, cols,
                                dx_r, dx_c, part, out, ctx->stream));
  HIPCHK(ctx, hipMemcpyAsync(normal, out, sizeof(double) * 9 * nseg, hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  return MFTX_OK;
}

int mftx_remove_tilt(mftx_ctx* ctx, const void* opd, int opd_dtype, int64_t ld_opd, const void* masks, int mask_dtype,
                     int64_t ld_mask, int64_t mask_stride, int32_t nseg, int32_t multi, int64_t rows, int64_t cols,
                     double dx_r, double dx_c, const double* tilt, double* out, int64_t ldo) {
  if (!ctx) return MFTX_EHANDLE;
  if (!opd || !masks || !tilt || !out) return fail(ctx, MFTX_EINVAL, "null array pointer");
  if ((opd_dtype != 1 && opd_dtype != 3) || (mask_dtype != 1 && mask_dtype != 3))
    return fail(ctx, MFTX_EINVAL, "opd and masks must be float32 or float64");
  if (rows <= 0 || cols <= 0 || ld_opd < cols || ld_mask < cols || ldo < cols || nseg <= 0 ||
      (!multi && nseg != 1) || (size_t)nseg * 2 * sizeof(double) > kSlotBytes ||
      (nseg > 1 && mask_stride < rows * ld_mask))
    return fail(ctx, MFTX_EINVAL, "bad tilt-removal shape");
  HIPCHK(ctx, hipSetDevice(ctx->device));
  void* dev = nullptr;
  const int rc = upload_desc(ctx, tilt, sizeof(double) * 2 * nseg, &dev);
  if (rc) return rc;
  HIPCHK(ctx, launch_remove_tilt(opd, opd_dtype, ld_opd, masks, mask_dtype, ld_mask, mask_stride, nseg, multi, rows,
                                 cols, dx_r, dx_c, (const double*)dev, out, ldo, ctx->stream));
  return MFTX_OK;
}

int mftx_zernike_basis(mftx_ctx* ctx, const double* rho, const double* theta, const void* mask, int mask_dtype,
                       int64_t npix, const int32_t* noll_nm, int32_t nmodes, int normalize, double* out) {
  return guarded(ctx, [&]() -> int {
  if (!ctx) return MFTX_EHANDLE;
  if (!rho || !theta || !mask || !noll_nm || !out) return fail(ctx, MFTX_EINVAL, "null array pointer");
  if (mask_dtype != 1 && mask_dtype != 3) return fail(ctx, MFTX_EINVAL, "mask must be float32 or float64");
  if (npix <= 0 || nmodes <= 0 || nmodes > 65535) return fail(ctx, MFTX_EINVAL, "bad basis shape");
  // radial coefficients (-1)^k (n-k)! / (k! ((n+m)/2-k)! ((n-m)/2-k)!) (zernike.py:104-107),
  // integers, exact in double while below 2^53
  std::vector<int> desc, pw;
  std::vector<double> coef, norm;
  for (int32_t i = 0; i < nmodes; ++i) {
    const int n = noll_nm[2 * i], m = noll_nm[2 * i + 1];
    const int am = std::abs(m);
    if (n < 0 || am > n || n > 60) return fail(ctx, MFTX_EINVAL, "bad Zernike (n, m)");
    desc.push_back(n);
    desc.push_back(m);
    desc.push_back((int)coef.size());
    int nk = 0;
    if ((n - am) % 2 == 0) {
      for (int k = 0; k <= (n - am) / 2; ++k) {
        // exact rational in long double, then rounded once (an integer)
        long double c = 1.0L;
        for (int q = 2; q <= n - k; ++q) c *= q;
        for (int q = 2; q <= k; ++q) c /= q;
        for (int q = 2; q <= (n + am) / 2 - k; ++q) c /= q;
        for (int q = 2; q <= (n - am) / 2 - k; ++q) c /= q;
        coef.push_back((double)((k % 2 ? -1.0L : 1.0L) * std::nearbyint((double)c)));
        pw.push_back(n - 2 * k);
        ++nk;
      }
    }
    desc.push_back(nk);
    norm.push_back(normalize ? (m == 0 ? std::sqrt((double)(n + 1)) : std::sqrt(2.0) * std::sqrt((double)(n + 1)))
                             : 1.0);
  }
  HIPCHK(ctx, hipSetDevice(ctx->device));
  const size_t o_desc = 0, o_norm = round_up(sizeof(int) * desc.size(), 16);
  const size_t o_coef = round_up(o_norm + sizeof(double) * norm.size(), 16);
  const size_t o_pw = round_up(o_coef + sizeof(double) * std::max<size_t>(coef.size(), 1), 16);
  const size_t bytes = o_pw + sizeof(int) * std::max<size_t>(pw.size(), 1);
  if (bytes > kSlotBytes) return fail(ctx, MFTX_EINVAL, "too many Zernike modes for one call");
  std::vector<char> host(bytes);
  std::memcpy(host.data() + o_desc, desc.data(), sizeof(int) * desc.size());
  std::memcpy(host.data() + o_norm, norm.data(), sizeof(double) * norm.size());
  if (!coef.empty()) std::memcpy(host.data() + o_coef, coef.data(), sizeof(double) * coef.size());
  if (!pw.empty()) std::memcpy(host.data() + o_pw, pw.data(), sizeof(int) * pw.size());
  void* dev = nullptr;
  const int rc = upload_desc(ctx, host.data(), bytes, &dev);
  if (rc) return rc;
  char* d = (char*)dev;
  HIPCHK(ctx, launch_zernike(rho, theta, mask, mask_dtype, npix, nmodes, (const int*)(d + o_desc),
                             (const double*)(d + o_coef), (const int*)(d + o_pw), (const double*)(d + o_norm), out,
                             ctx->stream));
  return MFTX_OK;
  });
}

int mftx_zero(mftx_ctx* ctx, void* p, int64_t bytes) {
  if (!ctx) return MFTX_EHANDLE;
  if (!p || bytes < 0) return fail(ctx, MFTX_EINVAL, "bad zero request");
  HIPCHK(ctx, hipSetDevice(ctx->device));
  HIPCHK(ctx, launch_zero(p, (size_t)bytes, ctx->stream));
  return MFTX_OK;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// batched plan
// ---------------------------------------------------------------------------

namespace {

// Problems with equal keys have one output grid and one stage-1 twiddle set
// (per member tile), so their stage-2 GEMMs concatenate along K.
struct ClassKey {
  int wave, M, N;
  double ar, ac, sr, sc;
  int64_t r0, c0;
  bool operator<(const ClassKey& o) const {
    return std::tie(wave, M, N, ar, ac, sr, sc, r0, c0) < std::tie(o.wave, o.M, o.N, o.ar, o.ac, o.sr, o.sc, o.r0, o.c0);
  }
};

struct Layout {
  size_t total = 256;  // leading pad: no real buffer sits at offset 0
  size_t take(size_t bytes) {
    const size_t off = total;
    total += (size_t)round_up((int64_t)bytes, 256);
    return off;
  }
};

struct ClassInfo {
  ClassKey key;
  std::vector<int> members;  // problem indices
  int group;
  bool col_first;
  int rblocks2 = 0;         // stage-2 row blocks: of N (row-first) or M (column-first) rows
  int64_t pairs1 = 0;       // K pairs of its longest stage-1 problem
  std::vector<int> nkb;     // stage-2 K blocks per member
  std::vector<size_t> abuf; // stage-2 operand per member
  size_t fbuf = 0;    // complex F (groups of the coherent launch)
  int p2 = -1;        // index of its stage-2 problem
  // its output grid: that of the key, or the box shared by its group's windows
  int M = 0, N = 0;
  double sr = 0, sc = 0;            // the key's shift seen from the grid's centre
  double about_r = 0, about_c = 0;  // shift of the core the grid is paired about
  int wr0 = 0, wc0 = 0;             // where the key's window starts in the grid

  void grids(OutGrid& g1, OutGrid& g2) const {
    g1 = make_grid(-(col_first ? key.ar : key.ac), col_first ? sr : sc, col_first ? M : N, col_first ? about_r : about_c);
    g2 = make_grid(-(col_first ? key.ac : key.ar), col_first ? sc : sr, col_first ? N : M, col_first ? about_c : about_r);
  }
};

// Whether `classes` windows of one box, of `nkb` stage-2 K blocks each on
// average, are better summed on chip on the box's grid (box samples over
// window samples: `waste`) than stored as Fields and summed by the coherent
// launch.  Per 32 x 32 block and class, in ns on a full chip: on chip 0.65
// per K block (its fragments come from L2 for each block) and 1.5 for its end,
// four waves taking the classes in turn; as a Field 0.34 per K block (128 x 128
// tiles) and 11.5 for storing, reading and adding it.  Measured (whole image,
// as Fields -> on chip): 18 segments, K = 4: 160 -> 78 us at waste 1.0,
// 83 -> 57 at 2.0; K = 7: 2169 -> 805 at 1.0, 690 -> 396 at 1.45, 691 -> 505 at
// 2.0; 6 segments, K = 22: 621 -> 515 at 1.0, 282 -> 286 at 1.29.
bool sum_windows(double waste, double nkb, int classes) {
  const double turns = 4.0 * ((classes + 3) / 4) / classes;
  return waste * (0.65 * nkb * turns + 1.5) <= 0.34 * nkb + 11.5;
}

// How a class reaches the image.
enum ClassPath {
  PATH_INTENSITY,  // alone in its group: |F|^2 summed in registers
  PATH_WINDOWS,    // one of several windows of one grid: summed in LDS, then squared
  PATH_FIELDS      // one of several grids: F stored, summed and squared by the coherent launch
};

}  // namespace

extern "C" {

int mftx_plan_psf(mftx_ctx* ctx, const mftx_tile* tiles, int32_t ntiles, const double* wavelengths, int32_t nwave,
                  const mftx_problem* problems, int32_t nprob, int64_t image_rows, int64_t image_cols,
                  int32_t precision, int32_t lambda_group, int32_t tile_n, mftx_plan** out) {
  return guarded(ctx, [&]() -> int {
  if (!ctx) return MFTX_EHANDLE;
  if (!out || !tiles || !wavelengths || (!problems && nprob > 0)) return fail(ctx, MFTX_EINVAL, "null argument");
  *out = nullptr;
  if (ntiles <= 0 || nwave <= 0 || nprob < 0) return fail(ctx, MFTX_EINVAL, "empty plan");
  if (precision != MFTX_PREC_FP32 && precision != MFTX_PREC_BF16X3) return fail(ctx, MFTX_EINVAL, "unknown precision");
  if (image_rows <= 0 || image_cols <= 0 || image_rows > (1 << 20) || image_cols > (1 << 20))
    return fail(ctx, MFTX_EINVAL, "bad image shape");
  if (lambda_group <= 0) lambda_group = 8;
  if (tile_n != 0 && tile_n != 64 && tile_n != 128) return fail(ctx, MFTX_EINVAL, "tile_n must be 0, 64 or 128");
  const int fixed_tile = tile_n == 64 ? TILE_MID : tile_n == 128 ? TILE_BIG : -1;
  for (int t = 0; t < ntiles; ++t) {
    const mftx_tile& T = tiles[t];
    if (!T.amp || !T.opd || T.m <= 0 || T.n <= 0 || T.m > (1 << 20) || T.n > (1 << 20) || T.ld_amp < T.n ||
        T.ld_opd < T.n || (T.amp_dtype != 1 && T.amp_dtype != 3) || (T.opd_dtype != 1 && T.opd_dtype != 3))
      return fail(ctx, MFTX_EINVAL, "bad tile " + std::to_string(t));
  }
  for (int w = 0; w < nwave; ++w)
    if (!(wavelengths[w] > 0)) return fail(ctx, MFTX_EINVAL, "wavelengths must be positive");
  for (int i = 0; i < nprob; ++i) {
    const mftx_problem& P = problems[i];
    if (P.tile < 0 || P.tile >= ntiles || P.wave < 0 || P.wave >= nwave || P.M <= 0 || P.N <= 0 ||
        P.M > (1 << 20) || P.N > (1 << 20) || std::llabs(P.out_r0) > (1 << 30) || std::llabs(P.out_c0) > (1 << 30) ||
        !std::isfinite(P.alpha_r) || !std::isfinite(P.alpha_c) ||
        !std::isfinite(P.shift_r) || !std::isfinite(P.shift_c) || !std::isfinite(P.offset_r) ||
        !std::isfinite(P.offset_c) || !std::isfinite(P.weight))
      return fail(ctx, MFTX_EINVAL, "bad problem " + std::to_string(i));
  }
  HIPCHK(ctx, hipSetDevice(ctx->device));
  const int prec = precision;

  // ---- classes and coherent groups ---------------------------------------------
  std::map<ClassKey, int> class_of;
  std::vector<ClassInfo> cls;
  for (int i = 0; i < nprob; ++i) {
    const mftx_problem& P = problems[i];
    const ClassKey k{P.wave, P.M, P.N, P.alpha_r, P.alpha_c, P.shift_r, P.shift_c, P.out_r0, P.out_c0};
    auto it = class_of.find(k);
    if (it == class_of.end()) {
      it = class_of.emplace(k, (int)cls.size()).first;
      ClassInfo c;
      c.key = k;
      c.group = P.group;
      cls.push_back(c);
    }
    if (cls[it->second].group != P.group)
      return fail(ctx, MFTX_EINVAL, "problems with identical output geometry must share a coherent group");
    cls[it->second].members.push_back(i);
  }
  std::map<std::pair<int, int>, std::vector<int>> groups;  // (wave, group) -> classes
  for (size_t c = 0; c < cls.size(); ++c) groups[{cls[c].key.wave, cls[c].group}].push_back((int)c);
  // A group with one class runs the intensity path.  The classes of a group
  // with several are windows of one grid, the box around them, where the box
  // is little larger than they are (their shifts differ by a few pixels, as
  // segment tilts do): transformed on that grid they are summed on chip.
  // Far apart, each would compute mostly what it drops; then their Fields are
  // stored and summed by the coherent launch (sum_windows draws the line).
  bool fast = true;  // every group has one class
  std::vector<ClassPath> path(cls.size(), PATH_INTENSITY);
  struct Box { int64_t r0, r1, c0, c1; };
  std::map<std::pair<int, int>, Box> boxes;  // of the groups of windows
  for (auto& c : cls) {
    c.M = c.key.M;
    c.N = c.key.N;
    c.sr = c.about_r = c.key.sr;
    c.sc = c.about_c = c.key.sc;
  }
  for (auto& g : groups) {
    if (g.second.size() < 2) continue;
    fast = false;
    const ClassKey& k0 = cls[g.second[0]].key;
    Box b{k0.r0, k0.r0, k0.c0, k0.c0};
    double area = 0, nkb = 0;
    bool same = true;
    for (int c : g.second) {
      const ClassKey& k = cls[c].key;
      for (int i : cls[c].members) {
        const mftx_tile& T = tiles[problems[i].tile];
        nkb += 0.5 * (pair_blocks(T.m) + pair_blocks(T.n)) / (double)g.second.size();
      }
      b.r0 = std::min(b.r0, k.r0);
      b.r1 = std::max(b.r1, k.r0 + k.M);
      b.c0 = std::min(b.c0, k.c0);
      b.c1 = std::max(b.c1, k.c0 + k.N);
      area += (double)k.M * k.N;
      same = same && k.ar == k0.ar && k.ac == k0.ac;
    }
    const double all = (double)(b.r1 - b.r0) * (double)(b.c1 - b.c0) * (double)g.second.size();
    const bool windows = same && sum_windows(all / area, nkb, (int)g.second.size()) && b.r1 - b.r0 <= (1 << 20) && b.c1 - b.c0 <= (1 << 20);
    for (int c : g.second) path[c] = windows ? PATH_WINDOWS : PATH_FIELDS;
    if (!windows) continue;
    boxes[g.first] = b;
    double mr = 0, mc = 0;
    for (int ci : g.second) {
      ClassInfo& c = cls[ci];
      c.M = (int)(b.r1 - b.r0);
      c.N = (int)(b.c1 - b.c0);
      c.wr0 = (int)(c.key.r0 - b.r0);
      c.wc0 = (int)(c.key.c0 - b.c0);
      // output coordinate (u - M / 2) - shift of one detector pixel in both grids
      c.sr = c.key.sr + c.wr0 + c.key.M / 2 - c.M / 2;
      c.sc = c.key.sc + c.wc0 + c.key.N / 2 - c.N / 2;
      mr += c.sr / (double)g.second.size();
      mc += c.sc / (double)g.second.size();
    }
    for (int ci : g.second) {
      cls[ci].about_r = mr;
      cls[ci].about_c = mc;
    }
  }

  // contraction order per class (all members share M, N), one for the classes of a group of windows
  auto costs = [&](const ClassInfo& c, double& row_first, double& col_first) {
    for (int i : c.members) {
      const mftx_tile& T = tiles[problems[i].tile];
      row_first += cost_row_first(T.m, T.n, c.M, c.N);
      col_first += cost_col_first(T.m, T.n, c.M, c.N);
    }
  };
  for (auto& g : groups) {
    double row_first = 0, col_first = 0;
    for (int c : g.second) {
      if (path[c] != PATH_WINDOWS) row_first = col_first = 0;
      costs(cls[c], row_first, col_first);
      cls[c].col_first = col_first < row_first;
    }
    if (path[g.second[0]] == PATH_WINDOWS)
      for (int c : g.second) cls[c].col_first = col_first < row_first;
  }

  // Each problem's stage-1 operand is its tile's phasor at its wavelength,
  // carrying the folds of its class's two output grids (stage 1's along K,
  // stage 2's along rows; the grids follow the shift and size, x0 the Field
  // offset).  Problems of one tile and orientation share an operand slot
  // when wavelength and folds agree, and get one each when they do not (the
  // same tile placed twice at one wavelength).
  using Slot = std::tuple<int, double, double, double, double>;  // wave, fold1, x01, fold2, x02
  std::vector<Slot> pslot(nprob);
  for (auto& c : cls) {
    const bool cf = c.col_first;
    for (int i : c.members) {
      const mftx_problem& P = problems[i];
      const mftx_tile& T = tiles[P.tile];
      OutGrid g1, g2;
      c.grids(g1, g2);
      pslot[i] = Slot{P.wave, g1.fold, cf ? -centre(T.m) + P.offset_r : -centre(T.n) + P.offset_c, g2.fold,
                      cf ? -centre(T.n) + P.offset_c : -centre(T.m) + P.offset_r};
    }
  }

  // ---- workspace layout ----------------------------------------------------------
  Layout lay;
  // phasor operands per (tile, orientation): every slot the pair is used with
  std::map<std::pair<int, int>, std::vector<Slot>> tile_slots_of;
  for (auto& c : cls)
    for (int i : c.members) tile_slots_of[{problems[i].tile, c.col_first ? 1 : 0}].push_back(pslot[i]);
  struct TileOp { int64_t R, K; size_t off; std::map<Slot, int> slot; int wave_off; int nslot; };
  std::map<std::pair<int, int>, TileOp> tops;
  std::vector<Slot> wave_slots;  // every phasor slot, grouped by (tile, orientation)
  for (auto& kv : tile_slots_of) {
    auto v = kv.second;
    std::sort(v.begin(), v.end());
    v.erase(std::unique(v.begin(), v.end()), v.end());
    const mftx_tile& T = tiles[kv.first.first];
    const bool tr = kv.first.second == 1;
    TileOp op;
    op.R = tr ? T.n : T.m;
    op.K = tr ? T.m : T.n;
    op.wave_off = (int)wave_slots.size();
    op.nslot = (int)v.size();
    for (size_t j = 0; j < v.size(); ++j) {
      op.slot[v[j]] = (int)j;
      wave_slots.push_back(v[j]);
    }
    op.off = lay.take(folded_bytes(op.R, op.K) * v.size());
    tops[kv.first] = op;
  }
  // stage-2 operands per class and member
  for (auto& c : cls) {
    const int64_t rows2 = c.col_first ? c.M : c.N;
    c.rblocks2 = (int)blocks32(rows2);
    for (int i : c.members) {
      const mftx_tile& T = tiles[problems[i].tile];
      const int nkb = pair_blocks(c.col_first ? T.n : T.m);
      c.nkb.push_back(nkb);
      c.abuf.push_back(lay.take(plain_bytes(rows2, nkb)));
      c.pairs1 = std::max<int64_t>(c.pairs1, pairs(c.col_first ? T.m : T.n));
    }
    if (path[&c - cls.data()] == PATH_FIELDS) c.fbuf = lay.take(sizeof(float2) * (size_t)c.key.M * c.key.N);
  }
  // f16 form: one scale for all tiles that meet in a class (their products are
  // summed unscaled along K), from the maxima of their amplitudes, which lie
  // together.  Classes of one group undo their own scales before they are added:
  // with one scale for the group a segment 1e-7 as bright as its neighbour kept
  // 13 of its 22 bits, and its Field was 8e-5 off.
  std::vector<int> comp(ntiles);
  for (int t = 0; t < ntiles; ++t) comp[t] = t;
  auto root = [&](int t) {
    while (comp[t] != t) t = comp[t] = comp[comp[t]];
    return t;
  };
  for (auto& c : cls)
    for (int i : c.members) comp[root(problems[i].tile)] = root(problems[c.members[0]].tile);
  struct Comp { size_t part = 0, inv = 0; int n = 0; };  // workspace offsets of the maxima and the inverse scale
  std::map<int, Comp> comps;
  std::vector<MaxOp> maxes;
  std::vector<size_t> max_part;  // workspace offset of each job's maxima
  long long max_total = 0;
  if (prec == PREC_FP32) {
    for (int t = 0; t < ntiles; ++t) comps[root(t)].n += max_blocks(tiles[t].m, tiles[t].n);
    size_t inv = lay.take(sizeof(float) * comps.size());  // side by side: the stores of a group read them all
    for (auto& kv : comps) {
      kv.second.part = lay.take(sizeof(float) * kv.second.n);
      kv.second.inv = inv;
      inv += sizeof(float);
      size_t at = kv.second.part;
      for (int t = 0; t < ntiles; ++t) {
        if (root(t) != kv.first) continue;
        const mftx_tile& T = tiles[t];
        MaxOp mx = {};
        mx.src = T.amp;
        mx.dtype = T.amp_dtype;
        mx.m = T.m;
        mx.n = T.n;
        mx.ld = T.ld_amp;
        mx.nblk = max_blocks(T.m, T.n);
        mx.begin = max_total;
        max_total += mx.nblk;
        maxes.push_back(mx);
        max_part.push_back(at);
        at += sizeof(float) * mx.nblk;
      }
    }
  }

  // Weights all below 2^-60 meet the FP32 sums without their common power of
  // two, which the reduction multiplies in: the unitary scale and the f16 form's
  // would take them out of FP32's range.
  double most_weight = 0;
  for (int i = 0; i < nprob; ++i) most_weight = std::max(most_weight, std::fabs(problems[i].weight));
  const int wexp = most_weight > 0 && most_weight < 0x1p-60 ? std::ilogb(most_weight) : 0;

  // ---- descriptors ---------------------------------------------------------------
  // Segment addresses are workspace offsets (operand) and table indices until
  // the workspace exists.
  Tables tables;
  struct SegRef { size_t a; int table; };
  std::vector<Problem> p1, p2;  // stage 1 per (class, member); stage 2 per class
  std::vector<Seg> segs;
  std::vector<SegRef> refs;
  struct Patch { size_t dst, inv; };  // workspace offsets of the destination and the inverse scale (0: none)
  std::vector<Patch> patch1, patch2;
  std::vector<int> nkb1;              // K blocks of each stage-1 problem
  std::vector<std::vector<std::pair<Seg, SegRef>>> seg2(cls.size());
  std::vector<RowPhase> row_phases(cls.size(), RowPhase{});
  size_t row_phase_rows = 0;
  for (size_t ci = 0; ci < cls.size(); ++ci) {
    ClassInfo& c = cls[ci];
    const ClassKey& K = c.key;
    const bool cf = c.col_first;
    const bool single = path[ci] == PATH_INTENSITY && c.members.size() == 1;
    const double a1 = -(cf ? K.ar : K.ac), a2 = -(cf ? K.ac : K.ar);
    const int n1 = cf ? c.M : c.N, n2 = cf ? c.N : c.M;  // output columns of the stages
    OutGrid g1, g2;
    c.grids(g1, g2);
    double xc2 = 0;
    // stage 1, one problem per member
    for (size_t j = 0; j < c.members.size(); ++j) {
      const int i = c.members[j];
      const TileOp& op = tops[{problems[i].tile, cf ? 1 : 0}];
      const double xc1 = std::get<2>(pslot[i]) + 0.5 * (double)(op.K - 1);
      const double xc = std::get<4>(pslot[i]) + 0.5 * (double)(op.R - 1);
      Problem q = {};
      q.sbeg = (int)segs.size();
      q.send = q.sbeg + 1;
      q.rblocks = pair_blocks(op.R);
      q.sblocks = (int)blocks32(g1.slots);
      q.cols = g1.slots;
      q.ncols = n1;
      q.cp = g1.cp;
      q.cm = g1.cm;
      q.y0 = g1.y0;
      // the phase of stage 1's input midpoint is a phase of stage 2's rows,
      // which |F|^2 of a single segment does not see
      q.xrot = single ? 0.0 : a1 * xc1;
      q.scale = (float)stage1_scale(prec, c.pairs1);
      q.ldd = c.nkb[j];
      const int nkb = pair_blocks(op.K);
      segs.push_back(Seg{nullptr, nullptr, 0.0, nkb, nkb, 0, 0});
      refs.push_back(SegRef{op.off + (size_t)op.slot.at(pslot[i]) * folded_bytes(op.R, op.K),
                            tables.get(a1, g1.y0, op.K, g1.slots)});
      patch1.push_back(Patch{c.abuf[j], 0});
      p1.push_back(q);
      nkb1.push_back(nkb);
      // its stage-2 segment
      Seg sg = {};
      sg.nkb = sg.a_nkb = c.nkb[j];
      sg.rot = j ? a2 * (xc2 - xc) : 0.0;
      xc2 = xc;
      seg2[ci].push_back({sg, SegRef{c.abuf[j], tables.get(a2, g2.y0, op.R, g2.slots)}});
      if (single) {
        row_phases[ci] = RowPhase{a1 * xc1, g1.cm + g1.y0, nullptr, n1, 0};
        row_phase_rows += n1;
      }
    }
    // stage 2, one problem per class
    Problem q = {};
    q.rblocks = c.rblocks2;
    q.sblocks = (int)blocks32(g2.slots);
    q.i0 = cf ? c.wr0 : c.wc0;
    q.i1 = q.i0 + (cf ? K.M : K.N);
    q.j0 = cf ? c.wc0 : c.wr0;
    q.j1 = q.j0 + (cf ? K.N : K.M);
    q.cols = g2.slots;
    q.ncols = n2;
    q.cp = g2.cp;
    q.cm = g2.cm;
    q.y0 = g2.y0;
    q.xrot = a2 * xc2;
    q.trans = cf ? 0 : 1;
    q.wrows = K.M;
    q.wcols = K.N;
    const double unit = std::sqrt(std::fabs(K.ar * K.ac));  // unitary scale (fourier.py:100-101)
    const bool stored = path[ci] == PATH_FIELDS;
    if (!stored) {  // the scale is a power of two, so the weight is rounded once
      q.scale = (float)stage2_scale(prec, c.pairs1);
      q.weight = (float)(unit * unit * std::ldexp(problems[c.members[0]].weight, -wexp));
    } else {
      q.scale = (float)(unit * stage2_scale(prec, c.pairs1));
      q.ldd = K.N;  // F[u][v]
    }
    c.p2 = (int)p2.size();
    patch2.push_back(Patch{stored ? c.fbuf : 0, prec == PREC_FP32 ? comps[root(problems[c.members[0]].tile)].inv : 0});
    p2.push_back(q);
  }
  bool multi = false;  // a class of several segments along K
  for (auto& c : cls) multi = multi || c.members.size() > 1;

  // owned until returned: every failure or exception path frees the plan and its workspace
  std::unique_ptr<mftx_plan, int (*)(mftx_plan*)> owned(new mftx_plan(), mftx_plan_destroy);
  mftx_plan* plan = owned.get();
  plan->ctx = ctx;
  plan->prec = prec;
  plan->img_rows = image_rows;
  plan->img_cols = image_cols;

  // stage-1 works: runs of consecutive problems with one tiling and K length
  // (the wavelengths of a tile) share a work item, so the load pipeline runs
  // on across their K loops instead of refilling for every short one
  std::vector<Work> w1;
  plan->tile1 = list_works(w1, p1, nkb1, fixed_tile, 8);

  // stage-2 works: λ-groups of classes with one output window and orientation
  // accumulate |F|^2 in registers (the intensity path); a class of a
  // several-class group gets a complex-store work set of its own.
  // A work item maps every problem's slots through its first problem's output
  // grid (store_partial), so classes share a λ-group only when their stage-2
  // grids agree too: the pairing columns (cp, cm) and the slot count, which
  // follow from the sub-pixel shift (DispersiveTilt moves it per wavelength
  // while the integer placement stays).  Partial images are indexed by output
  // pixel, so every λ-group of one window, whatever its grid, is summed by
  // that window's single reduction.
  struct GeoInfo { std::vector<std::vector<int>> lgroups; size_t partial; int64_t prow, pcol; };
  std::vector<GeoInfo> geos;
  auto class_nkb = [&](int c) {
    int n = 0;
    for (int k : cls[c].nkb) n += k;
    return n;
  };
  {
    using Grid = std::tuple<int, int, int>;  // stage-2 (cp, cm, slots)
    std::map<std::tuple<int, int, int64_t, int64_t, int>, std::map<Grid, std::vector<int>>> geo;
    for (size_t c = 0; c < cls.size(); ++c) {
      if (path[c] != PATH_INTENSITY) continue;
      const Problem& q = p2[cls[c].p2];
      geo[{cls[c].key.M, cls[c].key.N, cls[c].key.r0, cls[c].key.c0, cls[c].col_first ? 1 : 0}][{q.cp, q.cm, q.cols}]
          .push_back((int)c);
    }
    // the tile and the λ-group length (lambda_group at most: shorter where
    // that fills the chip better) follow the grid with most classes
    const std::vector<int>* top = nullptr;
    int64_t nfast = 0;
    for (auto& kv : geo)
      for (auto& sub : kv.second) {
        nfast += sub.second.size();
        if (!top || sub.second.size() > top->size()) top = &sub.second;
      }
    Schedule sch{multi ? TILE_MULTI : TILE_MID, lambda_group};
    if (top) {
      const Problem& q = p2[cls[(*top)[0]].p2];
      sch = pick_schedule(multi && fixed_tile == TILE_BIG ? TILE_MULTI : fixed_tile == TILE_MID && multi ? TILE_MULTI : fixed_tile,
                          multi, q.rblocks, q.sblocks, class_nkb((*top)[0]), nfast, lambda_group);
    }
    plan->tile2 = sch.tile;
    for (auto& kv : geo) {
      GeoInfo gi;
      for (auto& sub : kv.second) {
        const auto& cl = sub.second;
        // groups of nearly equal length, none longer than the schedule's
        const size_t ng = (cl.size() + sch.run - 1) / sch.run;
        for (size_t s = 0; s < ng; ++s)
          gi.lgroups.emplace_back(cl.begin() + s * cl.size() / ng, cl.begin() + (s + 1) * cl.size() / ng);
      }
      gi.prow = round_up(std::get<0>(kv.first), 128);  // partial[u][v]
      gi.pcol = round_up(std::get<1>(kv.first), 128);
      gi.partial = lay.take(sizeof(float) * gi.prow * gi.pcol * gi.lgroups.size());
      geos.push_back(gi);
    }
  }
  // stage-2 problem lists in launch order (λ-groups contiguous), intensity and
  // complex-store, each problem followed by copies of its class's segments
  std::vector<Problem> p2_launch, p2c_launch, p2w_launch;
  std::vector<Patch> patch2_launch, patch2c_launch, patch2w_launch;
  std::vector<Work> w2, w2c, w2w, wf;
  auto push2 = [&](std::vector<Problem>& list, std::vector<Patch>& patches, int c) {
    Problem q = p2[cls[c].p2];
    q.sbeg = (int)segs.size();
    for (auto& sr : seg2[c]) {
      segs.push_back(sr.first);
      refs.push_back(sr.second);
    }
    q.send = (int)segs.size();
    list.push_back(q);
    patches.push_back(patch2[cls[c].p2]);
  };
  for (auto& gi : geos)
    for (size_t g = 0; g < gi.lgroups.size(); ++g) {
      const int pb = (int)p2_launch.size();
      int nch = 0;
      for (int c : gi.lgroups[g]) {
        push2(p2_launch, patch2_launch, c);
        nch += class_nkb(c);
      }
      const ClassInfo& c0 = cls[gi.lgroups[g][0]];
      const size_t poff = gi.partial + sizeof(float) * gi.prow * gi.pcol * g;
      // the partial image offset rides in the pointer field until the workspace exists
      add_tiles(w2, plan->tile2, pb, (int)p2_launch.size(), nch, c0.rblocks2, p2[c0.p2].sblocks,
                (float*)(uintptr_t)poff, (long long)gi.pcol, c0.key.M, c0.key.N);
    }
  // groups of windows: a partial image per group, those of one box together
  struct WindowGeo { Box box; size_t partial; int64_t prow, pcol; int n; };
  std::vector<WindowGeo> wgeos;
  {
    std::map<std::tuple<int64_t, int64_t, int64_t, int64_t>, std::vector<std::pair<int, int>>> by_box;
    for (auto& kv : boxes) by_box[{kv.second.r0, kv.second.r1, kv.second.c0, kv.second.c1}].push_back(kv.first);
    for (auto& kv : by_box) {
      WindowGeo wg;
      wg.box = boxes[kv.second[0]];
      wg.n = (int)kv.second.size();
      wg.prow = round_up(wg.box.r1 - wg.box.r0, 128);
      wg.pcol = round_up(wg.box.c1 - wg.box.c0, 128);
      wg.partial = lay.take(sizeof(float) * wg.prow * wg.pcol * wg.n);
      for (int i = 0; i < wg.n; ++i) {
        const std::vector<int>& cl = groups[kv.second[i]];
        const int pb = (int)p2w_launch.size();
        int nch = 0;
        for (int c : cl) {
          push2(p2w_launch, patch2w_launch, c);
          nch += class_nkb(c);
        }
        const ClassInfo& c0 = cls[cl[0]];
        const Problem& q = p2[c0.p2];
        // the partial image offset rides in the pointer field until the workspace exists
        float* partial = (float*)(uintptr_t)(wg.partial + sizeof(float) * wg.prow * wg.pcol * i);
        for (int r = 0; r < c0.rblocks2; ++r)
          for (int t = 0; t < q.sblocks; ++t)
            w2w.push_back(Work{pb, (int)p2w_launch.size(), r, t, partial, (long long)wg.pcol, c0.M, c0.N, nch, 0});
      }
      wgeos.push_back(wg);
    }
  }
  {
    // Complex stores: neighbouring classes of one shape share a work item, so
    // its load pipeline runs on under the stores (64 weighted fields of 512^2,
    // two rounds of workgroups with one class each: 111 us, now 90).
    auto cplx_works = [&](const std::vector<int>& cl, std::vector<Work>& works) {
      if (cl.empty()) return 0;
      std::vector<Problem> ps;
      std::vector<int> nkb;
      for (int c : cl) {
        ps.push_back(p2[cls[c].p2]);
        nkb.push_back(class_nkb(c));
      }
      return list_works(works, ps, nkb, multi && fixed_tile >= 0 ? TILE_MULTI : fixed_tile, 8, multi);
    };
    std::vector<int> slow, every;
    for (size_t c = 0; c < cls.size(); ++c) {
      every.push_back((int)c);
      if (path[c] == PATH_FIELDS) slow.push_back((int)c);
    }
    for (int c : slow) push2(p2c_launch, patch2c_launch, c);
    // the complex-field set: each class's stage-2 problem
    std::vector<Patch> patch_f;
    for (int c : every) {
      push2(plan->pf, patch_f, c);
      plan->class_first.push_back(cls[c].members[0]);
    }
    plan->tile2c = cplx_works(slow, w2c);
    plan->tile_f = cplx_works(every, wf);
  }
  // executed MFMA FLOPs of the two launches: 12 instructions of 32 x 32 x 16
  // per 32 x 32 block and K block
  auto mfma = [](const std::vector<Work>& ws, int tile) {
    double f = 0;
    for (auto& w : ws) f += (double)w.nch * tile_rows(tile) * tile_slots(tile) * 12.0 * 32768.0;
    return f;
  };
  const double mf1 = mfma(w1, plan->tile1), mf2 = mfma(w2, plan->tile2) + mfma(w2c, plan->tile2c) +
                     mfma(w2w, TILE_SMALL);
  w1 = xcd_order(w1);
  w2 = xcd_order(w2);
  w2c = xcd_order(w2c);
  w2w = xcd_order(w2w);
  wf = xcd_order(wf);

  const size_t o_tab = lay.total;
  lay.take(tables.place(o_tab));
  const size_t o_rowph = lay.take(sizeof(float2) * std::max<size_t>(row_phase_rows, 1));
  const size_t o_rpops = lay.take(sizeof(RowPhase) * std::max<size_t>(cls.size(), 1));
  const size_t o_w1 = lay.take(sizeof(Work) * std::max<size_t>(w1.size(), 1));
  const size_t o_w2 = lay.take(sizeof(Work) * std::max<size_t>(w2.size(), 1));
  const size_t o_p1 = lay.take(sizeof(Problem) * std::max<size_t>(p1.size(), 1));
  const size_t o_p2 = lay.take(sizeof(Problem) * std::max<size_t>(p2_launch.size(), 1));
  const size_t o_w2c = lay.take(sizeof(Work) * std::max<size_t>(w2c.size(), 1));
  const size_t o_p2c = lay.take(sizeof(Problem) * std::max<size_t>(p2c_launch.size(), 1));
  const size_t o_w2w = lay.take(sizeof(Work) * std::max<size_t>(w2w.size(), 1));
  const size_t o_p2w = lay.take(sizeof(Problem) * std::max<size_t>(p2w_launch.size(), 1));
  const size_t o_segs = lay.take(sizeof(Seg) * std::max<size_t>(segs.size(), 1));
  const size_t o_iw = lay.take(sizeof(PhasorWave) * std::max<size_t>(wave_slots.size(), 1));
  const size_t o_ops = lay.take(sizeof(PhasorOp) * std::max<size_t>(tops.size(), 1));
  const size_t o_max = lay.take(sizeof(MaxOp) * std::max<size_t>(maxes.size(), 1));
  const size_t o_top = lay.take(sizeof(TableOp) * std::max<size_t>(tables.ops.size(), 1));
  const size_t o_wf = lay.take(sizeof(Work) * std::max<size_t>(wf.size(), 1));
  const size_t o_pf = lay.take(sizeof(Problem) * std::max<size_t>(plan->pf.size(), 1));
  // groups with several output grids: their classes' fields in map order
  std::vector<CoherentGroup> cgroups;
  std::vector<int> cadd_class;
  for (auto& kv : groups) {
    if (path[kv.second[0]] != PATH_FIELDS) continue;
    cgroups.push_back(CoherentGroup{(int)cadd_class.size(), (int)kv.second.size(),
                                    problems[cls[kv.second[0]].members[0]].weight});
    cadd_class.insert(cadd_class.end(), kv.second.begin(), kv.second.end());
  }
  const size_t o_red = lay.take(sizeof(ReduceOp) * std::max<size_t>(geos.size() + wgeos.size(), 1));
  const size_t o_cg = lay.take(sizeof(CoherentGroup) * std::max<size_t>(cgroups.size(), 1));
  const size_t o_ca = lay.take(sizeof(CoherentAdd) * std::max<size_t>(cadd_class.size(), 1));

  if (!try_malloc(&plan->ws, lay.total)) {
    plan->ws = nullptr;
    return fail(ctx, MFTX_ENOMEM, "plan workspace allocation of " + std::to_string(lay.total) + " bytes failed");
  }
  char* base = (char*)plan->ws;
  for (size_t t = 0; t < tables.ops.size(); ++t) tables.ops[t].dst = base + tables.off[t];
  for (size_t i = 0; i < segs.size(); ++i) {
    segs[i].a = base + refs[i].a;
    segs[i].b = base + tables.off[refs[i].table];
    segs[i].b_nkb = tables.ops[refs[i].table].nkb;
  }
  auto rebase = [&](std::vector<Problem>& ps, const std::vector<Patch>& patches) {
    for (size_t i = 0; i < ps.size(); ++i) {
      ps[i].dst = patches[i].dst ? (void*)(base + patches[i].dst) : nullptr;
      ps[i].inv = patches[i].inv ? (const float*)(base + patches[i].inv) : nullptr;
    }
  };
  rebase(p1, patch1);
  rebase(p2_launch, patch2_launch);
  rebase(p2c_launch, patch2c_launch);
  rebase(p2w_launch, patch2w_launch);
  for (auto* ws : {&w2, &w2w})
    for (auto& w : *ws)
      if (w.partial) w.partial = (float*)(base + (size_t)(uintptr_t)w.partial);
  {
    float2* rp = (float2*)(base + o_rowph);
    for (size_t c = 0; c < cls.size(); ++c) {
      Problem& q = plan->pf[c];
      const Patch& pt = patch2[cls[c].p2];
      q.dst = nullptr;
      q.wmap = nullptr;
      q.inv = pt.inv ? (const float*)(base + pt.inv) : nullptr;
      plan->field_scale.push_back(stage2_scale(prec, cls[c].pairs1));
      if (row_phases[c].rows) {
        row_phases[c].table = rp;
        q.rowph = rp;
        rp += row_phases[c].rows;
        plan->max_rows = std::max(plan->max_rows, row_phases[c].rows);
      }
    }
    plan->row_phases = (RowPhase*)(base + o_rpops);
  }
  std::vector<PhasorWave> iw(wave_slots.size());
  for (size_t i = 0; i < wave_slots.size(); ++i) {
    const Slot& sl = wave_slots[i];
    iw[i] = PhasorWave{4.0 / wavelengths[std::get<0>(sl)], 4.0 * std::get<1>(sl), std::get<2>(sl),
                       4.0 * std::get<3>(sl), std::get<4>(sl)};
  }
  for (size_t i = 0; i < maxes.size(); ++i) maxes[i].part = (float*)(base + max_part[i]);

  plan->works1 = (Work*)(base + o_w1);
  plan->works2 = (Work*)(base + o_w2);
  plan->probs1 = (Problem*)(base + o_p1);
  plan->probs2 = (Problem*)(base + o_p2);
  plan->segs = (Seg*)(base + o_segs);
  plan->waves = (PhasorWave*)(base + o_iw);
  plan->nwork1 = (int)w1.size();
  plan->nwork2 = (int)w2.size();
  plan->works2c = (Work*)(base + o_w2c);
  plan->probs2c = (Problem*)(base + o_p2c);
  plan->nwork2c = (int)w2c.size();
  plan->works2w = (Work*)(base + o_w2w);
  plan->probs2w = (Problem*)(base + o_p2w);
  plan->nwork2w = (int)w2w.size();
  plan->works_f = (Work*)(base + o_wf);
  plan->probs_f = (Problem*)(base + o_pf);
  plan->nwork_f = (int)wf.size();
  plan->max_ops = (MaxOp*)(base + o_max);
  plan->n_max_ops = (int)maxes.size();
  plan->max_blocks = max_total;
  // the descriptors lie together from o_rpops to the workspace's end, so one copy
  // takes them all (15 copies of a few KB: 306 -> 350 us for a plan of 64^2)
  std::vector<char> desc(lay.total - o_rpops);
  auto up = [&](void* d, const void* s, size_t n) {
    if (n) std::memcpy(desc.data() + ((char*)d - base - o_rpops), s, n);
  };
  up(plan->works1, w1.data(), sizeof(Work) * w1.size());
  up(plan->works2, w2.data(), sizeof(Work) * w2.size());
  up(plan->probs1, p1.data(), sizeof(Problem) * p1.size());
  up(plan->probs2, p2_launch.data(), sizeof(Problem) * p2_launch.size());
  up(plan->works2c, w2c.data(), sizeof(Work) * w2c.size());
  up(plan->probs2c, p2c_launch.data(), sizeof(Problem) * p2c_launch.size());
  up(plan->works2w, w2w.data(), sizeof(Work) * w2w.size());
  up(plan->probs2w, p2w_launch.data(), sizeof(Problem) * p2w_launch.size());
  up(plan->segs, segs.data(), sizeof(Seg) * segs.size());
  up(plan->waves, iw.data(), sizeof(PhasorWave) * iw.size());
  std::vector<CoherentAdd> cadds;
  for (int c : cadd_class)
    cadds.push_back(CoherentAdd{(const float2*)(base + cls[c].fbuf), cls[c].key.M, cls[c].key.N, (int)cls[c].key.r0,
                                (int)cls[c].key.c0});
  plan->cgroups = (CoherentGroup*)(base + o_cg);
  plan->cadds = (CoherentAdd*)(base + o_ca);
  plan->n_cgroups = (int)cgroups.size();
  up(plan->cgroups, cgroups.data(), sizeof(CoherentGroup) * cgroups.size());
  up(plan->cadds, cadds.data(), sizeof(CoherentAdd) * cadds.size());
  up(plan->row_phases, row_phases.data(), sizeof(RowPhase) * row_phases.size());
  up(plan->max_ops, maxes.data(), sizeof(MaxOp) * maxes.size());
  up(plan->works_f, wf.data(), sizeof(Work) * wf.size());
  up(base + o_top, tables.ops.data(), sizeof(TableOp) * tables.ops.size());

  std::vector<PhasorOp> ops;
  long long pthreads = 0, quads = 0;
  for (auto& kv : tops) quads += operand_quads(kv.second.R, kv.second.K, kv.second.nslot);
  plan->split = operand_split(quads);
  for (auto& kv : tops) {
    const TileOp& op = kv.second;
    const mftx_tile& T = tiles[kv.first.first];
    PhasorOp ph = {};
    ph.amp = T.amp;
    ph.opd = T.opd;
    ph.amp_dtype = T.amp_dtype;
    ph.opd_dtype = T.opd_dtype;
    ph.ld_amp = T.ld_amp;
    ph.ld_opd = T.ld_opd;
    ph.m = (int)T.m;
    ph.n = (int)T.n;
    ph.trans = kv.first.second;
    ph.nwave = op.nslot;
    ph.waves = plan->waves + op.wave_off;
    ph.dst = base + op.off;
    ph.wave_stride = (long long)folded_bytes(op.R, op.K);
    if (prec == PREC_FP32) {
      const Comp& cm = comps[root(kv.first.first)];
      ph.sc = ScaleSrc{(const float*)(base + cm.part), (float*)(base + cm.inv), cm.n, 0};
    }
    ph.begin = group_begin(pthreads);
    pthreads = ph.begin + operand_threads(op.R, op.K, ph.nwave, plan->split);
    ops.push_back(ph);
  }
  plan->phasor_ops = (PhasorOp*)(base + o_ops);
  plan->n_phasor_ops = (int)ops.size();
  plan->phasor_threads = pthreads;
  up(plan->phasor_ops, ops.data(), sizeof(PhasorOp) * ops.size());
  for (auto& gi : geos) {
    const ClassInfo& c0 = cls[gi.lgroups[0][0]];
    plan->reduces.push_back(ReduceOp{(const float*)(base + gi.partial), (long long)(gi.prow * gi.pcol),
                                     (long long)gi.pcol, (int)gi.lgroups.size(), c0.key.M, c0.key.N, (int)c0.key.r0,
                                     (int)c0.key.c0, 0});
  }
  for (auto& wg : wgeos)
    plan->reduces.push_back(ReduceOp{(const float*)(base + wg.partial), (long long)(wg.prow * wg.pcol), (long long)wg.pcol,
                                     wg.n, (int)(wg.box.r1 - wg.box.r0), (int)(wg.box.c1 - wg.box.c0), (int)wg.box.r0,
                                     (int)wg.box.c0, 0});
  plan->reduce_ops = (ReduceOp*)(base + o_red);
  plan->unit = std::ldexp(1.0, wexp);
  up(plan->reduce_ops, plan->reduces.data(), sizeof(ReduceOp) * plan->reduces.size());
  hipError_t e = hipMemcpy(base + o_rpops, desc.data(), desc.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess)  // the twiddle tables, once for the plan's life
    e = launch_tables(prec, (const TableOp*)(base + o_top), (int)tables.ops.size(), tables.threads, ctx->stream);
  if (e != hipSuccess) return hipfail(ctx, e, "plan descriptor upload");
  // ---- info: algorithmic FLOPs are 8 per complex MAC of the cheaper order -------
  double fl = 0, g1 = 0, g2 = 0;
  for (auto& c : cls)
    for (int i : c.members) {
      const mftx_problem& P = problems[i];
      const double m = (double)tiles[P.tile].m, n = (double)tiles[P.tile].n, M = P.M, N = P.N;
      fl += 8.0 * std::min(cost_row_first(m, n, M, N), cost_col_first(m, n, M, N));
      g1 += 8.0 * (c.col_first ? M * m * n : m * n * N);
      g2 += 8.0 * (c.col_first ? M * n * N : M * m * N);
    }
  plan->info.flops = fl;
  plan->info.gemm_flops[0] = g1;
  plan->info.gemm_flops[1] = g2;
  plan->info.mfma_flops[0] = mf1;
  plan->info.mfma_flops[1] = mf2;
  double bytes = 0;
  for (auto& ph : ops) bytes += 2.0 * (double)ph.wave_stride * ph.nwave;  // write + read
  for (auto& c : cls)
    for (int k : c.nkb) bytes += 2.0 * (double)c.rblocks2 * k * A_BLOCK;
  bytes += 4.0 * image_rows * image_cols;
  plan->info.bytes_hbm_min = bytes;
  double bph = 0, bre = 0;
  for (auto& ph : ops)
    bph += (double)ph.m * ph.n * ((ph.amp_dtype == MFTX_DTYPE_F64 ? 8.0 : 4.0) + (ph.opd_dtype == MFTX_DTYPE_F64 ? 8.0 : 4.0)) +
           (double)ph.wave_stride * ph.nwave;
  for (auto& r : plan->reduces) {
    const int64_t r1 = (int64_t)r.r0 + r.rows, c1 = (int64_t)r.c0 + r.cols;
    const double vr = (double)std::max<int64_t>(0, std::min<int64_t>(r1, image_rows) - std::max(r.r0, 0));
    const double vc = (double)std::max<int64_t>(0, std::min<int64_t>(c1, image_cols) - std::max(r.c0, 0));
    bre += 4.0 * r.ngroups * vr * vc + 4.0 * vr * vc;
  }
  plan->info.bytes_phasor = bph;
  plan->info.bytes_reduce = bre;
  plan->info.coherent_fast = fast ? 1 : 0;
  plan->info.n_stage1 = (int)p1.size();
  plan->info.n_stage2 = (int)cls.size();
  plan->info.n_work1 = plan->nwork1;
  plan->info.n_work2 = plan->nwork2 + plan->nwork2c + plan->nwork2w;
  int nl = (maxes.empty() ? 0 : 1) + (ops.empty() ? 0 : 1) + 1 + (w2.empty() ? 0 : 1) + (w2c.empty() ? 0 : 1) +
           (w2w.empty() ? 0 : 1) + (plan->reduces.empty() ? 0 : 1);
  nl += plan->n_cgroups ? 1 : 0;
  plan->info.n_launch = nl;
  *out = owned.release();
  return MFTX_OK;
  });
}

}  // extern "C"

static hipError_t launch_phasors(const mftx_plan* plan, hipStream_t s) {
  const hipError_t e = launch_absmax(plan->max_ops, plan->n_max_ops, plan->max_blocks, s);
  if (e != hipSuccess) return e;
  return launch_operands(plan->prec, false, plan->split, plan->phasor_ops, plan->n_phasor_ops, plan->phasor_threads, s);
}

// Stage 2: the intensity launch (classes alone in their coherent group), the
// launch of the groups of windows and the complex-store launch (the classes of
// the other groups).
static hipError_t launch_stage2(const mftx_plan* plan, hipStream_t s) {
  hipError_t e = hipSuccess;
  if (plan->nwork2)
    e = launch_gemm(plan->prec, EPI_INTENSITY, plan->tile2, plan->works2, plan->nwork2, plan->probs2, plan->segs, s);
  if (e == hipSuccess && plan->nwork2w)
    e = launch_gemm_coherent(plan->prec, plan->works2w, plan->nwork2w, plan->probs2w, plan->segs, s);
  if (e == hipSuccess && plan->nwork2c)
    e = launch_gemm(plan->prec, EPI_STORE_CPLX, plan->tile2c, plan->works2c, plan->nwork2c, plan->probs2c, plan->segs,
                    s);
  return e;
}

// The image: one launch sums the partial images into it (or clears it where a
// plan has none), then the several-class groups add their |sum of fields|^2.
static hipError_t launch_finish(const mftx_plan* plan, void* image, int dtype, int64_t ldi, int accumulate,
                                hipStream_t s) {
  if (!plan->reduces.empty() || !plan->n_cgroups) {
    const hipError_t e = launch_reduce(plan->reduce_ops, (int)plan->reduces.size(), image, dtype, ldi,
                                       (int)plan->img_rows, (int)plan->img_cols, accumulate, plan->unit, s);
    if (e != hipSuccess || !plan->n_cgroups) return e;
    accumulate = 1;
  }
  return launch_coherent(plan->cgroups, plan->n_cgroups, plan->cadds, image, dtype, ldi, (int)plan->img_rows,
                         (int)plan->img_cols, accumulate, s);
}

static int plan_launch(mftx_plan* plan, void* image, int dtype, int64_t ldi, int accumulate) {
  mftx_ctx* ctx = plan->ctx;
  hipStream_t s = ctx->stream;
  HIPCHK(ctx, launch_phasors(plan, s));
  HIPCHK(ctx, launch_gemm(plan->prec, EPI_STORE_PACKED, plan->tile1, plan->works1, plan->nwork1, plan->probs1, plan->segs, s));
  HIPCHK(ctx, launch_stage2(plan, s));
  HIPCHK(ctx, launch_finish(plan, image, dtype, ldi, accumulate, s));
  return MFTX_OK;
}

extern "C" {

int mftx_plan_execute(mftx_plan* plan, void* image, int32_t image_dtype, int64_t ldi, int32_t accumulate) {
  return guarded(plan ? plan->ctx : nullptr, [&]() -> int {
  if (!plan || !plan->ctx) return MFTX_EHANDLE;
  mftx_ctx* ctx = plan->ctx;
  if (!image) return fail(ctx, MFTX_EINVAL, "null image");
  if (image_dtype != 1 && image_dtype != 3) return fail(ctx, MFTX_EINVAL, "image must be float32 or float64");
  if (ldi < plan->img_cols) return fail(ctx, MFTX_EINVAL, "image row stride too small");
  HIPCHK(ctx, hipSetDevice(ctx->device));
  // Launched one by one: a plan is 3 to 8 launches, 3 to 4 us of host time each,
  // and replaying them from a graph took longer on either side (host 13 -> 28 us
  // and 324 -> 329 us an image for 64 wavelengths of 1024^2, 17 -> 23 and 19 ->
  // 25 us for three of 64^2), besides 150 us to capture and instantiate one.
  return plan_launch(plan, image, image_dtype, ldi, accumulate);
  });
}

// The plan's launch groups in execute order (phasors, stage-1 GEMM, stage-2
// GEMM, reduction), the first `upto` of them; with `ev`, an event
// is recorded before the first and after each.
static hipError_t profile_launches(mftx_plan* plan, void* image, int dtype, int64_t ldi, hipStream_t s, int upto,
                                   const hipEvent_t* ev) {
  hipError_t e = ev ? hipEventRecord(ev[0], s) : hipSuccess;
  for (int k = 0; k < upto && e == hipSuccess; ++k) {
    if (k == 0) e = launch_phasors(plan, s);
    if (k == 1)
      e = launch_gemm(plan->prec, EPI_STORE_PACKED, plan->tile1, plan->works1, plan->nwork1, plan->probs1, plan->segs,
                      s);
    if (k == 2) e = launch_stage2(plan, s);
    if (k == 3) e = launch_finish(plan, image, dtype, ldi, 0, s);
    if (e == hipSuccess && ev) e = hipEventRecord(ev[k + 1], s);
  }
  return e;
}

// Graph mode of mftx_plan_profile: one graph per prefix of the launch groups
// (the first k of them, k = 1..4), each replayed `repeats` times back to back
// between two stream events, twice; group k's time is the difference of the
// mean replay times of prefixes k + 1 and k, so every launch runs as in an
// execute, after its producer, with no event between launches.
// Returns the runtime's error when it cannot capture.
static hipError_t profile_graphs(mftx_plan* plan, void* image, int dtype, int64_t ldi, int repeats, double* ms) {
  hipStream_t s = plan->ctx->stream;
  hipStream_t cap = nullptr;
  hipGraphExec_t x[4] = {nullptr, nullptr, nullptr, nullptr};
  hipEvent_t a = nullptr, b = nullptr;
  hipError_t e = hipStreamCreateWithFlags(&cap, hipStreamNonBlocking);
  for (int k = 0; k < 4 && e == hipSuccess; ++k) {
    hipGraph_t g = nullptr;
    e = hipStreamBeginCapture(cap, hipStreamCaptureModeThreadLocal);
    if (e == hipSuccess) {
      const hipError_t l = profile_launches(plan, image, dtype, ldi, cap, k + 1, nullptr);
      e = hipStreamEndCapture(cap, &g);
      if (e == hipSuccess) e = l;
    }
    if (e == hipSuccess) e = hipGraphInstantiate(&x[k], g, nullptr, nullptr, 0);
    if (g) (void)hipGraphDestroy(g);
  }
  if (e == hipSuccess) e = hipEventCreate(&a);
  if (e == hipSuccess) e = hipEventCreate(&b);
  // two full replays first: caches and clocks as in a run of executes
  for (int r = 0; r < 2 && e == hipSuccess; ++r) e = hipGraphLaunch(x[3], s);
  // prefixes timed in the order 1 2 3 4 4 3 2 1: a slow drift of the clock
  // over the measurement adds the same to both timings of every prefix
  double t[4] = {0, 0, 0, 0};
  for (int i = 0; i < 8 && e == hipSuccess; ++i) {
    const int k = i < 4 ? i : 7 - i;
    e = hipEventRecord(a, s);
    for (int r = 0; r < repeats && e == hipSuccess; ++r) e = hipGraphLaunch(x[k], s);
    if (e == hipSuccess) e = hipEventRecord(b, s);
    if (e == hipSuccess) e = hipEventSynchronize(b);
    float f = 0;
    if (e == hipSuccess) e = hipEventElapsedTime(&f, a, b);
    t[k] += 0.5 * (double)f / repeats;
  }
  for (auto& g : x)
    if (g) (void)hipGraphExecDestroy(g);
  if (a) (void)hipEventDestroy(a);
  if (b) (void)hipEventDestroy(b);
  if (cap) (void)hipStreamDestroy(cap);
  if (e != hipSuccess) return e;
  ms[0] = t[0];
  for (int k = 1; k < 4; ++k) ms[k] = t[k] - t[k - 1];
  return hipSuccess;
}

int mftx_plan_profile(mftx_plan* plan, void* image, int32_t image_dtype, int64_t ldi, int32_t repeats, double* ms) {
  if (!plan || !plan->ctx) return MFTX_EHANDLE;
  mftx_ctx* ctx = plan->ctx;
  if (!image || !ms || repeats <= 0 || repeats > 4096) return fail(ctx, MFTX_EINVAL, "bad profile request");
  if (image_dtype != 1 && image_dtype != 3) return fail(ctx, MFTX_EINVAL, "image must be float32 or float64");
  if (ldi < plan->img_cols) return fail(ctx, MFTX_EINVAL, "image row stride too small");
  return guarded(ctx, [&]() -> int {
  HIPCHK(ctx, hipSetDevice(ctx->device));
  if (plan->use_graph) {
    double g[4];
    if (profile_graphs(plan, image, image_dtype, ldi, repeats, g) == hipSuccess) {
      for (int k = 0; k < 4; ++k) ms[k] = g[k];
      ms[4] = 1.0;
      return MFTX_OK;
    }
    (void)hipGetLastError();  // the runtime refused a capture: time eagerly instead
  }
  // eager: every repeat back to back on the context stream with events
  // between the launch groups, one wait at the end
  hipStream_t s = ctx->stream;
  std::vector<hipEvent_t> ev(5 * (size_t)repeats, nullptr);
  hipError_t e = hipSuccess;
  for (auto& x : ev)
    if (e == hipSuccess) e = hipEventCreate(&x);
  for (int r = 0; r < repeats && e == hipSuccess; ++r)
    e = profile_launches(plan, image, image_dtype, ldi, s, 4, &ev[5 * (size_t)r]);
  if (e == hipSuccess) e = hipEventSynchronize(ev.back());
  double acc[4] = {0, 0, 0, 0};
  for (int r = 0; r < repeats && e == hipSuccess; ++r)
    for (int k = 0; k < 4 && e == hipSuccess; ++k) {
      float t = 0;
      e = hipEventElapsedTime(&t, ev[5 * (size_t)r + k], ev[5 * (size_t)r + k + 1]);
      acc[k] += t;
    }
  for (auto& x : ev)
    if (x) (void)hipEventDestroy(x);
  if (e != hipSuccess) return hipfail(ctx, e, "plan profile");
  for (int k = 0; k < 4; ++k) ms[k] = acc[k] / repeats;
  ms[4] = 0.0;
  return MFTX_OK;
  });
}

int mftx_plan_set_fields(mftx_plan* plan, void* const* dst, int64_t ldd, const void* const* wmap, int32_t wmap_dtype,
                         int64_t ldw, const double* scale) {
  if (!plan || !plan->ctx) return MFTX_EHANDLE;
  mftx_ctx* ctx = plan->ctx;
  return guarded(ctx, [&]() -> int {
    if (!dst || !scale) return fail(ctx, MFTX_EINVAL, "null argument");
    if (wmap && wmap_dtype != 1 && wmap_dtype != 3) return fail(ctx, MFTX_EINVAL, "weight map must be float32 or float64");
    // every argument is checked before any descriptor changes
    for (size_t c = 0; c < plan->pf.size(); ++c) {
      const Problem& q = plan->pf[c];
      const int i = plan->class_first[c];
      const int64_t N = q.trans ? q.i1 - q.i0 : q.j1 - q.j0;  // the class's F is M x N, row stride ldd
      if (!dst[i]) return fail(ctx, MFTX_EINVAL, "null field pointer for problem " + std::to_string(i));
      if (ldd < N || (wmap && wmap[i] && ldw < N)) return fail(ctx, MFTX_EINVAL, "field row stride too small");
      if (!std::isfinite(scale[i])) return fail(ctx, MFTX_EINVAL, "non-finite field scale");
    }
    for (size_t c = 0; c < plan->pf.size(); ++c) {
      Problem& q = plan->pf[c];
      const int i = plan->class_first[c];
      q.dst = dst[i];
      q.ldd = ldd;
      q.wmap = wmap ? wmap[i] : nullptr;
      q.wdtype = wmap_dtype;
      q.ldw = ldw;
      q.scale = (float)(scale[i] * plan->field_scale[c]);
    }
    HIPCHK(ctx, hipSetDevice(ctx->device));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    if (!plan->pf.empty())
      HIPCHK(ctx, hipMemcpy(plan->probs_f, plan->pf.data(), sizeof(Problem) * plan->pf.size(), hipMemcpyHostToDevice));
    if (!plan->fields_ready)  // once: the phases stage 1 leaves out
      HIPCHK(ctx, launch_row_phases(plan->row_phases, (int)plan->pf.size(), plan->max_rows, ctx->stream));
    plan->fields_ready = 1;
    return MFTX_OK;
  });
}

int mftx_plan_execute_fields(mftx_plan* plan) {
  if (!plan || !plan->ctx) return MFTX_EHANDLE;
  mftx_ctx* ctx = plan->ctx;
  if (!plan->fields_ready) return fail(ctx, MFTX_EINVAL, "mftx_plan_set_fields has not been called");
  HIPCHK(ctx, hipSetDevice(ctx->device));
  HIPCHK(ctx, launch_gemm(plan->prec, EPI_STORE_CPLX, plan->tile_f, plan->works_f, plan->nwork_f, plan->probs_f,
                          plan->segs, ctx->stream));
  return MFTX_OK;
}

int mftx_plan_set_graph(mftx_plan* plan, int32_t use_graph) {
  if (!plan) return MFTX_EHANDLE;
  plan->use_graph = use_graph ? 1 : 0;
  return MFTX_OK;
}

int mftx_plan_get_info(const mftx_plan* plan, mftx_plan_info* info) {
  if (!plan || !info) return MFTX_EHANDLE;
  *info = plan->info;
  return MFTX_OK;
}

int mftx_plan_destroy(mftx_plan* plan) {
  if (!plan) return MFTX_EHANDLE;
  if (plan->ctx) {
    (void)hipSetDevice(plan->ctx->device);
    (void)hipStreamSynchronize(plan->ctx->stream);
  }
  if (plan->ws) (void)hipFree(plan->ws);
  delete plan;
  return MFTX_OK;
}

}  // extern "C"
