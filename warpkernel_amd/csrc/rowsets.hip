// rowsets.hip -- several right-hand sides on the matrix cores, for layouts whose
// neighbouring rows share their columns (the three unknowns of an elasticity
// node): Y[4 rows, k] += A[4 rows, 4 steps] X[4 steps, k] by
// v_mfma_f64_4x4x4, four such row sets per wave.
//
// The instruction adds its four products to the accumulator one after another,
// each by an IEEE fma (checked bit for bit on the device against a chain of
// fma, subnormals, infinities and signed zeros included), so with a set's steps
// in order every row sums as in the other kernels: the first product rounded,
// then one fma per further slot, pads included.
//
// Why: with a row per lane every product reads its own 8 bytes of x from LDS, and
// a k-tile's window leaves a few waves per CU (hex elasticity 32^3 k=16: LDS
// 23% busy at 1.65 waves per SIMD).  Here one read of x serves the set's rows,
// the values stay in registers whatever k, and no window limits residency
// (12 or 16 waves per CU).  Hex elasticity FP64, against the window kernels, one
// set of inputs repeated: 32^3 k=16 58.4 -> 25.1 us, k=32 100 -> 38.4; 64^3 k=16
// 421 -> 248, k=32 803 -> 382 (other inputs from pass to pass: 32^3 k=16 58.5 ->
// 33.6, 48^3 k=32 365 -> 167).  What bounds it: a wave first waits for its
// record, then for its values (64^3 k=4: 61 us without the values, 133 without
// x, 175 with both);
// from k = 16 on the reads of x through L1, 67 us per 8 columns at 64^3 where
// the matrix instructions alone take 18.  Measured and not kept: x through an
// LDS window filled by direct-to-LDS loads (64^3 k=8 221 us, k=32 489), values
// through LDS in 16-byte pieces (k=8 193), a ring of 3 or 21 steps (k=8 187,
// 217), 20 waves per CU (spills: 307), each lane's 32 bytes of a line of x as 16 of
// each half (48^3 k=32 177 against 168), nontemporal values, whose lines the
// neighbouring waves then miss (32^3 k=16 34.8 against 26.3).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "spmv_device.hpp"
#include "wk_internal.hpp"

namespace wk {
namespace {

constexpr int kMaxChunks = 3;   // groups of at most 84 steps
constexpr int kSetChunk = 7;    // matrix steps (28 slots) per chunk
constexpr int kSetBlock = 4;    // waves per block of the product

__host__ __device__ constexpr int32_t set_chunks(int32_t len) {
  return (len + 4 * kSetChunk - 1) / (4 * kSetChunk);
}

}  // namespace

// Four row sets of one group: one wave of the product.
struct SetRec {
  int64_t base;      // first slot of the group
  int32_t len;       // its steps
  int32_t row0;      // its first row
  uint8_t first[8];  // first lane of sets 0..3 and past the last; 64: no such set
  int32_t col0[4];   // least column of each set (uint16 columns)
  int32_t pad[2];
};

namespace {

struct SetArgs {
  const SetRec *rec;  // [nwaves]
  const void *cols;   // [nwaves][kMaxChunks][16][8] uint16 from the set's least column, or int32
  int32_t nwaves;
};

// Columns of one lane: chunk c's seven steps (of eight fields).
template <class I>
struct SetCols {
  I c[kMaxChunks][8];
};

// One wave: four row sets.  Lane 16k + 4b + i holds A's entry (row i of set b,
// step 4s + k) for every s in registers, loaded once; per k-tile it reads the B
// operand of its four steps straight from x (set b's column at step 4s + k,
// right-hand sides j*E .. j*E+E-1 of the tile, j = lane & 3) into a ring of
// seven steps: step s + 7's read goes out when step s has been multiplied.
template <class P, int OUT, int NC, int E, class I>
__device__ __forceinline__ void rowset_wave(const SpmvArgs &a, const SetRec *rec, const SetCols<I> &sc,
                                            int32_t col0, int32_t lane, int32_t ntiles) {
  using V = typename P::V;
  using X = typename P::X;
  constexpr int CS = kSetChunk;
  constexpr int KS = NC * CS;
  constexpr int KT = 4 * E;
  constexpr int RING = kSetChunk;  // divides KS: a step's ring slot is the same in every tile
  const int32_t len = rec->len;
  const int32_t i4 = lane & 3, b = (lane >> 2) & 3, k4 = lane >> 4;
  const uint64_t fb = *reinterpret_cast<const uint64_t *>(rec->first);
  const int32_t f0 = (int32_t)(fb >> (8 * b)) & 255, f1 = (int32_t)(fb >> (8 * b + 8)) & 255;
  uint32_t xo[KS];  // byte offset of the row of x of step s
  const uint32_t ldb = (uint32_t)(a.ldx * (int64_t)sizeof(X));
#pragma unroll
  for (int s = 0; s < KS; s++) xo[s] = (uint32_t)(col0 + (int32_t)sc.c[s / CS][s % CS]) * ldb;
  V raw[KS];
  {
    const int32_t row = f0 + i4 < f1 ? f0 + i4 : (f0 < 63 ? f0 : 63);
    const char *vb = reinterpret_cast<const char *>(static_cast<const V *>(a.vals) + rec->base);
#pragma unroll
    for (int s = 0; s < KS; s++) {
      int32_t step = 4 * s + k4;
      if (s >= KS - CS) step = step < len ? step : len - 1;  // only the last chunk passes the end
      const uint32_t vo = (uint32_t)(row + 64 * step) * (uint32_t)sizeof(V);
      __builtin_memcpy(&raw[s], vb + vo, sizeof(V));
    }
  }
  const int32_t r_out = f0 + k4;  // D's lane 16i + 4b + j: row i of set b
  const int32_t rowid = rec->row0 + r_out;
  const bool writer = r_out < f1 && rowid < a.nznrows;
  // (read for every lane: a guarded read would be waited for here)
  const int32_t dst = OUT == OUT_RUNX ? rowid : a.row_map[rowid < a.nznrows ? rowid : a.nznrows - 1];

  // The lane's first column of tile t.  In a last tile of fewer than KT columns
  // lanes move left onto columns that others hold too: the same sums (y is
  // stored twice), and no masked reads (k >= E).
  auto column = [&](int32_t t) {
    const int32_t c = t * KT + i4 * E;
    return c < a.k - E ? c : a.k - E;
  };
  X xv[RING][E];
  const char *xb = static_cast<const char *>(a.x);
  auto load = [&](int s, uint32_t tb) { __builtin_memcpy(xv[s % RING], xb + (xo[s] + tb), E * sizeof(X)); };
  double av[KS];
  double acc[E];
  auto mul = [&](int s) {
#pragma unroll
    for (int e = 0; e < E; e++) {
      double bv = (double)xv[s % RING][e];
      // steps past the end (last chunk only): -0 * 0 changes nothing
      if (s >= KS - CS) bv = 4 * s + k4 < len ? bv : 0.0;
      acc[e] = __builtin_amdgcn_mfma_f64_4x4x4f64(av[s], bv, acc[e], 0, 0, 0);
    }
  };
  auto store = [&](int32_t t) {
    if (!writer) return;
    const int32_t e0 = column(t);
    double *yr = a.y + (int64_t)dst * a.ldy + e0;
    if constexpr (OUT == OUT_RESID) {
      // r may be b: of a column that several lanes hold, only the one whose place
      // it is in the tile may write, and all of b is read before
      const double *br = a.b + (int64_t)dst * a.ldb + e0;
      const int32_t others = t * KT + i4 * E - e0;  // leading columns of other lanes
      double bv[E];
#pragma unroll
      for (int e = 0; e < E; e++) bv[e] = br[e];
      if (others <= 0) {
#pragma unroll
        for (int e = 0; e < E; e++) yr[e] = bv[e] - acc[e];
      } else {
#pragma unroll
        for (int e = 1; e < E; e++)
          if (e >= others) yr[e] = bv[e] - acc[e];
      }
    } else {
#pragma unroll
      for (int e = 0; e < E; e++) yr[e] = acc[e];
    }
  };
  uint32_t tb = (uint32_t)column(0) * (uint32_t)sizeof(X);
#pragma unroll
  for (int s = 0; s < RING; s++) load(s, tb);
#pragma unroll
  for (int s = 0; s < KS; s++) av[s] = s < KS - CS || 4 * s + k4 < len ? (double)raw[s] : -0.0;
  int32_t t = 0;
  // (tiles of 4 and 8 columns come alone, launch_rowsets: without the loop the
  // residual's kernel for 5 to 8 columns does not spill, blocks of
  // three unknowns on 56^3 nodes k=8 164 -> 130 us)
  for (; (E == 4 || OUT != OUT_RESID) && t + 1 < ntiles; t++) {
    const uint32_t tn = (uint32_t)column(t + 1) * (uint32_t)sizeof(X);
#pragma unroll
    for (int e = 0; e < E; e++) acc[e] = -0.0;
#pragma unroll
    for (int s = 0; s < KS; s++) {
      mul(s);
      if (s + RING < KS)
        load(s + RING, tb);
      else
        load(s + RING - KS, tn);
    }
    store(t);
    tb = tn;
  }
#pragma unroll
  for (int e = 0; e < E; e++) acc[e] = -0.0;
#pragma unroll
  for (int s = 0; s < KS; s++) {
    mul(s);
    if (s + RING < KS) load(s + RING, tb);
  }
  store(t);
}

// Waves per SIMD: three hold 168 registers each, four 128.
template <class P, int E>
constexpr int set_waves() {
  return E * (int)sizeof(typename P::X) < 32 ? 4 : 3;
}

template <class P, int OUT, int E, class I>
__global__ __launch_bounds__(kSetBlock * 64, (set_waves<P, E>())) void spmv_rowset_kernel(
    SpmvArgs a, SetArgs w, int32_t nwork, int32_t ntiles, int32_t remap) {
  const int32_t tid = threadIdx.x;
  const int32_t bid = blockIdx.x;
  if (bid >= nwork) {
    const int64_t p = (int64_t)a.nznrows + (int64_t)(bid - nwork) * (kSetBlock * 64) + tid;
    if (p >= a.nrows) return;
    const int64_t dst = OUT == OUT_RUNX ? p : (int64_t)a.row_map[p];
    for (int32_t t = 0; t < a.k; t++)
      a.y[dst * a.ldy + t] = OUT == OUT_RESID ? a.b[dst * a.ldb + t] : 0.0;
    return;
  }
  const int32_t wv = __builtin_amdgcn_readfirstlane(work_id(bid, nwork, remap) * kSetBlock + (tid >> 6));
  if (wv >= w.nwaves) return;
  const int32_t lane = tid & 63;
  // the record and the columns depend on the wave's number alone, so both are
  // one memory latency away
  const SetRec *rec = w.rec + wv;
  int32_t col0 = 0;
  if (sizeof(I) == 2) col0 = rec->col0[(lane >> 2) & 3];
  SetCols<I> sc;
  const I *cp = static_cast<const I *>(w.cols) + ((int64_t)wv * (kMaxChunks * 16) + (lane >> 2)) * 8;
#pragma unroll
  for (int c = 0; c < kMaxChunks; c++) __builtin_memcpy(sc.c[c], cp + c * 128, 8 * sizeof(I));
  const int32_t nc = set_chunks(rec->len);
  if (nc == 3)
    rowset_wave<P, OUT, 3, E, I>(a, rec, sc, col0, lane, ntiles);
  else if (nc == 2)
    rowset_wave<P, OUT, 2, E, I>(a, rec, sc, col0, lane, ntiles);
  else
    rowset_wave<P, OUT, 1, E, I>(a, rec, sc, col0, lane, ntiles);
}

// Row sets of one group per wave: lanes in order, a lane joins the set of the
// lane before it when both read the same column at every step, in Kr numbering
// too, and the set has fewer than four lanes.  (A pad and an entry of column 0
// read the same column of x but not of x in Kr numbering, where pads read column
// 0 too.)  Pass 1 writes a bit per lane that starts a set and the widest column
// span of a lane.
constexpr int kBuildWaves = 4;
__global__ __launch_bounds__(kBuildWaves * 64) void row_set_kernel(
    const int32_t *__restrict__ cols, const int32_t *__restrict__ cols_kr,
    const int64_t *__restrict__ warp_offsets, const uint32_t *__restrict__ max_nz_rows, int32_t ngroups,
    uint64_t *__restrict__ starts, uint32_t *__restrict__ span) {
  const int32_t lane = threadIdx.x & 63;
  const int32_t g = __builtin_amdgcn_readfirstlane((int32_t)(blockIdx.x * kBuildWaves + (threadIdx.x >> 6)));
  if (g >= ngroups) return;
  const int64_t base = warp_offsets[g];
  const int32_t len = (int32_t)max_nz_rows[g];
  bool same = lane > 0;
  int32_t lo = INT32_MAX, hi = 0;
  constexpr int U = 9;  // loads in flight; past the end the last step again
  for (int32_t t0 = 0; t0 < len; t0 += U) {
    int32_t p[U];
#pragma unroll
    for (int u = 0; u < U; u++) p[u] = cols[base + lane + 64 * (int64_t)(t0 + u < len ? t0 + u : len - 1)];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int32_t before = __shfl_up(p[u], 1);  // by every lane, also those that differ already
      same = same && before == p[u];
      if (cols_kr && __ballot(p[u] == 0)) {
        const int32_t kr = cols_kr[base + lane + 64 * (int64_t)(t0 + u < len ? t0 + u : len - 1)];
        same = __shfl_up(kr, 1) == kr && same;
      }
      lo = min(lo, p[u]);
      hi = max(hi, p[u]);
    }
  }
  const uint64_t m = __ballot(same);
  uint64_t st = 0;
  uint32_t size = 0;
  for (int l = 0; l < 64; l++) {
    if (!((m >> l) & 1u) || size == 4) {
      st |= 1ull << l;
      size = 0;
    }
    size++;
  }
  uint32_t s = (uint32_t)(hi - lo);
  for (int o = 32; o > 0; o >>= 1) s = max(s, (uint32_t)__shfl_xor((int)s, o));
  if (lane == 0) {
    starts[g] = st;
    span[g] = s;
  }
}

// Pass 2, one block per group, one wave per four sets: their record and
// columns.  Field u < 7 of chunk c, lane group 4k + b: set b's column at step
// 4 (7c + u) + k.  Steps past the end repeat the last one; missing sets hold
// column 0 (nothing of theirs is stored).
template <class I>
__global__ __launch_bounds__(1024) void row_set_cols_kernel(
    const int32_t *__restrict__ cols, const int64_t *__restrict__ warp_offsets,
    const uint32_t *__restrict__ max_nz_rows, const uint64_t *__restrict__ starts,
    const uint32_t *__restrict__ woff, I *__restrict__ out, SetRec *__restrict__ rec) {
  const int32_t lane = threadIdx.x & 63;
  const int32_t g = blockIdx.x;
  const uint32_t q = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t w0 = woff[g], nq = woff[g + 1] - w0;
  if (q >= nq) return;
  const int64_t base = warp_offsets[g];
  const int32_t len = (int32_t)max_nz_rows[g], nc = set_chunks(len);
  const int32_t kb = lane & 15, k4 = kb >> 2, b = kb & 3, c = lane >> 4;
  uint64_t rest = starts[g];
  for (uint32_t j = 0; j < 4 * q; j++) rest &= rest - 1;
  int32_t first[5];  // of the wave's four sets, and past them
  for (int j = 0; j < 5; j++) {
    first[j] = rest ? __builtin_ctzll(rest) : 64;
    rest &= rest - 1;
  }
  const int32_t f0 = b == 0 ? first[0] : b == 1 ? first[1] : b == 2 ? first[2] : first[3];
  const int32_t *cp = cols + base + (f0 < 64 ? f0 : 63);
  int32_t col[8];
#pragma unroll
  for (int u = 0; u < 8; u++) {
    const int32_t step = 4 * (kSetChunk * c + u) + k4;
    col[u] = cp[64 * (int64_t)(step < len ? step : len - 1)];
    if (f0 >= 64) col[u] = 0;
  }
  int32_t c0 = 0;
  if (sizeof(I) == 2) {
    // the set's least column: lane groups c < 3 hold every step, the fourth
    // repeats some
    c0 = col[0];
    for (int u = 1; u < 8; u++) c0 = min(c0, col[u]);
    for (int o = 4; o < 64; o <<= 1) c0 = min(c0, __shfl_xor(c0, o));  // over the lanes of set b
  }
  if (rec) {
    SetRec *r = rec + w0 + q;
    if (lane == 0) {
      r->base = base;
      r->len = len;
      r->row0 = g * 64;
      for (int j = 0; j < 8; j++) r->first[j] = (uint8_t)(j < 5 ? first[j] : 64);
    }
    if (lane < 4) r->col0[lane] = c0;
  }
  if (c < kMaxChunks) {
    I *dst = out + (((int64_t)(w0 + q) * kMaxChunks + c) * 16 + kb) * 8;
#pragma unroll
    for (int u = 0; u < 8; u++) dst[u] = u < kSetChunk && c < nc ? (I)(col[u] - c0) : (I)0;
  }
}

using SetFn = void (*)(const SpmvArgs &, const SetArgs &, dim3, int32_t, int32_t, int32_t, hipStream_t);

template <class P, int OUT, int E, class I>
void launch_set(const SpmvArgs &a, const SetArgs &w, dim3 grid, int32_t nwork, int32_t ntiles, int32_t remap,
                hipStream_t s) {
  hipLaunchKernelGGL((spmv_rowset_kernel<P, OUT, E, I>), grid, dim3(kSetBlock * 64), 0, s, a, w, nwork, ntiles,
                     remap);
}

template <class P, int OUT, class I>
SetFn pick_set_e(int e) {
  if (e == 1) return &launch_set<P, OUT, 1, I>;
  if (e == 2) return &launch_set<P, OUT, 2, I>;
  return &launch_set<P, OUT, 4, I>;
}

template <class P, int OUT>
SetFn pick_set_i(int e, bool narrow) {
  return narrow ? pick_set_e<P, OUT, uint16_t>(e) : pick_set_e<P, OUT, int32_t>(e);
}

// e: right-hand sides per lane, a quarter of the k-tile (1, 2 or 4).  Kr columns
// are always int32: a set's span reaches over the whole numbering.
SetFn pick_set(int prec, int out, int e, bool narrow) {
  if (prec == 0) {
    if (out == OUT_RUN) return pick_set_i<PF64, OUT_RUN>(e, narrow);
    if (out == OUT_RUNX) return pick_set_e<PF64, OUT_RUNX, int32_t>(e);
    return pick_set_i<PF64, OUT_RESID>(e, narrow);
  }
  if (out == OUT_RUNX) return pick_set_e<PF32D, OUT_RUNX, int32_t>(e);
  return pick_set_i<PF32D, OUT_RUN>(e, narrow);
}

// Row sets pay where they hold at least this many rows on average: a matrix
// instruction computes four rows per set whether or not the set has them.
constexpr double kSetRows = 2.0;

}  // namespace

bool launch_rowsets(const DevLayout &D, int prec, int out, const SpmvArgs &a0, int32_t k, int32_t remap,
                    hipStream_t stream) {
  const bool kr = out == OUT_RUNX;
  if (!D.rs_waves || D.win_max <= 0 || prec == 1 || !row_sets_take(D, k) || (kr && !D.rs_cols_kr)) return false;
  SpmvArgs a = a0;
  if (!row_sets_reach(D, prec == 0 ? WK_F64 : WK_F32, a.ldx)) return false;
  // Tiles of 4, 8 or 16 columns.  The widest that k fills: it costs one pass
  // over a wave's columns, and 16 FP64 values are a whole 128-byte line of x
  // (hex elasticity 64^3 k=32, 16-column tiles 382 us, 8-column ones 506).
  const int e = k <= 4 ? 1 : k <= 8 ? 2 : 4;
  SetFn fn = pick_set(prec, out, e, D.rs_narrow);
  const SetArgs w{static_cast<const SetRec *>(D.rs_rec), kr ? D.rs_cols_kr : D.rs_cols, D.rs_waves};
  const int32_t ntiles = (k + 4 * e - 1) / (4 * e);
  const int64_t nwork = ((int64_t)D.rs_waves + kSetBlock - 1) / kSetBlock;
  const int64_t nfill = ((int64_t)D.nrows - D.nznrows + kSetBlock * 64 - 1) / (kSetBlock * 64);
  if (nwork + nfill > INT32_MAX) fail(WK_ERR_LIMIT, "grid too large");
  a.k = k;
  fn(a, w, dim3((uint32_t)(nwork + nfill)), (int32_t)nwork, ntiles, remap, stream);
  hip_check(hipGetLastError(), "spmv launch");
  return true;
}

bool row_sets_begin(DevLayout &D, uint64_t *starts, uint32_t *span, hipStream_t stream) {
  D.rs_waves = 0;
  const int32_t G = D.ngroups;
  if (D.variant != 1 || D.W != 64 || D.win_max <= 0 || G <= 0 || !D.cols) return false;
  // (a group without steps, which only arrays from elsewhere can hold, has no last
  // step to repeat)
  for (int32_t g = 0; g < G; g++)
    if (!D.h_max_nz_rows[g] || set_chunks((int32_t)D.h_max_nz_rows[g]) > kMaxChunks) return false;
  const int64_t blocks = ((int64_t)G + kBuildWaves - 1) / kBuildWaves;
  hipLaunchKernelGGL(row_set_kernel, dim3((uint32_t)blocks), dim3(kBuildWaves * 64), 0, stream, D.cols,
                     D.cols_kr, D.warp_offsets, D.max_nz_rows, G, starts, span);
  hip_check(hipGetLastError(), "row set launch");
  return true;
}

void row_sets_finish(wk_engine *E, DevLayout &D, const uint64_t *starts, uint32_t *span, const uint64_t *hs,
                     const uint32_t *hw, hipStream_t stream) {
  const int32_t G = D.ngroups;
  std::vector<uint32_t> woff((size_t)G + 1, 0);
  int64_t sets = 0, waves = 0;
  uint32_t widest = 0;
  int most = 0;  // waves of one group
  for (int32_t g = 0; g < G; g++) {
    // (lanes past the last row hold no set)
    const int32_t rows = std::min(64, D.nznrows - 64 * g);
    const int n = __builtin_popcountll(hs[g] & (~0ull >> (64 - rows)));
    sets += n;
    waves += (n + 3) / 4;
    most = std::max(most, (n + 3) / 4);
    widest = std::max(widest, hw[g]);
    woff[g + 1] = (uint32_t)waves;
  }
  if (waves > INT32_MAX / 64 || (double)D.nznrows < kSetRows * (double)sets) return;
  D.rs_narrow = widest <= 65535;
  hip_check(hipMemcpyAsync(span, woff.data(), 4 * woff.size(), hipMemcpyHostToDevice, stream), "row sets");
  // records, columns and Kr columns in one allocation
  const size_t n = (size_t)waves * kMaxChunks * 128;
  const size_t rec_bytes = sizeof(SetRec) * (size_t)waves, col_bytes = n * (D.rs_narrow ? 2 : 4);
  char *mem = dev_alloc<char>(E, (int64_t)(rec_bytes + col_bytes + (D.cols_kr ? 4 * n : 0)));
  SetRec *rec = reinterpret_cast<SetRec *>(mem);
  D.rs_rec = rec;
  D.rs_cols = mem + rec_bytes;
  const dim3 grid((uint32_t)G), block(64 * (uint32_t)most);
  if (D.rs_narrow)
    hipLaunchKernelGGL(row_set_cols_kernel<uint16_t>, grid, block, 0, stream, D.cols, D.warp_offsets, D.max_nz_rows,
                       starts, span, static_cast<uint16_t *>(D.rs_cols), rec);
  else
    hipLaunchKernelGGL(row_set_cols_kernel<int32_t>, grid, block, 0, stream, D.cols, D.warp_offsets, D.max_nz_rows,
                       starts, span, static_cast<int32_t *>(D.rs_cols), rec);
  hip_check(hipGetLastError(), "row set launch");
  if (D.cols_kr) {
    D.rs_cols_kr = mem + rec_bytes + col_bytes;
    hipLaunchKernelGGL(row_set_cols_kernel<int32_t>, grid, block, 0, stream, D.cols_kr, D.warp_offsets,
                       D.max_nz_rows, starts, span, static_cast<int32_t *>(D.rs_cols_kr), nullptr);
    hip_check(hipGetLastError(), "row set launch");
  }
  // woff goes, and the engine may be used on another stream
  hip_check(hipStreamSynchronize(stream), "row sets");
  D.rs_waves = (int32_t)waves;
}

}  // namespace wk
