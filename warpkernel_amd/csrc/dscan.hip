// dscan.hip -- the scan/process step on the GPU: a device CSR becomes an
// engine without the matrix visiting the host.
//
// The result is the layout of structure::scan / structure2::scan
// (warpkernel.hpp:309-365, 578-736) at group width 64 and the padded arrays of
// process (hpp:379-398, 749-769), bit for bit the host scan's; only the way
// they are computed differs:
//   1. one pass checks the CSR (rowptr monotone from 0 to nnz, columns in
//      range) and finds the longest row; nothing else runs on a malformed CSR;
//   2. per block of rows (one wave), a histogram of row lengths in LDS; the
//      histograms in (length descending, block ascending) order are
//      prefix-summed on the host: the start of every (length, block) run of
//      the sorted order;
//   3. each block walks its rows in order, 64 at a time, and ranks the rows of
//      one length with ballots, so placement is stable: length descending, row
//      ascending (checkPairOrder, hpp:222-225);
//   4. the longest row of each group comes back to the host (G values), where
//      WPK2's split rule (shared with the host scan) and the group offsets are
//      computed; one kernel then writes the padded values, columns, Kr columns
//      and the CSR-to-slot map with coalesced stores.
// Limits: group width 64, rows of at most 8191 entries (the LDS histogram),
// no transposed layout (the adjoint engine is built by wk_engine_create).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "wk_internal.hpp"

namespace wk {
namespace {

constexpr int32_t kMaxLen = 8191;
constexpr int64_t kMaxCounts = int64_t(1) << 24;  // histogram entries, all blocks

// part[b] = longest row seen by block b, part[nb + b] = error bits
// (1: rowptr ends, 2: rowptr decreases, 4: column out of range)
__global__ __launch_bounds__(256) void csr_check_kernel(const int32_t *__restrict__ rowptr,
                                                        int32_t nrows,
                                                        const int32_t *__restrict__ colind,
                                                        int64_t nnz, int32_t ncols,
                                                        int32_t *__restrict__ part) {
  __shared__ int32_t red_max[256], red_bad[256];
  int32_t m = 0, bad = 0;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (int64_t r = t0; r < nrows; r += stride) {
    const int32_t len = rowptr[r + 1] - rowptr[r];
    if (len < 0) bad |= 2;
    m = max(m, len);
  }
  // four columns a load where colind allows it (hex elasticity 40^3, 16M columns,
  // 32 -> 16 us)
  const int64_t n4 = ((uintptr_t)colind & 15) == 0 ? nnz / 4 : 0;
  const int4 *c4 = reinterpret_cast<const int4 *>(colind);
#pragma unroll 4
  for (int64_t e = t0; e < n4; e += stride) {
    const int4 c = c4[e];
    const uint32_t most = max(max((uint32_t)c.x, (uint32_t)c.y), max((uint32_t)c.z, (uint32_t)c.w));
    if (most >= (uint32_t)ncols) bad |= 4;
  }
  for (int64_t e = 4 * n4 + t0; e < nnz; e += stride)
    if ((uint32_t)colind[e] >= (uint32_t)ncols) bad |= 4;
  if (t0 == 0 && (rowptr[0] != 0 || (int64_t)rowptr[nrows] != nnz)) bad |= 1;
  red_max[threadIdx.x] = m;
  red_bad[threadIdx.x] = bad;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      red_max[threadIdx.x] = max(red_max[threadIdx.x], red_max[threadIdx.x + o]);
      red_bad[threadIdx.x] |= red_bad[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[blockIdx.x] = red_max[0];
    part[gridDim.x + blockIdx.x] = red_bad[0];
  }
}

// counts[(maxlen - len) * nblk + b] = rows of length len among block b's rows
__global__ __launch_bounds__(64) void len_hist_kernel(const int32_t *__restrict__ rowptr,
                                                      int32_t nrows, int32_t rpb, int32_t maxlen,
                                                      int32_t nblk, int32_t *__restrict__ counts) {
  extern __shared__ int32_t hist[];
  const int32_t b = blockIdx.x;
  for (int32_t l = threadIdx.x; l <= maxlen; l += 64) hist[l] = 0;
  __syncthreads();
  const int64_t r0 = (int64_t)b * rpb;
  for (int32_t t = threadIdx.x; t < rpb; t += 64) {
    const int64_t r = r0 + t;
    if (r < nrows) atomicAdd(&hist[rowptr[r + 1] - rowptr[r]], 1);
  }
  __syncthreads();
  for (int32_t l = threadIdx.x; l <= maxlen; l += 64)
    counts[(int64_t)(maxlen - l) * nblk + b] = hist[l];
}

// Stable placement: starts[(maxlen - len) * nblk + b] is the sorted position
// of block b's first row of length len.  One wave per block; per chunk of 64
// rows, one round per distinct length among them.
__global__ __launch_bounds__(64) void place_kernel(const int32_t *__restrict__ rowptr,
                                                   int32_t nrows, int32_t rpb, int32_t maxlen,
                                                   int32_t nblk, const int32_t *__restrict__ starts,
                                                   int32_t *__restrict__ row_map,
                                                   int32_t *__restrict__ row_map_inv,
                                                   uint32_t *__restrict__ slen) {
  extern __shared__ int32_t next[];  // next free sorted position per length
  const int32_t b = blockIdx.x;
  const int32_t lane = threadIdx.x;
  for (int32_t l = lane; l <= maxlen; l += 64) next[l] = starts[(int64_t)(maxlen - l) * nblk + b];
  __syncthreads();
  const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;  // lanes under this one
  for (int32_t c = 0; c < rpb; c += 64) {
    const int64_t r = (int64_t)b * rpb + c + lane;
    const int32_t len = r < nrows ? rowptr[r + 1] - rowptr[r] : -1;
    bool pending = r < nrows;
    uint64_t act;
    while ((act = __ballot(pending)) != 0) {
      const int32_t src = __ffsll((unsigned long long)act) - 1;
      const int32_t v = __shfl(len, src);  // this round's length, wave-uniform
      const bool mine = pending && len == v;
      const uint64_t same = __ballot(mine);
      const int32_t base = next[v];
      if (mine) {
        const int32_t pos = base + (int32_t)__popcll(same & below);
        row_map[pos] = (int32_t)r;
        row_map_inv[r] = pos;
        slen[pos] = (uint32_t)len;
        pending = false;
      }
      __builtin_amdgcn_wave_barrier();
      if (lane == src) next[v] = base + (int32_t)__popcll(same);
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// aw[g] = length of sorted row 64 g, the longest of group g; aw[ngroups] that of
// the last nonempty row, the shortest
__global__ __launch_bounds__(256) void group_len_kernel(const uint32_t *__restrict__ slen,
                                                        int32_t ngroups, int32_t nznrows,
                                                        uint32_t *__restrict__ aw) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g <= ngroups) aw[g] = slen[g < ngroups ? g * 64 : nznrows - 1];
}

// One block per (sub-)group w: lane l holds chunk l % tpr of sorted row
// row_off[w] + l / tpr (WPK1: tpr 1, rows 64 w + l); its slots are
// warp_offsets[w] + l + 64 i, i < A_w; slots past the chunk are pads (0, col 0).
// The rows' entries are read kFillSteps at a time, 256 bytes of values per row
// together, turned around in LDS and written a step (64 slots) at a time, so
// reads, padded arrays and the CSR-to-slot map are all whole lines.  (A lane
// per row walking its own entries read 64 scattered lines per load and wrote
// the map 4 bytes to a line: hex elasticity 40^3, 16M entries, 725 us against
// 107.)
constexpr int kFillSteps = 32;
constexpr int kFillThreads = 256;

template <class T>
__global__ __launch_bounds__(kFillThreads) void fill_kernel(
    const int32_t *__restrict__ rowptr, const int32_t *__restrict__ colind,
    const double *__restrict__ vals, const int32_t *__restrict__ row_map,
    const int32_t *__restrict__ row_map_inv, const int64_t *__restrict__ wo,
    const uint32_t *__restrict__ aw, const uint32_t *__restrict__ tpr_a,
    const uint32_t *__restrict__ row_off, int32_t nznrows, T *__restrict__ pv,
    int32_t *__restrict__ pc, int32_t *__restrict__ pkr, uint32_t *__restrict__ slot_of_nz,
    int2 *__restrict__ lane_src) {
  constexpr int PER = kFillSteps * 64 / kFillThreads;
  __shared__ int32_t first[64], count[64];        // each lane's first CSR entry, entries
  __shared__ T sv[64][kFillSteps + 1];            // odd row length: the turned reads spread
  __shared__ int32_t sc[64][kFillSteps + 1];
  const int32_t w = blockIdx.x;
  const int32_t tid = threadIdx.x;
  const uint32_t A = aw[w];
  if (tid < 64) {
    const uint32_t tpr = tpr_a ? tpr_a[w] : 1u;
    const uint32_t p = (tpr_a ? row_off[w] : (uint32_t)w * 64u) + (uint32_t)tid / tpr;
    const uint32_t chunk = (uint32_t)tid & (tpr - 1);
    int32_t rb = 0, n = 0;
    if (p < (uint32_t)nznrows) {
      const int32_t r = row_map[p];
      const int32_t b1 = rowptr[r + 1];
      rb = rowptr[r] + (int32_t)(chunk * A);
      n = max(0, min(b1 - rb, (int32_t)A));
    }
    first[tid] = rb;
    count[tid] = n;
    lane_src[(int64_t)w * 64 + tid] = int2{rb, n};
  }
  __syncthreads();
  const int64_t base = wo[w];
  for (uint32_t i0 = 0; i0 < A; i0 += kFillSteps) {
    T v[PER];
    int32_t c[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) {
      const int32_t l = (tid + j * kFillThreads) / kFillSteps;
      const int32_t i = (int32_t)i0 + tid % kFillSteps;
      v[j] = T(0);
      c[j] = 0;
      if (i < count[l]) {
        const int32_t e = first[l] + i;
        v[j] = (T)vals[e];
        c[j] = colind[e];
        slot_of_nz[e] = (uint32_t)(base + l + 64 * (int64_t)i);
      }
    }
#pragma unroll
    for (int j = 0; j < PER; j++) {
      const int32_t l = (tid + j * kFillThreads) / kFillSteps;
      sv[l][tid % kFillSteps] = v[j];
      sc[l][tid % kFillSteps] = c[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PER; j++) {
      const int32_t l = tid & 63, t = (tid + j * kFillThreads) >> 6;
      const uint32_t i = i0 + (uint32_t)t;
      if (i < A) {
        const int64_t slot = base + l + 64 * (int64_t)i;
        const int32_t col = sc[l][t];
        pv[slot] = sv[l][t];
        pc[slot] = col;
        if (pkr) pkr[slot] = (int32_t)i < count[l] ? row_map_inv[col] : 0;
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------- x windows
// The windows of build_windows (scan.cpp), built on the device, one block per
// group: the distinct slot keys (the entry's column, -1 for a pad) in ascending
// order, and each slot's position among them.
//
// Where the group's columns span at most kWinBits (every banded ordering) they are
// read once, into registers, set bits of an LDS bitmap, and a key's position is the
// number of bits below its own: the words' running counts plus one popcount
// (window_kernel; spans of at most kBandBits first, with 12 KB of LDS and so the
// occupancy of the registers, then the others).  Wider groups sort their keys in
// LDS (window_sort_kernel).  The keys go to a stash, since where they belong is
// known only when every group has been counted; window_place_kernel copies them
// there.  Hex elasticity 40^3, 3,231 groups of 5,184 slots: sorting every group,
// once to count and once to write, took 1.01 + 1.38 ms; the bitmap in two such
// passes, which read the columns five times, 88 + 117 us; 52 + 24 us here, and 7 to place.  Groups of
// more than kWinSlots slots are not handled: the engine then has no windows.
constexpr int32_t kWinSlots = 8192;
constexpr int32_t kWinBits = kWinSlots * 32;  // the bitmap takes the sort's LDS
constexpr int32_t kBandBits = 65536;
constexpr int kWinThreads = 256;

struct WinBuild {
  const int32_t *rowptr, *row_map, *row_map_inv, *cols;
  const int64_t *wo;
  const uint32_t *aw, *tpr, *row_off;
  int32_t nznrows;
};

// Entries of each lane of group g (the fill kernel's chunk rule).
__device__ void lane_entries(const WinBuild &b, int32_t g, int32_t *lane_n) {
  const int32_t tid = threadIdx.x;
  if (tid < 64) {
    const uint32_t A = b.aw[g];
    const uint32_t tpr = b.tpr ? b.tpr[g] : 1u;
    const uint32_t p = (b.tpr ? b.row_off[g] : (uint32_t)g * 64u) + (uint32_t)tid / tpr;
    const uint32_t chunk = (uint32_t)tid & (tpr - 1);
    int32_t n = 0;
    if (p < (uint32_t)b.nznrows) {
      const int32_t r = b.row_map[p];
      const int32_t rb = b.rowptr[r] + (int32_t)(chunk * A);
      n = max(0, min(b.rowptr[r + 1] - rb, (int32_t)A));
    }
    lane_n[tid] = n;
  }
  __syncthreads();
}

// Sorted keys of group g in keys[0, N) (INT_MAX past the S slots).
__device__ void sort_group_keys(const WinBuild &b, int32_t g, int32_t S, int32_t *keys,
                                const int32_t *lane_n, int32_t &N) {
  const int32_t tid = threadIdx.x;
  N = 64;
  while (N < S) N <<= 1;
  const int64_t base = b.wo[g];
  for (int32_t t = tid; t < N; t += kWinThreads)
    keys[t] = t < S ? ((t >> 6) < lane_n[t & 63] ? b.cols[base + t] : -1) : INT32_MAX;
  __syncthreads();
  for (int32_t k = 2; k <= N; k <<= 1)
    for (int32_t j = k >> 1; j > 0; j >>= 1) {
      for (int32_t t = tid; t < N; t += kWinThreads) {
        const int32_t o = t ^ j;
        if (o > t) {
          const int32_t a = keys[t], c = keys[o];
          if ((a > c) == ((t & k) == 0)) {
            keys[t] = c;
            keys[o] = a;
          }
        }
      }
      __syncthreads();
    }
}

// The least and greatest column of the group's entries and whether it has a
// pad, over the whole block (red: kWinThreads ints).
struct Span {
  int32_t lo, hi, pad;
};
__device__ Span block_span(int32_t lo, int32_t hi, int32_t pad, int32_t *red) {
  const int32_t tid = threadIdx.x;
  for (int o = 32; o > 0; o >>= 1) {
    lo = min(lo, __shfl_xor(lo, o));
    hi = max(hi, __shfl_xor(hi, o));
    pad |= __shfl_xor(pad, o);
  }
  if ((tid & 63) == 0) {
    red[tid >> 6] = lo;
    red[8 + (tid >> 6)] = hi;
    red[16 + (tid >> 6)] = pad;
  }
  __syncthreads();
  for (int w = 0; w < kWinThreads / 64; w++) {
    lo = min(lo, red[w]);
    hi = max(hi, red[8 + w]);
    pad |= red[16 + w];
  }
  __syncthreads();
  return {lo, hi, pad};
}

// Inclusive sum of every thread's c over the block; total: the whole sum (red:
// kWinThreads / 64 ints, free again after the next barrier).
__device__ int32_t block_scan(int32_t c, int32_t *red, int32_t &total) {
  const int32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int o = 1; o < 64; o <<= 1) {
    const int32_t v = __shfl_up(c, o);
    if (lane >= o) c += v;
  }
  if (lane == 63) red[wave] = c;
  __syncthreads();
  total = 0;
  for (int w = 0; w < kWinThreads / 64; w++) {
    if (w < wave) c += red[w];
    total += red[w];
  }
  return c;
}

// count[g]: distinct keys, -1 where they are more than kMaxWindow, kWide where the
// columns span more than BITS.  stash[g][stride]: the keys.  R: slots of a thread,
// kWinThreads R at least the longest group's.  The kernel for more than kBandBits
// takes only the groups that the one before it has marked.
constexpr int32_t kWide = -2;
template <int R, int BITS>
__global__ __launch_bounds__(kWinThreads) void window_kernel(WinBuild b, int32_t stride,
                                                             int32_t *__restrict__ count,
                                                             int32_t *__restrict__ stash,
                                                             uint16_t *__restrict__ win_idx) {
  __shared__ uint32_t bits[BITS / 32];
  __shared__ uint16_t below[BITS / 32];  // bits in the words before
  __shared__ int32_t lane_n[64];
  __shared__ int32_t red[32];
  const int32_t g = blockIdx.x;
  const int32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (BITS > kBandBits && count[g] != kWide) return;
  const int32_t A = (int32_t)b.aw[g];
  const int64_t base = b.wo[g] + tid;
  int32_t c[R];
#pragma unroll
  for (int j = 0; j < R; j++) c[j] = wave + 4 * j < A ? b.cols[base + kWinThreads * j] : 0;
  lane_entries(b, g, lane_n);
  const int32_t n = lane_n[lane];
  int32_t lo = INT32_MAX, hi = -1, pad = 0;
#pragma unroll
  for (int j = 0; j < R; j++) {
    const int32_t i = wave + 4 * j;
    if (i < n) {
      lo = min(lo, c[j]);
      hi = max(hi, c[j]);
    } else if (i < A) {
      pad = 1;
    }
  }
  const Span sp = block_span(lo, hi, pad, red);
  if (sp.hi - sp.lo >= BITS) {
    if (tid == 0) count[g] = kWide;
    return;
  }
  const int32_t words = sp.hi < sp.lo ? 0 : (sp.hi - sp.lo + 32) >> 5;
  for (int32_t t = tid; t < words; t += kWinThreads) bits[t] = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < R; j++)
    if (wave + 4 * j < n) {
      const uint32_t k = (uint32_t)(c[j] - sp.lo), bit = 1u << (k & 31);
      // most columns come from several slots: only the first pay the atomic
      if (!(bits[k >> 5] & bit)) atomicOr(&bits[k >> 5], bit);
    }
  __syncthreads();
  const int32_t per = ((words + kWinThreads - 1) / kWinThreads) | 1;  // odd: no bank conflicts
  const int32_t t0 = min(words, tid * per), t1 = min(words, t0 + per);
  int32_t sum = 0, total;
  for (int32_t t = t0; t < t1; t++) sum += __popc(bits[t]);
  int32_t rank = block_scan(sum, red, total) - sum + sp.pad;  // a pad's key is the first
  total += sp.pad;
  if (tid == 0) count[g] = total > kMaxWindow ? -1 : total;
  if (total > kMaxWindow) return;
  int32_t *keys = stash + (int64_t)g * stride;
  if (tid == 0 && sp.pad) keys[0] = -1;
  for (int32_t t = t0; t < t1; t++) {
    below[t] = (uint16_t)rank;
    for (uint32_t m = bits[t]; m; m &= m - 1) keys[rank++] = sp.lo + 32 * t + (__ffs((int)m) - 1);
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < R; j++) {
    const int32_t i = wave + 4 * j;
    if (i < A) {
      int32_t p = 0;
      if (i < n) {
        const uint32_t k = (uint32_t)(c[j] - sp.lo);
        p = below[k >> 5] + __popc(bits[k >> 5] & ((1u << (k & 31)) - 1u));
      }
      win_idx[base + kWinThreads * j] = (uint16_t)p;
    }
  }
}

// The groups that are still marked.
__global__ __launch_bounds__(kWinThreads) void window_sort_kernel(WinBuild b, int32_t stride,
                                                                  int32_t *__restrict__ count,
                                                                  int32_t *__restrict__ stash,
                                                                  uint16_t *__restrict__ win_idx) {
  __shared__ int32_t keys[kWinSlots];
  __shared__ int32_t uniq[kMaxWindow];
  __shared__ int32_t lane_n[64];
  __shared__ int32_t red[32];
  const int32_t g = blockIdx.x;
  const int32_t tid = threadIdx.x;
  if (count[g] != kWide) return;
  const int32_t S = (int32_t)b.aw[g] * 64;  // at most kWinSlots
  const int64_t base = b.wo[g];
  lane_entries(b, g, lane_n);
  int32_t N = 0, n;  // the keys in LDS: S rounded up to a power of two
  sort_group_keys(b, g, S, keys, lane_n, N);
  // ranks of the distinct keys: each thread counts a contiguous chunk of the
  // sorted keys, then an inclusive scan of the chunk counts
  const int32_t per = N / kWinThreads > 0 ? N / kWinThreads : 1;
  const int32_t t0 = min(N, tid * per), t1 = min(N, t0 + per);
  int32_t c = 0;
  for (int32_t t = t0; t < t1; t++) c += keys[t] != INT32_MAX && (t == 0 || keys[t] != keys[t - 1]);
  int32_t rank = block_scan(c, red, n) - c;
  if (tid == 0) count[g] = n > kMaxWindow ? -1 : n;
  if (n > kMaxWindow) return;
  for (int32_t t = t0; t < t1; t++) {
    const int32_t k = keys[t];
    if (k != INT32_MAX && (t == 0 || k != keys[t - 1])) {
      uniq[rank] = k;
      stash[(int64_t)g * stride + rank] = k;
      rank++;
    }
  }
  __syncthreads();
  // each slot's position among the distinct keys (ascending; a pad's key -1,
  // when present, is the first)
  for (int32_t t = tid; t < S; t += kWinThreads) {
    const int32_t key = (t >> 6) < lane_n[t & 63] ? b.cols[base + t] : -1;
    int32_t lo = 0, hi = n;
    while (lo < hi) {
      const int32_t mid = (lo + hi) >> 1;
      if (uniq[mid] < key)
        lo = mid + 1;
      else
        hi = mid;
    }
    win_idx[base + t] = (uint16_t)lo;
  }
}

__global__ __launch_bounds__(kWinThreads) void window_place_kernel(const int32_t *__restrict__ stash, int32_t stride,
                                                                   const uint32_t *__restrict__ off,
                                                                   const int32_t *__restrict__ row_map_inv,
                                                                   int32_t *__restrict__ win_cols,
                                                                   int32_t *__restrict__ win_cols_kr) {
  const int32_t g = blockIdx.x;
  const uint32_t w0 = off[g], n = off[g + 1] - w0;
  for (uint32_t t = threadIdx.x; t < n; t += kWinThreads) {
    const int32_t k = stash[(int64_t)g * stride + t];
    win_cols[w0 + t] = k < 0 ? 0 : k;
    if (win_cols_kr) win_cols_kr[w0 + t] = k < 0 ? 0 : row_map_inv[k];
  }
}

template <int R>
void launch_windows(const WinBuild &b, int32_t ngroups, int32_t ncols, int32_t stride, int32_t *count,
                    int32_t *stash, uint16_t *win_idx, hipStream_t s) {
  const dim3 grid((uint32_t)ngroups), block(kWinThreads);
  hipLaunchKernelGGL((window_kernel<R, kBandBits>), grid, block, 0, s, b, stride, count, stash, win_idx);
  if (ncols > kBandBits)
    hipLaunchKernelGGL((window_kernel<R, kWinBits>), grid, block, 0, s, b, stride, count, stash, win_idx);
  if (ncols > kWinBits)
    hipLaunchKernelGGL(window_sort_kernel, grid, block, 0, s, b, stride, count, stash, win_idx);
  hip_check(hipGetLastError(), "windows");
}

template <class T>
std::vector<T> download(const T *d, int64_t n, hipStream_t s) {
  std::vector<T> h((size_t)n);
  if (n) {
    hip_check(hipMemcpyAsync(h.data(), d, sizeof(T) * (size_t)n, hipMemcpyDeviceToHost, s),
              "download");
    hip_check(hipStreamSynchronize(s), "download");
  }
  return h;
}

template <class T>
void launch_fill(const DevLayout &D, const int32_t *rowptr, const int32_t *colind,
                 const double *vals, hipStream_t s) {
  if (!D.ngroups) return;
  hipLaunchKernelGGL(fill_kernel<T>, dim3((uint32_t)D.ngroups), dim3(kFillThreads), 0, s, rowptr,
                     colind, vals, D.row_map, D.row_map_inv, D.warp_offsets, D.max_nz_rows, D.tpr,
                     D.row_off, D.nznrows, static_cast<T *>(D.vals), D.cols, D.cols_kr, D.slot_of_nz,
                     reinterpret_cast<int2 *>(D.lane_src));
  hip_check(hipGetLastError(), "fill");
}

// Device memory for a part of the scan, given back at its end; idle: nothing uses
// it any more (on an error its kernels may still run).
struct Stash {
  int device;
  size_t bytes;
  int32_t *p;
  bool idle = false;
  Stash(int dev, size_t n)
      : device(dev), bytes(n), p(n ? static_cast<int32_t *>(block_take(bytes)) : nullptr) {}
  ~Stash() {
    if (!p) return;
    if (!idle) (void)hipDeviceSynchronize();
    block_give(device, p, bytes);
  }
  Stash(const Stash &) = delete;
  Stash &operator=(const Stash &) = delete;
};

// Scan + process of one device CSR into E->fwd.
void device_scan(wk_engine *E, int32_t variant, int32_t threshold, int32_t max_tpr, bool kr,
                 const int32_t *rowptr, const int32_t *colind, const double *vals,
                 hipStream_t s) {
  const int32_t nrows = E->nrows, ncols = E->ncols;
  const int64_t nnz = E->nnz;
  DevLayout &D = E->fwd;
  D.variant = variant;
  D.W = 64;
  D.nrows = nrows;
  D.ncols = ncols;

  // 1. check the CSR, find the longest row
  const int64_t work = std::max<int64_t>(nrows, nnz);
  const int32_t nb = (int32_t)std::min<int64_t>(std::max<int64_t>((work + 1023) / 1024, 1), 1024);
  int32_t *part = dev_alloc<int32_t>(E, 2 * (int64_t)nb);
  hipLaunchKernelGGL(csr_check_kernel, dim3(nb), dim3(256), 0, s, rowptr, nrows, colind, nnz,
                     ncols, part);
  hip_check(hipGetLastError(), "csr_check");
  const std::vector<int32_t> hp = download(part, 2 * (int64_t)nb, s);
  int32_t maxlen = 0, bad = 0;
  for (int32_t b = 0; b < nb; b++) {
    maxlen = std::max(maxlen, hp[b]);
    bad |= hp[nb + b];
  }
  if (bad & 1) fail(WK_ERR_CSR, "rowptr must start at 0 and end at nnz");
  if (bad & 2) fail(WK_ERR_CSR, "rowptr decreases");
  if (bad & 4) fail(WK_ERR_CSR, "column index out of range");
  if (maxlen > kMaxLen)
    fail(WK_ERR_LIMIT, "rows longer than " + std::to_string(kMaxLen) +
                           " entries: scan on the host (wk_scan1 / wk_scan2)");
  if (nrows == 0) return;

  // 2. histograms of row lengths per block; run starts
  int32_t rpb = 1024;
  while ((int64_t)(maxlen + 1) * ((nrows + (int64_t)rpb - 1) / rpb) > kMaxCounts) rpb *= 2;
  const int32_t nblk = (int32_t)((nrows + (int64_t)rpb - 1) / rpb);
  const int64_t ncount = (int64_t)(maxlen + 1) * nblk;
  const size_t lds = sizeof(int32_t) * (size_t)(maxlen + 1);
  D.row_map = dev_alloc<int32_t>(E, nrows);
  D.row_map_inv = dev_alloc<int32_t>(E, nrows);
  uint32_t *slen = dev_alloc<uint32_t>(E, nrows);
  int32_t *counts = dev_alloc<int32_t>(E, ncount);
  hipLaunchKernelGGL(len_hist_kernel, dim3(nblk), dim3(64), lds, s, rowptr, nrows, rpb, maxlen,
                     nblk, counts);
  hip_check(hipGetLastError(), "len_hist");
  std::vector<int32_t> starts = download(counts, ncount, s);
  int64_t acc = 0;
  for (int64_t t = 0; t < ncount; t++) {
    const int32_t c = starts[t];
    starts[t] = (int32_t)acc;
    acc += c;
  }
  if (acc != nrows) fail(WK_ERR_STATE, "row histogram does not add up to nrows");
  // rows of length 0 form the last run
  const int32_t nznrows = starts[(int64_t)maxlen * nblk];
  hip_check(hipMemcpyAsync(counts, starts.data(), sizeof(int32_t) * (size_t)ncount,
                           hipMemcpyHostToDevice, s),
            "upload");
  hipLaunchKernelGGL(place_kernel, dim3(nblk), dim3(64), lds, s, rowptr, nrows, rpb, maxlen, nblk,
                     counts, D.row_map, D.row_map_inv, slen);
  hip_check(hipGetLastError(), "place");
  D.nznrows = nznrows;

  // 3. groups and their split
  const int32_t G0 = (nznrows + 63) / 64;
  std::vector<uint32_t> aw0;
  uint32_t shortest = 0;
  if (G0) {
    uint32_t *daw = dev_alloc<uint32_t>(E, (int64_t)G0 + 1);
    hipLaunchKernelGGL(group_len_kernel, dim3((uint32_t)(G0 / 256 + 1)), dim3(256), 0, s, slen,
                       G0, nznrows, daw);
    hip_check(hipGetLastError(), "group_len");
    aw0 = download(daw, (int64_t)G0 + 1, s);
    shortest = aw0.back();
    aw0.pop_back();
  }
  std::vector<uint32_t> A, rows_nominal, rows_actual;
  if (variant == 2)
    split_groups(aw0, nznrows, 64, threshold, max_tpr, A, rows_nominal, rows_actual);
  else
    A = aw0;
  const int32_t G = (int32_t)A.size();
  std::vector<int64_t> wo((size_t)G + 1, 0);
  for (int32_t g = 0; g < G; g++) wo[g + 1] = wo[g] + (int64_t)A[g] * 64;
  if (wo[G] > (int64_t)UINT32_MAX) fail(WK_ERR_LIMIT, "padded layout exceeds 2^32 slots");
  D.ngroups = G;
  D.allocate_nz = wo[G];
  D.h_max_nz_rows = A;
  D.warp_offsets = dev_upload(E, wo.data(), (int64_t)wo.size(), s);
  D.max_nz_rows = dev_upload(E, A.data(), G, s);
  std::vector<uint32_t> tpr, roff;  // (uploads: alive until the next wait)
  if (variant == 2) {
    tpr.resize((size_t)G);
    roff.assign((size_t)G + 1, 0);
    for (int32_t w = 0; w < G; w++) {
      tpr[w] = 64u / rows_nominal[w];
      roff[w + 1] = roff[w] + rows_actual[w];
    }
    roff[G] = (uint32_t)nrows;  // sentinel (hpp:716)
    D.tpr = dev_upload(E, tpr.data(), G, s);
    D.row_off = dev_upload(E, roff.data(), G + 1, s);
  }

  // 4. padded arrays and the CSR -> slot map
  D.cols = dev_alloc<int32_t>(E, D.allocate_nz);
  D.cols_kr = kr ? dev_alloc<int32_t>(E, D.allocate_nz) : nullptr;
  const int64_t even = nnz + (nnz & 1);  // (first entry, entries) pairs follow the map
  D.slot_of_nz = dev_alloc<uint32_t>(E, even + 128 * (int64_t)G);
  D.lane_src = reinterpret_cast<int32_t *>(D.slot_of_nz + even);
  if (E->dtype == WK_F64) {
    D.vals = dev_alloc<double>(E, D.allocate_nz);
    launch_fill<double>(D, rowptr, colind, vals, s);
  } else {
    D.vals = dev_alloc<float>(E, D.allocate_nz);
    launch_fill<float>(D, rowptr, colind, vals, s);
  }

  // 5. x windows, when every group fits
  const uint32_t longest = G ? *std::max_element(A.begin(), A.end()) : 0;
  D.longest = longest;
  const bool windows = G && (int64_t)longest * 64 <= kWinSlots;
  // the uploads' host arrays go, and the caller may use the engine on another
  // stream or free the CSR (with windows, their counts' download waits)
  if (!windows) hip_check(hipStreamSynchronize(s), "device scan");
  if (windows) {
    WinBuild wb{rowptr, D.row_map, D.row_map_inv, D.cols, D.warp_offsets, D.max_nz_rows,
                D.tpr, D.row_off, nznrows};
    const int32_t stride = std::min((int32_t)longest * 64, kMaxWindow);
    const int64_t keys = (int64_t)stride * G;
    const bool small = keys <= 65536;  // an allocation less
    // (counts: read and written before build_compact_columns takes them)
    int32_t *dcount = dev_alloc<int32_t>(E, compact_words(G) + (small ? keys : 0));
    Stash taken(E->device, small ? 0 : sizeof(int32_t) * (size_t)keys);
    int32_t *stash = small ? dcount + compact_words(G) : taken.p;
    uint16_t *idx = dev_alloc<uint16_t>(E, D.allocate_nz);
    const auto launch = longest <= 16   ? launch_windows<4>
                        : longest <= 32 ? launch_windows<8>
                        : longest <= 96 ? launch_windows<24>
                                        : launch_windows<32>;
    launch(wb, G, ncols, stride, dcount, stash, idx, s);
    const std::vector<int32_t> cnt = download(dcount, G, s);
    taken.idle = true;
    bool fits = true;
    std::vector<uint32_t> off((size_t)G + 1, 0);
    int32_t most = 0;
    for (int32_t g = 0; g < G && fits; g++) {
      if (cnt[g] < 0) fits = false;
      off[g + 1] = off[g] + (uint32_t)std::max(cnt[g], 0);
      most = std::max(most, cnt[g]);
    }
    if (fits) {
      D.win_off = dev_upload(E, off.data(), (int64_t)off.size(), s);
      D.win_cols = dev_alloc<int32_t>(E, off[G]);
      D.win_cols_kr = kr ? dev_alloc<int32_t>(E, off[G]) : nullptr;
      D.win_idx = idx;
      taken.idle = false;
      hipLaunchKernelGGL(window_place_kernel, dim3((uint32_t)G), dim3(kWinThreads), 0, s, stash, stride, D.win_off,
                         D.row_map_inv, D.win_cols, D.win_cols_kr);
      hip_check(hipGetLastError(), "window place");
      D.win_max = most;
      D.win_total = off[G];
      build_packed_positions(E, D, s);
      hip_check(hipStreamSynchronize(s), "window place");
      taken.idle = true;
      build_compact_columns(E, D, reinterpret_cast<uint32_t *>(dcount), s);
    } else {
      dev_give(E, idx);
    }
  }

  wk_layout_info &I = E->info;
  I.nznrows = nznrows;
  I.nwarps = G;
  I.allocate_nz = D.allocate_nz;
  if (variant == 2) {
    // min_nz starts at nrows (hpp:607)
    I.min_nz = nznrows ? std::min<uint32_t>(shortest, (uint32_t)nrows) : (uint32_t)nrows;
    I.max_nz = (uint32_t)maxlen;
  }
}

}  // namespace

}  // namespace wk

using namespace wk;

extern "C" int wk_engine_create_device(int32_t variant, int32_t threshold, int32_t max_tpr,
                                       int32_t nrows, int32_t ncols, int64_t nnz,
                                       const int32_t *rowptr_dev, const int32_t *colind_dev,
                                       const double *vals_dev, int32_t values_dtype,
                                       uint32_t flags, void *stream, wk_engine **out) {
  return guarded([&] {
    if (!out) fail(WK_ERR_ARG, "out is NULL");
    *out = nullptr;
    if (variant != 1 && variant != 2) fail(WK_ERR_ARG, "variant must be 1 or 2");
    if (nrows < 0 || ncols < 0) fail(WK_ERR_ARG, "negative matrix dimension");
    if (nnz < 0 || nnz > INT32_MAX) fail(WK_ERR_LIMIT, "nnz must be in [0, 2^31)");
    if (!rowptr_dev || (nnz && (!colind_dev || !vals_dev))) fail(WK_ERR_ARG, "NULL argument");
    if (values_dtype != WK_F64 && values_dtype != WK_F32) fail(WK_ERR_ARG, "unknown values dtype");
    if (flags & ~(uint32_t)WK_ENGINE_KR)
      fail(WK_ERR_ARG, "only WK_ENGINE_KR is supported here (the adjoint layout is built by "
                       "wk_engine_create)");
    const bool kr = flags & WK_ENGINE_KR;
    if (kr && nrows != ncols) fail(WK_ERR_ARG, "the Kr form needs a square matrix");
    if (variant == 2) {
      if (threshold < 0) fail(WK_ERR_ARG, "threshold must be >= 0");
      if (max_tpr < 2 || max_tpr > 64 || (max_tpr & (max_tpr - 1)))
        fail(WK_ERR_ARG, "max_tpr must be a power of two in [2, 64]");
    }
    auto *E = new wk_engine();
    try {
      hip_check(hipGetDevice(&E->device), "hipGetDevice");
      E->dtype = values_dtype;
      E->nrows = nrows;
      E->ncols = ncols;
      E->nnz = nnz;
      wk_layout_info &I = E->info;
      I.variant = variant;
      I.group_width = 64;
      I.threshold = variant == 2 ? threshold : 0;
      I.max_tpr = variant == 2 ? max_tpr : 32;
      I.nrows = nrows;
      I.ncols = ncols;
      I.nz = nnz;
      if (variant == 2) I.min_nz = (uint32_t)nrows;
      device_scan(E, variant, threshold, max_tpr, kr, rowptr_dev, colind_dev, vals_dev,
                  static_cast<hipStream_t>(stream));
    } catch (...) {
      wk_engine_destroy(E);
      throw;
    }
    *out = E;
  });
}

extern "C" int wk_engine_download(const wk_engine *E, int32_t which, void *host_dst,
                                  int64_t *count) {
  return guarded([&] {
    if (!E) fail(WK_ERR_ARG, "engine is NULL");
    const DevLayout &D = E->fwd;
    const void *src = nullptr;
    size_t esz = 4;
    int64_t n = 0;
    switch (which) {
      case WK_ROW_MAP: src = D.row_map; n = D.row_map ? D.nrows : 0; break;
      case WK_ROW_MAP_INV: src = D.row_map_inv; n = D.row_map_inv ? D.nrows : 0; break;
      case WK_REORDER_ROWS: src = D.slot_of_nz; n = D.slot_of_nz ? E->nnz : 0; break;
      case WK_WARP_OFFSETS: src = D.warp_offsets; n = D.warp_offsets ? D.ngroups + 1 : 0; esz = 8; break;
      case WK_MAX_NZ_ROWS: src = D.max_nz_rows; n = D.max_nz_rows ? D.ngroups : 0; break;
      case WK_THREADS_PER_ROW: src = D.tpr; n = D.tpr ? D.ngroups : 0; break;
      case WK_ROW_OFFSET_WARP: src = D.row_off; n = D.row_off ? D.ngroups + 1 : 0; break;
      case WK_ENGINE_VALUES:
        src = D.vals;
        n = D.vals ? D.allocate_nz : 0;
        esz = E->dtype == WK_F64 ? 8 : 4;
        break;
      case WK_ENGINE_COLS: src = D.cols; n = D.cols ? D.allocate_nz : 0; break;
      case WK_ENGINE_COLS_KR: src = D.cols_kr; n = D.cols_kr ? D.allocate_nz : 0; break;
      case WK_ENGINE_WIN_IDX: src = D.win_idx; n = D.win_idx ? D.allocate_nz : 0; esz = 2; break;
      case WK_ENGINE_WIN_OFF: src = D.win_off; n = D.win_off ? D.ngroups + 1 : 0; break;
      case WK_ENGINE_WIN_COLS:
      case WK_ENGINE_WIN_COLS_KR: {
        src = which == WK_ENGINE_WIN_COLS ? D.win_cols : D.win_cols_kr;
        uint32_t total = 0;
        if (src && D.win_off)
          hip_check(hipMemcpy(&total, D.win_off + D.ngroups, sizeof total, hipMemcpyDeviceToHost), "download");
        n = src ? total : 0;
        break;
      }
      case WK_ENGINE_ND_COLS: src = D.nd_cols; n = D.nd_cols ? D.win_total : 0; break;
      case WK_ENGINE_ND_CNT: src = D.nd_cnt; n = D.nd_cnt ? D.ngroups : 0; break;
      case WK_ENGINE_ND_COLS_KR: src = D.nd_cols_kr; n = D.nd_cols_kr ? 3 * D.win_total : 0; break;
      case WK_ENGINE_ND_OFF: src = D.nd_off; n = D.nd_off ? D.ngroups + 1 : 0; break;
      case WK_ENGINE_ND_POS: {
        src = D.nd_pos;
        uint32_t words = 0;
        if (src && D.nd_off)
          hip_check(hipMemcpy(&words, D.nd_off + D.ngroups, sizeof words, hipMemcpyDeviceToHost), "download");
        n = src ? (int64_t)words * 64 : 0;
        break;
      }
      default: fail(WK_ERR_ARG, "unknown engine array");
    }
    if (!count) fail(WK_ERR_ARG, "count is NULL");
    if (!host_dst) {
      *count = n;
      return;
    }
    if (*count != n) fail(WK_ERR_ARG, "count must be " + std::to_string(n) + " for this array");
    if (!n) return;
    int cur = 0;
    hip_check(hipGetDevice(&cur), "hipGetDevice");
    hip_check(hipSetDevice(E->device), "hipSetDevice");
    const hipError_t e = hipMemcpy(host_dst, src, esz * (size_t)n, hipMemcpyDeviceToHost);
    (void)hipSetDevice(cur);
    hip_check(e, "download");
  });
}
