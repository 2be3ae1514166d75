// process.hip -- new matrix values into an engine's layouts (wk_engine_update_values):
// the reference's process step (warpkernel.hpp:379-398, 749-769) for values
// alone, on the device.
//
// Layouts whose lanes hold runs of CSR entries (every forward layout without
// the row sort), unless small or with a group that is a bottleneck: one block per
// group reads its rows' entries 4 to 64 at a time, turns them around in LDS and
// writes whole steps.  It streams 16 bytes per FP64 entry, both ways in whole lines,
// with no index array.  (One thread per entry writing through the CSR-to-slot map
// put 8 bytes into each 128-byte line: hex elasticity 48^3, 27.4M entries, 305 us
// against 77.)  The transposed layout, where its entries lie near each other and
// few slots are pads, reads the entry of each slot instead: indices and values
// written in order, the 8-byte reads land on lines that the same group's other
// steps read too (hex diffusion 48^3, both layouts 31 us as two scatters, 23 here
// in one launch).  The others go through the map.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "spmv_device.hpp"
#include "wk_internal.hpp"

namespace wk {
namespace {

constexpr int kThreads = 256;
// slots per thread of the transposed layout (hex diffusion 48^3, the training
// step: 54.9 us with 4, 57.0 with 8)
constexpr int kGatherPer = 4;

struct UpdateArgs {
  const void *src;                // CSR values
  void *dst;                      // padded values
  const int2 *lane_src;           // [ngroups * W] first CSR entry and entries of each lane
  const int64_t *warp_offsets;
  const uint32_t *max_nz_rows;
  int32_t ngroups;
  void *dst_t;                    // padded values of the transposed layout
  const int32_t *src_of_slot;     // its slots' CSR entries, -1 for a pad
  int64_t slots_t;
  int32_t nblocks_t;              // blocks of the transposed layout
};

// S: steps of a group turned at a time, by TH threads
template <class T, int W, int S, int TH>
__device__ __forceinline__ void turn_group(const UpdateArgs &u, int32_t g) {
  constexpr int PER = S * W / TH;
  static_assert(PER * TH == S * W, "whole passes");
  __shared__ int2 ls[W];
  __shared__ T tile[W][S + 1];  // odd row length: the turned reads spread over the banks
  const int32_t tid = threadIdx.x;
  const T *src = static_cast<const T *>(u.src);
  T *dst = static_cast<T *>(u.dst) + u.warp_offsets[g];
  const int32_t len = (int32_t)u.max_nz_rows[g];
  if (tid < W) ls[tid] = u.lane_src[(int64_t)g * W + tid];
  __syncthreads();
  for (int32_t i0 = 0; i0 < len; i0 += S) {
    T v[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) {
      const int2 s = ls[(tid + j * TH) / S];
      const int32_t i = i0 + (tid + j * TH) % S;
      v[j] = i < s.y ? src[s.x + i] : T(0);
    }
#pragma unroll
    for (int j = 0; j < PER; j++) tile[(tid + j * TH) / S][(tid + j * TH) % S] = v[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PER; j++) {
      const int32_t l = tid % W, t = (tid + j * TH) / W;
      if (i0 + t < len) dst[l + (int64_t)W * (i0 + t)] = tile[l][t];
    }
    __syncthreads();
  }
}

template <class T, int TH>
__device__ __forceinline__ void gather_slots(const UpdateArgs &u, int32_t b) {
  const T *src = static_cast<const T *>(u.src);
  T *dst = static_cast<T *>(u.dst_t);
  const int64_t s0 = (int64_t)b * (TH * kGatherPer) + threadIdx.x;
  int32_t e[kGatherPer];
#pragma unroll
  for (int j = 0; j < kGatherPer; j++) {
    const int64_t s = s0 + (int64_t)j * TH;
    e[j] = s < u.slots_t ? u.src_of_slot[s] : -1;
  }
  T v[kGatherPer];
#pragma unroll
  for (int j = 0; j < kGatherPer; j++) v[j] = e[j] >= 0 ? src[e[j]] : T(0);
#pragma unroll
  for (int j = 0; j < kGatherPer; j++)
    if (e[j] >= 0) dst[s0 + (int64_t)j * TH] = v[j];
}

// Blocks [0, ngroups): groups of the forward layout; then the transposed
// layout's slots, each XCD a contiguous range of them.
template <class T, int W, int S, int TH>
__global__ __launch_bounds__(TH) void update_kernel(UpdateArgs u) {
  const int32_t b = blockIdx.x;
  if (b < u.ngroups)
    turn_group<T, W, S, TH>(u, b);
  else
    gather_slots<T, TH>(u, work_id(b - u.ngroups, u.nblocks_t, 1));
}

// The other layouts: entry i to slot[i].
template <class T>
__global__ __launch_bounds__(kThreads) void scatter_kernel(const T *__restrict__ src,
                                                           const uint32_t *__restrict__ slot,
                                                           T *__restrict__ dst, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    dst[slot[i]] = src[i];
}

// Entry i of the CSR to slot[i].
template <class T>
void scatter(const DevLayout &D, const void *vals, int64_t nnz, hipStream_t s) {
  if (!D.slot_of_nz) fail(WK_ERR_STATE, "layout has no device scatter map");
  const int64_t blocks = std::min<int64_t>((nnz + kThreads - 1) / kThreads, 65536);
  hipLaunchKernelGGL(scatter_kernel<T>, dim3((uint32_t)blocks), dim3(kThreads), 0, s,
                     static_cast<const T *>(vals), D.slot_of_nz, static_cast<T *>(D.vals), nnz);
  hip_check(hipGetLastError(), "scatter launch");
}

template <class T>
void update_values(const wk_engine *E, const void *vals, hipStream_t s) {
  const DevLayout &D = E->fwd;
  UpdateArgs u{};
  u.src = vals;
  // The steps turned at a time, by mean row length.  Up to 4 and 8, where there are
  // groups enough, one wave a group: most of a 16-step tile and three of its waves
  // would be empty (threshold 5, P1 tets 54^3, 10,399 groups, 14.1 -> 8.5 us, 9.6 by
  // the map; threshold 4, 2D Laplacian 400^2 11.4 -> 6.4; with 2,246 groups level).
  // Up to 16, half the LDS of 32 and twice the blocks in flight (2D Laplacian 407^2,
  // 9 entries, residual with new values 15.1 -> 14.6); 32; and for longer rows 64 by eight waves, a whole
  // group in two turns (hex elasticity, 81 entries: 48^3 residual with new values
  // 129.1 -> 122.1 us, 123.2 with 32 steps and eight waves; 16^3 update 5.9 -> 5.1;
  // but hex diffusion 60^3, 27 entries, 16.1 -> 17.4, and FP32 elasticity 28^3 8.4
  // -> 9.0).  Width 32 knows two tiles (tets 96^3 at threshold 5, both layouts, 174 us by
  // the maps, 238 with 32 steps, 148 with 8)
  const int64_t slots = (int64_t)D.W * D.ngroups;
  const bool many = D.ngroups >= 4096;
  const int steps = D.W != 64 ? (D.ngroups >= 2048 && D.allocate_nz <= 16 * slots ? 8 : 32)
                    : many && D.allocate_nz <= 4 * slots            ? 4
                    : many && D.allocate_nz <= 8 * slots            ? 8
                    : D.allocate_nz <= 16 * slots                   ? 16
                    : sizeof(T) == 4 || D.allocate_nz <= 32 * slots ? 32
                                                                    : 64;
  const int threads = steps <= 8 ? 64 : steps == 64 ? 512 : kThreads;
  // A block turns its group's steps one tile after another, about 1.1 us each, while
  // the map takes 11 us per million FP64 entries of long rows, 6 per million FP32
  // ones: layouts with a group too long for its share of the entries keep the map
  // (200,000 rows of 9 entries and one of 100,000: 9.8 us, 1,568 turned; 64 of 8,000
  // 13.6, 419; 1,500 rows of 1,500, 24 groups, 25.4, 39.2; but 20,000 of 500 147, 37.9;
  // 4,096 of 300, FP64 16.4, 10.3, FP32 11.4, 13.2; in a graph, 1,000 rows of 81 2.9, 4.6,
  // but FP32 elasticity 12^3, both layouts in one launch, 9.3, 5.8).
  // So do small ones, whose map stays in L2, unless the transposed layout takes its
  // values in the same launch (in a graph: 20,000 rows of 9 entries 2.8, 3.0, of 16
  // 3.0, 3.2; elasticity 8^3 3.3, 4.6; both layouts of the 9 6.1 as two maps, 4.5), and
  // larger ones of the shortest rows, whose groups hold too little (400,000 rows of 2
  // 3.9, 4.8, FP32 3.1, 4.3; of 4 7.4, 6.1, FP32 4.2, 4.8; 100,000 of 9 5.1, 4.6)
  constexpr bool f64 = sizeof(T) == 8;
  const int64_t turns = ((int64_t)D.longest + steps - 1) / steps;
  const bool shared = E->has_adj && E->adj.src_of_slot;
  const bool by_map = !D.lane_src || turns > (shared ? 3 : 1) + E->nnz / (f64 ? 131072 : 262144) ||
                      (!shared && (E->nnz <= 327680 ||
                                   (D.allocate_nz <= 6 * slots && E->nnz <= (f64 ? 1 << 20 : 1 << 21))));
  if (!by_map) {
    u.dst = D.vals;
    u.lane_src = reinterpret_cast<const int2 *>(D.lane_src);
    u.warp_offsets = D.warp_offsets;
    u.max_nz_rows = D.max_nz_rows;
    u.ngroups = D.ngroups;
  } else {
    scatter<T>(D, vals, E->nnz, s);
  }
  if (shared) {
    u.dst_t = E->adj.vals;
    u.src_of_slot = E->adj.src_of_slot;
    u.slots_t = E->adj.allocate_nz;
    u.nblocks_t = (int32_t)((u.slots_t + threads * kGatherPer - 1) / (threads * kGatherPer));
  } else if (E->has_adj) {
    scatter<T>(E->adj, vals, E->nnz, s);
  }
  const int64_t blocks = (int64_t)u.ngroups + u.nblocks_t;
  if (blocks > INT32_MAX) fail(WK_ERR_LIMIT, "grid too large");
  if (blocks == 0) return;
  const auto kernel = D.W != 64     ? (steps == 8 ? update_kernel<T, 32, 8, 64> : update_kernel<T, 32, 32, kThreads>)
                      : steps == 4  ? update_kernel<T, 64, 4, 64>
                      : steps == 8  ? update_kernel<T, 64, 8, 64>
                      : steps == 16 ? update_kernel<T, 64, 16, kThreads>
                      : steps == 32 ? update_kernel<T, 64, 32, kThreads>
                                    : update_kernel<T, 64, 64, 512>;
  hipLaunchKernelGGL(kernel, dim3((uint32_t)blocks), dim3((uint32_t)threads), 0, s, u);
  hip_check(hipGetLastError(), "update launch");
}

}  // namespace

void launch_update_values(const wk_engine *E, const void *vals_csr, hipStream_t stream) {
  if (E->nnz <= 0) return;
  if (E->dtype == WK_F64)
    update_values<double>(E, vals_csr, stream);
  else
    update_values<float>(E, vals_csr, stream);
}

}  // namespace wk
