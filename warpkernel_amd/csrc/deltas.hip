// deltas.hip -- one right-hand side with 16-bit column offsets, for banded
// layouts of short rows (P1 tetrahedra, the 2D Laplacian), whose x windows do not
// pay.
//
// Each slot's column is its row plus a signed 16-bit offset (column 0, which
// pads read, has a code of its own), four steps of a lane to one 8-byte word.
// The direct kernel loads 4 bytes of column per slot with an instruction per
// step; here it is 2 bytes and a quarter of the column loads: P1 tets 96^3
// (13.5M entries, 155 MB instead of 182) 30.4 -> 27.8 us, 60^3 9.5 -> 7.5, where
// the 155 MB alone take 21.8 at the streaming rate; the rest goes to the x
// gathers, an instruction per step.  Products and their order are the direct
// kernel's, so results are equal bit for bit.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "spmv_device.hpp"
#include "wk_internal.hpp"

namespace wk {
namespace {

template <class P, bool SPLIT, int OUT, int U>
__global__ __launch_bounds__(512) void spmv_delta_kernel(SpmvArgs a, const uint2 *__restrict__ words,
                                                         const uint32_t *__restrict__ off, int32_t nwork,
                                                         int32_t remap) {
  using V = typename P::V;
  using X = typename P::X;
  using Acc = typename P::Acc;
  const int32_t lane = threadIdx.x & 63;
  const int32_t wpb = blockDim.x >> 6;
  const int32_t bid = blockIdx.x;
  if (bid >= nwork) {
    const int64_t pos = (int64_t)a.nznrows + (int64_t)(bid - nwork) * blockDim.x + threadIdx.x;
    if (pos >= a.nrows) return;
    const int64_t dst = a.row_map[pos];
    a.y[dst * a.ldy] = OUT == OUT_RESID ? a.b[dst * a.ldb] : 0.0;
    return;
  }
  const int32_t g = __builtin_amdgcn_readfirstlane(work_id(bid, nwork, remap) * wpb + (int32_t)(threadIdx.x >> 6));
  if (g >= a.ngroups) return;
  const uint32_t len = a.max_nz_rows[g];
  const uint32_t tpr = SPLIT ? a.tpr[g] : 1u;
  const uint32_t rowid = (SPLIT ? a.row_off[g] : (uint32_t)g * 64u) + (uint32_t)lane / tpr;
  const bool row = rowid < (uint32_t)a.nznrows;
  const int32_t dst = a.row_map[row ? rowid : (uint32_t)a.nznrows - 1];
  const V *vp = static_cast<const V *>(a.vals) + a.warp_offsets[g] + lane;
  const uint2 *wp = words + (int64_t)off[g] * 64 + lane;
  Acc acc = delta_steps<P, U>(vp, wp, static_cast<const X *>(a.x), a.ldx, len, dst);
  if constexpr (SPLIT) {
    // lockstep pairwise tree of hpp:157-162: lane t adds lane t+o's partial
    for (uint32_t o = 1; o < tpr; o <<= 1) {
      Acc other = P::shfl_down(acc, (int)o, 64);
      P::add(acc, other);
    }
  }
  if (((uint32_t)lane & (tpr - 1)) != 0 || !row) return;
  const double res = P::result(acc);
  if constexpr (OUT == OUT_RESID)
    a.y[(int64_t)dst * a.ldy] = a.b[(int64_t)dst * a.ldb] - res;
  else
    a.y[(int64_t)dst * a.ldy] = res;
}

// One wave per group: the group's words, and whether every slot has an offset.
constexpr int kBuildWaves = 4;
__global__ __launch_bounds__(kBuildWaves * 64) void delta_build_kernel(SpmvArgs a, int32_t split,
                                                                      const uint32_t *__restrict__ off,
                                                                      uint32_t *__restrict__ fits,
                                                                      uint2 *__restrict__ words) {
  const int32_t lane = threadIdx.x & 63;
  const int32_t g = __builtin_amdgcn_readfirstlane((int32_t)(blockIdx.x * kBuildWaves + (threadIdx.x >> 6)));
  if (g >= a.ngroups) return;
  const uint32_t len = a.max_nz_rows[g];
  const uint32_t tpr = split ? a.tpr[g] : 1u;
  const uint32_t rowid = (split ? a.row_off[g] : (uint32_t)g * 64u) + (uint32_t)lane / tpr;
  const int32_t row = a.row_map[rowid < (uint32_t)a.nznrows ? rowid : (uint32_t)a.nznrows - 1];
  const int32_t *cp = a.cols + a.warp_offsets[g] + lane;
  bool ok = true;
  for (uint32_t i = 0; i < len; i += 4) {
    uint32_t w[2] = {0u, 0u};
#pragma unroll
    for (uint32_t u = 0; u < 4; u++) {
      int32_t d = kDeltaZero;
      if (i + u < len) {
        const int32_t c = cp[64 * (int64_t)(i + u)];
        if (c) {
          d = c - row;
          ok = ok && d > kDeltaZero && d < -kDeltaZero;
        }
      }
      w[u / 2] |= ((uint32_t)d & 0xffffu) << (16 * (u & 1));
    }
    words[((int64_t)off[g] + i / 4) * 64 + lane] = uint2{w[0], w[1]};
  }
  ok = __ballot(!ok) == 0;
  if (lane == 0) fits[g] = ok ? 1u : 0u;
}

using DeltaFn = void (*)(const SpmvArgs &, const DevLayout &, dim3, dim3, int32_t, int32_t, hipStream_t);

template <class P, bool SPLIT, int OUT, int U>
void launch_delta(const SpmvArgs &a, const DevLayout &D, dim3 grid, dim3 block, int32_t nwork, int32_t remap,
                  hipStream_t s) {
  hipLaunchKernelGGL((spmv_delta_kernel<P, SPLIT, OUT, U>), grid, block, 0, s, a,
                     reinterpret_cast<const uint2 *>(D.dl_words), D.dl_off, nwork, remap);
}

template <class P, int U>
DeltaFn pick_delta_out(bool split, int out) {
  if (out == OUT_RUN) return split ? &launch_delta<P, true, OUT_RUN, U> : &launch_delta<P, false, OUT_RUN, U>;
  if constexpr (std::is_same_v<P, PF64>)
    if (out == OUT_RESID)
      return split ? &launch_delta<P, true, OUT_RESID, U> : &launch_delta<P, false, OUT_RESID, U>;
  return nullptr;
}

template <class P>
DeltaFn pick_delta_u(bool split, int out, int u) {
  if constexpr (std::is_same_v<P, PF64>)
    if (u == 28) return pick_delta_out<P, 28>(split, out);
  return u == 8    ? pick_delta_out<P, 8>(split, out)
         : u == 12 ? pick_delta_out<P, 12>(split, out)
                   : pick_delta_out<P, 16>(split, out);
}

SpmvArgs layout_args(const DevLayout &D) {
  SpmvArgs a{};
  a.vals = D.vals;
  a.cols = D.cols;
  a.row_map = D.row_map;
  a.warp_offsets = D.warp_offsets;
  a.max_nz_rows = D.max_nz_rows;
  a.tpr = D.tpr;
  a.row_off = D.row_off;
  a.ngroups = D.ngroups;
  a.nznrows = D.nznrows;
  a.nrows = D.nrows;
  return a;
}

}  // namespace

bool launch_deltas(const DevLayout &D, int prec, int out, const SpmvArgs &a, int wpb, int unroll, int32_t remap,
                   hipStream_t stream) {
  if (!D.dl_words || D.win_max <= 0) return false;
  const bool split = D.variant == 2;
  // A lane's whole row in flight, and no more, since steps past the row cost
  // their branches: P1 tets 96^3 (15 steps) 27.8 us with 16, 28.7 with 8; hex
  // diffusion 48^3 (27) 7.06 with 28, 7.27 with 16 (FP32 5.9 and 5.6); 2D
  // Laplacian 400^2 (9) 4.01 with 12, 4.61 with 8, 4.09 with 16; WPK2's groups of
  // a few steps, tets 96^3 at threshold 5, 32.9 with 8, 42.0 with 16
  const int64_t slots = (int64_t)64 * D.ngroups;
  const int u = unroll == 16                      ? 16
                : D.allocate_nz <= 8 * slots      ? 8
                : D.allocate_nz <= 12 * slots     ? 12
                : D.allocate_nz <= 20 * slots     ? 16
                : prec == 0                       ? 28
                                                  : 16;
  DeltaFn fn = prec == 0 ? pick_delta_u<PF64>(split, out, u)
                         : prec == 1 ? pick_delta_u<PF32C>(split, out, u) : pick_delta_u<PF32D>(split, out, u);
  if (!fn) return false;
  const int64_t nwork = ((int64_t)D.ngroups + wpb - 1) / wpb;
  const int64_t nfill = ((int64_t)D.nrows - D.nznrows + wpb * 64 - 1) / (wpb * 64);
  if (nwork + nfill > INT32_MAX) fail(WK_ERR_LIMIT, "grid too large");
  fn(a, D, dim3((uint32_t)(nwork + nfill)), dim3((uint32_t)wpb * 64), (int32_t)nwork, remap, stream);
  hip_check(hipGetLastError(), "spmv launch");
  return true;
}

// The words do not depend on whether they fit, so they are written at once and
// given back by deltas_finish if some group's do not.
bool deltas_begin(wk_engine *E, DevLayout &D, std::vector<uint32_t> &off, uint32_t *fits, uint32_t *dev_off,
                  hipStream_t stream) {
  const int32_t G = D.ngroups;
  // short rows whose windows do not pay by themselves (swapped columns turn
  // the windows off, and the offsets with them); lanes past the last row with
  // entries read its place in row_map, so there has to be one
  if (D.W != 64 || D.nznrows <= 0 || D.win_max <= 0 || D.nd_max > 0 || G <= 0 ||
      (double)D.allocate_nz >= 40.0 * 64.0 * (double)G || (double)D.allocate_nz < 1.25 * (double)D.win_total)
    return false;
  off.assign((size_t)G + 1, 0);
  for (int32_t g = 0; g < G; g++) {
    const uint64_t words = (uint64_t)off[g] + (D.h_max_nz_rows[g] + 3) / 4;
    if (words > UINT32_MAX) return false;
    off[g + 1] = (uint32_t)words;
  }
  D.dl_words = dev_alloc<uint32_t>(E, (int64_t)off.back() * 128);
  D.dl_off = dev_off;
  hip_check(hipMemcpyAsync(dev_off, off.data(), 4 * off.size(), hipMemcpyHostToDevice, stream), "deltas");
  hipLaunchKernelGGL(delta_build_kernel, dim3((uint32_t)(((int64_t)G + kBuildWaves - 1) / kBuildWaves)),
                     dim3(kBuildWaves * 64), 0, stream, layout_args(D), D.variant == 2, D.dl_off, fits,
                     reinterpret_cast<uint2 *>(D.dl_words));
  hip_check(hipGetLastError(), "delta launch");
  return true;
}

void deltas_finish(wk_engine *E, DevLayout &D, const uint32_t *fits) {
  for (int32_t g = 0; g < D.ngroups; g++)
    if (!fits[g]) {
      dev_give(E, D.dl_words);
      D.dl_words = nullptr;
      D.dl_off = nullptr;
      return;
    }
}

}  // namespace wk
