// tune.cpp -- per-engine launch configurations and the autotuner.
//
// The reference tunes by sweeping warps/block (1..16) and the WPK2 threshold
// in its drivers and keeping the fastest (wpk1.cu:138-257, wpk2.cu:156-302).
// Here every engine keeps one launch configuration per (operation, k): a
// layout-based choice until wk_tune measures the candidates on the device.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <utility>
#include <vector>

#include "wk_internal.hpp"

namespace wk {

namespace {

int64_t cfg_key(int32_t op, int32_t k) { return ((int64_t)op << 32) | (uint32_t)k; }

int pow2_at_most(int v) {
  int p = 1;
  while (p * 2 <= v) p *= 2;
  return p;
}

int pow2_at_least(int v) {
  int p = 1;
  while (p < v) p *= 2;
  return p;
}

const DevLayout &layout_for(const wk_engine *E, int32_t op) { return op == WK_OP_ADJOINT ? E->adj : E->fwd; }

// Whether stage 6 is the row sets.
bool row_sets_run(const DevLayout &D, int32_t dtype, int32_t k, int32_t sums) {
  return D.rs_waves > 0 && D.win_max > 0 && row_sets_take(D, k) && (dtype == WK_F64 || sums == WK_ACC_F64);
}

// The sums of an FP32 engine that is not told: FP64 ones from kRowSetDefault where
// the layout has row sets, whichever kernel runs, so that they depend on k and the
// matrix's structure and not on its size (they did: compensated up to k = 8 from
// 8,192 groups, where 64^3 k=5 took 186 us against 122 here).  Exact products:
// closer to the exact result than the compensated sums (1e-16 against 2e-14
// normwise on 32^3), and faster (32^3 k=8 13.7 us against 23.5).
int32_t default_sums(const DevLayout &D, int32_t k) {
  return D.rs_waves > 0 && k >= kRowSetDefault ? WK_ACC_F64 : WK_ACC_TWOSUM;
}

// Where the row sets beat the layout's other kernels, by the rows a wave sums (8
// where sets hold two rows, 10 to 12 three, 16 four), the mean row length and
// the groups.  Blocks of dof rows over a band of w nodes, d = dof, n = d w entries a
// row, us by the other kernels and by the row sets:
//   two rows a set, from 640 groups: short rows lose below k = 9 (3,750 groups, d 2:
//   n 4 k=5 16.2 / 20.9, n 10 19.0 / 21.1, n 18 23.2 / 21.5; 936 groups, n 4 k=8 5.8 /
//   6.7; 468 groups, n 4 k=8 4.0 / 3.9), and the shortest above (n 2 k=12 23.3 / 30.1,
//   n 4 42.2 / 29.9); FP32 values with FP64 sums longer ones on large layouts
//   (3,750 groups, n 18 k=5 15.7 / 18.7; 936 groups, n 6 5.8 / 5.8);
//   two, the largest layouts: whole window tiles, and k = 5 (n 18, 4,005 groups k=8 25.1 /
//   23.0, 6,133 32.7 / 39.3, 8,002 41.2 / 51.0, k=12 68.7 / 73.2, but k=5 55.9 / 46.4, k=7
//   94.3 / 50.5, k=16 107 / 82; 25,313 groups k=8 138 / 184, k=5 155 / 176; n 54, 8,192
//   groups, k=8 106 / 100);
//   three, large layouts: the shortest (3,750 groups, d 3: n 3 k=5 13.1 / 16.8, n 6 17.2 /
//   16.8; FP32 n 3 10.5 / 14.6, n 6 14.3 / 14.6);
//   up to three and fewer than 4 entries: k = 8, one tile of the direct kernel (249
//   groups, d 3 n 3 2.6 / 2.8; 468 groups, d 2 n 2 3.0 / 3.8).
// FP32 layouts of 8,192 groups or more keep the windows up to k = 8 (hex elasticity
// 64^3 k=8 114 us against 126; k=5 122 either way).
bool row_sets_pay(const DevLayout &D, int32_t dtype, int32_t k, double mean_len) {
  const bool f64 = dtype == WK_F64;
  const double rows = (double)D.nznrows / (double)D.rs_waves;
  const bool two = rows < 10.0, three = rows < 14.0;  // at most
  if (two && mean_len < 32.0 && D.ngroups >= 5120 &&
      ((k < 16 && k % 4 == 0) || (k == 5 && D.ngroups >= 10240)))
    return false;
  if (k >= 9) return !(two && mean_len < 4.0 && D.ngroups >= 640);
  if (!f64 && D.ngroups >= 8192) return false;
  if (k == 8 && three && mean_len < 4.0) return false;
  if (two && D.ngroups >= 640 && mean_len < (f64 ? 12.0 : D.ngroups >= 2048 ? 24.0 : 6.0)) return false;
  return !(three && D.ngroups >= 2048 && mean_len < (f64 ? 5.0 : 6.0));
}

// One right-hand side: where x windows that pay (3 slots or more an entry) beat the
// 16-bit column offsets, by mean row length, the longest group against it, the
// groups, and reuse.  Few groups leave the windows' fill uncovered; long rows, and
// long groups among short ones, take several of the offsets' batches, whose x
// gathers the windows' LDS reads outrun.  us by offsets and by windows (bands of
// random columns unless named; r: slots an entry):
//   39 entries, FP64 1,000 groups 6.8 / 6.6, 1,563 9.8 / 8.2, 6,250 32.4 / 27.1;
//     FP32 313 4.9 / 5.2, 1,000 6.6 / 6.0, 4,063 14.1 / 11.2, 9,375 r 4.0 32.8 / 27.0
//   27 entries, FP64 1,563 6.6 / 6.6, 2,657 10.4 / 9.7; FP32 1,000 5.6 / 5.2, 4,063
//     10.3 / 8.3, 9,375 r 4.0 23.5 / 20.9; hex diffusion r 3.0 to 3.4, FP64 48^3 (1,839) 7.2 / 7.6, 60^3 (3,547)
//     13.6 / 12.7, 100^3 (16,098) 52.3 / 49.9, FP32 60^3 8.1 / 8.5, 100^3 29.9 / 33.3
//   20 entries, FP64 2,032 6.3 / 6.8, 2,657 8.5 / 7.9; FP32 2,032 5.4 / 5.3, 2,657 6.5 / 5.4
//   16 entries, FP64 4,063 9.5 / 9.9, 9,375 r 4.3 20.6 / 23.5, r 10 level
//   1 to 39 entries, mean 17, FP64 858 7.1 / 7.1, 1,139 8.9 / 8.0, 4,018 24.9 / 23.3;
//     FP32 737 6.3 / 5.1; 12 to 27, mean 18, FP64 2,032 8.2 / 8.4, 2,657 11.6 / 10.2, 9,375
//     25.4 / 30.6; FP32 1,000 5.2 / 4.7, 9,375 19.3 / 21.1; 1 to 17, mean 7.5, 37.5 / 58.1
bool windows_beat_offsets(const DevLayout &D, int32_t dtype, double mean_len, double reuse) {
  const bool f64 = dtype == WK_F64;
  const int32_t G = D.ngroups;
  const double mix = (double)D.pk_longest / std::max(1.0, mean_len);
  if (mean_len >= 32.0) return G >= (f64 ? 1280 : 768);
  if (G >= 8192) return reuse >= (f64 ? 4.5 : 4.0) || (f64 && mean_len >= 20.0);
  if (mean_len < 16.0) return false;
  if (mix >= 1.8) return G >= (f64 ? 1024 : 512);
  if (mix >= 1.4) return G >= (f64 ? 2304 : 768);
  if (f64) return mean_len >= 20.0 && G >= 2304;
  return reuse >= 4.0 && mean_len >= 20.0 && G >= (mean_len >= 24.0 ? 768 : 2304);
}

// Candidate set: the knobs that change speed but not results.
std::vector<wk_launch> candidates(const DevLayout &D, int32_t dtype, const wk_launch &base, int32_t k) {
  std::vector<wk_launch> out;
  const size_t vsz = dtype == WK_F64 ? 8 : 4;
  for (int wpb : {1, 2, 4, 8})
    for (int remap : {0, 1}) {
      wk_launch c = base;
      c.waves_per_block = wpb;
      c.xcd_remap = remap;
      c.blocks_per_cu = 0;
      if (k == 1 || D.W == 32) {
        c.k_tile = 1;
        for (int u : {8, 16}) {
          c.unroll = u;
          c.rows_per_lane = 1;
          c.stage_lds = 0;
          out.push_back(c);
          if (D.dl_words) {
            // the columns themselves where 0 takes their offsets
            c.stage_lds = 9;
            out.push_back(c);
            c.stage_lds = 0;
          }
          if (u == 8 && D.W == 64) {
            // the index stream nontemporal too (scattered x gathers keep more L2)
            c.nontemporal = 2;
            out.push_back(c);
            c.nontemporal = base.nontemporal;
          }
          if (D.W == 64 && (size_t)wpb * u * 64 * (vsz + 4) <= 65536) {
            for (int st : {1, 2}) {
              c.stage_lds = st;
              out.push_back(c);
            }
            // x windows, with 16-bit or packed 10-bit positions (the launcher
            // falls back where a window does not fit)
            if (D.win_max > 0) {
              c.stage_lds = 3;
              out.push_back(c);
              if (D.win_pk) {
                c.stage_lds = 5;
                out.push_back(c);
              }
              if (D.nd_max > 0) {
                c.stage_lds = 7;
                out.push_back(c);
              }
            }
            c.stage_lds = 0;
          }
        }
        if (D.W == 64) {
          c.unroll = 8;
          c.rows_per_lane = 2;
          out.push_back(c);
          c.nontemporal = 2;
          out.push_back(c);
          c.nontemporal = base.nontemporal;
          // four groups per wave (scattered columns)
          c.rows_per_lane = 4;
          for (int u : {4, 8}) {
            c.unroll = u;
            out.push_back(c);
          }
          c.unroll = 8;
        }
      } else {
        c.unroll = 8;
        c.rows_per_lane = 1;
        c.stage_lds = 0;
        for (int kt = 1; kt <= std::min(32, pow2_at_least(k)); kt *= 2) {
          c.k_tile = kt;
          out.push_back(c);
          if (D.win_max > 0 && kt >= 2 && kt <= 8) {
            // windowed passes, values through slices or straight into registers
            // (the latter also with 16-step batches at k-tiles 4 and 8, one or
            // two waves per window); the launcher falls back where the window
            // does not fit
            for (int st : {3, 4}) {
              c.stage_lds = st;
              out.push_back(c);
            }
            if (kt >= 4 && wpb <= 2) {
              c.stage_lds = 4;
              c.unroll = 16;
              out.push_back(c);
              c.unroll = 8;
            }
            c.stage_lds = 0;
          }
        }
        // the row sets (one shape), and the group's values held in registers
        // across 32-byte k-tiles (the launcher falls back where groups are
        // longer than 84 steps)
        const bool sets = row_sets_run(D, dtype, k, base.accumulate);
        if (sets && wpb == 1) {
          c.stage_lds = 6;
          c.k_tile = std::min(8, pow2_at_most(k));
          out.push_back(c);
          c.stage_lds = 0;
        }
        if (D.win_pk && k >= (int)(32 / vsz) && wpb <= 4) {
          c.stage_lds = sets ? 8 : 6;
          c.k_tile = std::min(32, pow2_at_most(k));
          out.push_back(c);
          c.stage_lds = 0;
        }
      }
    }
  return out;
}

}  // namespace

wk_launch heuristic_launch(const DevLayout &D, int32_t dtype, int32_t k, bool kr, int32_t sums, int64_t ldx) {
  wk_launch c;
  wk_launch_default(&c);
  bool masked = false;  // k-tiles may exceed k (windowed multi-RHS)
  const double mean_len =
      D.ngroups ? (double)D.allocate_nz / ((double)D.ngroups * D.W) : 0.0;
  // x windows pay where each window entry serves enough slots to amortise its
  // fill: at k = 1, hex elasticity (7.6 slots per entry for WPK1, 6.0 for
  // WPK2 at threshold 27) gains 10-30%, while hex diffusion (3.4), P1 tets
  // (2.1) and the 2D Laplacian (2.9) lose.  With several right-hand sides
  // each entry serves k_tile products per slot: hex diffusion gains 35-45%
  // from k=2 (k=32: 128 -> 68 us), P1 tets from k=16 in FP64 (620 -> 476 us)
  // and from k=2 in FP32; the tiny 2D Laplacian only at k=32.
  const bool win_ok = D.W == 64 && D.win_max > 0 && D.win_total > 0;
  const double reuse = win_ok ? (double)D.allocate_nz / (double)D.win_total : 0.0;
  // (k = 1 with packed positions from 3 slots per entry: hex diffusion 48^3,
  // 3.4, forward and adjoint 7.16 us against 7.76 staged; P1 tets, 2.1, and
  // the 2D Laplacian, 2.9, stay faster without windows)
  // (WPK2 layouts from k = 8 at 2.5: hex diffusion 48^3 at threshold 5, 2.74
  // slots per entry, k=8 25.0 us against 32.3 direct)
  const bool windows =
      win_ok && (k == 1 ? reuse >= (D.win_pk ? 3.0 : 4.5)
                        : reuse >= 3.0 || (reuse >= 2.0 && (k >= 16 || (dtype != WK_F64 &&
                                                                         D.ngroups >= 1024))) ||
                              (D.variant == 2 && k >= 8 && reuse >= 2.5) ||
                              (dtype == WK_F64 && D.variant == 1 && k >= 4 && reuse >= 2.0 &&
                               mean_len < 20.0 && D.ngroups >= 4096));
  const bool keep_windows = windows && windows_beat_offsets(D, dtype, mean_len, reuse);
  if (k == 1 && !kr && D.dl_words && win_ok && D.nd_max == 0 && !keep_windows) {
    // 16-bit column offsets (deltas.hip).  P1 tets 96^3 30.4 -> 27.8 us (FP32
    // 23.9 -> 18.8), 60^3 9.5 -> 7.5; large layouts without the remap (96^3 27.8
    // against 28.8, FP32 18.8 against 21.6; 60^3 7.6 against 7.4).  Ahead of the
    // windows too, most on small layouts, where filling them is a serial step (2D
    // Laplacian 27^2 2.3 us against 3.3, hex diffusion 22^3 4.0 against 5.0, 48^3
    // 7.1 against 7.4) and on WPK2's short groups (threshold 5: tets 96^3 32.9
    // against 39.7 direct, 2D Laplacian 600^2 8.8 against 15.7, hex diffusion
    // 48^3 10.5 against 17.5)
    c.stage_lds = 0;
    c.unroll = 8;  // (the steps in flight: launch_deltas)
    c.waves_per_block = 2;
    c.xcd_remap = D.variant == 2 || D.ngroups < 8192;
  } else if (k == 1 && windows) {
    // 10 bytes per slot, x from the group's window in LDS; one wave per
    // block, a contiguous range of groups per XCD, and 16-step batches for
    // long groups (hex elasticity 64^3: 99.3 us against 104 with 8-step
    // batches and no remap; WPK2 at threshold 27, 21-step groups: 8-step
    // batches, 109.7 us against 139 with 16).  Where every window has at
    // most 1024 entries the positions are packed 10 bits each, 9.3 bytes per
    // slot (stage 5: 24- or 12-step batches; 64^3: 96.7 us, 32^3: 13.8
    // against 15.0, WPK2 64^3: 107.5 against 110.2).  FP32 values take the
    // 12-step batches at every length (32^3 compensated 9.3 us against 9.6,
    // FP64 accumulation 8.8 against 12.1; 64^3 58.4 / 58.5, 58.2 / 71.4).
    // Where slots read x by whole nodes (elasticity) the node window takes
    // 10 bits of position per three slots (stage 7), with 27-step batches
    // on long groups and 18-step ones otherwise: 64^3 90.0 against 97.3 us,
    // 32^3 12.6 against 14.4, WPK2 at threshold 27 106.3 against 108.6 and
    // 16.0 against 17.5; FP32 64^3 51.4 against 58.6 (compensated) and 50.4
    // against 58.9 (FP64 accumulation), 32^3 7.8 against 9.7 and 7.3 against
    // 9.3
    c.stage_lds = D.win_pk ? 5 : 3;
    c.unroll = mean_len >= 40.0 && dtype == WK_F64 ? 16 : 8;
    c.waves_per_block = 1;
    if (D.nd_max > 0) {
      c.stage_lds = 7;
      c.unroll = mean_len >= 40.0 ? 16 : 8;
      // groups of at most 27 steps (their values straight into registers,
      // no slice): four waves per block on large layouts (WPK2 at threshold
      // 27, hex elasticity 64^3, 49,189 groups: 101.8 us against 103.5 with
      // one; 48^3, 20,764 groups: 45.3 against 45.9; 32^3, 6,164: level)
      if (D.pk_longest <= 27 && D.ngroups >= 16384) c.waves_per_block = 4;
    }
    c.xcd_remap = 1;
  } else if (k >= 2 && windows) {
    // (k-tiles may pass k: the launcher runs a rest of 3 or more columns as
    // one masked tile of the next power of two: hex elasticity 64^3 k=3 as
    // one 4-wide pass, k=7 as one 8-wide pass 207 us against 385 as 4 + 2 +
    // 1)
    masked = true;
    // several right-hand sides through windows of k-tile values per column,
    // all k-tiles in one launch, a group's tiles on one XCD (remap) so its
    // values and positions come from HBM once.  Up to k = 16 the values and
    // positions go straight into registers (stage 4): the x reads dominate
    // the LDS traffic, and staging would add to it.  Measured on hex
    // elasticity 32^3 and 64^3: FP64 k=4 17.3 / 119 us (stage 3: 23.7 /
    // 128), k=8 and 16 with k-tile 8 shared by two waves; at k=32 the
    // staged form with one wave per window stays ahead (111 / 817 us).  FP32
    // (compensated) is bound by its arithmetic; on 32^3 a window per wave
    // below k = 16 (k=2 11.2, k=4 15.6, k=8 22.4 us, against 12.7 / 19.0 /
    // 24.9 with windows shared one right-hand side per wave), and from k = 16
    // two waves sharing a k-tile-8 window; from k = 8 16-step batches (two in
    // flight: 32^3 k=32 84.3 us against 89.6 with 8-step ones, 64^3 k=16 304
    // against 323).
    c.unroll = 8;
    c.xcd_remap = 1;
    if (dtype == WK_F64) {
      if (k <= 4 || (k < 16 && D.ngroups < 2048 && mean_len >= 40.0)) {
        // (k = 8 on small layouts of long rows: k-tile 4, one wave per window;
        // elasticity 32^3, 1685 groups, 30.8 us against 32.4 with k-tile 8
        // over two waves; 40^3, 3231 groups, 56.6 against 55.4; hex diffusion
        // 48^3, 27-entry rows, 17.6 against 16.9.  There k = 7 runs as 4 + a
        // masked 4 in one launch, 33.2 us against 35.3 as one masked 8.
        // Elsewhere k = 5 to 7 take the k = 8 shape below as one masked
        // pass: hex diffusion k=7 19.3 us against 30.4 as 4 + 2 + 1)
        c.stage_lds = 4;
        c.k_tile = std::min(4, pow2_at_least(k));
        c.waves_per_block = 1;
      } else if (k < 16 || (k == 16 && D.ngroups < 4096) || mean_len < 40.0) {
        // (short rows keep the register-fed form at every k: hex diffusion
        // k=32 68 us against 86 staged; at k = 16 the staged form pays from a
        // few thousand groups: elasticity 48^3 181 against 191 us, 64^3 421
        // against 453, 32^3 62.8 against 60.8)
        c.stage_lds = 4;
        c.k_tile = 8;
        c.waves_per_block = 2;
      } else {
        c.stage_lds = 3;
        c.k_tile = 8;
        c.waves_per_block = 1;
      }
      if ((D.win_pk && D.pk_longest <= 84 && mean_len >= 40.0 &&
           (k >= 32 || (k >= 16 && D.ngroups < 4096))) ||
          (D.variant == 1 && D.win_pk && D.pk_longest <= 36 && mean_len >= 20.0 && k >= 8)) {
        // the group's values in registers across 4-wide passes (stage 6):
        // elasticity 32^3 k=16 58.3 against 61.1 us, k=32 99.9 against 111.6;
        // 64^3 k=32 803 against 819, but k=16 446 against 423.  Groups of at
        // most 36 steps from k = 8: hex diffusion 48^3 (27-entry rows) k=8
        // 15.8 against 17.0 us, k=16 35.5 against 37.3, k=32 65.7 against
        // 68.1; P1 tets (15-entry rows) lose (k=16 69.5 against 68.5)
        c.stage_lds = 6;
        c.k_tile = 8;
        c.waves_per_block = 1;
      }
      if (D.variant == 1 && mean_len < 20.0 && D.ngroups >= 4096) {
        // short rows with 2-3 slots per window entry (P1 tets 96^3, 15-entry
        // rows, 2.1): 16-step batches, one wave per k-tile-4 window below
        // k = 8 (k=4 44.5 us against 49.6 direct), the values in registers
        // at k = 8 (83.5 against 89.5), k-tile 8 over two waves from k = 16
        // (k=16 215.5 against 229.6, k=32 452.5 against 475.9)
        c.unroll = 16;
        if (k < 8) {
          c.stage_lds = 4;
          c.k_tile = std::min(4, pow2_at_most(k));
          c.waves_per_block = 1;
        } else if (k < 16 && D.win_pk && D.pk_longest <= 36) {
          c.stage_lds = 6;
          c.k_tile = 8;
          c.waves_per_block = 1;
          c.unroll = 8;
        } else {
          c.stage_lds = 4;
          c.k_tile = 8;
          c.waves_per_block = 2;
        }
      }
      if (D.variant == 2 && k >= 8) {
        // WPK2's split groups are a few steps long: one wave per window and
        // 16-step batches (hex elasticity 32^3 at threshold 27, k=8 28.5 us
        // against 32.8, k=16 59.2 against 64.9; hex diffusion 48^3 at
        // threshold 5, k=16 52.4 against 76.0; P1 tets 96^3 at threshold 5,
        // k=16 256 against 323), and from k = 32 the values in registers
        // (hex diffusion 95.0 against 145, tets 535 against 661; from 4,096
        // groups: the 2D Laplacian 128^2 at threshold 5, 521 groups, k=32
        // 15.1 against 9.3), four waves to a block (tets 535.5 against 586.0
        // with one, elasticity 64^3 846.8 against 872.1, 32^3 112.3 against
        // 115.6; hex diffusion 96.1 against 94.7)
        c.stage_lds = 4;
        c.k_tile = 8;
        c.waves_per_block = 1;
        c.unroll = 16;
        if (k >= 32 && D.win_pk && D.pk_longest <= 84 && D.ngroups >= 4096) {
          c.stage_lds = 6;
          c.unroll = 8;
          c.waves_per_block = 4;
        }
      }
    } else if (mean_len < 20.0 && k >= 16 && D.ngroups >= 4096) {
      // FP32 values on short rows from k = 16: the direct kernel with wide
      // k-tiles outruns the windows (P1 tets 96^3: k=16 111 us against 120,
      // k=32 279 against 329), except on small layouts, whose few waves it
      // leaves idle (the 2D Laplacian 128^2, 261 groups: k=32 11.6 against 6.7)
      c.stage_lds = 0;
      c.unroll = 8;
      c.k_tile = std::min(32, pow2_at_most(k));
      c.waves_per_block = k >= 32 ? 1 : 2;
    } else {
      // (below k = 16 rows shorter than 40 share a window between two
      // waves: hex diffusion 48^3 k=4 7.6 us against 9.0, P1 tets k=8 53.5
      // against 66.0; hex elasticity keeps one, 22.5 against 22.7)
      c.stage_lds = 4;
      c.k_tile = std::min(8, pow2_at_least(k));
      c.waves_per_block = k < 16 && mean_len >= 40.0 ? 1 : 2;
      c.unroll = k < 8 ? 8 : 16;
    }
  } else if (k == 1 && win_ok && reuse < 1.25 && D.variant == 1) {
    // scattered columns: nearly every slot of a group reads its own column of
    // x (a randomly numbered mesh), so each slot costs a separate line fetch
    // and the rate is set by the gathers in flight; four groups per wave with
    // four slots each in flight (P1 tets 96^3, randomly permuted, 1.00 slots
    // per window entry: 96.5 us against 120.8 with one group per wave at
    // unroll 8, 108.3 with two groups per wave; FP32 values 76.5 against
    // 77.2).  WPK2 layouts, whose split groups are a few steps long, keep one
    // group per wave (threshold 5: 129.2 us against 132.8)
    c.stage_lds = 0;
    c.rows_per_lane = 4;
    c.unroll = 4;
    c.waves_per_block = 2;
    c.xcd_remap = 1;
  } else if (k == 1 && D.W == 64 && mean_len >= 20.0) {
    // 16-byte batch copies through LDS, next batch in flight during the FMAs
    // (measured best on hex diffusion, 27-entry rows)
    c.stage_lds = 2;
    c.unroll = 8;
    c.waves_per_block = 4;
    c.xcd_remap = 0;
  } else {
    // short rows (P1 tets, 15 entries: 11% faster than staging)
    c.stage_lds = 0;
    c.unroll = 8;
    c.waves_per_block = 2;
    c.xcd_remap = 1;
    c.k_tile = std::min(8, pow2_at_most(std::max(1, k)));
    if (win_ok && reuse < 1.25 && k >= 16) {
      // scattered columns from k = 16: eight waves per block (randomly
      // numbered P1 tets, k=16: FP64 343 us against 375; FP32 with k-tiles
      // of k and no remap 240 against 355, k=32 315 against 517)
      c.waves_per_block = 8;
      if (dtype != WK_F64) {
        c.k_tile = std::min(32, pow2_at_most(k));
        c.xcd_remap = 0;
      }
    }
  }
  if (dtype != WK_F64) c.accumulate = sums != kDefaultSums ? sums : default_sums(D, k);
  if (win_ok && k >= kRowSetDefault && row_sets_run(D, dtype, k, c.accumulate) && row_sets_pay(D, dtype, k, mean_len) &&
      row_sets_reach(D, dtype, ldx)) {
    // row sets on the matrix cores (stage 6, rowsets.hip), all of k in one
    // launch.  Hex elasticity, FP64, one set of inputs repeated: 32^3 k=5 18.1 us
    // against 36.4, k=8 18.7 against 30.9, k=16 25.1 against 58.4 (other inputs
    // from pass to pass 33.6 against 58.5), k=32 38.4 against 100; 64^3 k=5
    // 176 against 194, k=8 181 against 204, k=16 248 against 421, k=32 382
    // against 803.  FP32 values with FP64 sums: 32^3 k=8 13.7 us, 48^3 36.4.
    c.stage_lds = 6;
    c.unroll = 8;
    c.k_tile = 8;
    c.waves_per_block = 1;
    c.rows_per_lane = 1;
    c.xcd_remap = 1;
  } else if (c.stage_lds == 6 && row_sets_run(D, dtype, k, c.accumulate)) {
    c.stage_lds = 8;  // the register kernel, as chosen above
  }
  // as the launcher uses it (a masked last tile where the windows run it)
  c.k_tile = std::min(c.k_tile, masked ? pow2_at_least(std::max(1, k)) : pow2_at_most(std::max(1, k)));
  return c;
}

wk_launch engine_launch(wk_engine *E, int32_t op, int32_t k, int32_t sums, int64_t ldx) {
  const DevLayout &D = layout_for(E, op);
  {
    std::lock_guard<std::mutex> g(E->cfg_mu);
    auto it = E->launch_cfg.find(cfg_key(op, k));
    if (it != E->launch_cfg.end()) {
      wk_launch c = it->second;
      if (E->dtype == WK_F64 || sums == kDefaultSums || sums == c.accumulate) return c;
      if (sums == WK_ACC_F64 || c.stage_lds != 6 || !row_sets_run(D, E->dtype, k, WK_ACC_F64)) {
        c.accumulate = sums;
        return c;
      }
    }
  }
  return heuristic_launch(D, E->dtype, k, op == WK_OP_RUN_X, sums, ldx);
}

}  // namespace wk

using namespace wk;

extern "C" {

int wk_engine_get_launch(const wk_engine *E, int32_t op, int32_t k, wk_launch *cfg) {
  if (!E || !cfg || op < 0 || op > 2 || k < 1) {
    set_last_error("bad argument");
    return WK_ERR_ARG;
  }
  *cfg = engine_launch(const_cast<wk_engine *>(E), op, k);
  return WK_OK;
}

int wk_engine_get_launch_sums(const wk_engine *E, int32_t op, int32_t k, int32_t accumulate, wk_launch *cfg) {
  if (!E || !cfg || op < 0 || op > 2 || k < 1) {
    set_last_error("bad argument");
    return WK_ERR_ARG;
  }
  *cfg = engine_launch(const_cast<wk_engine *>(E), op, k, accumulate == WK_ACC_F64 ? WK_ACC_F64 : WK_ACC_TWOSUM);
  return WK_OK;
}

int wk_engine_set_launch(wk_engine *E, int32_t op, int32_t k, const wk_launch *cfg) {
  if (!E || !cfg || op < 0 || op > 2 || k < 1) {
    set_last_error("bad argument");
    return WK_ERR_ARG;
  }
  std::lock_guard<std::mutex> g(E->cfg_mu);
  E->launch_cfg[cfg_key(op, k)] = *cfg;
  return WK_OK;
}

int wk_tune(wk_engine *E, int32_t op, const wk_launch *base, const void *x_dev, double *y_dev,
            int32_t k, int64_t ldx, int64_t ldy, int32_t reps, void *stream, wk_launch *best,
            float *best_ms) {
  if (!E || op < 0 || op > 2 || k < 1 || reps < 1) {
    set_last_error("bad argument");
    return WK_ERR_ARG;
  }
  if (op == WK_OP_ADJOINT && !E->has_adj) {
    set_last_error("engine was created without WK_ENGINE_ADJOINT");
    return WK_ERR_STATE;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  wk_launch b0 = base ? *base : engine_launch(E, op, k);
  const DevLayout &D = layout_for(E, op);
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
    set_last_error("hipEventCreate failed");
    return WK_ERR_HIP;
  }
  // one timing of c: two untimed launches, then reps timed ones (WK_ERR_ARG:
  // a shape this layout does not offer)
  auto time_cfg = [&](const wk_launch &c, float &ms) -> int {
    auto launch = [&]() {
      if (op == WK_OP_RUN) return wk_run(E, &c, x_dev, y_dev, k, ldx, ldy, stream);
      if (op == WK_OP_RUN_X) return wk_run_x(E, &c, x_dev, y_dev, k, ldx, ldy, stream);
      return wk_run_adjoint(E, &c, x_dev, y_dev, k, ldx, ldy, stream);
    };
    int r = launch();
    for (int w = 0; w < 2 && r == WK_OK; w++) r = launch();
    if (r != WK_OK) return r;
    (void)hipEventRecord(e0, s);
    for (int i = 0; i < reps && r == WK_OK; i++) r = launch();
    (void)hipEventRecord(e1, s);
    if (r != WK_OK) return r;
    if (hipEventSynchronize(e1) != hipSuccess) {
      set_last_error("tuning timing failed");
      return WK_ERR_HIP;
    }
    (void)hipEventElapsedTime(&ms, e0, e1);
    ms /= (float)reps;
    return WK_OK;
  };
  // every candidate once, then the three fastest twice more, keeping each
  // one's best time: a single timing taken while the clocks move must not
  // decide between shapes a few percent apart
  std::vector<std::pair<float, wk_launch>> timed;
  int rc = WK_OK;
  for (const wk_launch &c : candidates(D, E->dtype, b0, k)) {
    float ms = 0;
    rc = time_cfg(c, ms);
    if (rc == WK_ERR_ARG) {
      rc = WK_OK;  // shape not offered for this layout
      continue;
    }
    if (rc != WK_OK) break;
    timed.push_back({ms, c});
  }
  float best_t = INFINITY;
  wk_launch best_c = b0;
  if (rc == WK_OK && !timed.empty()) {
    std::stable_sort(timed.begin(), timed.end(),
                     [](const std::pair<float, wk_launch> &p, const std::pair<float, wk_launch> &q) {
                       return p.first < q.first;
                     });
    const size_t top = std::min<size_t>(3, timed.size());
    // the incumbent (base, or the engine's launch: the layout default until
    // tuned) is timed beside them and kept unless one beats it by more than
    // 1%, so shapes within noise of it do not replace it by chance
    float inc_t = INFINITY;
    for (int pass = 0; pass < 3 && rc == WK_OK; pass++) {
      float ms = 0;
      rc = time_cfg(b0, ms);
      if (rc == WK_ERR_ARG) {
        rc = WK_OK;  // not a shape this layout offers: no incumbent
        break;
      }
      if (rc == WK_OK) inc_t = std::min(inc_t, ms);
      if (pass == 2) break;
      for (size_t i = 0; i < top && rc == WK_OK; i++)
        if ((rc = time_cfg(timed[i].second, ms)) == WK_OK) timed[i].first = std::min(timed[i].first, ms);
    }
    for (size_t i = 0; i < top; i++)
      if (timed[i].first < best_t) {
        best_t = timed[i].first;
        best_c = timed[i].second;
      }
    if (std::isfinite(inc_t) && !(best_t < 0.99f * inc_t)) {
      best_t = inc_t;
      best_c = b0;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (rc != WK_OK) return rc;
  if (!std::isfinite(best_t)) {
    set_last_error("no launch configuration ran");
    return WK_ERR_ARG;
  }
  {
    std::lock_guard<std::mutex> g(E->cfg_mu);
    E->launch_cfg[cfg_key(op, k)] = best_c;
  }
  if (best) *best = best_c;
  if (best_ms) *best_ms = best_t;
  return WK_OK;
}

}  // extern "C"
