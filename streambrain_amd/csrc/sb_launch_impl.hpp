// Definitions of the launchers declared in sb_launch.hpp; included once per element type by
// sb_kernels_f32.hip / sb_kernels_f64.hip, which instantiate them explicitly.
#pragma once
#include "sb_kernels.hpp"
#include "sb_k_train.hpp"
#include "sb_k_forward_rows.hpp"
#include "sb_k_forward_chains.hpp"
#include "sb_k_skinny.hpp"
#include "sb_launch.hpp"

#include <algorithm>
#include <hip/hip_ext.h>
#include <cstdlib>
#include <type_traits>

namespace sb {

static inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
static inline long cdiv(long a, long b) { return (a + b - 1) / b; }

#define SB_LAUNCH_CHECK() SB_HIP(hipGetLastError())

static inline int device_cu_count() {
  static const int n = [] {
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess) {
      hipDeviceProp_t prop;
      if (hipGetDeviceProperties(&prop, dev) == hipSuccess) cus = prop.multiProcessorCount;
    }
    return cus;
  }();
  return n;
}

// ------------------------------------------------------------------------------------------- forward
template <typename T, int NG, bool FUSE, int LW = Real<T>::VW>
static int forward_variant(hipStream_t st, ForwardArgs<T> a, bool vec) {
  ProfScope prof_(st, K_FORWARD);
  a.by_batch_tiles = FastDiv::of(a.batch_tiles);
  // 8 workgroup ids per round of XCDs; ids beyond the last tile exit at once
  const long ntiles = a.col_tiles * a.batch_tiles;
  const long grid = 8 * cdiv(ntiles, 8);
  if (grid >= (1L << 31)) {
    set_error("launch_forward: too many tiles for one launch");
    return -1;
  }
  if (vec)
    hipLaunchKernelGGL((k_forward<T, NG, FUSE, true, 8, LW>), dim3((unsigned)grid), dim3(512), 0, st, a);
  else
    hipLaunchKernelGGL((k_forward<T, NG, FUSE, false, 8, LW>), dim3((unsigned)grid), dim3(512), 0, st, a);
  SB_LAUNCH_CHECK();
  return 0;
}

// The softmax behind a pass whose hypercolumns are spread over workgroups (TPR: as of the fused kernel it stands in for).
template <typename T, int TPR>
static int launch_softmax_as_fused(hipStream_t st, T *act, long B, long H, long Mc) {
  SB_REQUIRE(Mc <= 16 * TPR, "hypercolumn too wide");
  const long groups = B * H, blocks = cdiv(groups, 256 / TPR);
  SB_REQUIRE(blocks < (1L << 31), "too many groups");
  hipLaunchKernelGGL((k_softmax_as_fused<T, TPR>), dim3((unsigned)blocks), dim3(256), 0, st, act, groups, Mc);
  SB_LAUNCH_CHECK();
  return 0;
}

template <typename T>
int launch_forward(hipStream_t st, T *act, const T *x, const T *W, const T *bias, long B, long N,
                   long H, long Mc, bool softmax, long like) {
  return launch_forward_classify<T>(st, act, x, W, bias, B, N, H, Mc, softmax, nullptr, nullptr, nullptr, like);
}

// The fused kernel runs one workgroup per hypercolumn and 16 batch rows, one workgroup per CU.  For wide
// hypercolumns (more than two column groups) whose tiles fill their last round of workgroups badly,
// tiles of two column groups plus a separate softmax pass are faster (1568 -> Hx200, batch 128, fused
// against separate: H = 16: 31.7 / 23.4 us, H = 30: 33.9 / 40.0, H = 48: 63.4 / 57.1, H = 64: 66.1 / 74.5).
// (The separate pass, k_softmax, has the library's exponential and divides: other bits.)
template <typename T>
static bool forward_fuses(long B, long H, long Mc) {
  const long need = cdiv(Mc, 16 * Real<T>::VW), max_fused = sizeof(T) == 4 ? 4 : 7;
  const long tiles = H * cdiv(B, 16), cus = device_cu_count();
  return need <= max_fused && (need <= 2 || 20 * tiles >= 17 * cdiv(tiles, cus) * cus);
}

template <typename T>
int launch_forward_classify(hipStream_t st, T *act, const T *x, const T *W, const T *bias, long B, long N,
                            long H, long Mc, bool softmax, const T *labels, int32_t *pred,
                            unsigned long long *correct, long like) {
  constexpr int VW = Real<T>::VW;
  constexpr int GW = 16 * VW;
  SB_REQUIRE(act && x && W && bias, "null pointer");
  SB_REQUIRE(B > 0 && N > 0 && H > 0 && Mc > 0, "sizes must be positive");
  const long M = H * Mc;
  SB_REQUIRE(M < (1L << 31) && N < (1L << 31), "dimension too large");
  // A handful of output units: plain vector arithmetic, one workgroup per batch row.  Its time grows with M
  // where the MFMA kernel's is flat (3000 inputs, batch 128: float 7.1 us at M = 10, 15.6 at 32, MFMA 15.9;
  // double 12.2 at 10, 17.2 at 16, 30.9 at 32, MFMA 17.5).
  if (M <= (sizeof(T) == 4 ? 32 : 16)) {
    SB_REQUIRE(B < (1L << 31), "batch too large for one launch");
    ProfScope prof_(st, K_FORWARD);
    SB_REQUIRE(!labels || correct, "labels need a counter");
    hipLaunchKernelGGL((k_forward_skinny<T>), dim3((unsigned)B), dim3(256), 0, st, act, x, W, bias, N, M, Mc,
                       softmax ? 1 : 0, labels, pred, correct);
    SB_LAUNCH_CHECK();
    return 0;
  }
  if (labels || pred) {  // wider layers: the forward pass, then the classification kernel
    int rc = launch_forward<T>(st, act, x, W, bias, B, N, H, Mc, softmax, like);
    if (rc) return rc;
    return launch_argmax_rows<T>(st, act, labels, B, M, pred, correct);
  }
  // per-lane byte offsets inside one chunk of 16 rows of x or W are 32-bit
  SB_REQUIRE(16 * (N > M ? N : M) * (long)sizeof(T) < (1L << 31), "layer too wide for the forward kernel");
  ForwardArgs<T> a{act, x, W, bias, B, N, M, Mc, 0, cdiv(B, 16), {}};
  const bool base_vec = (N % VW == 0) && (M % VW == 0) && aligned16(x) && aligned16(W);
  const long need = cdiv(Mc, GW);
  const long fused_tiles = H * cdiv(B, 16), cus_ = device_cu_count();
  if (softmax && forward_fuses<T>(like > 0 ? like : B, H, Mc)) {
    const bool vec = base_vec && (Mc % VW == 0);
    // Hypercolumns of two column groups whose tiles leave half the CUs idle and that have a long reduction: a
    // workgroup per group, then the softmax.  Every sum as in the fused kernel, except in the four columns that
    // it takes as 4x4 products, so not those.  (Time fused over time this way, 120 tiles: 101 columns, 512 inputs
    // 0.93, 1024 1.13, 2048 1.34, 4096 1.40; doubles, 50 columns 0.92, 1.07, 1.18, 1.27.  2048 inputs, 160 tiles 1.29 and
    // 1.17, 240 tiles, where a CU gets two of these workgroups, 0.76 and 0.68.  The second launch costs 1 to 2 us.)
    const bool tail4 = sizeof(T) == 4 && vec && Mc == 100;
    if (need == 2 && 2 * fused_tiles <= cus_ && N >= 2048 && !tail4) {
      a.col_tiles = cdiv(M, GW);
      int rc = forward_variant<T, 1, false>(st, a, base_vec);
      if (rc) return rc;
      return launch_softmax_as_fused<T, 32>(st, act, B, H, Mc);
    }
    a.col_tiles = H;
    // Hypercolumns that need 7 column blocks of 16 (97..112 columns, e.g. 100).
    const long nblocks = cdiv(Mc, 16);
    if (vec && nblocks == 7) {
      constexpr int NGL = 8 / VW, LWL = 7 - (NGL - 1) * VW;  // float: 2 groups, 3 blocks; double: 4, 1
      // Large batches: 64 or 32 rows per workgroup instead of 16 while there still are enough tiles for
      // eight rounds / one round of workgroups, so that W crosses the L2 -> L1 path a quarter / half as
      // often (64 rows with fewer rounds lose more to the last, partly filled round than they gain).  A vector of
      // the last group may straddle the hypercolumn's end here (1568 -> 30 x 104, 16 rows a workgroup / as many as
      // this says: batch 512 62 / 56 us, 4096 414 / 373; 60 x 104, batch 256 62 / 56).
      const long cus = device_cu_count();
      // (double: at most 32 rows, 64 do not fit the register file)
      long rb = sizeof(T) == 4 && H * cdiv(B, 64) >= 8 * cus ? 4 : (H * cdiv(B, 32) >= cus ? 2 : 1);
      // (32-bit byte offsets inside the tile's rows)
      while (rb > 1 && 16 * rb * N * (long)sizeof(T) >= (1L << 31)) rb /= 2;
      a.batch_tiles = cdiv(B, 16 * rb);
      a.by_batch_tiles = FastDiv::of(a.batch_tiles);
      ProfScope prof_(st, K_FORWARD);
      const long grid = 8 * cdiv(a.col_tiles * a.batch_tiles, 8);
      SB_REQUIRE(grid < (1L << 31), "too many tiles for one launch");
      const dim3 g((unsigned)grid);
      if constexpr (sizeof(T) == 4) {
        // 100 columns = 6 blocks of 16 + 4: the last four as 4x4 products instead of a seventh block
        if (Mc == 6 * 16 + 4) {
          if (rb == 4) hipLaunchKernelGGL((k_forward<T, 2, true, true, 8, 2, 4, true>), g, dim3(512), 0, st, a);
          else if (rb == 2) hipLaunchKernelGGL((k_forward<T, 2, true, true, 8, 2, 2, true>), g, dim3(512), 0, st, a);
          else hipLaunchKernelGGL((k_forward<T, 2, true, true, 8, 2, 1, true>), g, dim3(512), 0, st, a);
          SB_LAUNCH_CHECK();
          return 0;
        }
        if (rb == 4) hipLaunchKernelGGL((k_forward<T, NGL, true, true, 8, LWL, 4>), g, dim3(512), 0, st, a);
      }
      if (rb == 4) {
      } else if (rb == 2)
        hipLaunchKernelGGL((k_forward<T, NGL, true, true, 8, LWL, 2>), g, dim3(512), 0, st, a);
      else
        hipLaunchKernelGGL((k_forward<T, NGL, true, true, 8, LWL>), g, dim3(512), 0, st, a);
      SB_LAUNCH_CHECK();
      return 0;
    }
    // As many blocks of 16 columns as the hypercolumn has, up to 8; wider ones in whole groups.
    auto blocks = [&](auto count) {
      constexpr int NB = decltype(count)::value, NG = (NB + VW - 1) / VW;
      return forward_variant<T, NG, true, NB - (NG - 1) * VW>(st, a, vec);
    };
    switch (nblocks) {
      case 1: return blocks(std::integral_constant<int, 1>{});
      case 2: return blocks(std::integral_constant<int, 2>{});
      case 3: return blocks(std::integral_constant<int, 3>{});
      case 4: return blocks(std::integral_constant<int, 4>{});
      case 5: return blocks(std::integral_constant<int, 5>{});
      case 6: return blocks(std::integral_constant<int, 6>{});
      case 7: return blocks(std::integral_constant<int, 7>{});
      case 8: return blocks(std::integral_constant<int, 8>{});
    }
    if constexpr (sizeof(T) == 4) return forward_variant<T, 4, true>(st, a, vec);
    else return forward_variant<T, 7, true>(st, a, vec);
  }
  // Tiles of two column groups, of one where the former leave half the CUs idle (time of two over time of one, 5 to 128
  // tiles: 64 inputs 1.0 to 1.1, 200 1.3, 300 1.4, 1000 1.55; doubles 1.0, 1.25, 1.3, 1.5; at 192 tiles 0.75 to 0.9 for all)
  const bool narrow = 2 * cdiv(M, 2 * GW) * cdiv(B, 16) <= cus_;
  a.col_tiles = cdiv(M, narrow ? GW : 2 * GW);
  int rc = narrow ? forward_variant<T, 1, false>(st, a, base_vec) : forward_variant<T, 2, false>(st, a, base_vec);
  if (rc) return rc;
  if (softmax) return launch_softmax<T>(st, act, B, H, Mc);
  return 0;
}

// ------------------------------------------------------------------- forward over the connected rows
template <typename T>
bool forward_rows_supported(const T *W, long N, long H, long Mc) {
  constexpr int VW = Real<T>::VW;
  const long M = H * Mc;
  return M > 32 && M % VW == 0 && Mc % VW == 0 && aligned16(W) &&
         cdiv(Mc, 16 * VW) <= (sizeof(T) == 4 ? 4 : 7) && 16 * N * (long)sizeof(T) < (1L << 31);
}

// Column groups of a hypercolumn in k_forward_rows, and column blocks of the last one (LW; 0: whole groups).
struct RowsGroups {
  int n, last;
};
template <typename T>
static RowsGroups forward_rows_groups(long Mc) {
  constexpr int VW = Real<T>::VW, GW = 16 * VW, NGL = 8 / VW, LWL = 7 - (NGL - 1) * VW;
  // hypercolumns of 7 column blocks of 16 (97..112 columns): the last group runs with 3 (float) or 1
  // (double) blocks, provided none of its vectors straddles the end of the hypercolumn (this kernel's loads of W
  // know no bounds)
  if (cdiv(Mc, 16) == 7 && (Mc - (NGL - 1) * GW) % LWL == 0) return {NGL, LWL};
  // and of 13 column blocks (193..208 columns, 200 among them): one block in the last group
  // (float: 4 groups, 12 + 1 blocks; double: 7, 12 + 1)
  if (cdiv(Mc, 16) == 13) return {VW == 2 ? 7 : 4, 1};
  const long need = cdiv(Mc, GW);
  return {need <= 1 ? 1 : need <= 2 ? 2 : need <= 4 ? 4 : 7, 0};
}
// Row blocks per workgroup.  Large batches: 64 or 32 rows while there are tiles for eight rounds / three quarters
// of a round of workgroups (much as in launch_forward), as long as the kernel then still fits two wavefronts per SIMD:
// two workgroups per CU with fewer rows each beat one with more (204 against 240 us at 1568 -> 30x100,
// batch 8192; 70 against 83 us at 1568 -> 100x100 in double, batch 512)
template <typename T>
static int forward_rows_blocks(int groups, long B, long N, long H) {
  const long cus = device_cu_count();
  const bool fits4 = forward_rows_regs<T>(groups, 4) <= kRowsRegsTwoWaves;
  int rb = fits4 && H * cdiv(B, 64) >= 8 * cus ? 4 : (4 * H * cdiv(B, 32) >= 3 * cus ? 2 : 1);
  while (rb > 1 && forward_rows_regs<T>(groups, rb) > kRowsRegsTwoWaves) rb /= 2;
  // (32-bit byte offsets inside the tile's rows)
  while (rb > 1 && 16 * rb * N * (long)sizeof(T) >= (1L << 31)) rb /= 2;
  return rb;
}
// Short lists, few rows: a segment of 256 list entries and partial sums that meet in one step (see the kernel).
template <typename T>
static bool forward_rows_short(long B, long N, long H, long Mc, long cap) {
  return cap <= 256 && forward_rows_blocks<T>(forward_rows_groups<T>(Mc).n, B, N, H) == 1;
}

template <typename T>
bool forward_bits_equal(long B1, long B2, long N, long H, long Mc, long cap) {
  if (cap > 0) return forward_rows_short<T>(B1, N, H, Mc, cap) == forward_rows_short<T>(B2, N, H, Mc, cap);
  return H * Mc <= (sizeof(T) == 4 ? 32 : 16) || forward_fuses<T>(B1, H, Mc) == forward_fuses<T>(B2, H, Mc);
}

// `like`: batch size whose order of sums is taken
template <typename T, int NG, int LW = Real<T>::VW>
static int forward_rows_variant(hipStream_t st, ForwardRowsArgs<T> a, long like) {
  ProfScope prof_(st, K_FORWARD);
  // four wavefronts measured best (8: 8.8 us, 4: 8.2 us, 2: 9.9 us, 16: 10.7 us at 1568 -> 30x100, density 0.1)
  constexpr int NW = 4;
  const long H = a.f.col_tiles, B = a.f.B;
  constexpr bool fits4 = forward_rows_regs<T>(NG, 4) <= kRowsRegsTwoWaves;
  const int rb = forward_rows_blocks<T>(NG, B, a.f.N, H);
  a.f.batch_tiles = cdiv(B, 16 * rb);
  a.f.by_batch_tiles = FastDiv::of(a.f.batch_tiles);
  const long grid = 8 * cdiv(a.f.col_tiles * a.f.batch_tiles, 8);
  SB_REQUIRE(grid < (1L << 31), "too many tiles for one launch");
  const dim3 g((unsigned)grid), blk(64 * NW);
  const bool is_short = forward_rows_short<T>(like, a.f.N, H, a.f.Mc, a.cap);
  const bool wide = a.f.N * a.f.M * (long)sizeof(T) > (1L << 32);
  auto launch_rb = [&](auto blocked, auto row_blocks) {  // (with the batch at hand in blocks of 16 rows, or without)
    constexpr bool XT = decltype(blocked)::value;
    constexpr int RB = decltype(row_blocks)::value;
    if (wide && is_short) hipLaunchKernelGGL((k_forward_rows<T, NG, NW, RB, XT, LW, 256, true>), g, blk, 0, st, a);
    else if (wide) hipLaunchKernelGGL((k_forward_rows<T, NG, NW, RB, XT, LW, 2048, true>), g, blk, 0, st, a);
    else if (is_short) hipLaunchKernelGGL((k_forward_rows<T, NG, NW, RB, XT, LW, 256>), g, blk, 0, st, a);
    else hipLaunchKernelGGL((k_forward_rows<T, NG, NW, RB, XT, LW>), g, blk, 0, st, a);
  };
  auto launch = [&](auto blocked) {
    if constexpr (fits4) {
      if (rb == 4) return launch_rb(blocked, std::integral_constant<int, 4>{});
    }
    if constexpr (forward_rows_regs<T>(NG, 2) <= kRowsRegsTwoWaves) {
      if (rb == 2) return launch_rb(blocked, std::integral_constant<int, 2>{});
    }
    launch_rb(blocked, std::integral_constant<int, 1>{});
  };
  if (a.xt) launch(std::true_type{});
  else launch(std::false_type{});
  SB_LAUNCH_CHECK();
  return 0;
}

// Few tiles: a workgroup of k_forward_rows per column group of a hypercolumn, then the softmax, every sum as in the fused
// kernel.  The second launch costs about a microsecond.  Time this way over time fused, at 8 / 40 / 80 / 128 / 152 tiles:
// 100 columns, lists of 300 1.09 / 1.11 / 1.12 / 1.13 / -, of 600 0.95 / 0.95 / 0.96 / 0.97 / 1.19, of 6000 0.68 / 0.67 / 0.69 /
// 0.71 / 1.07; 200 columns, lists of 300 0.81 / 0.82 / 0.94 / 0.99 / -, of 6000 0.41 / 0.42 / 0.66 / 0.72 / 0.94; doubles, 64
// columns, lists of 300 1.12 / 1.13 / 1.13 / 1.14 / -, of 600 0.98 / 0.98 / 1.00 / 1.01 / 1.19, of 6000 0.84 / 0.85 / 0.86 / 0.87
// / 1.06; 128 columns, lists of 300 0.82 / 0.85 / 0.97 / 0.99 / -, of 1200 0.54 / 0.62 / 0.76 / 0.77 / 0.93, of 6000 0.50 / 0.51 /
// 0.63 / 0.65 / 0.83.
template <typename T>
static bool forward_rows_splits(long B, long H, long Mc, long cap) {
  const long tiles = H * cdiv(B, 16), cus = device_cu_count(), blocks = cdiv(Mc, 16);
  if (blocks <= Real<T>::VW || cap <= 256) return false;  // (one column group; lists that may be summed in another order)
  if (2 * tiles <= cus) return cap >= 608 || blocks >= (sizeof(T) == 4 ? 10 : 8);
  return sizeof(T) == 8 && blocks >= 7 && 5 * tiles <= 3 * cus && cap >= 1280;
}

// How k_forward_chains covers a pass; no workgroups: it does not run.
template <typename T>
struct ChainsPlan {
  long workgroups = 0;
  int waves = 4;
  ForwardChainsArgs<T> args{};
};
// Pieces of a hypercolumn: as many (of one to four blocks of 16 columns) as workgroups of four wavefronts find a CU each;
// where even the fewest do not, workgroups of eight, whose wavefronts share the CU's SIMDs evenly.
template <typename T>
static ChainsPlan<T> forward_chains_plan(long B, long N, long H, long Mc, long cap, long like) {
  ChainsPlan<T> plan;
  const long M = H * Mc, cus = device_cu_count(), rbs = cdiv(B, 16), tiles = H * rbs;
  if (forward_rows_short<T>(like > 0 ? like : B, N, H, Mc, cap)) return plan;  // (another order of the four sums)
  if (N * M * (long)sizeof(T) > (1L << 32)) return plan;
  const long blocks = cdiv(Mc, 16), fewest = cdiv(blocks, 4);
  const bool few = 6 * tiles <= cus;
  if (2 * tiles > (blocks == 1 ? 3 * cus : cus)) return plan;
  // One and two blocks of columns: where the lists pay for the second launch (time of k_forward_rows over time this way:
  // 12 columns, lists of 2400 0.84, of 3600 0.88 at 36 tiles, 1.1 from 112, of 6000 0.95 at 16, 1.25 from 40; 32 columns, of 900
  // 0.9 to 0.98, of 1800 1.2; doubles, 12 columns, of 1800 0.82 up to 48 tiles, 1.08 from 112, of 3600 1.35; 32 columns, of 900
  // 0.88, of 1800 1.08 to 1.19).
  if (blocks <= 2) {
    const long from = blocks == 2 ? (sizeof(T) == 4 ? 1152 : 1408)
                                  : sizeof(T) == 4 ? (few ? 6016 : 3600) : (few ? 3072 : 1792);
    if (cap < from) return plan;
  } else if (cap < 640) {
    return plan;
  }
  ForwardChainsArgs<T> &c = plan.args;
  c.waves_rows = rbs >= 4 ? 4 : rbs >= 2 ? 2 : 1;
  c.row_groups = (int)cdiv(rbs, c.waves_rows);
  auto groups = [&](long pieces) { return cdiv(pieces, std::min<long>(4 / c.waves_rows, pieces)); };
  const long around = H * c.row_groups * kChains;
  long pieces = blocks;
  while (pieces > fewest && around * groups(pieces) > cus) pieces--;
  c.pieces = (int)pieces;
  c.waves_cols = (int)std::min<long>(4 / c.waves_rows, pieces);
  if (around * groups(pieces) > cus) {
    plan.waves = 8;
    if (2 * c.waves_cols <= c.pieces) c.waves_cols *= 2;
    else c.waves_rows *= 2, c.row_groups = (int)cdiv(rbs, c.waves_rows);
  }
  c.col_groups = (int)cdiv(c.pieces, c.waves_cols);
  const long workgroups = H * kChains * c.row_groups * c.col_groups;
  if (blocks > 2) {
    // Wider hypercolumns: which way the fullest CU is done first, by what 1300 shapes took (3 to 14 blocks, 8 to 128
    // tiles, lists of 600 to 15800): microseconds per list entry, and per entry and block that a SIMD has in all (this way:
    // wavefronts of a SIMD times blocks of a piece; k_forward_rows: workgroups on a CU, three at a time), and per million
    // logits that pass through memory.  Estimates are within a tenth of the measured times in nine of ten; the way they choose
    // is on average 0.7 % slower than the better one, k_forward_rows alone 13 % (doubles, 80 tiles of 200 columns, lists of
    // 1200: 25.5 us there, 33.8 this way; 14 blocks of 16 batch rows, which fill neither, 9 x 160 columns, lists of 3600:
    // 59 and 93; 27648 -> 15 x 200, lists of 15800, batch 128: 162 and 134).
    const double L = (double)(cap - 24), logits = 1e-6 * (double)(B * M);  // (a list and its padding)
    const long on_cu = cdiv(workgroups, cus) * (plan.waves / 4);
    const double load = (double)(on_cu * cdiv(blocks, pieces));
    const bool f = sizeof(T) == 4;
    const double here = f ? 7.1 + L * (0.0014 + 0.00087 * load - (on_cu > 1 ? 0.0008 : 0)) + 19 * logits
                          : 8.1 + L * (0.0025 + 0.0016 * load - (on_cu > 1 ? 0.0006 : 0)) + 27 * logits;
    double there;
    if (blocks <= Real<T>::VW) {
      there = 3.9 + L * (0.0023 + 0.00083 * (double)blocks);
    } else {
      const long all = tiles * cdiv(blocks, Real<T>::VW), rounds = cdiv(all, 3 * cus);
      const double load_there = (double)(3 * (rounds - 1) + cdiv(all - 3 * cus * (rounds - 1), cus));
      there = f ? 6.2 + L * (0.0016 * (double)rounds + 0.0039 * load_there) + 4.3 * logits
                : 4.9 + L * (0.0053 * (double)rounds + 0.0028 * load_there) + 15 * logits;
    }
    if (here >= there) return plan;
  }
  plan.workgroups = workgroups;
  return plan;
}
template <typename T>
size_t forward_rows_bytes(long B, long N, long H, long Mc, long cap, long like) {
  if (B <= 0 || N <= 0 || H <= 0 || Mc <= 0 || H * Mc >= (1L << 31) || N >= (1L << 31)) return 0;
  return forward_chains_plan<T>(B, N, H, Mc, cap, like).workgroups > 0 ? kChains * sizeof(T) * (size_t)B * (size_t)(H * Mc) : 0;
}

template <typename T>
int launch_forward_rows(hipStream_t st, T *act, const T *x, const T *W, const T *bias, const int *rows,
                        const int *row_cnt, long cap, long B, long N, long H, long Mc, const T *x_blocked, long like,
                        void *scratch) {
  SB_REQUIRE(act && x && W && bias && rows && row_cnt, "null pointer");
  SB_REQUIRE(B > 0 && N > 0 && H > 0 && Mc > 0, "sizes must be positive");
  SB_REQUIRE(H * Mc < (1L << 31) && N < (1L << 31), "dimension too large");
  SB_REQUIRE(cap > 0 && cap % 16 == 0, "row lists must be padded to a multiple of 16");
  SB_REQUIRE(forward_rows_supported<T>(W, N, H, Mc), "shape not supported by the row-list forward kernel");
  ForwardRowsArgs<T> a{{act, x, W, bias, B, N, H * Mc, Mc, H, cdiv(B, 16), {}}, rows, row_cnt, cap, x_blocked};
  if (scratch) {
    ChainsPlan<T> plan = forward_chains_plan<T>(B, N, H, Mc, cap, like);
    if (plan.workgroups > 0) {
      ProfScope prof_(st, K_FORWARD);
      plan.args.r = a;
      plan.args.part = (T *)scratch;
      const dim3 g((unsigned)(8 * cdiv(plan.workgroups, 8))), blk(64 * plan.waves);
      const bool mixed = plan.args.waves_cols > 1 && cdiv(Mc, 16) % plan.args.pieces != 0;
      if (x_blocked && mixed) hipLaunchKernelGGL((k_forward_chains<T, true, true>), g, blk, 0, st, plan.args);
      else if (x_blocked) hipLaunchKernelGGL((k_forward_chains<T, true, false>), g, blk, 0, st, plan.args);
      else if (mixed) hipLaunchKernelGGL((k_forward_chains<T, false, true>), g, blk, 0, st, plan.args);
      else hipLaunchKernelGGL((k_forward_chains<T, false, false>), g, blk, 0, st, plan.args);
      SB_LAUNCH_CHECK();
      hipLaunchKernelGGL((k_softmax_of_chains<T>), dim3((unsigned)cdiv(B * H, 8)), dim3(128), 0, st, act,
                         (const T *)plan.args.part, bias, B, H, Mc);
      SB_LAUNCH_CHECK();
      return 0;
    }
  }
  constexpr int VW = Real<T>::VW, GW = 16 * VW;
  if (forward_rows_splits<T>(B, H, Mc, cap)) {
    ProfScope prof_(st, K_FORWARD);
    a.f.by_batch_tiles = FastDiv::of(a.f.batch_tiles);
    const dim3 g((unsigned)(8 * cdiv(H * a.f.batch_tiles, 8)), (unsigned)cdiv(Mc, GW)), blk(256);
    const bool wide = N * H * Mc * (long)sizeof(T) > (1L << 32);
    auto launch = [&](auto blocked) {
      constexpr bool XT = decltype(blocked)::value;
      if (wide) hipLaunchKernelGGL((k_forward_rows<T, 1, 4, 1, XT, VW, 2048, true, true>), g, blk, 0, st, a);
      else hipLaunchKernelGGL((k_forward_rows<T, 1, 4, 1, XT, VW, 2048, false, true>), g, blk, 0, st, a);
    };
    if (x_blocked) launch(std::true_type{});
    else launch(std::false_type{});
    SB_LAUNCH_CHECK();
    return launch_softmax_as_fused<T, 16>(st, act, B, H, Mc);
  }
  if (like <= 0) like = B;
  constexpr int NGL = 8 / VW, LWL = 7 - (NGL - 1) * VW, NGM = VW == 2 ? 7 : 4;
  const RowsGroups groups = forward_rows_groups<T>(Mc);
  if (groups.last > 0 && cdiv(Mc, 16) == 7) return forward_rows_variant<T, NGL, LWL>(st, a, like);
  if (groups.last > 0) return forward_rows_variant<T, NGM, 1>(st, a, like);
  if (Mc <= 16) return forward_rows_variant<T, 1, 1>(st, a, like);  // (one block of columns)
  if (groups.n == 1) return forward_rows_variant<T, 1>(st, a, like);
  if (groups.n == 2) return forward_rows_variant<T, 2>(st, a, like);
  if (groups.n == 4) return forward_rows_variant<T, 4>(st, a, like);
  if constexpr (sizeof(T) == 8) return forward_rows_variant<T, 7>(st, a, like);
  return -1;
}

template <typename T>
int launch_softmax(hipStream_t st, T *act, long B, long H, long Mc) {
  SB_REQUIRE(act, "null pointer");
  SB_REQUIRE(B > 0 && H > 0 && Mc > 0, "sizes must be positive");
  const long groups = B * H;
  SB_REQUIRE(cdiv(groups, 4) < (1L << 31), "too many groups");
  ProfScope prof_(st, K_SOFTMAX);
  hipLaunchKernelGGL((k_softmax<T>), dim3((unsigned)cdiv(groups, 4)), dim3(256), 0, st, act, groups,
                     Mc);
  SB_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------------------------------- fused training
// One round of workgroups: every one finds a slot at once (five per CU for floats of whole vectors, else four).
template <typename T>
static long train_tiles_of_one_round() { return (long)train_waves_per_simd<T, true, 1>() * device_cu_count(); }

// Floats go through k_trace_sums<float, true> and k_train_split in layers of 2.5 rounds of 64 x 64 tiles and more where
// that is faster, sums included (the numbers: time of whole steps with k_train_fused over that with k_train_split, at
// 96 to 20000 columns, 100 to 700 MiB of Cij and W, 32 to 600 batch rows):
//   Cij and W beyond the memory-side cache: any batch (from 32 rows, see k_train_split: 12670 x 3000 1.7, 9500 x 4000
//   1.3, 3800 x 10000 1.7; 64 rows 2.2, 1.2, 1.7; 300 rows 2.0, 1.6, 1.7).  In it the matrix instructions have to
//   gain what the split costs: rows that are no whole number of 128-byte lines from 65 rows (77 rows, 4600 to 8700 x
//   3000 0.99 to 1.06, 2929 columns 1.10 to 1.15; 64 rows 0.98 to 0.99 and 1.0), others from 97 (100 rows, 3440 to 6550 x
//   4000 1.03 to 1.10, 128 rows 1.05 to 1.10; 77 rows 0.97 to 1.00, 33 rows 0.89 to 0.92);
//   not for few columns, between which the split of x cannot be shared out: from 192 columns (200: 1.0 to 2.0, below 100
//   MB or beyond 200 rows down to 0.95; 100 columns: 0.7 to 1.2), or from 640 where rows are whole lines (640: 0.94 at 700
//   MB to 1.4; 320: 0.8 to 1.15), which k_train_fused writes at full rate.
// The layers below the 2.5 rounds, which train for epochs in moments, keep the rounding of their trajectories (after a
// few dozen steps those tell one order of sums from another); there are up to 15 % to gain there.
// Its windows hold 128 rows of Cij and 32 split batch rows.
template <typename T>
size_t train_split_bytes(long B, long N, long H, long Mc) {
  if constexpr (sizeof(T) != 4) return 0;
  if (B < kSplitBatch || N <= 0 || H <= 0 || Mc <= 0) return 0;
  const long M = H * Mc;
  const bool whole_lines = M % 32 == 0;
  if (M < (whole_lines ? 640 : 192) || 2 * cdiv(N, 64) * cdiv(M, 64) < 5 * train_tiles_of_one_round<T>()) return 0;
  const bool cached = 2 * N * M * (long)sizeof(T) <= (256L << 20);
  if (cached && B <= (whole_lines ? 96 : 64)) return 0;
  const long xw = cdiv(N, kSplitTileI) * kSplitTileI, yw = cdiv(M, kSplitTileJ) * kSplitTileJ;
  const long wider = xw > yw ? xw : yw;
  if (128 * M * 4 >= (1L << 31) || wider * (kSplitRows / 8) * 3 * 16 >= (1L << 31)) return 0;
  return (size_t)(xw + yw) * 6 * (size_t)(cdiv(B, kSumRows) * kSumRows) + (size_t)(xw + yw) / 64 * sizeof(int);
}

// x^T y through the pieces: the scratch is there, the layer is one for it, and the factor of the sums stays normal with the
// pieces' scale in it.
template <typename T>
static bool train_splits(const void *split, long B, long N, long H, long Mc, T tau) {
  return sizeof(T) == 4 && split && train_split_bytes<T>(B, N, H, Mc) > 0 &&
         (float)((T)1 / (T)B * tau) * kSplitUnscale >= 0x1p-126f;
}

// Every tile adds up the batch's x and y columns for its own rows and columns, which with many tile
// rows and columns is most of the kernel's vector arithmetic (43 % at 65536 x 100000, batch 1024).
// From one and a half rounds of workgroups on (floats with more than 32 rows; doubles: two and a half), a small launch
// computes the new traces once and the tiles read them (floats: where k_train_split does not run).  Timed, 4096
// inputs, batch 128, floats, with / without that launch: 23.7 / 22.5 us at 1.05 rounds, 29.3 / 29.9 at 1.5, 34.6 /
// 35.6 at 2, 45.5 / 48.5 at 3, 67.1 / 69.2 at 5; doubles: 48.1 / 47.3 at 1.6 rounds, 55.8 / 54.3 at 2, 110.3 /
// 113.7 at 2.5.  (Whole vectors only.)
template <typename T>
static bool train_sums_apart(long B, long N, long H, long Mc) {
  const long pre_from = sizeof(T) == 8 ? 5 * 4 : 3 * 5;  // in half workgroups per CU
  return H * Mc > 32 && Mc % Real<T>::VW == 0 &&
         2 * cdiv(N, 64) * cdiv(H * Mc, 64) >= pre_from * device_cu_count() && (sizeof(T) == 8 || B > 32);
}
// A launch of its own that forms the traces reads and writes each once, in one thread, and nobody else reads the old ones.
template <typename T>
bool train_in_place_supported(const void *split, long B, long N, long H, long Mc, T taupdt) {
  if (B <= 0 || N <= 0 || H <= 0 || Mc <= 0) return false;
  return train_splits<T>(split, B, N, H, Mc, TraceScalars<T>::from(taupdt, T(0)).tau) || train_sums_apart<T>(B, N, H, Mc);
}

template <typename T>
int launch_train_fused(hipStream_t st, const T *x, const T *y, T *Cij, T *W, const T *Ci, const T *Cj,
                       T *Ci_next, T *Cj_next, const uint8_t *wmask, int bias_mode, T *bias, T *kbi,
                       long B, long N, long H, long Mc, T taupdt, T cthr, T khalf, T pmin, T taubdt,
                       bool w_masked, const void *prefetch, size_t prefetch_bytes, void *split) {
  constexpr int VW = Real<T>::VW;
  SB_REQUIRE(x && y && Cij && Ci && Cj && Ci_next && Cj_next, "null pointer");  // W may be null: traces only
  SB_REQUIRE(bias_mode == 0 || (bias && kbi), "bias update needs bias and kbi");
  const bool in_place = Ci == Ci_next && Cj == Cj_next;
  SB_REQUIRE(in_place || (Ci != Ci_next && Cj != Cj_next), "old and new traces: the same buffers or distinct ones");
  SB_REQUIRE(B > 0 && N > 0 && H > 0 && Mc > 0, "sizes must be positive");
  const long M = H * Mc;
  SB_REQUIRE(M < (1L << 31) && N < (1L << 31) && B < (1L << 31), "dimension too large");
  const TraceScalars<T> s = TraceScalars<T>::from(taupdt, cthr);
  TrainArgs<T> a;
  a.x = x; a.y = y; a.Cij = Cij; a.W = W; a.Ci = Ci; a.Cj = Cj; a.Ci_next = Ci_next; a.Cj_next = Cj_next;
  a.wmask = wmask; a.w_masked = (wmask && w_masked) ? 1 : 0;
  a.bias_mode = bias_mode; a.bias = bias; a.kbi = kbi;
  a.B = B; a.N = N; a.M = M; a.H = H; a.Mc = Mc;
  a.tau = s.tau; a.omt = s.omt; a.fB = (T)B; a.invB = (T)1 / (T)B; a.cthr = s.cthr; a.cthr4 = s.cthr4;
  // traces up to cthr^2 * 2^48 keep every argument max(Cij, cthr^4) / (Ci Cj) of the float weight
  // logarithm at or above 2^-96; doubles have no such limit
  if constexpr (sizeof(T) == 4) a.lim = s.cthr * s.cthr * 0x1p48f;
  else a.lim = (T)INFINITY;
  a.khalf = khalf; a.pmin = pmin; a.taubdt = taubdt;
  a.tiles_i = cdiv(N, 64); a.tiles_j = cdiv(M, 64);
  // tile order (see the kernel): column-major while a batch of x fits an L2 with room to spare, beyond that
  // panels of 16 tile columns while a panel's y slabs (16 x 64 columns of the batch) stay within 2 MiB, else
  // of 8.  x is fetched once per panel: at 55296 x 20000, batch 256, 7.0 GB per launch with panels of 8, 5.7 GB
  // with 16 (32: 5.8 GB); the launch takes the same time either way (4.41 / 4.43 / 4.40 ms), it is not bound by
  // that traffic.
  const bool wide_panels = 16L * 64 * B * (long)sizeof(T) <= (2L << 20);
  a.panel_cols = B * N * (long)sizeof(T) > (2L << 20) ? (wide_panels ? 16u : 8u) : 1u;
  a.by_panel = FastDiv::of(a.tiles_i * a.panel_cols); a.by_Mc = FastDiv::of(Mc);
  // (a region beyond 64 MiB would push more out of the memory-side cache than it brings in)
  const bool pf = prefetch && prefetch_bytes > 0 && prefetch_bytes <= ((size_t)64 << 20);
  a.prefetch = pf ? prefetch : nullptr;
  a.prefetch_bytes = pf ? (unsigned)prefetch_bytes : 0u;
  a.prefetch_lines = (a.prefetch_bytes + 127) / 128;
  // a line per thread: what limits a cold fetch is how many misses one CU keeps in flight (a single workgroup
  // needs 29 us for the 6272 lines of a 128 x 1568 float batch, 25 workgroups on as many CUs finish inside the
  // tiles' 15 us), so the lines are spread over as many workgroups as there are lines / 256, at most 512
  // (a multiple of 8: they come first in the grid, and the tiles behind them keep their XCDs)
  a.prefetch_groups = a.prefetch_lines ? (unsigned)std::min<long>(512, 8 * cdiv(a.prefetch_lines, 8 * 256)) : 0u;
  if (M <= 32) {  // a handful of output units: plain vector arithmetic
    SB_REQUIRE(!in_place, "traces of this layer cannot be updated in place");
    const long rows = skinny_train_rows(M);
    SB_REQUIRE(cdiv(N, rows) < (1L << 31), "too many rows for one launch");
    ProfScope prof_(st, K_TRAIN_FUSED, true);
    // batch rows staged per chunk (see the kernel)
    long bc = kSkinnyLoads * (256 / rows) < kSkinnyLoads * (256 / M) ? kSkinnyLoads * (256 / rows) : kSkinnyLoads * (256 / M);
    if (bc > kSkinnyStage / (rows + M)) bc = kSkinnyStage / (rows + M);
    if (bc > ((1L << 31) - 1) / (N * (long)sizeof(T))) bc = ((1L << 31) - 1) / (N * (long)sizeof(T));
    if (bc > B) bc = B;
    SB_REQUIRE(bc >= 1, "layer too wide for the small-output training kernel");
    if (prof_.carries())
      hipExtLaunchKernelGGL((k_train_skinny<T>), dim3((unsigned)cdiv(N, rows)), dim3(256), 0, st, prof_.start(),
                            prof_.stop(), 0, a, (int)bc);
    else
      hipLaunchKernelGGL((k_train_skinny<T>), dim3((unsigned)cdiv(N, rows)), dim3(256), 0, st, a, (int)bc);
    SB_LAUNCH_CHECK();
    return 0;
  }
  SB_REQUIRE(a.tiles_i * a.tiles_j < (1L << 31) - 8, "too many tiles for one launch");
  // the kernel addresses a chunk of x and y rows and one 64-row band of Cij / W through buffer windows
  // with 32-bit offsets
  SB_REQUIRE(64 * (N > M ? N : M) * (long)sizeof(T) <= (1L << 31),
             "layer too wide: 64 rows of it must stay below 2 GiB");
  // 16-byte stores of Cij and W need rows that are whole vectors (a vector must not run into the next
  // row); loads are 16-byte accesses for every shape, and neither needs more than element alignment
  const bool vec = M % VW == 0;
  // one workgroup per tile (+ the few that prefetch, which the kernel tells apart by their index)
  const dim3 grid((unsigned)(a.tiles_i * a.tiles_j) + a.prefetch_groups);
  // batch rows per turn of two chunks.  Floats: 32, 18 KiB of LDS per workgroup, so five workgroups share a
  // CU.  Doubles: 16 -- the staging registers of two chunks of 8 rows leave the kernel without spills at four
  // wavefronts per SIMD (1 % faster than 32 at 1568 x 10000, batch 512).
  constexpr int KCH = sizeof(T) == 8 ? 16 : 32;
  const bool one_byte = Mc % VW == 0;  // every vector of VW columns lies inside one hypercolumn
  ProfScope prof_(st, K_TRAIN_FUSED, true);
  // one launch, or the sum launch and the tile launch, with the profile's events riding on them
  auto launch = [&](auto kernel, dim3 g, bool first, bool last, auto... more) {
    if (prof_.carries())
      hipExtLaunchKernelGGL(kernel, g, dim3(256), 0, st, first ? prof_.start() : nullptr,
                            last ? prof_.stop() : nullptr, 0, a, more...);
    else
      hipLaunchKernelGGL(kernel, g, dim3(256), 0, st, a, more...);
  };
  const dim3 sums((unsigned)(cdiv(N, 64) + cdiv(M, 64)));
  if constexpr (sizeof(T) == 4) {
    if (train_splits<T>(split, B, N, H, Mc, a.tau)) {
      SplitBatch sp;
      sp.x_width = (unsigned)(cdiv(N, kSplitTileI) * kSplitTileI);
      sp.y_width = (unsigned)(cdiv(M, kSplitTileJ) * kSplitTileJ);
      sp.x = (const bf16x8 *)split;
      const long octets = cdiv(B, kSumRows) * kSumRows / 8;
      sp.y = sp.x + octets * 3 * sp.x_width;
      sp.x_odd = (const int *)(sp.y + octets * 3 * sp.y_width);
      sp.y_odd = sp.x_odd + sp.x_width / 64;
      a.tiles_i = cdiv(N, kSplitTileI);
      a.tiles_j = cdiv(M, kSplitTileJ);
      // (always in panels: column by column the split batch of x, six bytes a value, does not stay in an L2: 5570 x 4000,
      // batch 100, 1.25 times the time)
      a.panel_cols = wide_panels ? 16u : 8u;
      a.by_panel = FastDiv::of(a.tiles_i * a.panel_cols);
      launch(k_trace_sums<T, true>, sums, true, false, sp);
      const dim3 tiles((unsigned)(a.tiles_i * a.tiles_j) + a.prefetch_groups);
      // Non-temporal loads of Cij from 320 MiB of it (time without over with them: rows of whole lines, 4000 to 20000
      // columns, 100 to 256 batch rows, 244 MiB 0.99, 343 MiB 1.06 to 1.08, 600 MiB to 4.2 GiB 1.05 to 1.23; 32 batch rows
      // 1.0; 6000 columns, 1.1 GiB 1.07), where rows are whole half lines or many batch rows pass by (3000 to 13400
      // columns, 256 and 300 rows 1.05 to 1.12; up to 128 rows, 450 MiB to 1.1 GiB, 0.77 to 0.89).
      const bool stream = N * M * (long)sizeof(T) > (320L << 20) && (M % 16 == 0 || B >= 192);
      auto launch_tiles = [&](auto streamed) {
        constexpr bool S = decltype(streamed)::value;
        if (vec && one_byte) launch(k_train_split<true, 1, S>, tiles, false, true, sp);
        else if (vec) launch(k_train_split<true, VW, S>, tiles, false, true, sp);
        else launch(k_train_split<false, VW, S>, tiles, false, true, sp);  // (one_byte implies vec)
      };
      if (stream) launch_tiles(std::true_type{});
      else launch_tiles(std::false_type{});
      SB_LAUNCH_CHECK();
      return 0;
    }
  }
  const long ntiles = a.tiles_i * a.tiles_j;
  const bool one_round = ntiles <= train_tiles_of_one_round<T>();
  const bool apart = train_sums_apart<T>(B, N, H, Mc);
  SB_REQUIRE(!in_place || apart, "traces of this layer cannot be updated in place");
  if constexpr (sizeof(T) == 8) {
    // Cij and W together beyond what the memory-side cache keeps: non-temporal stores (whole steps, batch 128, written
    // through / non-temporal: 7208 x 3000, 330 MiB, 190 / 141 us, 9174 x 3000, 420 MiB, 238 / 180, 20000 rows
    // 1364 / 626; rows of whole cache lines, 10000 columns, batch 512, 239 MiB 412 / 407, batch 128, 420 MiB 190 / 177;
    // time written through over time non-temporal between batches of 16 and 300: at 220 MiB 0.9 to 1.1, at 235
    // 0.95 to 1.4, at 265 1.0 to 1.6)
    if (2 * N * M * (long)sizeof(T) > (230L << 20) && (!vec || one_byte)) {
      if (vec) {
        launch(k_trace_sums<T>, sums, true, false, SplitBatch{});
        launch(k_train_fused<T, KCH, true, 1, true, false, true>, grid, false, true);
      } else {
        launch(k_train_fused<T, KCH, false, VW, false, false, true>, grid, true, true);
      }
      SB_LAUNCH_CHECK();
      return 0;
    }
  }
  if (apart) {
    launch(k_trace_sums<T>, sums, true, false, SplitBatch{});
    launch(k_train_fused<T, KCH, true, 1, true>, grid, false, true);
  } else if (vec && one_byte && one_round)
    launch(k_train_fused<T, KCH, true, 1, false, true>, grid, true, true);
  else if (vec && one_byte)
    launch(k_train_fused<T, KCH, true, 1>, grid, true, true);
  else if (vec)
    launch(k_train_fused<T, KCH, true, VW>, grid, true, true);
  else if (one_byte)
    launch(k_train_fused<T, KCH, false, 1>, grid, true, true);
  else
    launch(k_train_fused<T, KCH, false, VW>, grid, true, true);
  SB_LAUNCH_CHECK();
  return 0;
}

template <typename T>
bool train_skinny_epoch_supported(long M) { return M <= 32; }
// Floats and up to 16 units: always (whole epochs of 4096 to 8192 rows, time of a launch per batch, shuffled inputs included,
// over time of one launch, at batches of 16 / 128 / 512 / 2048 rows: 784 x 10 7.0 / 4.2 / 2.8 / 2.3, 3000 x 10 6.9 / 4.4 / 3.0
// / 2.4, 20000 x 32 2.0 / 1.6 / 1.2 / 1.1, 50000 x 32 - / 1.5 / 1.2 / 1.1; doubles 3000 x 10 7.8 / 4.3 / 3.0 / 2.5, 50000 x
// 16 - / 2.7 / 2.0 / 1.9).  Doubles of 17 to 32 units are bound by what the fullest CU has to do either way, and a workgroup
// here has three quarters of the rows that one of k_train_skinny has: batches of 768 rows and more, which share the cost of
// their launch among many rows, only where that leaves the fullest CU at most 4/3 as many workgroups (time as above,
// at 512 / 768 / 1024 / 4096 rows: 3000 x 32, 2 and 2 of them, 1.29 / 1.28 / 1.23 / 1.15; 6000 x 28, 4 and 3, 1.20 / 1.16
// / 1.12 / 1.02; 50000 x 32, 33 and 25, 1.10 / - / 1.03 / 0.99; 20000 x 32, 14 and 10, 1.05 / - / 0.99 / 0.94; 8000 x 28, 6
// and 4, 0.98 / 0.94 / 0.91 / 0.82; 4000 x 25, 3 and 2, 0.99 / 0.93 / 0.90 / 0.81).
template <typename T>
bool train_skinny_epoch_pays(long B, long N, long M) {
  if (!train_skinny_epoch_supported<T>(M)) return false;
  if (sizeof(T) == 4 || M <= 16 || B < 768) return true;
  const long cus = device_cu_count();
  const long here = cdiv(cdiv(N, skinny_epoch_rows(M)), cus), there = cdiv(cdiv(N, skinny_train_rows(M)), cus);
  return 3 * here <= 4 * there;
}

template <typename T>
int launch_train_skinny_epoch(hipStream_t st, const T *x, const int64_t *order, const T *y, T *Cij, T *W, const T *Ci,
                              const T *Cj, T *Ci_next, T *Cj_next, long B, long rows, long N, long H, long Mc, T taupdt,
                              T cthr) {
  SB_REQUIRE(x && order && y && Cij && W && Ci && Cj && Ci_next && Cj_next, "null pointer");
  SB_REQUIRE(Ci != Ci_next && Cj != Cj_next, "old and new traces must be distinct buffers");
  SB_REQUIRE(B > 0 && rows > 0 && N > 0 && H > 0 && Mc > 0, "sizes must be positive");
  const long M = H * Mc;
  SB_REQUIRE(train_skinny_epoch_supported<T>(M), "too many units");
  SB_REQUIRE(rows < (1L << 31), "too many rows");
  const TraceScalars<T> s = TraceScalars<T>::from(taupdt, cthr);
  SkinnyEpochArgs<T> e{};
  TrainArgs<T> &a = e.a;
  a.x = x; a.y = y; a.Cij = Cij; a.W = W; a.Ci = Ci; a.Cj = Cj; a.Ci_next = Ci_next; a.Cj_next = Cj_next;
  a.B = B < rows ? B : rows; a.N = N; a.M = M; a.H = H; a.Mc = Mc;
  a.tau = s.tau; a.omt = s.omt; a.fB = (T)a.B; a.invB = (T)1 / (T)a.B; a.cthr = s.cthr; a.cthr4 = s.cthr4;
  e.order = order;
  e.rows = rows;
  const long last = rows - (cdiv(rows, a.B) - 1) * a.B;
  e.fB_last = (T)last; e.invB_last = (T)1 / (T)last;
  const long groups = cdiv(N, skinny_epoch_rows(M));
  SB_REQUIRE(groups < (1L << 31) - 8, "too many rows for one launch");
  ProfScope prof_(st, K_TRAIN_FUSED, true);
  const dim3 g((unsigned)(8 * cdiv(groups, 8)));
  auto launch = [&](auto kernel) {
    if (prof_.carries()) hipExtLaunchKernelGGL(kernel, g, dim3(512), 0, st, prof_.start(), prof_.stop(), 0, e);
    else hipLaunchKernelGGL(kernel, g, dim3(512), 0, st, e);
  };
  if (M <= 16) launch(k_train_skinny_epoch<T, 16>);
  else launch(k_train_skinny_epoch<T, 32>);
  SB_LAUNCH_CHECK();
  return 0;
}

template <typename T>
int launch_weights_from_traces(hipStream_t st, T *W, const T *Ci, const T *Cj, const T *Cij, const uint8_t *wmask,
                               T cthr, long N, long H, long Mc, bool w_masked) {
  SB_REQUIRE(W && Ci && Cj && Cij, "null pointer");
  SB_REQUIRE(N > 0 && H > 0 && Mc > 0, "sizes must be positive");
  const long M = H * Mc;
  SB_REQUIRE(M < (1L << 31) && N < (1L << 31), "dimension too large");
  const TraceScalars<T> s = TraceScalars<T>::from(T(0), cthr);
  ProfScope prof_(st, K_WEIGHT_PASS);
  constexpr int VW = Real<T>::VW;
  // 16-byte vectors that lie inside one row (and one hypercolumn), and a turn's rows inside one window
  if (M % VW == 0 && (!wmask || Mc % VW == 0) && kRowsPerTurn * M * (long)sizeof(T) < (1L << 31)) {
    const long turns = cdiv(N, kRowsPerTurn);
    const dim3 grid((unsigned)cdiv(M, 256 * VW), (unsigned)(turns < 32768 ? turns : 32768));
    if (wmask)
      hipLaunchKernelGGL((k_weight_pass<T, true>), grid, dim3(256), 0, st, W, Ci, Cj, Cij, wmask, cthr, s.cthr4, N, M,
                         H, FastDiv::of(Mc), w_masked ? 1 : 0);
    else
      hipLaunchKernelGGL((k_weight_pass<T, false>), grid, dim3(256), 0, st, W, Ci, Cj, Cij, wmask, cthr, s.cthr4, N, M,
                         H, FastDiv::of(Mc), 0);
    SB_LAUNCH_CHECK();
    return 0;
  }
  hipLaunchKernelGGL((k_weights_from_traces<T>), dim3((unsigned)(N < 8192 ? N : 8192)), dim3(256), 0, st, W, Ci,
                     Cj, Cij, cthr, s.cthr4, N, M);
  SB_LAUNCH_CHECK();
  if (wmask) return launch_apply_mask<T>(st, W, wmask, N, H, Mc);
  return 0;
}

template <typename T>
int launch_add_bias(hipStream_t st, T *act, const T *bias, long B, long M) {
  SB_REQUIRE(act && bias, "null pointer");
  SB_REQUIRE(B > 0 && M > 0, "sizes must be positive");
  const long blocks = cdiv(B * M, 256) < 8192 ? cdiv(B * M, 256) : 8192;
  ProfScope prof_(st, K_UPDATE_BIAS);
  hipLaunchKernelGGL((k_add_bias<T>), dim3((unsigned)blocks), dim3(256), 0, st, act, bias, B, M);
  SB_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------------------------- bias
template <typename T>
int launch_update_bias(hipStream_t st, T *bias, const T *Cj, T cthr, long M) {
  SB_REQUIRE(bias && Cj, "null pointer");
  SB_REQUIRE(M > 0, "sizes must be positive");
  ProfScope prof_(st, K_UPDATE_BIAS);
  hipLaunchKernelGGL((k_update_bias<T>), dim3((unsigned)cdiv(M, 256)), dim3(256), 0, st, bias, Cj, cthr,
                     M);
  SB_LAUNCH_CHECK();
  return 0;
}

template <typename T>
int launch_update_bias_regularized(hipStream_t st, T *bias, T *kbi, const T *Cj, T cthr, T khalf,
                                   T pmin, T taubdt, long M) {
  SB_REQUIRE(bias && kbi && Cj, "null pointer");
  SB_REQUIRE(M > 0, "sizes must be positive");
  ProfScope prof_(st, K_UPDATE_BIAS_REG);
  hipLaunchKernelGGL((k_update_bias_regularized<T>), dim3((unsigned)cdiv(M, 256)), dim3(256), 0, st,
                     bias, kbi, Cj, cthr, khalf, pmin, taubdt, M);
  SB_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------------------------- mask
// W_fix != nullptr: the swap kernel also rewrites the weights of the rows that changed sides and (rows !=
// nullptr) rebuilds the hypercolumn's row list, when it can (*merged = true); see MaskArgs.
template <typename T>
static int update_mask_impl(hipStream_t st, uint8_t *wmask, const T *W, const T *Ci, const T *Cj,
                            const T *Cij, T cthr, long N, long H, long Mc, long h, long iterations, T *nom,
                            int *csum, T *W_fix, int *rows, int *row_cnt, long cap, bool *merged) {
  SB_REQUIRE(wmask && Ci && Cj && Cij && nom && csum, "null pointer");
  SB_REQUIRE(N > 0 && H > 0 && Mc > 0, "sizes must be positive");
  SB_REQUIRE(h >= 0 && h < H, "hypercolumn index out of range");
  SB_REQUIRE(iterations >= 0, "iterations must be non-negative");
  SB_REQUIRE(cdiv(N, 4) < (1L << 31), "in_features too large");
  const TraceScalars<T> s = TraceScalars<T>::from(T(0), cthr);
  MaskArgs<T> a;
  a.wmask = wmask; a.W = W; a.Ci = Ci; a.Cj = Cj; a.Cij = Cij; a.cthr = cthr; a.cthr4 = s.cthr4;
  a.N = N; a.M = H * Mc; a.H = H; a.Mc = Mc; a.h = h; a.iterations = iterations;
  a.nom = nom; a.score = nom + N;
  a.csum = csum; a.side = csum + N;
  // two rows change sides per iteration; the rows that did are noted and rewritten with 32-bit indices
  const bool merge = W_fix != nullptr && iterations > 0 && 2 * iterations <= kMaxChangedRows && N < (1L << 31) &&
                     N * Mc < (1L << 31);
  a.W_fix = merge ? W_fix : nullptr;
  a.rows = merge ? rows : nullptr;
  a.row_cnt = row_cnt;
  a.cap = cap;
  if (merged) *merged = merge;
  {
    ProfScope prof_(st, K_MASK_SCORES);
    if (N >= 16L * 2 * device_cu_count())  // two workgroups of sixteen rows for every CU
      hipLaunchKernelGGL((k_mask_scores<T, 16>), dim3((unsigned)cdiv(N, 16)), dim3(256), 0, st, a);
    else
      hipLaunchKernelGGL((k_mask_scores<T, 4>), dim3((unsigned)cdiv(N, 4)), dim3(256), 0, st, a);
    SB_LAUNCH_CHECK();
  }
  if (iterations > 0) {
    ProfScope prof_(st, K_MASK_SWAP);
    hipLaunchKernelGGL((k_mask_swap<T>), dim3(1), dim3(1024), 0, st, a);
    SB_LAUNCH_CHECK();
  }
  return 0;
}

template <typename T>
int launch_update_mask(hipStream_t st, uint8_t *wmask, const T *W, const T *Ci, const T *Cj,
                       const T *Cij, T cthr, long N, long H, long Mc, long h, long iterations, T *nom,
                       int *csum) {
  return update_mask_impl<T>(st, wmask, W, Ci, Cj, Cij, cthr, N, H, Mc, h, iterations, nom, csum, nullptr,
                             nullptr, nullptr, 0, nullptr);
}

template <typename T>
int launch_rewire(hipStream_t st, uint8_t *wmask, T *W, const T *Ci, const T *Cj, const T *Cij, T cthr, long N,
                  long H, long Mc, long h, long iterations, T *nom, int *csum, int *rows, int *row_cnt,
                  long cap) {
  SB_REQUIRE(W, "null pointer");
  SB_REQUIRE(!rows || (row_cnt && cap > 0 && cap % 16 == 0), "row list arguments");
  bool merged = false;
  int rc = update_mask_impl<T>(st, wmask, (const T *)nullptr, Ci, Cj, Cij, cthr, N, H, Mc, h, iterations, nom,
                               csum, W, rows, row_cnt, cap, &merged);
  if (rc || merged) return rc;
  return launch_mask_fix_weights<T>(st, W, wmask, Ci, Cj, Cij, cthr, N, H, Mc, h, rows, row_cnt, cap);
}

template <typename T>
int launch_mask_fix_weights(hipStream_t st, T *W, const uint8_t *wmask, const T *Ci, const T *Cj,
                            const T *Cij, T cthr, long N, long H, long Mc, long h, int *rows, int *row_cnt,
                            long cap) {
  SB_REQUIRE(W && wmask && Ci && Cj && Cij, "null pointer");
  SB_REQUIRE(h >= 0 && h < H, "hypercolumn index out of range");
  SB_REQUIRE(!rows || (row_cnt && cap > 0 && cap % 16 == 0), "row list arguments");
  SB_REQUIRE(cdiv(N * Mc, 256) + 1 < (1L << 31), "too many elements for one launch");
  const TraceScalars<T> s = TraceScalars<T>::from(T(0), cthr);
  ProfScope prof_(st, K_MASK_FIX);
  // with a row list, one more workgroup rebuilds the list of hypercolumn h
  const long blocks = cdiv(N * Mc, 256) + (rows ? 1 : 0);
  hipLaunchKernelGGL((k_mask_fix_weights<T>), dim3((unsigned)blocks), dim3(256), 0, st, W, wmask, Ci, Cj, Cij,
                     cthr, s.cthr4, N, H * Mc, H, Mc, h, rows, row_cnt, cap);
  SB_LAUNCH_CHECK();
  return 0;
}

template <typename T>
int launch_apply_mask(hipStream_t st, T *W, const uint8_t *wmask, long N, long H, long Mc) {
  SB_REQUIRE(W && wmask, "null pointer");
  SB_REQUIRE(N > 0 && H > 0 && Mc > 0, "sizes must be positive");
  SB_REQUIRE(H * Mc < (1L << 31), "dimension too large");
  const long blocks = N < 8192 ? N : 8192;
  ProfScope prof_(st, K_APPLY_MASK);
  constexpr int VW = Real<T>::VW;
  if (Mc % VW == 0 && aligned16(W)) {
    const long turns = cdiv(N, kRowsPerTurn);
    hipLaunchKernelGGL((k_apply_mask_vec<T>), dim3((unsigned)cdiv(H * Mc, 256 * VW), (unsigned)(turns < 4096 ? turns : 4096)),
                       dim3(256), 0, st, W, wmask, N, H * Mc, H, FastDiv::of(Mc));
    SB_LAUNCH_CHECK();
    return 0;
  }
  hipLaunchKernelGGL((k_apply_mask<T>), dim3((unsigned)blocks), dim3(256), 0, st, W, wmask, N, H * Mc, H,
                     FastDiv::of(Mc));
  SB_LAUNCH_CHECK();
  return 0;
}

// *count += number of entries of W that are non-zero under a zero mask byte
template <typename T>
int launch_count_unmasked(hipStream_t st, const T *W, const uint8_t *wmask, long N, long H, long Mc,
                          unsigned long long *count) {
  SB_REQUIRE(W && wmask && count, "null pointer");
  SB_REQUIRE(N > 0 && H > 0 && Mc > 0, "sizes must be positive");
  SB_REQUIRE(H * Mc < (1L << 31), "dimension too large");
  const long blocks = N < 4096 ? N : 4096;
  ProfScope prof_(st, K_APPLY_MASK);
  hipLaunchKernelGGL((k_count_unmasked<T>), dim3((unsigned)blocks), dim3(256), 0, st, W, wmask, N, H * Mc, H,
                     Mc, count);
  SB_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------------------------------- classification
template <typename T>
int launch_argmax_rows(hipStream_t st, const T *act, const T *labels, long B, long M, int32_t *pred,
                       unsigned long long *correct) {
  SB_REQUIRE(act, "null pointer");
  SB_REQUIRE(!labels || correct, "labels need a counter");
  SB_REQUIRE(B > 0 && M > 0, "sizes must be positive");
  ProfScope prof_(st, K_ARGMAX);
  hipLaunchKernelGGL((k_argmax_rows<T>), dim3((unsigned)cdiv(B, 4)), dim3(256), 0, st, act, labels, B,
                     M, pred, correct);
  SB_LAUNCH_CHECK();
  return 0;
}

template <typename T>
int launch_gather_rows(hipStream_t st, T *dst, const T *src, const int64_t *idx, long rows,
                       long cols) {
  SB_REQUIRE(dst && src && idx, "null pointer");
  SB_REQUIRE(rows > 0 && cols > 0 && rows < (1L << 31), "bad shape");
  ProfScope prof_(st, K_GATHER);
  hipLaunchKernelGGL((k_gather_rows<T>), dim3((unsigned)rows), dim3(256), 0, st, dst, src, idx, rows,
                     cols);
  SB_LAUNCH_CHECK();
  return 0;
}

template <typename T>
int launch_gather_rows_blocked(hipStream_t st, T *dst, T *plain, const T *src, const int64_t *idx, long rows,
                               long cols) {
  SB_REQUIRE(dst && src, "null pointer");
  SB_REQUIRE(rows > 0 && cols > 0 && cdiv(rows, 16) < (1L << 31), "bad shape");
  ProfScope prof_(st, K_GATHER);
  const long col_groups = cdiv(cols, 256) < 65535 ? cdiv(cols, 256) : 65535;
  hipLaunchKernelGGL((k_gather_rows_blocked<T>), dim3((unsigned)cdiv(rows, 16), (unsigned)col_groups), dim3(256), 0,
                     st, dst, plain, src, idx, rows, cols);
  SB_LAUNCH_CHECK();
  return 0;
}

template <typename T>
int launch_mfma_probe(hipStream_t st, T *sink, long workgroups, long iters) {
  SB_REQUIRE(sink, "null pointer");
  SB_REQUIRE(workgroups > 0 && workgroups < (1L << 31) && iters > 0 && iters <= (1L << 24), "bad sizes");
  hipLaunchKernelGGL((k_mfma_probe<T>), dim3((unsigned)workgroups), dim3(256), 0, st, sink, iters);
  SB_LAUNCH_CHECK();
  return 0;
}

template <typename T>
int launch_fill(hipStream_t st, T *dst, T value, size_t n) {
  if (n == 0) return 0;
  SB_REQUIRE(dst, "null pointer");
  const size_t blocks = (n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096;
  ProfScope prof_(st, K_FILL);
  hipLaunchKernelGGL((k_fill<T>), dim3((unsigned)blocks), dim3(256), 0, st, dst, value, n);
  SB_LAUNCH_CHECK();
  return 0;
}

template <typename T>
int launch_copy_pair(hipStream_t st, T *dst1, const T *src1, size_t n1, T *dst2, const T *src2, size_t n2) {
  if (n1 + n2 == 0) return 0;
  SB_REQUIRE(dst1 && src1 && dst2 && src2, "null pointer");
  const size_t blocks = (n1 + n2 + 255) / 256 < 4096 ? (n1 + n2 + 255) / 256 : 4096;
  ProfScope prof_(st, K_FILL);
  hipLaunchKernelGGL((k_copy_pair<T>), dim3((unsigned)blocks), dim3(256), 0, st, dst1, src1, n1, dst2, src2, n2);
  SB_LAUNCH_CHECK();
  return 0;
}

#define SB_INSTANTIATE_LAUNCHERS(T)                                                                   \
  template int launch_forward<T>(hipStream_t, T *, const T *, const T *, const T *, long, long, long, \
                                 long, bool, long);                                                   \
  template int launch_forward_classify<T>(hipStream_t, T *, const T *, const T *, const T *, long,    \
                                          long, long, long, bool, const T *, int32_t *,               \
                                          unsigned long long *, long);                                \
  template bool forward_bits_equal<T>(long, long, long, long, long, long);                            \
  template bool forward_rows_supported<T>(const T *, long, long, long);                               \
  template int launch_forward_rows<T>(hipStream_t, T *, const T *, const T *, const T *, const int *, \
                                      const int *, long, long, long, long, long, const T *, long,     \
                                      void *);                                                        \
  template size_t forward_rows_bytes<T>(long, long, long, long, long, long);                          \
  template int launch_gather_rows_blocked<T>(hipStream_t, T *, T *, const T *, const int64_t *, long, \
                                             long);                                                  \
  template int launch_softmax<T>(hipStream_t, T *, long, long, long);                                 \
  template int launch_train_fused<T>(hipStream_t, const T *, const T *, T *, T *, const T *, const T *, \
                                     T *, T *, const uint8_t *, int, T *, T *, long, long, long, long, \
                                     T, T, T, T, T, bool, const void *, size_t, void *);              \
  template size_t train_split_bytes<T>(long, long, long, long);                                       \
  template bool train_in_place_supported<T>(const void *, long, long, long, long, T);                 \
  template bool train_skinny_epoch_pays<T>(long, long, long);                                         \
  template int launch_train_skinny_epoch<T>(hipStream_t, const T *, const int64_t *, const T *, T *,  \
                                            T *, const T *, const T *, T *, T *, long, long, long,    \
                                            long, long, T, T);                                        \
  template int launch_update_bias<T>(hipStream_t, T *, const T *, T, long);                           \
  template int launch_weights_from_traces<T>(hipStream_t, T *, const T *, const T *, const T *,       \
                                             const uint8_t *, T, long, long, long, bool);             \
  template int launch_add_bias<T>(hipStream_t, T *, const T *, long, long);                           \
  template int launch_update_bias_regularized<T>(hipStream_t, T *, T *, const T *, T, T, T, T, long); \
  template int launch_update_mask<T>(hipStream_t, uint8_t *, const T *, const T *, const T *,         \
                                     const T *, T, long, long, long, long, long, T *, int *);         \
  template int launch_mask_fix_weights<T>(hipStream_t, T *, const uint8_t *, const T *, const T *,    \
                                          const T *, T, long, long, long, long, int *, int *, long);  \
  template int launch_rewire<T>(hipStream_t, uint8_t *, T *, const T *, const T *, const T *, T, long, \
                                long, long, long, long, T *, int *, int *, int *, long);              \
  template int launch_apply_mask<T>(hipStream_t, T *, const uint8_t *, long, long, long);             \
  template int launch_count_unmasked<T>(hipStream_t, const T *, const uint8_t *, long, long, long,    \
                                        unsigned long long *);                                        \
  template int launch_argmax_rows<T>(hipStream_t, const T *, const T *, long, long, int32_t *,        \
                                     unsigned long long *);                                           \
  template int launch_gather_rows<T>(hipStream_t, T *, const T *, const int64_t *, long, long);       \
  template int launch_mfma_probe<T>(hipStream_t, T *, long, long);                                    \
  template int launch_fill<T>(hipStream_t, T *, T, size_t);                                           \
  template int launch_copy_pair<T>(hipStream_t, T *, const T *, size_t, T *, const T *, size_t);

}  // namespace sb
