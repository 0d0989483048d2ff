// Forward pass over the connected rows for layers with few tiles and long lists: the four sums that the wavefronts of
// k_forward_rows form one after the other on one CU, on four.
#pragma once
#include "sb_k_forward_rows.hpp"

namespace sb {

// k_forward_rows deals the chunks of a hypercolumn's row list out to its four wavefronts (chunk c to wavefront c mod 4) and
// adds up their four sums at the end.  Here the chunks of one of them, in the same order, hence the same sum, are the
// whole reduction of a wavefront, and the four sums of a tile may be formed on four CUs: a wavefront takes 16 batch rows,
// a piece of 16 to 64 columns of a hypercolumn and one chain of four, and puts its sum into part[chain][B, M];
// k_softmax_of_chains adds the four up in k_forward_rows' order, so the activations have the same bits.
// Bound: the matrix instructions, which two wavefronts per SIMD keep busy and one nearly (12.9 and 17.5 ns each), as
// long as little else is issued between them.  So the list is staged as byte offsets, which costs an operand one addition
// of 32 bits (with the row index instead, multiplied by the row length in 64 bits at every use, 205 us where this takes
// 155); four chunks of operands in flight or in use (two 3 % slower, six no better); and the pieces are dealt in whole
// blocks of 16 columns (200 columns: 4 + 3 + 3 + 3 blocks, not 64 + 64 + 64 + 8 columns), two to a SIMD where the chip
// is filled twice.  W is read once per 64 or 128 batch rows, by wavefronts side by side on a CU.
// 27648 -> 15 x 200, lists of 15800, batch 128, floats: 151 us with the softmax where W is found in the memory-side cache,
// 202 where it has just been written past it (passes one after the other 134, a workgroup of k_forward_rows per column
// group 162).  Then the
// lines that a CU's L1 holds for what is on its way are the bound, a half line of x per entry and 16 batch rows among
// them: four or twelve chunks ahead, the same time.  32 rows (30 tiles, narrower pieces): 113 -> 64 us.
template <typename T>
struct ForwardChainsArgs {
  ForwardRowsArgs<T> r;
  T *part;                     // [kChains][B, M]
  int waves_rows, waves_cols;  // wavefronts of a workgroup along the batch and along a hypercolumn: 4 or 8 in all
  int pieces;                  // of a hypercolumn
  int row_groups, col_groups;  // workgroups along the batch and along a hypercolumn
};
constexpr int kChains = 4;
constexpr int kChainSeg = 4096;  // list entries of a chain staged at a time

// XT: as in k_forward_rows.  W stays below 4 GiB.
// MIXED: wavefronts of a workgroup may have pieces of different widths, each walked in code of its own, between barriers
// that all of them meet at.  Otherwise a workgroup is in one such code from start to end, with fewer registers
// (27648 -> 15 x 100, lists of 15800, batch 128, whose pieces are of four and of three blocks: 94 us this way, 88.5
// otherwise).
template <typename T, bool XT, bool MIXED>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(MIXED ? 2 : 3)))
void k_forward_chains(ForwardChainsArgs<T> ac) {
  const ForwardRowsArgs<T> &ar = ac.r;
  const ForwardArgs<T> &a = ar.f;
  constexpr int VW = Real<T>::VW, KC = 4 * VW, SEG = kChainSeg, SEGC = SEG / KC;
  constexpr int D = 4;  // chunks of operands in flight or being multiplied
  using acc_t = typename Real<T>::acc_t;
  typedef unsigned ivec_t __attribute__((ext_vector_type(VW)));
  // per entry: byte offsets of its row of W and of its column of x
  __shared__ __attribute__((aligned(16))) unsigned woff[SEG], xoff[SEG];

  // an XCD gets a contiguous run of workgroups, chains outermost: the x columns of a chain then stay in its L2
  const unsigned total = (unsigned)a.col_tiles * ac.row_groups * ac.col_groups * kChains;
  const unsigned per_xcd = (total + 7) / 8;
  unsigned rest = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (rest >= total) return;  // whole workgroup, before any barrier
  const unsigned rg = rest % ac.row_groups;
  rest /= ac.row_groups;
  const unsigned cg = rest % ac.col_groups;
  rest /= ac.col_groups;
  const unsigned ct = rest % (unsigned)a.col_tiles, ch = rest / (unsigned)a.col_tiles;

  const int tid = threadIdx.x, lane = tid & 63, p = lane & 15, q = lane >> 4, threads = blockDim.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wc = w / ac.waves_rows, wr = w - wc * ac.waves_rows;
  const long b0 = ((long)rg * ac.waves_rows + wr) * 16;
  // blocks of 16 columns, the first pieces have one more
  const int piece = cg * ac.waves_cols + wc, blocks = ((int)a.Mc + 15) / 16;
  const int each = blocks / ac.pieces, more = blocks - each * ac.pieces;
  const int nb = each + (piece < more ? 1 : 0);
  const int jg = (piece * each + (piece < more ? piece : more)) * 16;
  const bool active = b0 < a.B && piece < ac.pieces && wc < ac.waves_cols;  // (uniform) the others only stage the list
  const int ncol = (int)a.Mc - jg < 16 * nb ? (int)a.Mc - jg : 16 * nb;
  const long j0 = (long)ct * a.Mc + (active ? jg : 0);
  const int *list = ar.rows + (long)ct * ar.cap;
  const int cnt = ar.row_cnt[ct];
  const BufferWindow<T> xwin((XT ? ar.xt : a.x) + (active ? b0 : 0) * a.N,
                             active ? (XT ? (a.B + 15) / 16 * 16 - b0 : a.B - b0) * a.N : 0);
  const unsigned xat = XT ? (unsigned)(p * sizeof(T)) : (unsigned)((long)p * a.N * sizeof(T));
  constexpr unsigned XSTEP = (XT ? 16u : 1u) * (unsigned)sizeof(T);
  // chunks ch, ch + 4, .. of the list; the first one also where the list is shorter (padding), as in k_forward_rows
  const int chunks = (cnt + KC - 1) / KC;
  const int mine = chunks > (int)ch ? (chunks - 1 - (int)ch) / kChains + 1 : 1;

  // the lane's first column of group g; a vector that would run over the piece's end starts earlier (its columns are
  // computed twice, with the same result)
  auto first_col = [&](int g, int width) {
    const int c = g * 16 * VW + width * p, last = ncol - width;
    return c < last ? c : (last > 0 ? last : 0);
  };
  // adds up the n chunks of the staged segment (per wavefront: no barriers in here); acc: a sum per block of 16 columns
  auto walk = [&](auto nblocks, int n, auto &acc) {
    constexpr int NB = decltype(nblocks)::value, NG = (NB + VW - 1) / VW, LW = NB - (NG - 1) * VW;
    auto width = [](int g) { return g == NG - 1 ? LW : VW; };
    unsigned wcol[NG];
#pragma unroll
    for (int g = 0; g < NG; g++) wcol[g] = (unsigned)((j0 + first_col(g, width(g))) * sizeof(T));
    T xr[D][VW], wt[D][VW][NG][VW];
    auto request = [&](int c, T(&xo)[VW], T(&wo)[VW][NG][VW]) {
      const int at = (c < SEGC ? c : SEGC - 1) * KC + VW * q;
      const ivec_t wv = *reinterpret_cast<const ivec_t *>(&woff[at]), xv = *reinterpret_cast<const ivec_t *>(&xoff[at]);
#pragma unroll
      for (int s = 0; s < VW; s++) {
        T one[1];
        xwin.template load_n<1>(one, xat + xv[s]);
        xo[s] = one[0];
#pragma unroll
        for (int g = 0; g < NG; g++) {
          const char *const from = reinterpret_cast<const char *>(a.W) + (wcol[g] + wv[s]);
          if (width(g) == VW) {
            const PackedCols<T, VW> v = *reinterpret_cast<const PackedCols<T, VW> *>(from);
#pragma unroll
            for (int e = 0; e < VW; e++) wo[s][g][e] = v.v[e];
          } else {
            const PackedCols<T, LW> v = *reinterpret_cast<const PackedCols<T, LW> *>(from);
#pragma unroll
            for (int e = 0; e < LW; e++) wo[s][g][e] = v.v[e];
          }
        }
      }
    };
    auto compute = [&](const T(&xi)[VW], const T(&wi)[VW][NG][VW]) {
#pragma unroll
      for (int s = 0; s < VW; s++)
#pragma unroll
        for (int g = 0; g < NG; g++)
#pragma unroll
          for (int c = 0; c < VW; c++)
            if (c < width(g)) acc[g * VW + c] = Real<T>::mfma(xi[s], wi[s][g][c], acc[g * VW + c]);
    };
#pragma unroll
    for (int u = 0; u < D - 1; u++) request(u, xr[u], wt[u]);
    __builtin_amdgcn_sched_barrier(0);
    int i = 0;
    for (; i + D <= n; i += D) {
#pragma unroll
      for (int u = 0; u < D; u++) {
        request(i + u + D - 1, xr[(u + D - 1) % D], wt[(u + D - 1) % D]);
        __builtin_amdgcn_sched_barrier(0);
        compute(xr[u], wt[u]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int u = 0; u < D - 1; u++)
      if (i + u < n) compute(xr[u], wt[u]);
  };
  auto store = [&](auto nblocks, const auto &acc) {
    constexpr int NB = decltype(nblocks)::value, NG = (NB + VW - 1) / VW, LW = NB - (NG - 1) * VW;
    auto width = [](int g) { return g == NG - 1 ? LW : VW; };
    T *const out = ac.part + (long)ch * a.B * a.M + j0;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const long row = b0 + Real<T>::acc_row(q, v);
      if (row >= a.B) continue;
#pragma unroll
      for (int g = 0; g < NG; g++) {
        const int c0 = first_col(g, width(g));
#pragma unroll
        for (int e = 0; e < VW; e++)
          if (e < width(g) && c0 + e < ncol) out[row * a.M + c0 + e] = acc[g * VW + e][v];
      }
    }
  };
  auto with_blocks = [&](int count, auto what) {
    if (count == 4) what(std::integral_constant<int, 4>{});
    else if (count == 3) what(std::integral_constant<int, 3>{});
    else if (count == 2) what(std::integral_constant<int, 2>{});
    else what(std::integral_constant<int, 1>{});
  };
  // Stages the list segment by segment, all wavefronts together; `on_segment` of the active ones in between.
  auto segments = [&](auto on_segment) {
    int left = mine;
    for (int c0 = 0; left > 0; c0 += SEGC, left -= SEGC) {
      const int n = left < SEGC ? left : SEGC;
      if (c0 > 0) __syncthreads();  // everyone is done with the staged segment
      // (D - 1 chunks beyond the last one are requested and not used: padding)
      const int stage = (n + D - 1 < SEGC ? n + D - 1 : SEGC) * KC;
      constexpr int U = 4;
      for (int e0 = tid; e0 < stage; e0 += threads * U) {
        int r[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int e = e0 + threads * u;
          const long k = ((long)(c0 + e / KC) * kChains + ch) * KC + e % KC;
          const bool on = e < n * KC && k < ar.cap;
          r[u] = list[on ? k : 0];
          r[u] = on ? r[u] : -1;
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int e = e0 + threads * u;
          if (e < stage) {
            woff[e] = r[u] < 0 ? 0u : (unsigned)r[u] * (unsigned)(a.M * sizeof(T));
            xoff[e] = r[u] < 0 ? BufferWindow<T>::kOutside : (unsigned)r[u] * XSTEP;
          }
        }
      }
      __syncthreads();
      if (active) on_segment(n);
    }
  };
  if constexpr (MIXED) {
    acc_t acc[4] = {acc_t{0, 0, 0, 0}, acc_t{0, 0, 0, 0}, acc_t{0, 0, 0, 0}, acc_t{0, 0, 0, 0}};
    segments([&](int n) { with_blocks(nb, [&](auto nblocks) { walk(nblocks, n, acc); }); });
    if (active) with_blocks(nb, [&](auto nblocks) { store(nblocks, acc); });
  } else {
    const int first = cg * ac.waves_cols;  // (its width is that of all of the workgroup's pieces)
    with_blocks(each + (first < more ? 1 : 0), [&](auto nblocks) {
      acc_t acc[decltype(nblocks)::value];
#pragma unroll
      for (auto &sum : acc) sum = acc_t{0, 0, 0, 0};
      segments([&](int n) { walk(nblocks, n, acc); });
      if (active) store(nblocks, acc);
    });
  }
}

// act = softmax_per_hypercolumn(the four chains added up as forward_finish does + bias), with forward_finish's arithmetic
// for four wavefronts: 16 threads per (row, hypercolumn), thread lr has units lr + 16 t.
template <typename T>
__global__ __launch_bounds__(128) void k_softmax_of_chains(T *act, const T *part, const T *bias, long B, long H, long Mc) {
  constexpr int TPR = 16, PT = 16;
  const long groups = B * H, M = H * Mc;
  const long g = (long)blockIdx.x * (128 / TPR) + threadIdx.x / TPR;
  const int lr = threadIdx.x % TPR;
  const long gg = g < groups ? g : groups - 1;  // (lanes past the end take part in the exchanges)
  const long row = gg / H, j0 = (gg - row * H) * Mc;
  const T *const src = part + row * M + j0;
  const long plane = B * M;
  T vals[PT], mx = -INFINITY;
#pragma unroll
  for (int t = 0; t < PT; t++) {
    const long col = lr + TPR * t, c = col < Mc ? col : 0;
    const T s02 = src[2 * plane + c] + src[c], s13 = src[3 * plane + c] + src[plane + c];
    vals[t] = col < Mc ? (s02 + s13) + bias[j0 + c] : T(0);
    mx = (col < Mc && vals[t] > mx) ? vals[t] : mx;
  }
  mx = row16_reduce(mx, [](T x, T y) { return y > x ? y : x; });
  T sum = T(0);
#pragma unroll
  for (int t = 0; t < PT; t++)
    if (lr + TPR * t < Mc) {
      vals[t] = Real<T>::exp_nonpos(vals[t] - mx);
      sum += vals[t];
    }
  sum = row16_reduce(sum, [](T x, T y) { return x + y; });
  const T r = T(1) / sum;
  if (g >= groups) return;
  T *const out = act + row * M + j0;
#pragma unroll
  for (int t = 0; t < PT; t++)
    if (lr + TPR * t < Mc) out[lr + TPR * t] = sizeof(T) == 4 ? vals[t] * r : vals[t] / sum;
}

}  // namespace sb
