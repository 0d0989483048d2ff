// The greedy swap loop of the mask rewiring (omp.cc:289-315, where "omp.cc" =
// BCPNN/backend/_kernels/kernels_openmp_internal.cc of the reference), on the scores that k_mask_scores has left in
// memory.  One workgroup.
//
// An iteration changes nothing but the two rows it swaps, so over at most 16 iterations only the 16 best silent rows
// and the 16 worst active rows of the state they start from (plus rows that changed sides on the way) can ever be
// picked.  The kernel therefore works in rounds of 16 iterations:
//   phase A (whole workgroup): the 16 best rows of either side in the strict order (score, row index), which is the
//     order the picks take them in, equal scores included.  The rows are dealt into 64 bins; the 16th
//     largest of the 64 bins' best is a bound that at least 16 rows reach and few others do (about 3
//     more where the order knows nothing of the bins), the rows that reach it go to a list in LDS, and a
//     row's place is the number of listed rows ahead of it.  A lane's rows go into another bin in every wavefront: by
//     the index modulo 64 alone, images 64 pixels wide have whole columns in a bin, whose scores resemble each
//     other, and the list overflows (24576 rows, floats: 57 us instead of 18);
//   phase B (one wavefront, one candidate per lane and side): the iterations themselves, with the same picks, tie
//     rule, break conditions and score expression as a full scan.
// A round reads the N scores and sides twice (the second time from L2) and has seven barriers; its time is latency.
// What a round does not cover -- a side whose first candidate row has a NaN score or may come to have one, or a
// list that overflows -- is left to a full scan per iteration (swap_by_scans).
// 27648 rows, floats: 22 us; 318 us with the state in registers and a radix select on 2048-bin histograms, whose
// counters all threads hit together (scores share their leading bits), and a scan per iteration once any score is
// NaN, as the scores of inputs that are always on are (1 - Ci = 0).
#pragma once
#include "sb_kernels.hpp"

namespace sb {

// Monotone integer keys of the scores.
template <typename T>
struct ScoreKey;
template <>
struct ScoreKey<float> {
  using K = uint32_t;
  static __device__ __forceinline__ K of(float s) {
    const uint32_t b = __float_as_uint(s + 0.0f);  // -0 and +0 compare equal, so they share a key
    return b ^ ((b >> 31) ? 0xffffffffu : 0x80000000u);
  }
};
template <>
struct ScoreKey<double> {
  using K = uint64_t;
  static __device__ __forceinline__ K of(double s) {
    const uint64_t b = (uint64_t)__double_as_longlong(s + 0.0);
    return b ^ ((b >> 63) ? ~0ull : (1ull << 63));
  }
};
__device__ __forceinline__ float readlane_t(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double readlane_t(double v, int l) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// (key, row index) pairs and their wavefront-wide maximum; idx < 0 marks "no candidate"
template <typename K>
struct KeyIdx {
  K key;
  int idx;
};
template <typename K>
__device__ __forceinline__ KeyIdx<K> pick_key(KeyIdx<K> a, KeyIdx<K> b) {
  const bool take = b.idx >= 0 && (a.idx < 0 || b.key > a.key || (b.key == a.key && b.idx > a.idx));
  return take ? b : a;
}
__device__ __forceinline__ uint32_t readlane_k(uint32_t v, int l) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}
__device__ __forceinline__ uint64_t readlane_k(uint64_t v, int l) {
  const uint32_t lo = readlane_k((uint32_t)v, l), hi = readlane_k((uint32_t)(v >> 32), l);
  return ((uint64_t)hi << 32) | lo;
}
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_move_k(uint32_t v) {
  return (uint32_t)dpp_move<CTRL>((int)v);
}
template <int CTRL>
__device__ __forceinline__ uint64_t dpp_move_k(uint64_t v) {
  return ((uint64_t)dpp_move_k<CTRL>((uint32_t)(v >> 32)) << 32) | dpp_move_k<CTRL>((uint32_t)v);
}
template <typename K, int CTRL>
__device__ __forceinline__ KeyIdx<K> dpp_keyidx(KeyIdx<K> c) {
  return KeyIdx<K>{dpp_move_k<CTRL>(c.key), dpp_move<CTRL>(c.idx)};
}
template <typename K>
__device__ __forceinline__ KeyIdx<K> wave_pick(KeyIdx<K> c) {  // the result is wavefront-uniform
  c = pick_key<K>(c, dpp_keyidx<K, kDppSwap1>(c));
  c = pick_key<K>(c, dpp_keyidx<K, kDppSwap2>(c));
  c = pick_key<K>(c, dpp_keyidx<K, kDppHalfMirror>(c));
  c = pick_key<K>(c, dpp_keyidx<K, kDppMirror>(c));
  // every lane of a row of 16 now holds its row's pick; the four rows are combined from scalar
  // registers (a lane read is far cheaper than an exchange through the LDS crossbar)
  const KeyIdx<K> r0{readlane_k(c.key, 0), __builtin_amdgcn_readlane(c.idx, 0)};
  const KeyIdx<K> r1{readlane_k(c.key, 16), __builtin_amdgcn_readlane(c.idx, 16)};
  const KeyIdx<K> r2{readlane_k(c.key, 32), __builtin_amdgcn_readlane(c.idx, 32)};
  const KeyIdx<K> r3{readlane_k(c.key, 48), __builtin_amdgcn_readlane(c.idx, 48)};
  return pick_key<K>(pick_key<K>(r0, r1), pick_key<K>(r2, r3));
}

// 32-bit keys: (key, index + 1) packed into one 64-bit integer whose unsigned order is the order pick_key
// defines (0 = no candidate), so a pick is a 64-bit maximum: a third of the instructions.
__device__ __forceinline__ KeyIdx<uint32_t> wave_pick(KeyIdx<uint32_t> c) {
  uint64_t v = c.idx < 0 ? 0ull : ((uint64_t)c.key << 32) | (uint32_t)(c.idx + 1);
  auto larger = [](uint64_t a, uint64_t b) { return b > a ? b : a; };
  v = larger(v, dpp_move_k<kDppSwap1>(v));
  v = larger(v, dpp_move_k<kDppSwap2>(v));
  v = larger(v, dpp_move_k<kDppHalfMirror>(v));
  v = larger(v, dpp_move_k<kDppMirror>(v));
  const uint64_t m = larger(larger(readlane_k(v, 0), readlane_k(v, 16)),
                            larger(readlane_k(v, 32), readlane_k(v, 48)));
  return KeyIdx<uint32_t>{(uint32_t)(m >> 32), (int)(uint32_t)m - 1};
}

__device__ __forceinline__ void note_changed(int *changed, int *nchanged, long row) {
  const int at = atomicAdd(nchanged, 1);
  if (at < kMaxChangedRows) changed[at] = (int)row;
}

// reduction over a wavefront of an integer; the result is in every lane
template <typename Op>
__device__ __forceinline__ int wave_reduce(int v, Op op) {
  v = row16_reduce(v, op);
  return op(op(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
            op(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

template <typename T>
struct MaskSwap {
  using SK = ScoreKey<T>;
  using K = typename SK::K;
  static constexpr int NT = 1024, NWV = NT / 64, TOP = 16, LIST = 1024, U = 8;
  struct Shared {
    K bin_key[2][NWV][64];  // per side and wavefront: the best row of each bin ...
    int bin_idx[2][NWV][64];
    K list_key[2][LIST];  // ... and the rows at or beyond the bound
    int list_idx[2][LIST];
    K bound_key[2];
    int bound_idx[2], nlist[2], top[2][TOP];
    int rank[2][64];  // bins whose best row is ahead of this one's
    int nan_first[2], ahead[2];  // lowest row with a NaN score; rows with a score below it
    int swaps;
  };

  // This thread's rows i0 + tid, i0 + tid + NT, ..: scores and sides (2: no candidate, or no row), loads in flight
  // together.
  struct Rows {
    T s[U];
    int m[U];
  };
  static __device__ __forceinline__ void load_rows(const MaskArgs<T> &a, Rows &v, int i0) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const long i = (long)i0 + (int)threadIdx.x + NT * u;
      v.s[u] = a.score[i < a.N ? i : 0];
      v.m[u] = i < a.N ? a.side[i] : 2;
    }
  }
  // Calls f(row, side, score) for all of this thread's rows in ascending order.
  // `first`: the first NT * U rows, already loaded.  (No guards around the calls: what they hold is a few selects.)
  template <typename F>
  static __device__ __forceinline__ void for_rows(const MaskArgs<T> &a, const Rows &first, F &&f) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int u = 0; u < U; u++) f(tid + NT * u, first.m[u], first.s[u]);
    for (long i0 = NT * U; i0 < a.N; i0 += NT * U) {
      Rows v;
      load_rows(a, v, (int)i0);
#pragma unroll
      for (int u = 0; u < U; u++) f((int)i0 + tid + NT * u, v.m[u], v.s[u]);
    }
  }
  // in both groups the wanted rows are those with the LARGEST keys
  static __device__ __forceinline__ K key_of(int side, T s) {
    const K u = SK::of(s);
    return side == 0 ? u : (K)~u;
  }

  // One round of at most TOP iterations.  Returns the number of swaps, or -1: nothing was changed, and the
  // round has to be left to the full scan.  (uniform)
  static __device__ int round(const MaskArgs<T> &a, Shared &sh, int iterations, int *changed, int *nchanged) {
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int kNone = 0x7fffffff;
    if (tid < 2) sh.nlist[tid] = 0, sh.nan_first[tid] = kNone, sh.ahead[tid] = 0;
    if (tid < 128) sh.rank[tid >> 6][tid & 63] = 0;
    __syncthreads();
    // ---- phase A
    Rows first;
    load_rows(a, first, 0);
    KeyIdx<K> best[2] = {{0, -1}, {0, -1}};
    int nan_first[2] = {kNone, kNone};
    for_rows(a, first, [&](int i, int side, T s) {
      const bool num = s == s;
      const K key = key_of(side, s);  // (at least 1 for a number)
#pragma unroll
      for (int g = 0; g < 2; g++) {
        const bool take = num && side == g && key >= best[g].key;
        best[g].key = take ? key : best[g].key;
        best[g].idx = take ? i : best[g].idx;
      }
      if (!num) {
        if (side == 0) nan_first[0] = i < nan_first[0] ? i : nan_first[0];
        else if (side == 1) nan_first[1] = i < nan_first[1] ? i : nan_first[1];
      }
    });
#pragma unroll
    for (int g = 0; g < 2; g++) {
      const int bin = lane ^ (4 * wv);
      sh.bin_key[g][wv][bin] = best[g].key;
      sh.bin_idx[g][wv][bin] = best[g].idx;
      if (__ballot(nan_first[g] != kNone)) {  // one atomic per wavefront: they all hit one address
        const int lowest = wave_reduce(nan_first[g], [](int x, int y) { return y < x ? y : x; });
        if (lane == 0) atomicMin(&sh.nan_first[g], lowest);
      }
    }
    __syncthreads();
    // eight wavefronts per side: each has the side's 64 best rows, a lane each, and compares them with eight (one
    // wavefront with all 64: 3.5 us)
    const int g_of = wv / (NWV / 2);
    KeyIdx<K> b{0, -1};
#pragma unroll
    for (int w = 0; w < NWV; w++) b = pick_key<K>(b, KeyIdx<K>{sh.bin_key[g_of][w][lane], sh.bin_idx[g_of][w][lane]});
    {
      constexpr int PER = 64 / (NWV / 2);
      const int m0 = (wv % (NWV / 2)) * PER;
      int rank = 0;
#pragma unroll
      for (int m = 0; m < PER; m++) {
        const K km = readlane_k(b.key, m0 + m);
        const int im = __builtin_amdgcn_readlane(b.idx, m0 + m);
        rank += (im >= 0 && (km > b.key || (km == b.key && im > b.idx))) ? 1 : 0;
      }
      if (rank) atomicAdd(&sh.rank[g_of][lane], rank);
    }
    __syncthreads();
    if (wv % (NWV / 2) == 0) {
      const bool enough = __popcll(__ballot(b.idx >= 0)) >= TOP;  // else the side's rows are all listed
      if (enough ? (b.idx >= 0 && sh.rank[g_of][lane] == TOP - 1) : lane == 0) {
        sh.bound_key[g_of] = enough ? b.key : 0;
        sh.bound_idx[g_of] = enough ? b.idx : -1;
      }
    }
    __syncthreads();
    {
      const K bk[2] = {sh.bound_key[0], sh.bound_key[1]};
      const int bi[2] = {sh.bound_idx[0], sh.bound_idx[1]}, nf[2] = {sh.nan_first[0], sh.nan_first[1]};
      int ahead[2] = {0, 0};
      const bool nans = nf[0] != kNone || nf[1] != kNone;  // (uniform)
      for_rows(a, first, [&](int i, int side, T s) {
        const K key = key_of(side, s), bks = side == 0 ? bk[0] : bk[1];
        const bool num = side < 2 && s == s;
        if (num && key >= bks && (key > bks || i >= (side == 0 ? bi[0] : bi[1]))) {
          const int pos = atomicAdd(&sh.nlist[side], 1);
          if (pos < LIST) sh.list_key[side][pos] = key, sh.list_idx[side][pos] = i;
        }
        if (nans) {
#pragma unroll
          for (int g = 0; g < 2; g++) ahead[g] += (num && side == g && i < nf[g]) ? 1 : 0;
        }
      });
#pragma unroll
      for (int g = 0; g < 2; g++)
        if (nf[g] != kNone) {  // (uniform)
          const int sum = wave_reduce(ahead[g], [](int x, int y) { return x + y; });
          if (lane == 0) atomicAdd(&sh.ahead[g], sum);
        }
    }
    __syncthreads();
    int ntop[2];
#pragma unroll
    for (int g = 0; g < 2; g++) {
      if (sh.nlist[g] > LIST) return -1;
      ntop[g] = sh.nlist[g] < TOP ? sh.nlist[g] : TOP;
    }
    {
      const int g = tid >> 9, n = sh.nlist[g];
      for (int e = tid & 511; e < n; e += 512) {
        const K key = sh.list_key[g][e];
        const int idx = sh.list_idx[g][e];
        int rank = 0;
        constexpr int V = 8;  // entries whose LDS reads are in flight together
        for (int o0 = 0; o0 < n; o0 += V) {
          K ko[V];
          int io[V];
#pragma unroll
          for (int v = 0; v < V; v++) {  // (past the list: an entry that is not ahead of any)
            const int o = o0 + v < n ? o0 + v : e;
            ko[v] = sh.list_key[g][o], io[v] = sh.list_idx[g][o];
          }
#pragma unroll
          for (int v = 0; v < V; v++) rank += (ko[v] > key || (ko[v] == key && io[v] > idx)) ? 1 : 0;
        }
        if (rank < TOP) sh.top[g][rank] = idx;
      }
    }
    __syncthreads();
    // A NaN score counts only on a side's first candidate row.  While one of the scored rows ahead of the side's first
    // NaN is not among the rows that can be picked, that row (or one that joined the side ahead of it) is the first.
#pragma unroll
    for (int g = 0; g < 2; g++) {
      if (sh.nan_first[g] == kNone) continue;
      int pickable = 0;
      for (int k = 0; k < ntop[g]; k++) pickable += sh.top[g][k] < sh.nan_first[g] ? 1 : 0;
      if (sh.ahead[g] <= pickable) return -1;
    }
    if (wv == 0) {
      const int n = swaps_of_top(a, sh, iterations, ntop[0], ntop[1], changed, nchanged);
      if (lane == 0) sh.swaps = n;
    }
    __syncthreads();
    return sh.swaps;
  }

  // a row that has changed sides, as the next round and the caller find it
  static __device__ __forceinline__ void put_row(const MaskArgs<T> &a, int i, int side, int cs, T nom, int *changed,
                                                 int *nchanged) {
    a.wmask[(long)i * a.H + a.h] = (uint8_t)side;
    a.csum[i] = cs;
    a.side[i] = side;
    a.score[i] = mask_score<T>(nom, cs);
    note_changed(changed, nchanged, i);
  }

  // Phase B, by one wavefront: lane l holds the rank-l silent and the rank-l active candidate.  A pick is the maximum
  // of (key, row index) pairs -- the key orders the scores, the index settles equal scores in favour of the later
  // row, as the sequential >= / <= scans do.  A row that changes sides takes the score of its other side along
  // (csum +- 1), computed once up front, so the loop holds no division.
  static __device__ int swaps_of_top(const MaskArgs<T> &a, const Shared &sh, int iterations, int nS, int nA,
                                     int *changed, int *nchanged) {
    const int lane = threadIdx.x & 63;
    const int nS0 = nS, nA0 = nA;  // rows that change sides are appended from these slots on
    bool vS = lane < nS, vA = lane < nA;
    int iS = vS ? sh.top[0][lane] : 0, iA = vA ? sh.top[1][lane] : 0;
    int csS = vS ? a.csum[iS] : 0, csA = vA ? a.csum[iA] : 0;
    T nomS = vS ? a.nom[iS] : T(0), nomA = vA ? a.nom[iA] : T(0);
    // keys as seen from the silent side (largest score wins) and from the active side (smallest wins)
    K kS = SK::of(mask_score<T>(nomS, csS)), kS_other = (K)~SK::of(mask_score<T>(nomS, csS + 1));
    K kA = (K)~SK::of(mask_score<T>(nomA, csA)), kA_other = SK::of(mask_score<T>(nomA, csA - 1));
    // ---- All swaps at once, when that provably equals the loop below.  Iteration k of the loop picks the rank-k
    // candidates of both sides and swaps them unless the silent one scores lower, so the number of
    // swaps n is the length of the run of such pairs from rank 0 -- provided no row that changed sides
    // is ever picked again.  That holds when every new active row scores strictly above, and every new
    // silent row strictly below, the last pair the loop would look at; otherwise (blocks of equal scores,
    // dead inputs) the loop runs.  Both sides must also hold a candidate for every iteration that happens.
    {
      const int pairs = nS < nA ? nS : nA, kmax = iterations < pairs ? iterations : pairs;
      const K activeK = (K)~kA;  // (the key of the active candidate's score as the silent side has it)
      const unsigned long long keep_going = __ballot(lane < kmax && !(kS < activeK));
      const int n = __builtin_ctzll(~keep_going);  // (kmax <= 16: bit kmax is clear)
      if (n < kmax || kmax == iterations) {
        if (n == 0) return 0;  // nothing to swap
        const int last = n < kmax ? n : kmax - 1;  // the last pair the loop looks at
        const K lastS = readlane_k(kS, last), lastA = readlane_k(activeK, last);
        const bool swapped = lane < n;
        const bool again = swapped && (!((K)~kS_other > lastA) || !(kA_other < lastS));
        if (__ballot(again) == 0) {
          if (swapped) {
            put_row(a, iS, 1, csS + 1, nomS, changed, nchanged);
            put_row(a, iA, 0, csA - 1, nomA, changed, nchanged);
          }
          return n;
        }
      }
    }
    int it = 0;
    for (; it < iterations; it++) {
      KeyIdx<K> cmax{kS, vS ? iS : -1}, cmin{kA, vA ? iA : -1};
      cmax = wave_pick(cmax);
      cmin = wave_pick(cmin);
      if (cmax.idx < 0 || cmin.idx < 0) break;  // no silent or no active row
      if (cmax.key < (K)~cmin.key) break;       // vmax0 < vmin1
      const int lS = __builtin_ctzll(__ballot(vS && iS == cmax.idx));
      const int lA = __builtin_ctzll(__ballot(vA && iA == cmin.idx));
      const K wOther = readlane_k(kS_other, lS), wThis = cmax.key;  // winner: its active-side key, ...
      const K lOther = readlane_k(kA_other, lA), lThis = cmin.key;
      const int csW = __builtin_amdgcn_readlane(csS, lS), csL = __builtin_amdgcn_readlane(csA, lA);
      const T nomW = readlane_t(nomS, lS), nomL = readlane_t(nomA, lA);
      if (lane == lS) vS = false;
      if (lane == lA) vA = false;
      if (lane == nA) {  // the best silent row becomes active
        vA = true, iA = cmax.idx, csA = csW + 1, nomA = nomW;
        kA = wOther, kA_other = wThis;
      }
      if (lane == nS) {  // the worst active row becomes silent
        vS = true, iS = cmin.idx, csS = csL - 1, nomS = nomL;
        kS = lOther, kS_other = lThis;
      }
      nA++, nS++;
    }
    if (vS && lane >= nS0) put_row(a, iS, 0, csS, nomS, changed, nchanged);
    if (vA && lane >= nA0) put_row(a, iA, 1, csA, nomA, changed, nchanged);
    return it;
  }
};

// candidate row: score and row index (-1: none)
template <typename T>
struct Cand {
  T val;
  long idx;
};
// a sequential ascending scan with ">=" keeps the later of two equal maxima, with "<=" the later of two equal minima
template <typename T>
__device__ __forceinline__ Cand<T> better_max(Cand<T> a, Cand<T> b) {
  if (a.idx < 0) return b;
  if (b.idx < 0) return a;
  if (b.val > a.val || (b.val == a.val && b.idx > a.idx)) return b;
  return a;
}
template <typename T>
__device__ __forceinline__ Cand<T> better_min(Cand<T> a, Cand<T> b) {
  if (a.idx < 0) return b;
  if (b.idx < 0) return a;
  if (b.val < a.val || (b.val == a.val && b.idx > a.idx)) return b;
  return a;
}

// The iterations one by one, each a scan over all rows: what MaskSwap::round does not cover.
template <typename T>
__device__ void swap_by_scans(const MaskArgs<T> &a, long iterations, int *changed, int *nchanged) {
  __shared__ Cand<T> smax[16], smin[16];
  __shared__ long sfirst0[16], sfirst1[16];
  __shared__ int sstop;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  for (long it = 0; it < iterations; it++) {
    Cand<T> cmax{T(0), -1}, cmin{T(0), -1};
    long first0 = a.N, first1 = a.N;  // first candidate rows (for the NaN rule)
    for (long i = tid; i < a.N; i += 1024) {
      const int m = a.side[i];
      if (m > 1) continue;
      const T s = a.score[i];
      if (m == 0) {
        first0 = i < first0 ? i : first0;
        if (s == s) cmax = better_max<T>(cmax, Cand<T>{s, i});
      } else {
        first1 = i < first1 ? i : first1;
        if (s == s) cmin = better_min<T>(cmin, Cand<T>{s, i});
      }
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      Cand<T> o1{__shfl_xor(cmax.val, o), __shfl_xor(cmax.idx, o)};
      cmax = better_max<T>(cmax, o1);
      Cand<T> o2{__shfl_xor(cmin.val, o), __shfl_xor(cmin.idx, o)};
      cmin = better_min<T>(cmin, o2);
      const long f0 = __shfl_xor(first0, o), f1 = __shfl_xor(first1, o);
      first0 = f0 < first0 ? f0 : first0;
      first1 = f1 < first1 ? f1 : first1;
    }
    if (lane == 0) {
      smax[wv] = cmax;
      smin[wv] = cmin;
      sfirst0[wv] = first0;
      sfirst1[wv] = first1;
    }
    __syncthreads();
    if (tid == 0) {
      for (int k = 1; k < 16; k++) {
        cmax = better_max<T>(cmax, smax[k]);
        cmin = better_min<T>(cmin, smin[k]);
        first0 = sfirst0[k] < first0 ? sfirst0[k] : first0;
        first1 = sfirst1[k] < first1 ? sfirst1[k] : first1;
      }
      int stop = 0;
      if (first0 >= a.N || first1 >= a.N) {
        stop = 1;  // no silent or no active row
      } else {
        const T sf0 = a.score[first0], sf1 = a.score[first1];
        long imax0 = cmax.idx, imin1 = cmin.idx;
        T vmax0 = cmax.val, vmin1 = cmin.val;
        if (sf0 != sf0 || imax0 < 0) { imax0 = first0; vmax0 = sf0; }
        if (sf1 != sf1 || imin1 < 0) { imin1 = first1; vmin1 = sf1; }
        if (vmax0 < vmin1) {
          stop = 1;
        } else {
          const int cs1 = a.csum[imax0] + 1, cs0 = a.csum[imin1] - 1;
          a.wmask[imax0 * a.H + a.h] = 1;
          a.wmask[imin1 * a.H + a.h] = 0;
          a.csum[imax0] = cs1, a.side[imax0] = 1, a.score[imax0] = mask_score<T>(a.nom[imax0], cs1);
          a.csum[imin1] = cs0, a.side[imin1] = 0, a.score[imin1] = mask_score<T>(a.nom[imin1], cs0);
          note_changed(changed, nchanged, imax0);
          note_changed(changed, nchanged, imin1);
        }
      }
      sstop = stop;
    }
    __syncthreads();
    if (sstop) break;
    __syncthreads();
  }
}

// Steps 3 and 4 in the swap kernel's wake (a.W_fix != nullptr), by the whole workgroup: the weights of the
// rows that changed sides -- every other row of the hypercolumn already holds what its unchanged mask byte
// asks for -- and the hypercolumn's row list.  All threads of the workgroup call it.
template <typename T, int NT>
__device__ __forceinline__ void mask_swap_finish(const MaskArgs<T> &a, const int *changed, const int *nchanged) {
  if (a.W_fix == nullptr) return;  // uniform
  __syncthreads();                 // mask bytes and the list of changed rows are written
  if (a.rows != nullptr) mask_rows_block<NT>(a.rows, a.row_cnt, a.wmask, a.N, a.H, a.cap, a.h);
  // A thread owns a column (or every NT-th) and walks the rows, so that a reciprocal is formed once per row and once
  // per thread; one CU does all of this, and in doubles its vector unit is what it waits for.
  __shared__ T row_rci[kMaxChangedRows];
  const int nc = *nchanged < kMaxChangedRows ? *nchanged : kMaxChangedRows, tid = threadIdx.x;
  if (tid < nc) row_rci[tid] = trace_reciprocal<T>(a.Ci[changed[tid]], a.cthr);
  __syncthreads();
  const int cols = a.Mc < NT ? (int)a.Mc : NT, groups = NT / cols;
  if (tid >= groups * cols) return;
  constexpr int U = 8;  // rows whose loads are in flight together
  for (long c = tid % cols; c < a.Mc; c += cols) {
    const long j = a.h * a.Mc + c;
    const T rcj = trace_reciprocal<T>(a.Cj[j], a.cthr);
    for (int r0 = tid / cols; r0 < nc; r0 += groups * U) {
      long i[U];
      T cij[U];
      uint8_t on[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        i[u] = changed[r0 + groups * u < nc ? r0 + groups * u : r0];
        cij[u] = a.Cij[i[u] * a.M + j], on[u] = a.wmask[i[u] * a.H + a.h];
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int r = r0 + groups * u;
        if (r >= nc) break;
        a.W_fix[i[u] * a.M + j] = on[u] != 0 ? weight_from_traces<T>(cij[u], row_rci[r], rcj, a.cthr4) : T(0);
      }
    }
  }
}

template <typename T>
__global__ __launch_bounds__(1024) void k_mask_swap(MaskArgs<T> a) {
  using S = MaskSwap<T>;
  __shared__ typename S::Shared sh;
  __shared__ int changed[kMaxChangedRows], nchanged;  // rows that changed sides, see mask_swap_finish
  if (threadIdx.x == 0) nchanged = 0;                 // (published by the barriers of the first round)
  __syncthreads();
  for (long left = a.iterations; left > 0;) {
    const int n = (int)(left < S::TOP ? left : S::TOP);
    const int done = a.N < (1L << 31) ? S::round(a, sh, n, changed, &nchanged) : -1;  // (row indices are 32-bit there)
    if (done < 0) {
      __syncthreads();
      swap_by_scans<T>(a, left, changed, &nchanged);
      break;
    }
    if (done < n) break;
    left -= n;
  }
  mask_swap_finish<T, S::NT>(a, changed, &nchanged);
}

}  // namespace sb
