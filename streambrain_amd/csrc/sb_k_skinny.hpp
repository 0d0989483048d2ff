// Layers with very few output units (the 10-unit classification layer): forward and training passes on
// plain vector arithmetic.  With M <= 32 output columns an MFMA tile would be mostly padding, and the
// whole problem is a few million multiply-adds whose cost is latency, not arithmetic; what matters is
// that every load is coalesced and that no thread does more than a few hundred instructions.
//
// Thread layout shared by both kernels: R = 256 / M rows of W (or Cij) per pass, thread t < R*M owns
// column j = t % M of row r = t / M, so the R*M threads of a pass read R*M consecutive elements.
#pragma once
#include "sb_kernels.hpp"

namespace sb {

// act[b, :] = softmax_per_hypercolumn(x[b, :] . W + bias)      omp.cc:70-87 + kernels_numpy.py:13-25
// One workgroup per batch row.  Partial sums over the rows r, r + R, ... are added up in the order of r
// (fixed, so the result is deterministic).
// Classification in the same launch (_cpu_base_backend.py:239-241), when pred or labels is given: the
// row's first maximal unit goes to pred[b], and *correct counts the rows whose first maximal unit is the
// labels' first maximal unit -- the result k_argmax_rows gives on the stored activations.
template <typename T>
__global__ __launch_bounds__(256) void k_forward_skinny(T *act, const T *x, const T *W, const T *bias,
                                                        long N, long M, long Mc, int softmax,
                                                        const T *labels, int32_t *pred,
                                                        unsigned long long *correct) {
  __shared__ T part[256];
  __shared__ T logit[32];
  const int tid = threadIdx.x;
  const int R = 256 / (int)M;
  const int j = tid % (int)M, r = tid / (int)M;
  const T *xrow = x + (long)blockIdx.x * N;
  T acc = T(0);
  if (r < R) {
    // pointers advance by R rows per step, so a load costs one address addition and no multiplication
    const T *xq = xrow + r, *wq = W + (long)r * M + j;
    const long wstep = (long)R * M;
    long i = r;
    for (; i + 7 * R < N; i += 8 * R) {  // 8 rows of loads in flight
      T xv[8], wv[8];
#pragma unroll
      for (int k = 0; k < 8; k++) {
        xv[k] = *xq, wv[k] = *wq;
        xq += R, wq += wstep;
      }
#pragma unroll
      for (int k = 0; k < 8; k++) acc += xv[k] * wv[k];
    }
    for (; i < N; i += R, xq += R, wq += wstep) acc += *xq * *wq;
  }
  part[tid] = acc;
  __syncthreads();
  if (tid < M) {
    T s = T(0);
    for (int k = 0; k < R; k++) s += part[k * (int)M + tid];
    logit[tid] = s + bias[tid];
  }
  __syncthreads();
  T v = T(0);
  if (tid < M) {
    v = logit[tid];
    if (softmax) {
      const int h0 = (tid / (int)Mc) * (int)Mc;  // first unit of this thread's hypercolumn
      T mx = -INFINITY;
      for (int c = 0; c < Mc; c++) mx = logit[h0 + c] > mx ? logit[h0 + c] : mx;
      T sum = T(0);
      for (int c = 0; c < Mc; c++) sum += Real<T>::exp_(logit[h0 + c] - mx);
      v = Real<T>::exp_(v - mx) / sum;
    }
    act[(long)blockIdx.x * M + tid] = v;
  }
  if (pred == nullptr && labels == nullptr) return;  // uniform
  __syncthreads();  // everybody has read the logits
  if (tid < M) logit[tid] = v;
  __syncthreads();
  if (tid == 0) {
    int best = 0;
    for (int c = 1; c < M; c++) best = logit[c] > logit[best] ? c : best;
    if (pred) pred[blockIdx.x] = best;
    if (labels) {
      const T *lab = labels + (long)blockIdx.x * M;
      int lbest = 0;
      for (int c = 1; c < M; c++) lbest = lab[c] > lab[lbest] ? c : lbest;
      if (lbest == best) atomicAdd(correct, 1ull);
    }
  }
}

// The fused training pass of k_train_fused (same arguments, same results within rounding) for M <= 32:
// one workgroup per R rows of Cij (skinny_train_rows), thread (r, j) owning one element.  The workgroup stages its
// R columns of x and all of y in LDS, `bc` batch rows at a time, with every load of a chunk in flight at
// once (a row of x contributes R consecutive elements, a row of y all M); each thread then walks the
// chunk in LDS, accumulating its x^T y element and, in batch order and without FMA contraction, the
// column sums its row's Ci and its column's Cj are made of -- the reference's order, so the traces are
// bit-exact as in the tiled kernel.  Rows past the batch are staged as zeros, which change no sum.
// bc (set by the launcher): at most kSkinnyLoads passes of either staging loop, at most kSkinnyStage
// staged elements, byte offsets of a chunk of x below 2 GiB.
// Rows of Cij per workgroup: as many as fit 256 threads, at most 32 (with fewer columns than 8 some threads
// only stage; more rows would shorten the chunks the staging loops can cover).
__host__ __device__ constexpr int skinny_train_rows(long M) { return 256 / M < 32 ? (int)(256 / M) : 32; }
constexpr int kSkinnyLoads = 16;
constexpr int kSkinnyStage = 8192;
template <typename T>
__global__ __launch_bounds__(256) void k_train_skinny(TrainArgs<T> a, int bc) {
  using Rl = Real<T>;
  __shared__ T stage[kSkinnyStage];
  const int tid = threadIdx.x;
  const int M = (int)a.M;
  const int R = skinny_train_rows(M);
  const int j = tid % M, r = tid / M;
  const long i0 = (long)blockIdx.x * R, i = i0 + r;
  const bool mine = r < R && i < a.N;  // this thread owns an element of Cij
  T *xs = stage, *ys = stage + bc * R;
  // staging roles: x by (row xb of a pass, column xr), y by (row yb, column yj)
  const int xrows = 256 / R, xb = tid / R, xr = tid % R;  // xrows * R <= 256 threads load x
  const int yrows = 256 / M, yb = tid / M, yj = tid % M;
  const bool xload = xb < xrows && i0 + xr < a.N, yload = yb < yrows;
  constexpr unsigned ES = sizeof(T);
  const T cij_old = mine ? a.Cij[i * a.M + j] : T(0);  // requested first, used last
  T dot = T(0), sx = T(0), sy = T(0);
  for (long b0 = 0; b0 < a.B; b0 += bc) {
    const long left = a.B - b0;  // rows of this chunk inside the batch: min(left, bc)
    const BufferWindow<T> xwin(a.x + b0 * a.N + i0, (left - 1) * a.N + (a.N - i0)),
        ywin(a.y + b0 * a.M, left * a.M);
    T xv[kSkinnyLoads], yv[kSkinnyLoads];
#pragma unroll
    for (int k = 0; k < kSkinnyLoads; k++) {
      const int bx = xb + k * xrows, by = yb + k * yrows;
      T one[1];
      xwin.template load_n<1>(one, xload && bx < bc ? (unsigned)(((long)bx * a.N + xr) * ES)
                                                    : BufferWindow<T>::kOutside);
      xv[k] = one[0];
      ywin.template load_n<1>(one, yload && by < bc ? (unsigned)(((long)by * a.M + yj) * ES)
                                                    : BufferWindow<T>::kOutside);
      yv[k] = one[0];
    }
    if (b0 > 0) __syncthreads();  // the previous chunk has been consumed
#pragma unroll
    for (int k = 0; k < kSkinnyLoads; k++) {
      const int bx = xb + k * xrows, by = yb + k * yrows;
      if (xb < xrows && bx < bc) xs[bx * R + xr] = xv[k];
      if (yload && by < bc) ys[by * M + yj] = yv[k];
    }
    __syncthreads();
    if (mine) {
      const int rows = left < bc ? (int)left : bc;
      for (int b = 0; b < rows; b++) {
        const T xk = xs[b * R + r], yk = ys[b * M + j];
        dot += xk * yk;
        sx = Rl::add(sx, xk);
        sy = Rl::add(sy, yk);
      }
    }
  }
  if (!mine) return;
  const T ci = trace_next<T>(a.Ci[i], sx, a), cj = trace_next<T>(a.Cj[j], sy, a);
  if (j == 0) a.Ci_next[i] = ci;
  if (i == 0) {
    a.Cj_next[j] = cj;
    if (a.bias_mode == 1) {
      T kb = a.kbi[j];
      a.bias[j] = bias_regularized<T>(cj, kb, a.cthr, a.khalf, a.pmin, a.taubdt);
      a.kbi[j] = kb;
    }
  }
  T cn = cij_old * a.omt + dot * (a.invB * a.tau);
  cn = fmax(cn, T(0));
  a.Cij[i * a.M + j] = cn;
  const T wgt = weight_from_traces<T>(cn, trace_reciprocal<T>(ci, a.cthr), trace_reciprocal<T>(cj, a.cthr),
                                      a.cthr4);
  const bool on = a.wmask == nullptr || a.wmask[i * a.H + j / (int)a.Mc] != 0;
  if (a.W) a.W[i * a.M + j] = on ? wgt : T(0);
}

// k_train_skinny over many batches in one launch, for layers without mask and regularised bias (a classification layer whose
// inputs, the frozen activations of the layers below it, are all there): a workgroup keeps its elements of Cij and its
// traces in registers from batch to batch, and the weights, which nothing reads in between, are formed once at the end.
// Same sums in the same order, so the same bits as a launch per batch.
// A launch per batch takes 7.9 us at 3000 x 10, batch 128, and the shuffle of its inputs 115 us per 20000 rows: launch and
// completion, a round of cold loads, a walk over the batch, stores.  What is left here is the walk.  A wavefront issues
// a vector instruction every 4 ns at best, so the work is dealt out: wavefronts 4 to 7 bring kRows batch rows at a time
// to LDS, kAhead such chunks ahead of their use, while thread (r, j) of wavefronts 0 to 2 adds up the products of its
// element (i0 + r, j) and wavefront 3 the columns, lane r < R one of x, lane 32 + j one of y.  In LDS the batch rows of a column
// lie side by side, so that a thread takes a vector of them at a time.
// 3000 x 10, batch 128: 14.7 us for seven batches (with four wavefronts that do both 21.6, with two sets of loads between
// waits for all of them 34.8), 1.5 us for each further one.
template <typename T>
struct SkinnyEpochArgs {
  TrainArgs<T> a;        // of a whole batch
  const int64_t *order;  // batch row b is row order[b] of a.x and row b of a.y
  long rows;             // batch rows in all
  T fB_last, invB_last;  // of the last batch
};
constexpr int kSkinnyEpochRows = 64, kSkinnyEpochAhead = 4;
// Rows of Cij per workgroup: 192 threads' worth, at most 16 (a 64-byte run of a row of x in floats: more would be fewer
// workgroups than CUs at a few thousand inputs, fewer would share out each line among more CUs).
__host__ __device__ constexpr int skinny_epoch_rows(long M) { return 192 / M < 16 ? (int)(192 / M) : 16; }
// MAXM: 16 or 32, at least M.
template <typename T, int MAXM>
__global__ __launch_bounds__(512) void k_train_skinny_epoch(SkinnyEpochArgs<T> e) {
  using Rl = Real<T>;
  using vec_t = typename Rl::vec_t;
  constexpr int CB = kSkinnyEpochRows, AHEAD = kSkinnyEpochAhead, VW = Rl::VW, P = CB + VW;
  const TrainArgs<T> &a = e.a;
  __shared__ __attribute__((aligned(16))) T xs[2][16 * P], ys[2][MAXM * P];
  __shared__ T ci_s[16], cj_s[MAXM];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int M = (int)a.M, R = skinny_epoch_rows(M);
  const long N = a.N, groups = (N + R - 1) / R, per_xcd = (groups + 7) / 8;
  const long group = (long)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);  // neighbours, which share lines of x, on one XCD
  if ((long)(blockIdx.x >> 3) >= per_xcd || group >= groups) return;
  const long i0 = group * R;

  // Where a chunk lies: rows row .. row + left (at most CB) of a batch that ends at `end`.  Past the last row: none.
  struct Chunk {
    long row, end, rows, B;
    __device__ int size() const { return end - row < CB ? (int)(end - row) : CB; }
    __device__ bool completes() const { return row + CB >= end; }  // its batch
    __device__ bool last() const { return completes() && end == rows; }
    __device__ void next() {
      row += CB;
      if (row < end) return;
      row = end;
      end += rows - end < B ? rows - end : B;
    }
  };
  Chunk cur{0, a.B < e.rows ? a.B : e.rows, e.rows, a.B};

  if (w >= 4) {
    // ---- x by (row xb of a pass of 16, column xr), y by (row yb of a pass, column yj)
    constexpr int XL = CB * 16 / 256, YL = CB * MAXM / 256;  // loads per thread and chunk
    const int t = tid - 256, xb = t >> 4, xr = t & 15, ypass = 256 / M, yb = t / M, yj = t - yb * M;
    const bool xload = xr < R && i0 + xr < N, yload = yb < ypass;
    const T *const xcol = a.x + i0 + (xload ? xr : 0);
    const T *const ycol = a.y + (yload ? yj : 0);
    Chunk look = cur, req = cur;
    // Loads return in order: the data set's rows behind a chunk are looked up right behind the loads of the chunk AHEAD
    // before it, so that the addresses wait for nothing that is still wanted in flight.
    int at[AHEAD][XL];
    auto look_up = [&](int s) {
#pragma unroll
      for (int k = 0; k < XL; k++) {
        const long row = look.row + xb + 16 * k, in = row < e.rows ? row : e.rows - 1;
        at[s][k] = reinterpret_cast<const int *>(e.order)[2 * in];  // (the lower half: data sets are smaller than 2^31)
      }
      look.next();
    };
    T xv[AHEAD][XL], yv[AHEAD][YL];
    auto request = [&](int s) {  // (unguarded: what is not of the chunk is an element that is there, and zero when staged)
#pragma unroll
      for (int k = 0; k < XL; k++) xv[s][k] = xcol[(long)at[s][k] * N];
#pragma unroll
      for (int k = 0; k < YL; k++) {
        const long row = req.row + yb + k * ypass;
        yv[s][k] = ycol[(row < e.rows ? row : e.rows - 1) * M];
      }
      req.next();
      __builtin_amdgcn_sched_barrier(0);  // (the order of the loads is what the waits go by)
      look_up(s);
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int s = 0; s < AHEAD; s++) look_up(s);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < AHEAD; s++) request(s);
    auto turn = [&](auto set) {
      constexpr int s = decltype(set)::value, buf = s & 1;
      const int n = cur.size();
#pragma unroll
      for (int k = 0; k < XL; k++) xs[buf][xr * P + xb + 16 * k] = xload && xb + 16 * k < n ? xv[s][k] : T(0);
#pragma unroll
      for (int k = 0; k < YL; k++) {
        const int b = yb + k * ypass;
        if (yload && b < CB) ys[buf][yj * P + b] = b < n ? yv[s][k] : T(0);
      }
      request(s);
      __syncthreads();  // the chunk is there; the buffer written next has been read by now
      const bool done = cur.last();
      cur.next();
      return done;
    };
    static_assert(AHEAD == 4, "turns below");
    for (;;) {
      if (turn(std::integral_constant<int, 0>{})) break;  // (uniform)
      if (turn(std::integral_constant<int, 1>{})) break;
      if (turn(std::integral_constant<int, 2>{})) break;
      if (turn(std::integral_constant<int, 3>{})) break;
    }
    __syncthreads();
    return;
  }

  const bool adder = w == 3;
  const int j = tid % M, r = tid / M;
  const bool mine = !adder && r < R && i0 + r < N;
  const bool adds_x = adder && lane < R && i0 + lane < N, adds_y = adder && lane >= 32 && lane - 32 < M;
  const long i = i0 + r;
  // this thread's element of Cij and its product sum, or its trace and its column sum
  T state = *(mine ? a.Cij + i * M + j : adds_x ? a.Ci + i0 + lane : adds_y ? a.Cj + lane - 32 : a.Cj), acc = T(0);
  const int xfrom = mine ? r * P : 0, yfrom = (mine ? j : 0) * P;
  const int sfrom = adds_x ? lane * P : adds_y ? (lane - 32) * P : 0;
  // 16 rows at a time, the next 16 on their way from LDS (rows past the batch are zero, which changes no sum)
  constexpr int V = 16 / VW;
  for (int buf = 0;; buf ^= 1) {
    __syncthreads();  // the chunk is there
    const int n = cur.size();
    if (adder) {
      const T *const from = (adds_y ? ys[buf] : xs[buf]) + sfrom;
      vec_t v[2][V];
#pragma unroll
      for (int u = 0; u < V; u++) v[0][u] = *reinterpret_cast<const vec_t *>(from + u * VW);
#pragma unroll
      for (int g = 0; g < CB / 16; g++) {
        if (16 * g >= n) break;  // (uniform)
        if (g + 1 < CB / 16) {
#pragma unroll
          for (int u = 0; u < V; u++) v[(g + 1) & 1][u] = *reinterpret_cast<const vec_t *>(from + 16 * (g + 1) + u * VW);
        }
#pragma unroll
        for (int u = 0; u < V; u++)
#pragma unroll
          for (int k = 0; k < VW; k++) acc = Rl::add(acc, v[g & 1][u][k]);
      }
    } else {
      const T *const fx = xs[buf] + xfrom, *const fy = ys[buf] + yfrom;
      vec_t vx[2][V], vy[2][V];
#pragma unroll
      for (int u = 0; u < V; u++) {
        vx[0][u] = *reinterpret_cast<const vec_t *>(fx + u * VW);
        vy[0][u] = *reinterpret_cast<const vec_t *>(fy + u * VW);
      }
#pragma unroll
      for (int g = 0; g < CB / 16; g++) {
        if (16 * g >= n) break;  // (uniform)
        if (g + 1 < CB / 16) {
#pragma unroll
          for (int u = 0; u < V; u++) {
            vx[(g + 1) & 1][u] = *reinterpret_cast<const vec_t *>(fx + 16 * (g + 1) + u * VW);
            vy[(g + 1) & 1][u] = *reinterpret_cast<const vec_t *>(fy + 16 * (g + 1) + u * VW);
          }
        }
#pragma unroll
        for (int u = 0; u < V; u++)
#pragma unroll
          for (int k = 0; k < VW; k++) acc += vx[g & 1][u][k] * vy[g & 1][u][k];
      }
    }
    const bool done = cur.last();
    if (cur.completes()) {  // (uniform) a batch is complete
      TrainArgs<T> b = a;
      if (done) b.fB = e.fB_last, b.invB = e.invB_last;
      if (adder) {
        state = trace_next<T>(state, acc, b);
      } else {
        const T cn = state * b.omt + acc * (b.invB * b.tau);
        state = fmax(cn, T(0));
      }
      acc = T(0);
    }
    cur.next();
    if (done) break;
  }
  if (adds_x) ci_s[lane] = state, a.Ci_next[i0 + lane] = state;
  if (adds_y) {
    cj_s[lane - 32] = state;
    if (i0 == 0) a.Cj_next[lane - 32] = state;
  }
  __syncthreads();
  if (!mine) return;
  a.Cij[i * M + j] = state;
  a.W[i * M + j] = weight_from_traces<T>(state, trace_reciprocal<T>(ci_s[r], a.cthr), trace_reciprocal<T>(cj_s[j], a.cthr),
                                         a.cthr4);
}

}  // namespace sb
