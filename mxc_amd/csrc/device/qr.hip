// Householder factorizations of the basis construction, one matrix per
// workgroup (or per few waves), of variable sizes.
//
//  * qr:    Householder QR (Eigen HouseholderQR reflector convention,
//           h2matrix.cpp:78-79,102-105): beta = -sign(x0)||x||,
//           v = [1; x_tail/(x0 - beta)], tau = (beta - x0)/beta.
//  * cpqr:  column-pivoted QR with Eigen ColPivHouseholderQR semantics
//           (h2matrix.cpp:84-89): first-index argmax of the updated column
//           norms, LAPACK xGEQPF norm downdating with recomputation below
//           sqrt(eps), the "nonzero pivots" cut and rank() = #{|R_ii| > tol *
//           max pivot}. Stops as soon as the rank is settled.
//  * formq: the explicit Q of a QR.
//  * trsolve: X = R11^{-1} R12 of a pivoted QR.
// In all of them a wave holds whole columns, row lane + 64 j of a column in
// register j of a lane: loads are coalesced, and the wave's columns take part
// in one reduction together (wave_sums).
#include <cfloat>
#include <map>

#include "internal.hpp"
#include "wave.hpp"

namespace mxg {
namespace {

// This workgroup's task, its pointers known to be global ones.
__device__ inline QrTask read_task(const QrTask* __restrict__ tasks) {
  QrTask t = in_constant(tasks)[blockIdx.x];
  t.A = in_global(t.A);
  t.tau = in_global(t.tau);
  return t;
}
__device__ inline CpqrTask read_task(const CpqrTask* __restrict__ tasks) {
  CpqrTask t = in_constant(tasks)[blockIdx.x];
  t.A = in_global(t.A);
  t.perm = in_global(t.perm);
  t.rank_out = in_global(t.rank_out);
  t.work = in_global(t.work);
  return t;
}
__device__ inline FormQTask read_task(const FormQTask* __restrict__ tasks) {
  FormQTask t = in_constant(tasks)[blockIdx.x];
  t.P = in_global(t.P);
  t.tau = in_global(t.tau);
  t.Q = in_global(t.Q);
  t.R = in_global(t.R);
  return t;
}
__device__ inline TrTask read_task(const TrTask* __restrict__ tasks) {
  TrTask t = in_constant(tasks)[blockIdx.x];
  t.R0 = in_global(t.R0);
  t.X = in_global(t.X);
  return t;
}

// Rows a lane holds for n rows: the smallest of the compiled counts that fits.
constexpr int ROW_STEPS[] = {1, 2, 3, 4, 5, 6, 8, 12, 16};
inline int row_steps(int n) {
  for (int r : ROW_STEPS)
    if (n <= 64 * r) return r;
  return 0;
}
#define MXG_FOR_ROW_STEPS(CASE) CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(8) CASE(12) CASE(16)

// Entry k of a column held as x[j] = row lane + 64 j (k wave-uniform).
template <int R>
__device__ inline double col_entry(const double (&x)[R], int k) {
  double v = x[0];
#pragma unroll
  for (int j = 1; j < R; j++)
    if (j == (k >> 6)) v = x[j];
  return lane_get(v, k & 63);
}

// Reflector of rows k .. of the column x held by one wave: x becomes v (zero
// above k, 1 at k); returns beta and tau.
template <int R>
__device__ inline double wave_reflector(double (&x)[R], int k, int lane, double& tau) {
  double s = 0.;
#pragma unroll
  for (int j = 0; j < R; j++)
    if (lane + 64 * j > k) s += x[j] * x[j];
  s = wave_total(s);
  const double c0 = col_entry<R>(x, k);
  double beta = c0, sc = 0.;
  tau = 0.;
  if (!(s <= DBL_MIN)) {
    beta = sqrt(c0 * c0 + s);
    if (c0 >= 0.) beta = -beta;
    sc = 1. / (c0 - beta);
    tau = (beta - c0) / beta;
  }
#pragma unroll
  for (int j = 0; j < R; j++) {
    const int row = lane + 64 * j;
    x[j] = row > k ? (sc != 0. ? x[j] * sc : 0.) : (row == k ? 1. : 0.);
  }
  return beta;
}

struct Red {
  double v[4];
  int i[4];
};

__device__ inline double wg_sum(double v, Red& r) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) r.v[wave] = v;
  __syncthreads();
  return (r.v[0] + r.v[1]) + (r.v[2] + r.v[3]);
}

// max of v over the workgroup; ties resolved to the smallest index.
__device__ inline void wg_argmax(double v, int idx, Red& r, double& bv, int& bi) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    double ov = __shfl_xor(v, o, 64);
    int oi = __shfl_xor(idx, o, 64);
    if (ov > v || (ov == v && oi < idx)) { v = ov; idx = oi; }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) { r.v[wave] = v; r.i[wave] = idx; }
  __syncthreads();
  bv = r.v[0];
  bi = r.i[0];
  for (int w = 1; w < 4; w++)
    if (r.v[w] > bv || (r.v[w] == bv && r.i[w] < bi)) { bv = r.v[w]; bi = r.i[w]; }
}

// Householder reflector of x[0..len) (stride 1) in place; returns beta, writes tau.
// All threads participate; x[0] is left for the caller to overwrite with beta.
__device__ inline double make_reflector(double* x, int len, Red& r, double& tau) {
  double s = 0.;
  for (int i = 1 + threadIdx.x; i < len; i += 256) s += x[i] * x[i];
  s = wg_sum(s, r);
  const double c0 = x[0];
  double beta;
  if (s <= DBL_MIN) {
    tau = 0.;
    beta = c0;
    for (int i = 1 + threadIdx.x; i < len; i += 256) x[i] = 0.;
  } else {
    beta = sqrt(c0 * c0 + s);
    if (c0 >= 0.) beta = -beta;
    const double sc = 1. / (c0 - beta);
    for (int i = 1 + threadIdx.x; i < len; i += 256) x[i] *= sc;
    tau = (beta - c0) / beta;
  }
  return beta;
}

// Apply H = I - tau [1; v][1; v]^T (v = x[1..len)) to columns c of the block
// starting at row 0 of `base` (ld) for c in [c0, c1). Wave per column.
__device__ inline void apply_reflector(const double* x, int len, double tau, double* base, long long ld, int c0, int c1) {
  if (tau == 0.) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int c = c0 + wave; c < c1; c += 4) {
    double* col = base + (long long)c * ld;
    double w = (lane == 0) ? col[0] : 0.;
    for (int i = 1 + lane; i < len; i += 64) w += x[i] * col[i];
    w = wave_sum(w) * tau;
    if (lane == 0) col[0] -= w;
    for (int i = 1 + lane; i < len; i += 64) col[i] -= w * x[i];
  }
}

// Matrices of more rows or columns than the register kernel takes: the matrix
// stays in global memory.
__global__ void __launch_bounds__(256) k_qr(const QrTask* __restrict__ tasks) {
  __shared__ Red red;
  __shared__ double sh_tau;
  const QrTask t = read_task(tasks);
  const int size = min(t.m, t.n);
  for (int k = 0; k < size; k++) {
    double* col = t.A + k + (long long)k * t.lda;
    const int len = t.m - k;
    double tau;
    const double beta = make_reflector(col, len, red, tau);
    __syncthreads();
    if (threadIdx.x == 0) {
      col[0] = beta;
      t.tau[k] = tau;
      sh_tau = tau;
    }
    __syncthreads();
    apply_reflector(col, len, sh_tau, t.A + k, t.lda, k + 1, t.n);
    __syncthreads();
  }
  if (t.zero_lower)
    for (long long e = threadIdx.x; e < (long long)size * size; e += 256) {
      const int i = (int)(e % size), j = (int)(e / size);
      if (i > j) t.A[i + (long long)j * t.lda] = 0.;
    }
}

// f(integral_constant<int, I>) for I = 0 .. N - 1: a loop whose index can pick
// registers however long its body is.
template <int N, int I = 0, class F>
__device__ inline void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, I + 1>(f);
  }
}

// QR with the matrix in registers: eight waves, wave w holds columns w, w + 8,
// ... (C of them). Step k is one wave's reflector, which reaches the others
// through LDS (double-buffered by the parity of k, so one barrier a step),
// then every wave's update of its own columns. A column whose step is past
// takes part in the updates unread: it is stored when its step is done. The
// step is bound by its chain (reduction, square root, two divisions, barrier,
// reduction), not by the arithmetic: seven levels of up to 256 x 100 take 0.81
// ms, 11.9 ms with the matrix in global memory.
template <int R, int C>
__global__ void __launch_bounds__(512) k_qr_reg(const QrTask* __restrict__ tasks) {
  constexpr int G = C < 8 ? 4 : 8;
  __shared__ double vs[2][64 * R];
  __shared__ double taus[2];
  const QrTask t = read_task(tasks);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int size = min(t.m, t.n);
  double a[C][R];
#pragma unroll
  for (int i = 0; i < C; i++)
#pragma unroll
    for (int j = 0; j < R; j++) {
      const int row = lane + 64 * j, col = wave + 8 * i;
      a[i][j] = (row < t.m && col < t.n) ? t.A[row + (long long)col * t.lda] : 0.;
    }
  static_for<C>([&](auto step) {
    constexpr int i = decltype(step)::value;
    for (int w = 0; w < 8; w++) {
      const int k = 8 * i + w;
      if (k >= size) break;
      const int b = k & 1;
      if (wave == w) {
        double above[R], tau;
#pragma unroll
        for (int j = 0; j < R; j++) above[j] = a[i][j];
        const double beta = wave_reflector<R>(a[i], k, lane, tau);
        double* col = t.A + (long long)k * t.lda;
#pragma unroll
        for (int j = 0; j < R; j++) {
          const int row = lane + 64 * j;
          vs[b][row] = a[i][j];
          const double low = (t.zero_lower && row < size) ? 0. : a[i][j];
          if (row < t.m) col[row] = row < k ? above[j] : (row == k ? beta : low);
        }
        if (lane == 0) {
          taus[b] = tau;
          t.tau[k] = tau;
        }
      }
      __syncthreads();
      double v[R];
#pragma unroll
      for (int j = 0; j < R; j++) v[j] = vs[b][lane + 64 * j];
      const double tau = taus[b];
#pragma unroll
      for (int c0 = i; c0 < C; c0 += G) {
        double d[G], s[G / 4];
#pragma unroll
        for (int g = 0; g < G; g++) {
          d[g] = 0.;
          if (c0 + g < C)
#pragma unroll
            for (int j = 0; j < R; j++) d[g] += v[j] * a[c0 + g < C ? c0 + g : 0][j];
        }
        wave_sums<G>(d, s);
#pragma unroll
        for (int g = 0; g < G; g++)
          if (c0 + g < C) {
            const double wg = sum_of<G>(s, g) * tau;
#pragma unroll
            for (int j = 0; j < R; j++) a[c0 + g][j] -= wg * v[j];
          }
      }
    }
  });
  // columns past the last step (n > m) hold R entries only
#pragma unroll
  for (int i = 0; i < C; i++) {
    const int col = wave + 8 * i;
    if (col >= size && col < t.n)
#pragma unroll
      for (int j = 0; j < R; j++) {
        const int row = lane + 64 * j;
        if (row < t.m) t.A[row + (long long)col * t.lda] = a[i][j];
      }
  }
}

// Matrices beyond the blocked kernel's sizes: one reflector at a time on the
// matrix in global memory.
__global__ void __launch_bounds__(256) k_cpqr(const CpqrTask* __restrict__ tasks) {
  __shared__ Red red;
  __shared__ double sh_tau, sh_maxpivot;
  const CpqrTask t = read_task(tasks);
  const int K = t.K, M = t.M, size = min(K, M);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double* upd = t.work;
  double* dir = t.work + M;
  for (int j = threadIdx.x; j < M; j += 256) t.perm[j] = j;
  for (int j = wave; j < M; j += 4) {
    const double* col = t.A + (long long)j * t.lda;
    double s = 0.;
    for (int i = lane; i < K; i += 64) s += col[i] * col[i];
    s = wave_sum(s);
    if (lane == 0) upd[j] = dir[j] = sqrt(s);
  }
  __syncthreads();
  double mx = 0.;
  for (int j = threadIdx.x; j < M; j += 256) mx = fmax(mx, upd[j]);
  double maxnorm;
  int dummy;
  wg_argmax(mx, 0, red, maxnorm, dummy);
  const double eps = DBL_EPSILON;
  const double th_helper = (maxnorm * eps) * (maxnorm * eps) / (double)K;
  const double downdate_th = sqrt(eps);
  int nonzero = size, done = 0;
  double maxpivot = 0.;
  for (int k = 0; k < t.steps; k++) {
    double bv = -1.;
    int bi = M;
    for (int j = k + threadIdx.x; j < M; j += 256)
      if (upd[j] > bv) { bv = upd[j]; bi = j; }
    double gv;
    int gi;
    wg_argmax(bv, bi, red, gv, gi);
    if (gi >= M) gi = k;  // no comparable norm (NaN): the columns in order
    if (nonzero == size && gv * gv < th_helper * (double)(K - k)) nonzero = k;
    if (t.tol > 0. && nonzero < size) break;                      // rank counts i < nonzero only
    if (t.tol > 0. && k > 0 && gv <= t.tol * maxpivot) break;    // every later |R_ii| is below the threshold
    if (gi != k) {
      double* ck = t.A + (long long)k * t.lda;
      double* cb = t.A + (long long)gi * t.lda;
      for (int i = threadIdx.x; i < K; i += 256) {
        double a = ck[i];
        ck[i] = cb[i];
        cb[i] = a;
      }
      __syncthreads();
      if (threadIdx.x == 0) {
        double a = upd[k]; upd[k] = upd[gi]; upd[gi] = a;
        a = dir[k]; dir[k] = dir[gi]; dir[gi] = a;
        int p = t.perm[k]; t.perm[k] = t.perm[gi]; t.perm[gi] = p;
      }
    }
    __syncthreads();
    double* col = t.A + k + (long long)k * t.lda;
    const int len = K - k;
    double tau;
    const double beta = make_reflector(col, len, red, tau);
    __syncthreads();
    if (threadIdx.x == 0) {
      col[0] = beta;
      sh_tau = tau;
      sh_maxpivot = fmax(maxpivot, fabs(beta));
    }
    __syncthreads();
    maxpivot = sh_maxpivot;
    apply_reflector(col, len, sh_tau, t.A + k, t.lda, k + 1, M);
    __syncthreads();
    for (int j = k + 1 + threadIdx.x; j < M; j += 256) {
      if (upd[j] != 0.) {
        double q = fabs(t.A[k + (long long)j * t.lda]) / upd[j];
        q = (1. + q) * (1. - q);
        q = q < 0. ? 0. : q;
        const double r = upd[j] / dir[j];
        if (q * r * r <= downdate_th) {
          const double* cj = t.A + (long long)j * t.lda;
          double s = 0.;
          for (int i = k + 1; i < K; i++) s += cj[i] * cj[i];
          dir[j] = upd[j] = sqrt(s);
        } else {
          upd[j] *= sqrt(q);
        }
      }
    }
    __syncthreads();
    done = k + 1;
  }
  if (threadIdx.x == 0) {
    int rank;
    if (t.tol > 0.) {
      const double th = maxpivot * t.tol;
      const int lim = min(nonzero, done);
      rank = 0;
      for (int i = 0; i < lim; i++) rank += !(fabs(t.A[i + (long long)i * t.lda]) <= th);  // NaN counts
    } else {
      rank = done;
    }
    if (t.maxrank > 0) rank = min(rank, t.maxrank);
    *t.rank_out = rank;
  }
}

// Blocked column-pivoted QR (LAPACK xLAQPS's delayed updates): the last up to
// nb reflectors V and the products F = (tau A^T v, corrected) stay in LDS and
// the trailing matrix A - V F^T is formed only every nb steps. A step then
// reads the trailing matrix once (one product A^T v) and writes one row of it,
// where applying each reflector reads it twice and writes it once: with the
// matrices of a level larger than the caches that traffic is what bounds it.
// The pivot column, the row of a step and the norms recomputed under the
// downdating rule get the pending updates explicitly, so pivots, norms and
// rank are those of the unblocked algorithm up to rounding. Measured: eight
// 256 x 256 blocks to full rank 7.7 -> 1.4 ms; the levels of the sphere operator
// at N = 65536 (256 to 2 blocks of 256 to 350 columns) 85.8 -> 23.1 ms; seven
// levels of rank 100 at N = 32768 39.1 -> 8.4 ms. A step takes 9 to 14 us, most
// of it the chain of its phases (reflector, product, row, argmax) and the
// latency of the one pass over the trailing matrix.
// One matrix of K x M, K <= 64 R, per workgroup of eight waves; LDS: V nb x 64 R,
// F nb x mp, four arrays of mp and the flagged columns (mp >= M).
template <int R>
__global__ void __launch_bounds__(512) k_cpqr_blocked(const CpqrTask* __restrict__ tasks, int nb, int mp) {
  constexpr int KP = 64 * R;
  constexpr int G = R <= 4 ? 8 : 4;   // columns a wave takes at a time
  constexpr bool AHEAD = R <= 6;      // the next ones' loads in flight (registers allow it up to R = 6)
  extern __shared__ double sm[];
  double* Vs = sm;
  double* Fs = Vs + nb * KP;
  double* upd = Fs + nb * mp;
  double* dir = upd + mp;
  double* rowk = dir + mp;
  double* diag = rowk + mp;
  double* aux = diag + mp;
  int* flagged = reinterpret_cast<int*>(aux + nb);
  __shared__ int nflag, nrank;
  __shared__ double sh_tau, sh_beta;
  const CpqrTask t = read_task(tasks);
  const int K = t.K, M = t.M, size = min(K, M);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  double* A = t.A;
  const long long lda = t.lda;
  int rowc[R];  // rows of the lane, clamped: V is zero past K
#pragma unroll
  for (int r = 0; r < R; r++) rowc[r] = min(lane + 64 * r, K - 1);
  for (int j = tid; j < M; j += 512) t.perm[j] = j;
  for (int c0 = wave * G; c0 < M; c0 += 8 * G) {
    double d[G], s[G / 4];
#pragma unroll
    for (int g = 0; g < G; g++) {
      const double* col = A + (long long)min(c0 + g, M - 1) * lda;
      d[g] = 0.;
#pragma unroll
      for (int r = 0; r < R; r++) {
        const double x = col[rowc[r]];
        if (lane + 64 * r < K) d[g] += x * x;
      }
    }
    wave_sums<G>(d, s);
#pragma unroll
    for (int g = 0; g < G; g++) {
      const double nrm = sqrt(sum_of<G>(s, g));
      if (lane == 0 && c0 + g < M) upd[c0 + g] = dir[c0 + g] = nrm;
    }
  }
  if (tid == 0) nflag = nrank = 0;
  __syncthreads();
  const double eps = DBL_EPSILON;
  const double downdate_th = sqrt(eps);
  double th_helper = 0.;
  int nonzero = size, done = 0, j = 0;
  double maxpivot = 0.;
  for (int k = 0; k < t.steps; k++) {
    // pivot: the first column of largest norm (every wave finds it)
    double bv = -1.;
    int bi = M;
    for (int c = k + lane; c < M; c += 64) {
      const double u = upd[c];
      if (u > bv) { bv = u; bi = c; }
    }
    const double gv = wave_max(bv);
    const unsigned long long at = __ballot(bv == gv);
    int p = k;
    if (__popcll(at) == 1) {
      p = __builtin_amdgcn_readlane(bi, __ffsll((long long)at) - 1);
    } else {
      int m = bv == gv ? bi : M;
      for (int o = 32; o > 0; o >>= 1) m = min(m, __shfl_xor(m, o, 64));
      p = __builtin_amdgcn_readfirstlane(m);
    }
    if (p >= M) p = k;  // no comparable norm (NaN): the columns in order
    if (k == 0) th_helper = (gv * eps) * (gv * eps) / (double)K;
    if (nonzero == size && gv * gv < th_helper * (double)(K - k)) nonzero = k;
    if (t.tol > 0. && nonzero < size) break;                      // rank counts i < nonzero only
    if (t.tol > 0. && k > 0 && gv <= t.tol * maxpivot) break;    // every later |R_ii| is below the threshold
    // wave 0: the pivot column with its pending updates, and its reflector;
    // wave 1: column k, which takes the pivot column's place; wave 2: the
    // entries of F, the norms and the permutation that go with it
    double x[R], above[R], tau = 0., beta = 0., sw = 0., sw2 = 0.;
    int pp = 0, pk = 0;
    if (wave == 0) {
#pragma unroll
      for (int r = 0; r < R; r++) above[r] = x[r] = lane + 64 * r < K ? A[rowc[r] + p * lda] : 0.;
      for (int l = 0; l < j; l++) {
        const double f = Fs[l * mp + p];
#pragma unroll
        for (int r = 0; r < R; r++)
          if (lane + 64 * r >= k) x[r] -= Vs[l * KP + lane + 64 * r] * f;
      }
      beta = wave_reflector<R>(x, k, lane, tau);
    } else if (wave == 1) {
#pragma unroll
      for (int r = 0; r < R; r++) x[r] = A[rowc[r] + k * lda];
    } else if (wave == 2) {
      if (lane < j) sw = Fs[lane * mp + k];
      if (lane == 0) {
        sw2 = upd[k];
        tau = dir[k];
        pk = t.perm[k];
        pp = t.perm[p];
      }
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int r = 0; r < R; r++) {
        const int row = lane + 64 * r;
        Vs[j * KP + row] = x[r];
        if (row <= k && row < K) A[row + k * lda] = row < k ? above[r] : beta;
      }
      if (lane == 0) {
        sh_tau = tau;
        sh_beta = beta;
        diag[k] = fabs(beta);
        nflag = 0;
      }
    } else if (p != k) {
      if (wave == 1) {
#pragma unroll
        for (int r = 0; r < R; r++)
          if (lane + 64 * r < K) A[rowc[r] + p * lda] = x[r];
      } else if (wave == 2) {
        if (lane < j) Fs[lane * mp + p] = sw;
        if (lane == 0) {
          upd[p] = sw2;
          dir[p] = tau;
          t.perm[k] = pp;
          t.perm[p] = pk;
        }
      }
    }
    __syncthreads();
    tau = sh_tau;
    maxpivot = fmax(maxpivot, fabs(sh_beta));
    // A^T v over the columns right of k (rows from k on), and V^T v
    double v[R];
#pragma unroll
    for (int r = 0; r < R; r++) v[r] = Vs[j * KP + lane + 64 * r];
    const int rk = k >> 6, lk = k & 63;
    double a[G][R], an[AHEAD ? G : 1][R];
    auto load = [&](auto& q, int c0) {
#pragma unroll
      for (int g = 0; g < G; g++) {
        const double* col = A + (long long)min(c0 + g, M - 1) * lda;
#pragma unroll
        for (int r = 0; r < R; r++) q[g][r] = r >= rk ? col[rowc[r]] : 0.;
      }
    };
    int c0 = k + 1 + wave * G;
    if (AHEAD && c0 < M) load(a, c0);
    for (; c0 < M; c0 += 8 * G) {
      if constexpr (!AHEAD) load(a, c0);
      else if (c0 + 8 * G < M) load(an, c0 + 8 * G);
      double d[G], s[G / 4];
#pragma unroll
      for (int g = 0; g < G; g++) {
        d[g] = 0.;
#pragma unroll
        for (int r = 0; r < R; r++) d[g] += v[r] * a[g][r];
      }
      wave_sums<G>(d, s);
#pragma unroll
      for (int r = 0; r < R; r++)
        if (r == rk && lane == lk)
#pragma unroll
          for (int g = 0; g < G; g++)
            if (c0 + g < M) rowk[c0 + g] = a[g][r];
      if ((lane & 15) == 0) {
#pragma unroll
        for (int h = 0; h < G / 4; h++) {
          const int c = c0 + (lane >> 4) * (G / 4) + h;
          if (c < M) Fs[j * mp + c] = s[h];
        }
      }
      if constexpr (AHEAD)
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
          for (int r = 0; r < R; r++) a[g][r] = an[g][r];
    }
    for (int l = wave; l < j; l += 8) {
      double s = 0.;
#pragma unroll
      for (int r = 0; r < R; r++) s += Vs[l * KP + lane + 64 * r] * v[r];
      s = wave_total(s);
      if (lane == 0) aux[l] = s;
    }
    __syncthreads();
    // F's new row, row k of R and the norms, one column per thread
    for (int c = k + 1 + tid; c < M; c += 512) {
      double f = Fs[j * mp + c], akc = rowk[c];
      for (int l = 0; l < j; l++) {
        const double fl = Fs[l * mp + c];
        f -= fl * aux[l];
        akc -= Vs[l * KP + k] * fl;
      }
      f *= tau;
      akc -= f;
      Fs[j * mp + c] = f;
      A[k + c * lda] = akc;
      const double u = upd[c];
      if (u != 0.) {
        double q = fabs(akc) / u;
        q = (1. + q) * (1. - q);
        q = q < 0. ? 0. : q;
        const double rr = u / dir[c];
        if (q * rr * rr <= downdate_th)
          flagged[atomicAdd(&nflag, 1)] = c;
        else
          upd[c] = u * sqrt(q);
      }
    }
    __syncthreads();
    const int nf = nflag;
    done = k + 1;
    if (nf > 0) {  // norms recomputed from the updated columns
      for (int q = wave; q < nf; q += 8) {
        const int c = __builtin_amdgcn_readfirstlane(flagged[q]);
        double y[R], s = 0.;
#pragma unroll
        for (int r = 0; r < R; r++) y[r] = A[rowc[r] + c * lda];
        for (int l = 0; l <= j; l++) {
          const double f = Fs[l * mp + c];
#pragma unroll
          for (int r = 0; r < R; r++) y[r] -= Vs[l * KP + lane + 64 * r] * f;
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
          const int row = lane + 64 * r;
          if (row > k && row < K) s += y[r] * y[r];
        }
        s = sqrt(wave_total(s));
        if (lane == 0) upd[c] = dir[c] = s;
      }
      __syncthreads();
    }
    if (++j == nb) {  // A -= V F^T below row k
      for (int c0 = k + 1 + wave * 4; c0 < M; c0 += 32) {
        double y[4][R];
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
          for (int r = 0; r < R; r++) y[g][r] = A[rowc[r] + (long long)min(c0 + g, M - 1) * lda];
        for (int l = 0; l < nb; l++) {
          double f[4];
#pragma unroll
          for (int g = 0; g < 4; g++) f[g] = Fs[l * mp + min(c0 + g, M - 1)];
#pragma unroll
          for (int r = 0; r < R; r++) {
            const double vl = Vs[l * KP + lane + 64 * r];
#pragma unroll
            for (int g = 0; g < 4; g++) y[g][r] -= vl * f[g];
          }
        }
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
          for (int r = 0; r < R; r++) {
            const int row = lane + 64 * r;
            if (c0 + g < M && row > k && row < K) A[row + (long long)(c0 + g) * lda] = y[g][r];
          }
      }
      j = 0;
      __syncthreads();
    }
  }
  __syncthreads();
  if (t.tol > 0.) {
    const double th = maxpivot * t.tol;
    const int lim = min(nonzero, done);
    int mine = 0;
    for (int i = tid; i < lim; i += 512) mine += !(diag[i] <= th);  // NaN counts, so that it shows
    if (mine) atomicAdd(&nrank, mine);
    __syncthreads();
  }
  if (tid == 0) {
    int rank = t.tol > 0. ? nrank : done;
    if (t.maxrank > 0) rank = min(rank, t.maxrank);
    *t.rank_out = rank;
  }
}

__global__ void __launch_bounds__(256) k_formq(const FormQTask* __restrict__ tasks) {
  const FormQTask t = read_task(tasks);
  const int M = t.M;
  for (long long e = threadIdx.x; e < (long long)M * M; e += 256) {
    const int i = (int)(e % M), j = (int)(e / M);
    t.Q[e] = (i == j) ? 1. : 0.;
    t.R[e] = (j < t.r && i <= j) ? t.P[i + (long long)j * t.ldp] : 0.;
  }
  __syncthreads();
  for (int k = t.r - 1; k >= 0; k--) {
    apply_reflector(t.P + k + (long long)k * t.ldp, M - k, t.tau[k], t.Q + k, M, k, M);
    __syncthreads();
  }
}

// The columns of Q = H_0 ... H_{r-1} are independent of each other: a wave
// forms G of them in its registers, reflector by reflector, and only the
// reflectors (which all waves of a box share through L2) are read. No barrier.
// 0.57 ms for seven levels of rank 100 at N = 32768, 37.8 ms with Q in global
// memory and a barrier per reflector.
template <int R>
__global__ void __launch_bounds__(256) k_formq_reg(const FormQTask* __restrict__ tasks) {
  constexpr int G = R <= 8 ? 8 : 4;
  const FormQTask t = read_task(tasks);
  const int M = t.M;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c0 = (blockIdx.y * 4 + wave) * G;
  if (c0 >= M) return;
  double q[G][R], vn[R];
#pragma unroll
  for (int g = 0; g < G; g++)
#pragma unroll
    for (int j = 0; j < R; j++) q[g][j] = (lane + 64 * j == c0 + g) ? 1. : 0.;
  auto load = [&](int k) {
#pragma unroll
    for (int j = 0; j < R; j++) {
      const int row = lane + 64 * j;
      vn[j] = (row > k && row < M) ? t.P[row + (long long)k * t.ldp] : (row == k ? 1. : 0.);
    }
  };
  // reflector k leaves the columns left of k as they are (unit vectors e_c, c < k)
  int k = min(t.r, c0 + G) - 1;
  if (k >= 0) load(k);
  for (; k >= 0; k--) {
    double v[R];
#pragma unroll
    for (int j = 0; j < R; j++) v[j] = vn[j];
    if (k > 0) load(k - 1);
    const double tau = t.tau[k];
    double d[G], s[G / 4];
#pragma unroll
    for (int g = 0; g < G; g++) {
      d[g] = 0.;
#pragma unroll
      for (int j = 0; j < R; j++) d[g] += v[j] * q[g][j];
    }
    wave_sums<G>(d, s);
#pragma unroll
    for (int g = 0; g < G; g++) {
      const double w = sum_of<G>(s, g) * tau;
#pragma unroll
      for (int j = 0; j < R; j++) q[g][j] -= w * v[j];
    }
  }
#pragma unroll
  for (int g = 0; g < G; g++) {
    const int c = c0 + g;
    if (c < M)
#pragma unroll
      for (int j = 0; j < R; j++) {
        const int row = lane + 64 * j;
        if (row < M) {
          t.Q[row + (long long)c * M] = q[g][j];
          t.R[row + (long long)c * M] = (c < t.r && row <= c) ? t.P[row + (long long)c * t.ldp] : 0.;
        }
      }
  }
}

__global__ void __launch_bounds__(256) k_trsolve(const TrTask* __restrict__ tasks) {
  const TrTask t = read_task(tasks);
  const int r = t.r;
  for (int c = threadIdx.x; c < t.n; c += 256) {
    double* x = t.X + (long long)c * r;
    const double* b = t.R0 + (long long)(r + c) * t.ldr;
    for (int i = r - 1; i >= 0; i--) {
      double s = b[i];
      for (int j = i + 1; j < r; j++) s -= t.R0[i + (long long)j * t.ldr] * x[j];
      x[i] = s / t.R0[i + (long long)i * t.ldr];
    }
  }
}

// Back substitution by columns of R11, four right-hand sides per wave in its
// registers: step i divides entry i and subtracts column i of R11, whose load
// does not depend on the steps before it and is issued one step ahead (0.36 ms
// for seven levels at rank 100, about 5 ms with one right-hand side per thread).
template <int R>
__global__ void __launch_bounds__(256) k_trsolve_reg(const TrTask* __restrict__ tasks) {
  constexpr int G = 4;
  const TrTask t = read_task(tasks);
  const int r = t.r;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c0 = (blockIdx.y * 4 + wave) * G;
  if (c0 >= t.n) return;
  double x[G][R], cn[R];
#pragma unroll
  for (int g = 0; g < G; g++)
#pragma unroll
    for (int j = 0; j < R; j++) {
      const int row = lane + 64 * j;
      x[g][j] = (row < r && c0 + g < t.n) ? t.R0[row + (long long)(r + c0 + g) * t.ldr] : 0.;
    }
  auto load = [&](int i) {
#pragma unroll
    for (int j = 0; j < R; j++) {
      const int row = lane + 64 * j;
      cn[j] = row <= i ? t.R0[row + (long long)i * t.ldr] : 0.;
    }
  };
  load(r - 1);
#pragma unroll
  for (int jj = R - 1; jj >= 0; jj--) {
    for (int i = min(r, 64 * (jj + 1)) - 1; i >= 64 * jj; i--) {
      double c[R];
#pragma unroll
      for (int j = 0; j <= jj; j++) c[j] = cn[j];
      if (i > 0) load(i - 1);
      const int li = i & 63;
      const double d = lane_get(c[jj], li);
#pragma unroll
      for (int g = 0; g < G; g++) {
        const double xi = lane_get(x[g][jj], li) / d;
        const double kept = lane == li ? xi : (lane < li ? x[g][jj] - c[jj] * xi : x[g][jj]);
        x[g][jj] = kept;
#pragma unroll
        for (int j = 0; j < jj; j++) x[g][j] -= c[j] * xi;
      }
    }
  }
#pragma unroll
  for (int g = 0; g < G; g++)
    if (c0 + g < t.n)
#pragma unroll
      for (int j = 0; j < R; j++) {
        const int row = lane + 64 * j;
        if (row < r) t.X[row + (long long)(c0 + g) * r] = x[g][j];
      }
}

// One launch of kern over the tasks, grid (tasks, ydim), and a wait: the
// descriptor array is freed on return.
template <class Task, class Kern, class... Args>
void launch_tasks(const std::vector<Task>& tasks, Kern kern, int threads, unsigned ydim, size_t lds, hipStream_t s,
                  Args... args) {
  if (tasks.empty()) return;
  MXG_REQUIRE(tasks.size() < (1u << 31), "too many tasks");
  DevBuf<Task> dt;
  dt.upload(tasks, s);
  hipLaunchKernelGGL(kern, dim3((unsigned)tasks.size(), ydim), dim3(threads), lds, s, dt.p, args...);
  MXG_HIP(hipGetLastError());
  MXG_HIP(hipStreamSynchronize(s));
}

// Panel width and LDS bytes of the blocked pivoted QR: 16 reflectors where V
// and F fit beside the norms, else 8.
constexpr size_t CPQR_LDS = 156 * 1024;
inline size_t cpqr_lds(int R, int mp, int nb) {
  return sizeof(double) * ((size_t)nb * (64 * R + mp + 1) + 4 * (size_t)mp) + sizeof(int) * (size_t)mp;
}

template <int R>
void launch_cpqr(const std::vector<CpqrTask>& tasks, int nb, int mp, hipStream_t s) {
  const size_t lds = cpqr_lds(R, mp, nb);
  MXG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_cpqr_blocked<R>), hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)CPQR_LDS));
  launch_tasks(tasks, k_cpqr_blocked<R>, 512, 1, lds, s, nb, mp);
}

// Columns per wave of the register QR, 0 where it does not apply: R x C values
// must fit a lane's registers beside the reflector (80 of them and two waves
// per SIMD: at most 256 registers a lane).
inline int qr_cols(int R, int n) {
  for (int c : {4, 8, 13, 16})
    if (n <= 8 * c && R * c <= 80) return c;
  return 0;
}

}  // namespace

void qr_batched(const std::vector<QrTask>& tasks, hipStream_t s) {
  std::map<std::pair<int, int>, std::vector<QrTask>> by;  // (0, 0): the general kernel
  for (const QrTask& t : tasks) {
    if (t.m <= 0 || t.n <= 0) continue;
    const int R = row_steps(t.m) > 8 ? 0 : row_steps(t.m), C = R ? qr_cols(R, t.n) : 0;
    by[C ? std::make_pair(R, C) : std::make_pair(0, 0)].push_back(t);
  }
  for (const auto& kv : by) {
    const int R = kv.first.first, C = kv.first.second;
#define MXG_QR(RR, CC) if (R == RR && C == CC) { launch_tasks(kv.second, k_qr_reg<RR, CC>, 512, 1, 0, s); continue; }
#define MXG_QR_ROWS(RR) MXG_QR(RR, 4) MXG_QR(RR, 8) MXG_QR(RR, 13) MXG_QR(RR, 16)
    MXG_QR_ROWS(1) MXG_QR_ROWS(2) MXG_QR_ROWS(3) MXG_QR_ROWS(4) MXG_QR_ROWS(5)
    MXG_QR(6, 4) MXG_QR(6, 8) MXG_QR(6, 13) MXG_QR(8, 4) MXG_QR(8, 8)
#undef MXG_QR_ROWS
#undef MXG_QR
    MXG_REQUIRE(R == 0, "no QR kernel for this size");
    launch_tasks(kv.second, k_qr, 256, 1, 0, s);
  }
}

void formq_batched(const std::vector<FormQTask>& tasks, hipStream_t s) {
  std::map<int, std::vector<FormQTask>> by;
  std::map<int, int> mx;
  for (const FormQTask& t : tasks) {
    if (t.M <= 0) continue;
    const int R = row_steps(t.M);
    by[R].push_back(t);
    mx[R] = std::max(mx[R], t.M);
  }
  for (const auto& kv : by) {
    const unsigned y = ceil_div(mx[kv.first], kv.first <= 8 ? 32 : 16);
    switch (kv.first) {
#define MXG_CASE(RR) case RR: launch_tasks(kv.second, k_formq_reg<RR>, 256, y, 0, s); break;
      MXG_FOR_ROW_STEPS(MXG_CASE)
#undef MXG_CASE
      default: launch_tasks(kv.second, k_formq, 256, 1, 0, s);
    }
  }
}

void cpqr_batched(const std::vector<CpqrTask>& tasks, hipStream_t s) {
  std::map<std::pair<int, int>, std::vector<CpqrTask>> by;  // (rows a lane holds, panel width); (0, 0): the general kernel
  std::map<std::pair<int, int>, int> mx;
  for (const CpqrTask& t : tasks) {
    MXG_REQUIRE(t.steps <= std::min(t.K, t.M), "cpqr steps exceed min(K, M)");
    std::pair<int, int> key{0, 0};
    const int R = row_steps(t.K);
    if (R)
      for (int nb : {16, 8})
        if (cpqr_lds(R, t.M, nb) <= CPQR_LDS) {
          key = {R, nb};
          break;
        }
    by[key].push_back(t);
    mx[key] = std::max(mx[key], t.M);
  }
  for (const auto& kv : by) {
    const int nb = kv.first.second, mp = mx[kv.first];
    switch (kv.first.first) {
#define MXG_CASE(RR) case RR: launch_cpqr<RR>(kv.second, nb, mp, s); break;
      MXG_FOR_ROW_STEPS(MXG_CASE)
#undef MXG_CASE
      default: launch_tasks(kv.second, k_cpqr, 256, 1, 0, s);
    }
  }
}

void trsolve_batched(const std::vector<TrTask>& tasks, hipStream_t s) {
  std::map<int, std::vector<TrTask>> by;
  std::map<int, int> mx;
  for (const TrTask& t : tasks) {
    if (t.r <= 0 || t.n <= 0) continue;
    const int R = row_steps(t.r);
    by[R].push_back(t);
    mx[R] = std::max(mx[R], t.n);
  }
  for (const auto& kv : by) {
    const unsigned y = ceil_div(mx[kv.first], 16);
    switch (kv.first) {
#define MXG_CASE(RR) case RR: launch_tasks(kv.second, k_trsolve_reg<RR>, 256, y, 0, s); break;
      MXG_FOR_ROW_STEPS(MXG_CASE)
#undef MXG_CASE
      default: launch_tasks(kv.second, k_trsolve, 256, 1, 0, s);
    }
  }
}

}  // namespace mxg
