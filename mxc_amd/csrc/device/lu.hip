// Inverses of the rr blocks of the ULV factorization (h2matrix.cpp:435-441,
// Eigen PartialPivLU followed by products with its inverse), one matrix per
// workgroup, variable sizes up to 1024 rows.
//
// Gauss-Jordan elimination in place with partial pivoting, 16 columns at a
// time. With the panel's pivot rows R and the other rows O, a panel step turns
//   columns J: rows R -> P_R^{-1}, rows O -> -P_O P_R^{-1}   (together W, n x 16)
//   other columns: rows R -> W_R B, rows O -> A_O + W_O B    (B = A[R, :], 16 x n)
// so that after the last panel the matrix holds the inverse with its rows and
// columns permuted. A panel is eliminated by the whole workgroup with one row
// per thread in registers: each wave offers its largest candidate and that
// row's values through LDS (double-buffered), so a column costs one barrier.
// The update of the other columns is a product on the FP64 matrix cores, one
// strip of 16 columns per wave. The matrix stays in L2: it is read and written
// once per panel, and only W and the candidates are held in LDS. A panel is
// bound by its 16 dependent pivots (about 4 us), its update by the FP64 matrix
// cores; 115 registers a lane let two blocks of 512 threads share a CU, so
// that one's panels overlap the other's updates (512 blocks of 192 rows: 1.25
// -> 0.99 ms). Column-at-a-time elimination, with two barriers and a rank-1
// update per column, took 26.6 ms where this takes 1.9 (the seven levels of a
// factorization at N = 20000, rank 100: 64 blocks of 213 rows, then 100), and
// 6.1 ms where this takes 1.6 (N = 131072, rank 64, FP32).
//
// FP32 factorizations use it too, with FP64 arithmetic between FP32 input and
// output: the inverse formed in FP32 was what limited their accuracy (a
// fixed-rank preconditioner at N = 4096, rank 100, five seeds: substitutions
// 7e-5 to 1e-3 from those of the FP64 factorization, 4e-6 to 1e-5 with this).
#include <cfloat>
#include <map>

#include "internal.hpp"
#include "wave.hpp"

namespace mxg {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int GJ_NB = 16;

template <class T, int NT>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) k_gj_inverse(const LuTask<T>* __restrict__ tasks, int ldw) {
  constexpr int NW = NT / 64;
  extern __shared__ double Ws[];  // W[row][k] at Ws[k * ldw + row]
  __shared__ double cand[2][NW];
  __shared__ int candrow[2][NW];
  __shared__ __align__(16) double candval[2][NW][GJ_NB];
  __shared__ int rowof[NT], stepof[NT];  // pivot row of a step, step of a pivot row (-1: none yet)
  __shared__ double lg[NW];
  LuTask<T> task = in_constant(tasks)[blockIdx.x];
  task.A = in_global(task.A);
  task.inv = in_global(task.inv);
  task.work = in_global(task.work);
  task.info = in_global(task.info);
  const int n = task.n;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  double* S = task.work;
  for (int e = tid; e < n * n; e += NT) {
    const int i = e % n, j = e / n;
    S[e] = (double)task.A[i + (long long)j * task.lda];
  }
  stepof[tid] = -1;
  __syncthreads();
  bool open = tid < n;  // this thread's row has not been a pivot row
  double logdet = 0.;   // of the pivots of this thread's row
  int singular = 0;
  for (int j0 = 0; j0 < n; j0 += GJ_NB) {
    double a[GJ_NB];
#pragma unroll
    for (int c = 0; c < GJ_NB; c++) a[c] = (tid < n && j0 + c < n) ? S[tid + (j0 + c) * n] : 0.;
#pragma unroll
    for (int q = 0; q < GJ_NB; q++) {
      if (j0 + q >= n) break;
      const int b = q & 1;
      const double mag = fabs(a[q]);
      const double v = open ? (mag >= 0. ? mag : 0.) : -1.;  // NaN counts as zero
      const double m = wave_max(v);
      const int src = __ffsll((long long)__ballot(v == m)) - 1;
      if (lane == src) {
        cand[b][wave] = m;
        candrow[b][wave] = tid;
#pragma unroll
        for (int c = 0; c < GJ_NB; c++) candval[b][wave][c] = a[c];
      }
      __syncthreads();
      // the largest candidate, the lowest row among equals
      double best = cand[b][0];
      int w = 0;
#pragma unroll
      for (int u = 1; u < NW; u++) {
        const double o = cand[b][u];
        if (o > best) { best = o; w = u; }
      }
      const int p = candrow[b][w];
      double s[GJ_NB];
#pragma unroll
      for (int c = 0; c < GJ_NB; c++) s[c] = candval[b][w][c];
      const double d = s[q], inv = 1. / d;
      if (d == 0.) singular = 1;
      const double f = a[q];
#pragma unroll
      for (int c = 0; c < GJ_NB; c++) {
        s[c] = c == q ? inv : s[c] * inv;
        a[c] = tid == p ? s[c] : (c == q ? -f * inv : a[c] - f * s[c]);
      }
      if (tid == p) {
        open = false;
        rowof[j0 + q] = p;
        stepof[p] = j0 + q;
        logdet = log(fabs(d));
      }
    }
    if (tid < ldw)
#pragma unroll
      for (int c = 0; c < GJ_NB; c++) Ws[c * ldw + tid] = a[c];
    if (tid < n)
#pragma unroll
      for (int c = 0; c < GJ_NB; c++)
        if (j0 + c < n) S[tid + (j0 + c) * n] = a[c];
    __syncthreads();
    // the other columns: transposed 16 x 16 tiles (matrix-core rows are the
    // columns of S), so that the 16 lanes of a row of lanes touch 16
    // consecutive rows of one column
    for (int c0 = 16 * wave; c0 < n; c0 += 16 * NW) {
      if (c0 == j0) continue;
      double bf[4];  // B[k = lk + 4 t][column c0 + lr]
      const int cb = min(c0 + lr, n - 1);
#pragma unroll
      for (int t = 0; t < 4; t++) bf[t] = j0 + lk + 4 * t < n ? S[rowof[j0 + lk + 4 * t] + cb * n] : 0.;
      for (int r0 = 0; r0 < n; r0 += 64) {
        d4 acc[4];
        int st[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int row = r0 + 16 * u + lr;
          st[u] = row < n ? stepof[row] : -1;
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const int col = c0 + lk + 4 * q;
            acc[u][q] = (row < n && col < n) ? S[row + col * n] : 0.;
          }
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
          if (r0 + 16 * u >= n) break;
          const int row = r0 + 16 * u + lr;
          if (st[u] >= j0) acc[u] = d4{0., 0., 0., 0.};  // a pivot row of this panel
#pragma unroll
          for (int t = 0; t < 4; t++)
            acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(bf[t], Ws[(lk + 4 * t) * ldw + r0 + 16 * u + lr], acc[u], 0, 0, 0);
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const int col = c0 + lk + 4 * q;
            if (row < n && col < n) S[row + col * n] = acc[u][q];
          }
        }
      }
    }
    __syncthreads();
  }
  // entry (i, l) of S is entry (step of row i, pivot row of step l) of the inverse
  for (int e = tid; e < n * n; e += NT) {
    const int i = e % n, l = e / n;
    task.inv[stepof[i] + (long long)rowof[l] * n] = (T)S[e];
  }
  logdet = wave_total(logdet);
  if (lane == 0) lg[wave] = logdet;
  __syncthreads();
  if (tid == 0) {
    double sum = 0.;
    for (int w = 0; w < NW; w++) sum += lg[w];
    *task.info = (singular || sum <= log(DBL_MIN)) ? 1 : 0;
  }
}

template <class T, int NT>
void launch_gj(const std::vector<LuTask<T>>& tasks, hipStream_t s, Stage* st) {
  if (tasks.empty()) return;
  MXG_REQUIRE(tasks.size() < (1u << 31), "too many tasks");
  int nmax = 0;
  for (const LuTask<T>& t : tasks) nmax = std::max(nmax, t.n);
  // row stride 16 mod 32: two of a matrix-core operand's four k share no LDS bank
  const int ldw = std::min((nmax + 31) / 32 * 32 + 16, NT >= 1024 ? 1040 : NT + 16);
  const size_t lds = sizeof(double) * GJ_NB * (size_t)ldw;
  MXG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_gj_inverse<T, NT>), hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)(sizeof(double) * GJ_NB * 1040)));
  DevBuf<LuTask<T>> dt;
  const LuTask<T>* pt;
  if (st) {
    pt = st->put(tasks);
  } else {
    dt.upload(tasks, s);
    pt = dt.p;
  }
  const unsigned n = (unsigned)tasks.size();
  auto launch = [=] {
    hipLaunchKernelGGL((k_gj_inverse<T, NT>), dim3(n), dim3(NT), lds, s, pt, ldw);
    MXG_HIP(hipGetLastError());
  };
  if (st) {
    st->later(launch);
  } else {
    launch();
    MXG_HIP(hipStreamSynchronize(s));
  }
}

}  // namespace

template <class T>
void lu_inverse_batched(const std::vector<LuTask<T>>& tasks, hipStream_t s, Stage* st) {
  std::vector<LuTask<T>> small, medium, large;
  for (const LuTask<T>& t : tasks) {
    MXG_REQUIRE(t.n >= 0 && t.n <= 1024, "LU block larger than 1024");
    if (t.n == 0) continue;
    (t.n <= 64 ? small : t.n <= 512 ? medium : large).push_back(t);
  }
  launch_gj<T, 256>(small, s, st);
  launch_gj<T, 512>(medium, s, st);
  launch_gj<T, 1024>(large, s, st);
}

template void lu_inverse_batched<double>(const std::vector<LuTask<double>>&, hipStream_t, Stage*);
template void lu_inverse_batched<float>(const std::vector<LuTask<float>>&, hipStream_t, Stage*);

}  // namespace mxg
