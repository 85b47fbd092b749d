// Row reduction of the far-field block by a Rademacher sketch.
//
// For a box with M columns (its bodies or skeleton) and nf > M far rows, the
// shared-basis construction needs an M x M matrix with the row space of the
// far block G(t, j) = K(|far_t - col_j|). The reference takes the R factor of
// a Householder QR of G (h2matrix.cpp:78-79); here it is the sketch
// Y = Omega G with Omega(i, t) = +-1, which has the same column relations in
// exact arithmetic up to the subspace embedding (Halko, Martinsson, Tropp
// 2011) and costs one streaming pass: G is never stored.
//
// The product runs on the 8-bit integer matrix cores, exactly. Omega is +-1;
// an entry of G becomes a fixed-point number of 60 bits below a bound of the
// workgroup's entries, cut into eight signed bytes, and
// v_mfma_i32_16x16x64_i8 sums each byte's products in 32 bits (at most 8192
// rows of magnitude 128). The eight sums of an entry of Y are put together in
// 64-bit integers and rounded to FP64 once. The error is then that of the
// entries' own rounding to 2^-54 of the largest entry or better, where a sum
// in FP64 rounds at every step. The FP64 matrix cores do a 64th of the 8-bit
// rate, so that with eight bytes an entry the product costs an eighth.
//
// The bound: kernels decrease with the distance (for a negative alpha the
// largest distance counts too), so K at the smallest distance between the
// tile's columns and the slice's rows bounds all entries. The distance of the
// rows to the columns' bounding box gives it for well separated boxes; where
// that would waste more than 6 of the 60 bits (boxes that touch) the smallest
// distance is found exactly, at about a sixth of the evaluation's cost.
//
// Work decomposition: one 512-thread workgroup owns a tile of Y, all its rows
// up to 512 and 16 to 64 columns, and a contiguous slice of far rows; slices
// of one box are written as separate partial tiles and summed in a fixed
// order. Eight 32-bit accumulators per 16 x 16 tile limit a wave to four tiles
// (six for boxes of 257 to 384 columns). Per step of 64 (or 128) rows every
// thread evaluates 4 or 8 entries of one column and writes their bytes to LDS
// as the matrix cores read them, 16 rows of one byte and column side by side;
// the buffers alternate, so a step has one barrier. The signs come as bytes from
// a table shared by all boxes and filled once per call, or per window of a long
// list's rows: making the bytes of a wave's rows from sign bits in every step took a
// quarter of the vector instructions.
//
// Measured on the operator of the unit sphere at N = 65536 (eps 1e-12, boxes of
// 256 to 350 columns, 3.7e12 flops): 95.6 ms on the FP64 matrix cores, 28.9 ms
// (128 TFLOP/s of the FP64 product) now; the error of the operator against the
// dense product is the same (2.0e-13; four digits agree on seven problems). A
// step is bound by the eight bytes' reads from LDS and by the evaluation (52
// vector instructions an entry), which overlap only in part at two waves per
// SIMD. Tried: half of the waves evaluating while the other half multiplies
// (38.9 ms, the accumulators spill), twice the rows per wave (33.5), the entries'
// stages side by side (31.1), sign bits expanded in registers (33.0).
#include <map>

#include "internal.hpp"
#include "keval.hpp"
#include "wave.hpp"

namespace mxg {
namespace {

typedef int i4 __attribute__((ext_vector_type(4)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));

__device__ inline unsigned long long sketch_word(unsigned long long t, unsigned long long b) {
  unsigned long long z = t * 0x9E3779B97F4A7C15ull + b * 0xD1B54A32D192ED03ull + 0x632BE59BD9B4E019ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// Omega as signed bytes in the order the matrix cores take it: 16 rows (group
// g) x 64 far rows (block u) are 1024 contiguous bytes, lane 16 k + r holding
// rows r and far rows 64 u + 16 k .. + 15; the table holds nu blocks from block u0
// on. One thread per 16 bytes.
__global__ void __launch_bounds__(256) k_sketch_signs(u4* __restrict__ signs, int nu, int u0) {
  const long long e = (long long)blockIdx.x * 256 + threadIdx.x;  // u, then lane
  if (e >= 64ll * nu) return;
  const int g = blockIdx.y, lane = (int)(e & 63), row = 16 * g + (lane & 15);
  const long long t0 = (u0 + (e >> 6)) * 64 + 16 * (lane >> 4);
  u4 v;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    v[q] = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const unsigned neg = (unsigned)(sketch_word((unsigned long long)(t0 + 4 * q + i), (unsigned long long)(row >> 6)) >> (row & 63)) & 1u;
      v[q] |= (neg ? 0xFFu : 1u) << (8 * i);
    }
  }
  signs[64ll * nu * g + e] = v;
}

// Adding MAGIC rounds a double below 2^31 in magnitude to an integer, whose bits
// plus DIGITS are the sum's lower word; subtracting it again gives the integer.
// With DIGITS added (and taken out of each byte by an exclusive or) the bytes of
// the word are the integer's signed base-256 digits.
constexpr unsigned DIGITS = 0x80808080u;
constexpr double MAGIC = 6755399441055744.0 + 2155905152.0;  // 1.5 2^52 + DIGITS

// 4 x 4 bytes transposed: out[s] = byte s of a, b, c, d.
__device__ inline void bytes_of(unsigned a, unsigned b, unsigned c, unsigned d, unsigned (&out)[4]) {
  const unsigned ab0 = __builtin_amdgcn_perm(b, a, 0x05010400u), ab1 = __builtin_amdgcn_perm(b, a, 0x07030602u);
  const unsigned cd0 = __builtin_amdgcn_perm(d, c, 0x05010400u), cd1 = __builtin_amdgcn_perm(d, c, 0x07030602u);
  out[0] = __builtin_amdgcn_perm(cd0, ab0, 0x05040100u);
  out[1] = __builtin_amdgcn_perm(cd0, ab0, 0x07060302u);
  out[2] = __builtin_amdgcn_perm(cd1, ab1, 0x05040100u);
  out[3] = __builtin_amdgcn_perm(cd1, ab1, 0x07060302u);
}

// Eight waves, WR of them along the rows of Y: a wave owns RW x CT tiles of
// 16 x 16; KT far rows per step.
template <int KID, int WR, int RW, int CT, int KT>
__global__ void __launch_bounds__(512) k_sketch(const SketchTask* __restrict__ tasks, const double* __restrict__ bodies,
                                                EvalArgs ke, const u4* __restrict__ signs, int nu, int u0) {
  constexpr int WC = 8 / WR, TC = 16 * CT * WC;
  constexpr int E = KT * TC / 512;  // entries a thread evaluates per step: consecutive rows of one column
  constexpr int SUB = 16 / E;       // threads sharing 16 rows of a column
  constexpr int TG = KT / 16, NX = 3 * KT;
  static_assert((E == 4 || E == 8) && NX <= 512 && TG * TC * SUB == 512, "step shape");
  __shared__ __align__(16) unsigned char Gs[2][8][TG][TC][16];  // byte s of rows 16 g .. 16 g + 15 of a column
  __shared__ double Xr[2][KT][3];
  __shared__ double wmax[6][8];  // per wave
  __shared__ int widx[8];
  __shared__ unsigned char bad[TC];  // columns with entries that are not finite
  SketchTask tk = in_constant(tasks)[blockIdx.x];
  tk.rows = in_global(tk.rows);
  tk.cols = in_global(tk.cols);
  tk.out = in_global(tk.out);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  const double inf = __builtin_inf();

  // this thread's column (clamped: columns past M are not stored)
  const int tg = wave % TG, col = (wave / TG) * (64 / SUB) + lane / SUB, sub = lane % SUB;
  const long long cb = tk.cols[min(tk.j0 + col, tk.M - 1)];
  const double x0 = bodies[3 * cb], x1 = bodies[3 * cb + 1], x2 = bodies[3 * cb + 2];

  // ---- bound of the entries ----
  int shift;         // entries are K 2^shift, below 2^60
  bool odd = false;  // some distances are not for kernel_scaled: zero (the diagonal value), or
                     // beyond ke.far2, where entries are zero if they are finite
  bool flagged = false;  // bad is in use
  {
    // largest over the workgroup of N values, in every thread
    auto wg_max = [&](auto& v) {
      constexpr int N = sizeof(v) / sizeof(double);
#pragma unroll
      for (int d = 0; d < N; d++) v[d] = wave_max(v[d]);
      __syncthreads();
      if (lane == 0)
#pragma unroll
        for (int d = 0; d < N; d++) wmax[d][wave] = v[d];
      __syncthreads();
#pragma unroll
      for (int d = 0; d < N; d++) {
        v[d] = wmax[d][0];
#pragma unroll
        for (int w = 1; w < 8; w++) v[d] = fmax(v[d], wmax[d][w]);
      }
    };
    // the row nearest to the bounding box of the tile's columns, and how far any
    // row can be from a column
    bool nan = !(x0 == x0 && x1 == x1 && x2 == x2);
    double hull[6] = {x0, x1, x2, -x0, -x1, -x2};
    wg_max(hull);
    double best = inf, most = 0.;
    int at = tk.t0;
#pragma unroll 4
    for (int t = tk.t0 + tid; t < tk.t0 + SKETCH_ROWS; t += 512) {
      const int tc = min(t, tk.t1 - 1);
      const double* r = bodies + 3 * (long long)tk.rows[tc];
      double d2 = 0., far2 = 0.;
#pragma unroll
      for (int d = 0; d < 3; d++) {
        const double x = r[d], below = -hull[3 + d] - x, above = x - hull[d];
        const double g = fmax(fmax(below, above), 0.), f = fmin(below, above);
        nan = nan || !(x == x);
        d2 += g * g;
        far2 += f * f;
      }
      if (d2 < best) { best = d2; at = tc; }
      most = fmax(most, far2);
    }
    const double wbest = -wave_max(-best);
    const int src = __ffsll((long long)__ballot(best == wbest)) - 1;
    if (lane == src) widx[wave] = at;
    double lo[2] = {-wbest, most};
    wg_max(lo);
#pragma unroll
    for (int w = 0; w < 8; w++)
      if (wmax[0][w] == lo[0]) at = widx[w];
    const double lo2 = -lo[0];
    nan = __syncthreads_or(nan);
    // a distance that occurs: that row's smallest to the columns
    const double* r = bodies + 3 * (long long)tk.rows[at];
    const double e0 = r[0] - x0, e1 = r[1] - x1, e2 = r[2] - x2;
    double has[1] = {-(e0 * e0 + e1 * e1 + e2 * e2)};
    wg_max(has);
    const bool falls = KID == MXG_KERNEL_LAPLACE || ke.ch <= 0., plain = lo2 > 0. && lo[1] <= 0.5 * ke.far2;
    double bound = plain ? kernel_any<KID>(lo2, ke) : inf;
    if (!falls || !plain || has[0] == 0. || !(bound <= 64. * kernel_any<KID>(-has[0], ke))) {
      // the extreme distances over all pairs, the rows staged 512 at a time; a
      // coinciding pair has the diagonal value
      double* st = reinterpret_cast<double*>(&Gs[0][0][0][0][0]);
      double ext[3] = {-inf, 0., 0.};  // -smallest nonzero, largest, whether some are zero
      for (int tc = tk.t0; tc < tk.t1; tc += 512) {
        __syncthreads();
        if (tc + tid < tk.t1) {
          const double* q = bodies + 3 * (long long)tk.rows[tc + tid];
#pragma unroll
          for (int d = 0; d < 3; d++) st[3 * tid + d] = q[d];
        }
        __syncthreads();
        const int cnt = min(512, tk.t1 - tc);
        for (int t = tg * SUB + sub; t < cnt; t += TG * SUB) {
          const double dx = st[3 * t] - x0, dy = st[3 * t + 1] - x1, dz = st[3 * t + 2] - x2;
          const double d2 = dx * dx + dy * dy + dz * dz;
          ext[0] = fmax(ext[0], d2 != 0. ? -d2 : -inf);
          ext[1] = fmax(ext[1], d2);
          if (d2 == 0.) ext[2] = 1.;
        }
      }
      wg_max(ext);
      bound = ext[2] > 0. ? fabs(ke.diag) : 0.;
      const double nearest = ext[0] > -inf ? kernel_any<KID>(-ext[0], ke) : 0., farthest = ext[1] > 0. ? kernel_any<KID>(ext[1], ke) : 0.;
      // not a number, or infinite: at least one of the three is
      flagged = nan || !(bound < inf && nearest < inf && farthest < inf);
      bound = fmax(bound, fmax(nearest, farthest));
      odd = ext[2] > 0. || !(ext[1] <= ke.far2);
      __syncthreads();  // the staged rows have been read
    }
    flagged = flagged || nan;
    if (flagged) {
      // the columns of such entries will be NaN, as their sums are; the others' bound
      if (tid < TC) bad[tid] = 0;
      __syncthreads();
      double big[1] = {0.};
      for (int t = tk.t0 + tg * SUB + sub; t < tk.t1; t += TG * SUB) {
        const double* q = bodies + 3 * (long long)tk.rows[t];
        const double dx = q[0] - x0, dy = q[1] - x1, dz = q[2] - x2;
        const double v = fabs(kernel_any<KID>(dx * dx + dy * dy + dz * dz, ke));
        if (v < inf) big[0] = fmax(big[0], v);
        else bad[col] = 1;
      }
      wg_max(big);
      bound = big[0];
      odd = true;
    }
    shift = __builtin_amdgcn_readfirstlane(bound > 0. ? 59 - ilogb(bound) : 0);
  }

  // ---- Y = Omega G ----
  // far rows' coordinates, two steps ahead of the product (their indices three)
  const int xr = tid / 3, xc = tid - 3 * (tid / 3);
  auto row_index = [&](int t) { return (tid < NX && t < tk.t1) ? tk.rows[t] : -1; };
  auto row_coord = [&](int idx) { return idx >= 0 ? bodies[3 * (long long)idx + xc] : 0.; };
  const int wr = wave % WR, wc = wave / WR;
  const int g0 = (tk.i0 >> 4) + wr * RW;  // first row group (16 rows) of the wave
  const u4* sg = signs + 64ll * ((long long)nu * g0 - u0) + lane;
  constexpr bool AHEAD = RW * KT <= 128;  // signs loaded one step ahead, where registers allow it
  i4 om[AHEAD ? RW : 1];
  auto load_signs = [&](int i, int tb) { return *reinterpret_cast<const i4*>(sg + 64ll * (nu * i + (tb >> 6))); };
  auto evaluate = [&](int b, double (&v)[E]) {
#pragma unroll
    for (int e = 0; e < E; e++) {
      const int tt = 16 * tg + sub * E + e;
      const double dx = Xr[b][tt][0] - x0, dy = Xr[b][tt][1] - x1, dz = Xr[b][tt][2] - x2;
      v[e] = kernel_scaled<KID>(dx * dx + dy * dy + dz * dz, ke, shift - 30);
    }
  };
  // the bytes of this thread's entries of step tb into buffer b
  auto store = [&](int tb, int b, double (&v)[E]) {
    if (odd) {
#pragma unroll
      for (int e = 0; e < E; e++) {
        const int tt = 16 * tg + sub * E + e;
        const double dx = Xr[b][tt][0] - x0, dy = Xr[b][tt][1] - x1, dz = Xr[b][tt][2] - x2;
        const double d2 = dx * dx + dy * dy + dz * dz;
        v[e] = d2 == 0. ? ldexp(ke.diag, shift - 30) : d2 > ke.far2 ? 0. : v[e];
      }
    }
    if (tb + KT > tk.t1) {
#pragma unroll
      for (int e = 0; e < E; e++)
        if (tb + 16 * tg + sub * E + e >= tk.t1) v[e] = 0.;
    }
    unsigned h[E], l[E];
#pragma unroll
    for (int e = 0; e < E; e++) {  // v = hi + lo / 2^30, signed bytes of both
      const double hm = v[e] + MAGIC;
      h[e] = (unsigned)__double2loint(hm) ^ DIGITS;
      l[e] = (unsigned)__double2loint(fma(v[e] - (hm - MAGIC), 1073741824.0, MAGIC)) ^ DIGITS;
    }
#pragma unroll
    for (int e = 0; e < E; e += 4) {
      unsigned lo[4], hi[4];
      bytes_of(l[e], l[e + 1], l[e + 2], l[e + 3], lo);
      bytes_of(h[e], h[e + 1], h[e + 2], h[e + 3], hi);
#pragma unroll
      for (int s = 0; s < 4; s++) {
        *reinterpret_cast<unsigned*>(&Gs[b][s][tg][col][sub * E + e]) = lo[s];
        *reinterpret_cast<unsigned*>(&Gs[b][4 + s][tg][col][sub * E + e]) = hi[s];
      }
    }
  };
  i4 acc[RW][CT][8];
#pragma unroll
  for (int i = 0; i < RW; i++)
#pragma unroll
    for (int j = 0; j < CT; j++)
#pragma unroll
      for (int s = 0; s < 8; s++) acc[i][j][s] = i4{0, 0, 0, 0};

  auto multiply = [&](int tb, int b) {
#pragma unroll
    for (int kb = 0; kb < KT / 64; kb++) {
      i4 o[RW];
#pragma unroll
      for (int i = 0; i < RW; i++) {
        if constexpr (AHEAD) {
          o[i] = om[i];
          if (tb + KT < tk.t1) om[i] = load_signs(i, tb + KT);
        } else {
          o[i] = load_signs(i, tb + 64 * kb);
        }
      }
#pragma unroll
      for (int s = 0; s < 8; s++)
#pragma unroll
        for (int j = 0; j < CT; j++) {
          const i4 g = *reinterpret_cast<const i4*>(&Gs[b][s][4 * kb + lk][(wc * CT + j) * 16 + lr][0]);
#pragma unroll
          for (int i = 0; i < RW; i++) acc[i][j][s] = __builtin_amdgcn_mfma_i32_16x16x64_i8(o[i], g, acc[i][j][s], 0, 0, 0);
        }
    }
  };

  if (tid < NX) {
    Xr[0][xr][xc] = row_coord(row_index(tk.t0 + xr));
    Xr[1][xr][xc] = row_coord(row_index(tk.t0 + KT + xr));
  }
  double xnext = row_coord(row_index(tk.t0 + 2 * KT + xr));
  int inext = row_index(tk.t0 + 3 * KT + xr);
  if constexpr (AHEAD)
#pragma unroll
    for (int i = 0; i < RW; i++) om[i] = load_signs(i, tk.t0);
  __syncthreads();
  {
    double v[E];
    evaluate(0, v);
    store(tk.t0, 0, v);
  }
  int b = 0;
  for (int tb = tk.t0; tb < tk.t1; tb += KT, b ^= 1) {
    __syncthreads();  // this step's bytes and the next step's coordinates are there; Xr[b] has been read
    if (tid < NX) {
      Xr[b][xr][xc] = xnext;
      xnext = row_coord(inext);
      inext = row_index(tb + 4 * KT + xr);
    }
    // the next step's entries beside this step's products (after the last
    // step: entries nobody reads)
    multiply(tb, b);
    double v[E];
    evaluate(b ^ 1, v);
    store(tb + KT, b ^ 1, v);
  }
#pragma unroll
  for (int i = 0; i < RW; i++)
#pragma unroll
    for (int j = 0; j < CT; j++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int row = tk.i0 + (wr * RW + i) * 16 + 4 * lk + q;
        const int c = tk.j0 + (wc * CT + j) * 16 + lr;
        long long lo = 0, hi = 0;
#pragma unroll
        for (int s = 3; s >= 0; s--) {
          lo = lo * 256 + acc[i][j][s][q];
          hi = hi * 256 + acc[i][j][4 + s][q];
        }
        const double y = ldexp(fma((double)hi, 1073741824.0, (double)lo), -shift);
        const bool drop = flagged && bad[(wc * CT + j) * 16 + lr];
        if (row < tk.M && c < tk.M) tk.out[row + (long long)c * tk.M] = drop ? __builtin_nan("") : y;
      }
}

// dst[e] = sum_{s < nsplit} src[e + s * len], in order of s.
__global__ void __launch_bounds__(256) k_sum_slices(const SliceSum* __restrict__ tasks, const long long* __restrict__ prefix,
                                                    int ntasks) {
  const long long blk = blockIdx.x;
  const int t = find_task(prefix, ntasks, blk);
  SliceSum tk = tasks[t];
  tk.src = in_global(tk.src);
  tk.dst = in_global(tk.dst);
  const long long e = (blk - prefix[t]) * 256 + threadIdx.x;
  if (e >= tk.len) return;
  double s = 0.;
  for (int k = 0; k < tk.nsplit; k++) s += tk.src[e + (long long)k * tk.len];
  tk.dst[e] = s;
}

// Tile of a box: all its rows up to 512 in one, with as many columns as the
// accumulators leave room for (the entries of a column are evaluated once per
// tile of rows, so a taller tile is worth more than a wider one).
struct SketchShape {
  int rows, cols;
};
constexpr size_t SIGNS_BYTES = 64 << 20;  // of the sign table
constexpr SketchShape SKETCH_SHAPES[] = {{64, 64}, {128, 64}, {256, 32}, {384, 32}, {512, 16}};
int sketch_shape(int M) {
  int k = 0;
  while (k < 4 && M > SKETCH_SHAPES[k].rows) k++;
  return k;
}

template <int KID>
void launch_sketch(int shape, unsigned grid, const SketchTask* tasks, const double* bodies, mxg_kernel_t k,
                   const u4* signs, int nu, int u0, hipStream_t s) {
  const dim3 g(grid), blk(512);
  const EvalArgs ke = eval_args(k);
  switch (shape) {
    case 0: hipLaunchKernelGGL((k_sketch<KID, 4, 1, 2, 64>), g, blk, 0, s, tasks, bodies, ke, signs, nu, u0); break;
    case 1: hipLaunchKernelGGL((k_sketch<KID, 8, 1, 4, 64>), g, blk, 0, s, tasks, bodies, ke, signs, nu, u0); break;
    case 2: hipLaunchKernelGGL((k_sketch<KID, 8, 2, 2, 64>), g, blk, 0, s, tasks, bodies, ke, signs, nu, u0); break;
    case 3: hipLaunchKernelGGL((k_sketch<KID, 8, 3, 2, 64>), g, blk, 0, s, tasks, bodies, ke, signs, nu, u0); break;
    default: hipLaunchKernelGGL((k_sketch<KID, 8, 4, 1, 128>), g, blk, 0, s, tasks, bodies, ke, signs, nu, u0); break;
  }
  MXG_HIP(hipGetLastError());
}

}  // namespace

void sketch_rows(mxg_ctx_s* ctx, const std::vector<SketchBox>& boxes, const double* d_bodies, mxg_kernel_t k,
                 double* d_partial, hipStream_t s) {
  long long maxM = 0, maxnf = 0;
  for (const SketchBox& b : boxes) {
    if (b.M <= 0 || b.nf <= 0) continue;
    maxM = std::max<long long>(maxM, b.M);
    maxnf = std::max(maxnf, b.nf);
  }
  MXG_REQUIRE(maxnf < (1ll << 31), "far list too long");
  // The signs of every row group a tile can cover (up to 512 rows a tile), for
  // whole slices of far rows. Longer lists than SIGNS_BYTES have room for, 131072
  // rows with boxes of up to 512 columns, take turns in the table.
  const unsigned groups = (unsigned)((maxM + 511) / 512 * 32);
  const long long window = std::max<long long>(SIGNS_BYTES / (16 * std::max(groups, 1u)) / SKETCH_ROWS, 1) * SKETCH_ROWS;
  std::map<std::pair<long long, int>, std::vector<SketchTask>> tasks;  // by window and tile shape
  std::vector<SliceSum> sums;
  std::vector<long long> prefix{0};
  size_t poff = 0;
  double flops = 0.;
  for (const SketchBox& b : boxes) {
    if (b.M <= 0 || b.nf <= 0) continue;
    flops += 2. * b.M * (double)b.M * (double)b.nf;
    const int nsplit = (int)((b.nf + SKETCH_ROWS - 1) / SKETCH_ROWS);
    const long long len = (long long)b.M * b.M;
    double* base = nsplit == 1 ? b.Y : d_partial + poff;
    const int shape = sketch_shape(b.M);
    for (int sp = 0; sp < nsplit; sp++) {
      const int t0 = sp * SKETCH_ROWS, t1 = (int)std::min<long long>(b.nf, (long long)(sp + 1) * SKETCH_ROWS);
      for (int i0 = 0; i0 < b.M; i0 += SKETCH_SHAPES[shape].rows)
        for (int j0 = 0; j0 < b.M; j0 += SKETCH_SHAPES[shape].cols)
          tasks[{t0 / window, shape}].push_back(SketchTask{b.rows, b.cols, base + sp * len, t0, t1, b.M, i0, j0, 0});
    }
    if (nsplit > 1) {
      sums.push_back(SliceSum{base, b.Y, len, nsplit, 0});
      prefix.push_back(prefix.back() + (len + 255) / 256);
      poff += (size_t)nsplit * len;
    }
  }
  if (tasks.empty()) return;
  std::vector<DevBuf<SketchTask>> dts(tasks.size());
  size_t q = 0;
  for (const auto& kv : tasks) {
    MXG_REQUIRE(kv.second.size() < (1u << 31), "sketch grid too large");
    dts[q++].upload(kv.second, s);
  }
  const long long nu = (std::min(maxnf, window) + 127) / 128 * 2;  // whole steps of 128 far rows
  DevBuf<u4> signs;
  signs.alloc((size_t)(64 * nu) * groups);
  ProfScope prof(ctx, MXG_PROF_SKETCH, s, flops);
  q = 0;
  long long filled = -1;
  for (const auto& kv : tasks) {
    const int u0 = (int)(kv.first.first * window / 64);
    if (kv.first.first != filled) {
      hipLaunchKernelGGL(k_sketch_signs, dim3(ceil_div(64 * nu, 256), groups), dim3(256), 0, s, signs.p, (int)nu, u0);
      MXG_HIP(hipGetLastError());
      filled = kv.first.first;
    }
    const unsigned g = (unsigned)kv.second.size();
    const SketchTask* tp = dts[q++].p;
    const int shape = kv.first.second;
    if (k.id == MXG_KERNEL_GAUSSIAN) launch_sketch<MXG_KERNEL_GAUSSIAN>(shape, g, tp, d_bodies, k, signs.p, (int)nu, u0, s);
    else if (k.id == MXG_KERNEL_YUKAWA) launch_sketch<MXG_KERNEL_YUKAWA>(shape, g, tp, d_bodies, k, signs.p, (int)nu, u0, s);
    else launch_sketch<MXG_KERNEL_LAPLACE>(shape, g, tp, d_bodies, k, signs.p, (int)nu, u0, s);
  }
  DevBuf<SliceSum> ds;
  DevBuf<long long> dp;
  if (!sums.empty()) {
    ds.upload(sums, s);
    dp.upload(prefix, s);
    hipLaunchKernelGGL(k_sum_slices, dim3((unsigned)prefix.back()), dim3(256), 0, s, ds.p, dp.p, (int)sums.size());
    MXG_HIP(hipGetLastError());
  }
  prof.end();
  MXG_HIP(hipStreamSynchronize(s));
}

size_t sketch_partial_size(long long M, long long nf) {
  if (M <= 0 || nf <= 0) return 0;
  const long long nsplit = (nf + SKETCH_ROWS - 1) / SKETCH_ROWS;
  return nsplit > 1 ? (size_t)nsplit * M * M : 0;
}

}  // namespace mxg
