// Variable-size batched GEMM with K segments on CDNA4 matrix cores.
//
// Each task owns one output block C (m x n, column major) and a list of K
// segments; the result is C = alpha * sum_s op(A_s) op(B_s) + beta * C. This
// single primitive covers every dense contraction of the ULV factorization
// (two-sided basis rotations, Schur complements whose K dimension runs over a
// row of near blocks) and of the basis construction (triangular products).
//
// Tiling: a 256-thread workgroup computes up to 128 indices of one side of C
// (the F side) by 64 of the other. Each wave takes 16 of the 64 and all blocks
// of 16 of the F side, MI of them, which are dealt evenly to the tiles (100
// rows are one tile of 7 blocks, 313 three of 7), so that the ragged blocks of
// a factorization are padded to 16 and not to the tile; which side is F is
// chosen for the least padding. K advances in slabs of 16 or 32 rows staged
// through two LDS buffers, one barrier a slab; a slab's global loads are issued
// before the products of the slab in front of it. A slab never crosses a
// segment, so an element sums its products in the same order, four at a time,
// for every tile shape. Tiles of all tasks share one launch; a table gives each
// workgroup its tile, and consecutive tiles go to one XCD, whose L2 then serves
// the operands that the tiles of a task share.
//
// Large launches are bound by the FP64 or FP32 matrix cores (about 72 and 148
// TFLOP/s on long plain products), of which they reach 55 to 60%: what is left
// is the prologue and epilogue of a tile, 8 of its 80 us in FP64, and each
// slab's trip through LDS where too few other waves have products to issue.
// Small ones are bound by the latency of a tile's slabs. What it took, before
// and now, in the largest launches of a factorization at N = 20000 (rank 100,
// boxes of 313, FP64; rotations of 800 near blocks): 1174 -> 773 and 1133 ->
// 679 us, its Schur products 774 -> 472 us, the sums over 13 segments onto 64
// diagonal blocks 616 -> 296 us; N = 131072 (rank 64, boxes of 256, FP32,
// 3598 near blocks): 1185 -> 758, 1034 -> 665, 778 -> 557 and 218 -> 124 us;
// the launches of the upper levels 15 to 25 -> 5 to 10 us. Before, a tile was
// 64 x 64 with every load flat, predicated and with its own 64-bit address, and
// the workgroup found its task by a binary search in memory.
//
// MFMA 16x16x4 operand layout (wave64): lane l supplies A[l % 16][l / 16] and
// B[l / 16][l % 16] of the 16x4 and 4x16 operands. Accumulator entry q
// (q = 0..3) of lane l is C[4 * (l / 16) + q][l % 16] for f32 and
// C[l / 16 + 4 * q][l % 16] for f64 (checked on gfx950 by the GEMM tests).
#include "internal.hpp"

namespace mxg {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

__device__ inline d4 mfma(double a, double b, d4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
__device__ inline f4 mfma(float a, float b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

template <class T> struct Acc;
template <> struct Acc<double> { typedef d4 type; };
template <> struct Acc<float> { typedef f4 type; };

// One output tile of a launch. swap: the F side is the columns of C (its
// operand B), else the rows. f0, s0: the tile's first index of each side.
struct GemmTile {
  int task, f0, s0;
  short mi, swap;
};

// The tile of this workgroup: workgroups go to the XCDs in turn, and each XCD
// takes a consecutive run of the tiles.
__device__ inline GemmTile my_tile(const GemmTile* __restrict__ tiles) {
  const unsigned n = gridDim.x, x = blockIdx.x & 7, q = n >> 3, r = n & 7;
  return in_constant(tiles)[x * q + min(x, r) + (blockIdx.x >> 3)];
}

// Entry x of a slab's LDS row p stands at p * LD + (x ^ swizzle(p)): the 16
// consecutive x of four rows that a matrix-core operand reads, and the 16
// consecutive x or p that a slab's stores write, fall into different banks
// (64 of 4 bytes; 32 lanes of 8 bytes or 64 of 4 at a time). It permutes bits
// of p, so that swizzle(p + q) = swizzle(p) ^ swizzle(q) when p and q share none.
template <class T>
__device__ constexpr int swizzle(int p) {
  if (sizeof(T) == 8) return ((p & 1) << 4) | (((p >> 1) & 7) << 1) | ((p >> 4) & 1);
  return ((p & 2) << 3) | (((p >> 2) & 3) << 2) | (((p >> 4) & 1) << 1) | ((p >> 5) & 1);
}

// One operand's part of a tile, N blocks of 16 indices: a thread holds, of each
// block and of each 16 rows of a slab, one entry, with the lane along the
// operand's contiguous index. Indices past the edge read the last one: they
// reach no element of C. Entries past the end of k, or below a masked
// diagonal, are zeroed on the way to LDS.
template <class T, int N, int KH, int LD, class Off>
struct Panel {
  T r[KH][N];       // the slab loaded last
  const T* next;    // first entry of the slab to load next
  long long step;   // from one row (k) to the next
  Off off[N];       // byte offsets of a slab's entries from its first
  int even, odd;    // LDS positions of its blocks (bit 4 of the swizzle exchanges the blocks of a pair)
  int k, d;         // its row; stored row - stored column of its first entry, negated if k is the column
  int kend, mask, kcontig;
  __device__ void open(const T* p, int x0, int last, int ld, int kcontig_, int mask_) {
    kcontig = kcontig_;
    mask = mask_;
    step = kcontig ? 1 : ld;
    next = p + (kcontig ? (long long)x0 * ld : x0);
    const int p16 = threadIdx.x & 15, q16 = threadIdx.x >> 4, x = kcontig ? q16 : p16;
    k = kcontig ? p16 : q16;
#pragma unroll
    for (int u = 0; u < N; u++)
      off[u] = (Off)sizeof(T) * (kcontig ? (Off)p16 + (Off)min(q16 + 16 * u, last) * (Off)ld
                                         : (Off)min(p16 + 16 * u, last) + (Off)q16 * (Off)ld);
    const int sw = swizzle<T>(k), lo = k * LD + (x ^ (sw & 15));
    even = lo + (sw & 16);
    odd = lo + (16 ^ (sw & 16));
    d = kcontig ? k - x0 - x : x0 + x - k;
  }
  // issues the loads of the next slab, kend rows before the segment's end; rows
  // past the end read the last one
  __device__ void load(int kend_) {
    kend = kend_;
    auto at = [](const T* p, Off v) { return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + v); };
    if (kend >= 16 * KH) {
#pragma unroll
      for (int h = 0; h < KH; h++)
#pragma unroll
        for (int u = 0; u < N; u++) r[h][u] = at(next + 16 * h * step, off[u]);
    } else {
#pragma unroll
      for (int h = 0; h < KH; h++) {
        const Off back = (Off)(min(16 * h + k, kend - 1) - k) * (Off)(sizeof(T) * step);
#pragma unroll
        for (int u = 0; u < N; u++) r[h][u] = at(next, off[u] + back);
      }
    }
    next += 16 * KH * step;
  }
  __device__ void store(T* S) {
    if (kend < 16 * KH) {
#pragma unroll
      for (int h = 0; h < KH; h++) {
        const bool in = 16 * h + k < kend;
#pragma unroll
        for (int u = 0; u < N; u++) r[h][u] = in ? r[h][u] : T(0);
      }
    }
    if (mask) {
#pragma unroll
      for (int h = 0; h < KH; h++)
#pragma unroll
        for (int u = 0; u < N; u++) {
          const int e = kcontig ? d + 16 * h - 16 * u : d - 16 * h + 16 * u;
          r[h][u] = e > 0 ? T(0) : r[h][u];
        }
      d += kcontig ? 16 * KH : -16 * KH;
    }
#pragma unroll
    for (int h = 0; h < KH; h++)
#pragma unroll
      for (int u = 0; u < N; u++)
        S[((u & 1 ? odd : even) ^ (swizzle<T>(16 * h) & 15)) + 16 * h * LD + (u & ~1) * 16] = r[h][u];
  }
};

// LDS row stride for N blocks: of a row and the next, FP32 entries 32 banks apart
template <class T, int N>
constexpr int panel_ld = (N + 1) / 2 * 32 + (sizeof(T) == 8 || N % 4 == 2 || N == 1 ? 0 : 32);

template <class T, int MI, int KH, int LDF, int LDS, class Off>
__device__ inline void gemm_tile(const GemmTask<T>& task, const GemmSeg<T>* segs, const GemmTile& tile,
                                 T* __restrict__ Fs, T* __restrict__ Ss) {
  typedef typename Acc<T>::type V;
  constexpr int BK = 16 * KH;
  const int fn = tile.swap ? task.n : task.m, sn = tile.swap ? task.m : task.n;
  const int flast = min(16 * MI, fn - tile.f0) - 1, slast = min(64, sn - tile.s0) - 1;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  const bool idle = wave * 16 > slast;  // no column of the wave's block is in C
  V acc[MI];
#pragma unroll
  for (int i = 0; i < MI; i++) acc[i] = V{0, 0, 0, 0};

  Panel<T, MI, KH, LDF, Off> F;
  Panel<T, 4, KH, LDS, Off> S;
  GemmSeg<T> gn{};
  int cs = task.seg0, kleft = 0;  // next segment; rows left of the open one
  const int send = task.seg0 + task.nseg;
  if (cs < send) gn = segs[cs];
  // issues the loads of the next slab and returns its steps of 4 rows, 0 past the last slab
  auto load = [&]() {
    if (kleft <= 0) {
      GemmSeg<T> g;
      do {
        if (cs >= send) return 0;
        g = gn;
        if (++cs < send) gn = segs[cs];
      } while (g.k <= 0);
      kleft = g.k;
      const T* fp = tile.swap ? g.B : g.A;
      const T* sp = tile.swap ? g.A : g.B;
      F.open(in_global(fp), tile.f0, flast, tile.swap ? g.ldb : g.lda, tile.swap ? !g.tb : g.ta, tile.swap ? g.bmask : g.amask);
      S.open(in_global(sp), tile.s0, slast, tile.swap ? g.lda : g.ldb, tile.swap ? g.ta : !g.tb, tile.swap ? g.amask : g.bmask);
    }
    F.load(kleft);
    S.load(kleft);
    const int n = (min(BK, kleft) + 3) / 4;
    kleft -= BK;
    return n;
  };
  const int sw = swizzle<T>(lk), hi = sw & 16, lo = lr ^ (sw & 15);
  const int fe = lk * LDF + hi, fo = lk * LDF + (16 ^ hi), sb = lk * LDS + ((16 * wave) ^ hi);
  T a[2][MI], b[2];
  int steps = load();
  for (int buf = 0; steps; buf ^= 1) {
    T* fs = Fs + buf * (BK * LDF);
    T* ss = Ss + buf * (BK * LDS);
    F.store(fs);
    S.store(ss);
    __syncthreads();
    const int now = steps;
    steps = load();
    if (idle) continue;
    auto read = [&](int kk) {
      const int l = lo ^ (swizzle<T>(4 * kk) & 15);
#pragma unroll
      for (int i = 0; i < MI; i++) a[kk & 1][i] = fs[(i & 1 ? fo : fe) + l + kk * 4 * LDF + (i & ~1) * 16];
      b[kk & 1] = ss[sb + l + kk * 4 * LDS];
    };
    read(0);
#pragma unroll
    for (int kk = 0; kk < BK / 4; kk++) {
      if (kk >= now) break;
      if (kk + 1 < BK / 4) read(kk + 1);
      __builtin_amdgcn_sched_barrier(0);  // the next step's operands are on their way before this one's products
#pragma unroll
      for (int i = 0; i < MI; i++) acc[i] = mfma(b[kk & 1], a[kk & 1][i], acc[i]);
    }
  }

  const T alpha = (T)task.alpha, beta = (T)task.beta;
  T* const C = in_global(task.C);
  // all of C's entries are read before the first is written: one latency
  T c[MI][4];
  auto entry = [&](int i, int q, T*& p) {
    const int f = 16 * i + lr, x = 16 * wave + (sizeof(T) == 8 ? lk + 4 * q : 4 * lk + q);
    const int row = tile.swap ? tile.s0 + x : tile.f0 + f, col = tile.swap ? tile.f0 + f : tile.s0 + x;
    p = C + row + (long long)col * task.ldc;
    return f <= flast && x <= slast;
  };
  if (task.beta != 0.) {
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        T* p;
        c[i][q] = entry(i, q, p) ? *p : T(0);
      }
  }
#pragma unroll
  for (int i = 0; i < MI; i++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      T* p;
      if (entry(i, q, p)) {
        T v = alpha * acc[i][q];
        if (task.beta != 0.) v += beta * c[i][q];
        *p = v;
      }
    }
}

// 3 or 4 workgroups a CU: 168 or 128 registers a lane, and as much LDS
template <class T, int CAP, int KH, class Off>
__global__ void __launch_bounds__(256, sizeof(T) == 8 && CAP == 8 ? 3 : 4) k_bgemm(const GemmTask<T>* __restrict__ tasks, const GemmSeg<T>* __restrict__ segs,
                                                  const GemmTile* __restrict__ tiles) {
  constexpr int LDF = panel_ld<T, CAP>, LDS = panel_ld<T, 4>;
  __shared__ T Fs[2 * 16 * KH * LDF];
  __shared__ T Ss[2 * 16 * KH * LDS];
  const GemmTile tile = my_tile(tiles);
  const GemmTask<T> task = in_constant(tasks)[tile.task];
  switch (tile.mi) {
    case 1: gemm_tile<T, 1, KH, LDF, LDS, Off>(task, in_constant(segs), tile, Fs, Ss); break;
    case 2: if constexpr (CAP >= 2) gemm_tile<T, 2, KH, LDF, LDS, Off>(task, in_constant(segs), tile, Fs, Ss); break;
    case 3: if constexpr (CAP >= 3) gemm_tile<T, 3, KH, LDF, LDS, Off>(task, in_constant(segs), tile, Fs, Ss); break;
    case 4: if constexpr (CAP >= 4) gemm_tile<T, 4, KH, LDF, LDS, Off>(task, in_constant(segs), tile, Fs, Ss); break;
    case 5: if constexpr (CAP >= 5) gemm_tile<T, 5, KH, LDF, LDS, Off>(task, in_constant(segs), tile, Fs, Ss); break;
    case 6: if constexpr (CAP >= 6) gemm_tile<T, 6, KH, LDF, LDS, Off>(task, in_constant(segs), tile, Fs, Ss); break;
    case 7: if constexpr (CAP >= 7) gemm_tile<T, 7, KH, LDF, LDS, Off>(task, in_constant(segs), tile, Fs, Ss); break;
    case 8: if constexpr (CAP >= 8) gemm_tile<T, 8, KH, LDF, LDS, Off>(task, in_constant(segs), tile, Fs, Ss); break;
  }
}

// The FP32 tasks with bfloat16 inputs: op(A) and op(B) are rounded to
// bfloat16 (nearest even) as they are staged, and each 16-deep slab is one
// v_mfma_f32_16x16x16_bf16 per 16 x 16 accumulator (FP32 accumulation). Lane l
// supplies A[l % 16][4 (l / 16) + e] and B[4 (l / 16) + e][l % 16], e < 4; the
// accumulator layout is that of the FP32 instruction. Tiles go to the XCDs in runs,
// by the table, or (RUNS false) in launch order, each workgroup finding its task in
// the prefix sums of the tasks' tiles.
typedef short s4_t __attribute__((ext_vector_type(4)));
constexpr int BM = 64, BN = 64, BK = 16, PADH = 2;

__device__ inline unsigned short bf16_bits(float x) {
  const unsigned u = __float_as_uint(x);
  return (unsigned short)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

template <bool RUNS>
__global__ void __launch_bounds__(256) k_bgemm_bf16(const GemmTask<float>* __restrict__ tasks,
                                                    const GemmSeg<float>* __restrict__ segs,
                                                    const GemmTile* __restrict__ tiles,
                                                    const long long* __restrict__ prefix, int ntasks) {
  __shared__ unsigned short As[BK][BM + PADH];
  __shared__ unsigned short Bs[BK][BN + PADH];
  GemmTile tile;
  if constexpr (RUNS) {
    tile = my_tile(tiles);
  } else {
    tile.task = find_task(prefix, ntasks, blockIdx.x);
    const int local = (int)(blockIdx.x - prefix[tile.task]), tiles_m = (in_constant(tasks)[tile.task].m + BM - 1) / BM;
    tile.f0 = local % tiles_m * BM;
    tile.s0 = local / tiles_m * BN;
  }
  const GemmTask<float> task = in_constant(tasks)[tile.task];
  const int m0 = tile.f0, n0 = tile.s0;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave >> 1, wc = wave & 1;
  const int lr = lane & 15, lk = lane >> 4;

  f4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = f4{0, 0, 0, 0};

  for (int s = task.seg0; s < task.seg0 + task.nseg; s++) {
    const GemmSeg<float> g = in_constant(segs)[s];
    const float* gA = in_global(g.A);
    const float* gB = in_global(g.B);
    for (int k0 = 0; k0 < g.k; k0 += BK) {
#pragma unroll
      for (int e0 = 0; e0 < BM * BK; e0 += 256) {
        const int e = e0 + tid;
        int i, p;
        if (!g.ta) { i = e % BM; p = e / BM; } else { p = e % BK; i = e / BK; }
        const int gi = m0 + i, gp = k0 + p;
        float v = 0.f;
        if (gi < task.m && gp < g.k) {
          const int sr = g.ta ? gp : gi, sc = g.ta ? gi : gp;
          if (!(g.amask && sr > sc)) v = gA[sr + (long long)sc * g.lda];
        }
        As[p][i] = bf16_bits(v);
      }
#pragma unroll
      for (int e0 = 0; e0 < BK * BN; e0 += 256) {
        const int e = e0 + tid;
        int p, j;
        if (!g.tb) { p = e % BK; j = e / BK; } else { j = e % BN; p = e / BN; }
        const int gp = k0 + p, gj = n0 + j;
        float v = 0.f;
        if (gp < g.k && gj < task.n) {
          const int sr = g.tb ? gj : gp, sc = g.tb ? gp : gj;
          if (!(g.bmask && sr > sc)) v = gB[sr + (long long)sc * g.ldb];
        }
        Bs[p][j] = bf16_bits(v);
      }
      __syncthreads();
      s4_t a[2], b[2];
#pragma unroll
      for (int e = 0; e < 4; e++) {
#pragma unroll
        for (int i = 0; i < 2; i++) a[i][e] = (short)As[4 * lk + e][wr * 32 + i * 16 + lr];
#pragma unroll
        for (int j = 0; j < 2; j++) b[j][e] = (short)Bs[4 * lk + e][wc * 32 + j * 16 + lr];
      }
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[i], b[j], acc[i][j], 0, 0, 0);
      __syncthreads();
    }
  }

  const float alpha = (float)task.alpha, beta = (float)task.beta;
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int row = m0 + wr * 32 + i * 16 + 4 * lk + q;
        const int col = n0 + wc * 32 + j * 16 + lr;
        if (row < task.m && col < task.n) {
          float* c = in_global(task.C) + row + (long long)col * task.ldc;
          float v = alpha * acc[i][j][q];
          if (task.beta != 0.) v += beta * (*c);
          *c = v;
        }
      }
}

// Tiles of an m x n block with at most cap blocks of 16 on the F side.
struct Tiling {
  long long nf, ns;
  int mi, swap;
};
Tiling tiling(long long m, long long n, int cap) {
  Tiling best{};
  long long cost = 0;
  for (int swap = 0; swap < 2; swap++) {
    const long long bf = ((swap ? n : m) + 15) / 16, bs = ((swap ? m : n) + 15) / 16;
    const long long nf = (bf + cap - 1) / cap, ns = (bs + 3) / 4;
    const int mi = (int)((bf + nf - 1) / nf);
    const long long c = nf * mi * ns * 4;
    if (!swap || c < cost) {
      best = Tiling{nf, ns, mi, swap};
      cost = c;
    }
  }
  return best;
}

template <class T>
long long count_tiles(const std::vector<GemmTask<T>>& tasks, int cap) {
  long long n = 0;
  for (const GemmTask<T>& g : tasks) {
    if (g.m <= 0 || g.n <= 0) continue;
    const Tiling t = tiling(g.m, g.n, cap);
    n += t.nf * t.ns;
  }
  return n;
}

}  // namespace

template <class T>
void gemm_batched(const std::vector<GemmTask<T>>& tasks, const std::vector<GemmSeg<T>>& segs, hipStream_t s, bool bf16,
                  Stage* st) {
  if (tasks.empty()) return;
  MXG_REQUIRE(!bf16 || (std::is_same<T, float>::value), "bfloat16 inputs are for FP32 products");
  for (const GemmTask<T>& g : tasks)
    MXG_REQUIRE(g.seg0 >= 0 && g.nseg >= 0 && (size_t)(g.seg0 + g.nseg) <= segs.size(), "gemm task segment range");
  // The tallest F side that still gives two workgroups a CU: tall ones read
  // and stage less per product (the 800 blocks above: 773 us with 8, 841 with
  // 4, 955 with 2), short ones keep a small launch's chip busy (one tile of 16
  // to 128 rows of 64 Schur sums, K = 2660: 296, 307, 369 and 523 us with 1, 2,
  // 4 and 8 blocks).
  int cap = 8;
  while (!bf16 && cap > 1 && count_tiles(tasks, cap) < 512) cap /= 2;
  // byte offsets of a tile's entries in 32 bits, unless a column stride is 2^21 or more
  bool wide = false;
  for (const GemmSeg<T>& g : segs) wide = wide || std::max(g.lda, g.ldb) >= (1 << 21);
  if (wide) cap = 4;
  std::vector<GemmTile> tiles;
  std::vector<long long> prefix;  // of the bfloat16 tasks' tiles, if they go in launch order
  if (bf16) {
    prefix.push_back(0);
    for (const GemmTask<T>& g : tasks)
      prefix.push_back(prefix.back() +
                       (g.m > 0 && g.n > 0 ? (long long)((g.m + BM - 1) / BM) * ((g.n + BN - 1) / BN) : 0));
    MXG_REQUIRE(prefix.back() < (1ll << 31), "gemm grid too large");
    // The blocks of a factorization share their operands within a run (N = 20000,
    // rank 100, with bfloat16 Schur products: 7.5 ms, 8.0 in launch order). An XCD
    // that takes a run of a large block's columns reads all rows of op(A) at once,
    // beyond its L2: from 64 tiles on in launch order if A is stored as it is used
    // (4096 x 256 x 4096: 537 us, 580 in runs; 1000 x 1000 x 1000: 182 and 196), from
    // 1024 on if it is transposed (4096 x 4096 x 1024: 472 and 549; but 256 x 4096 x
    // 4096: 498 and 447, 1000 x 1000 x 1000: 200 and 181).
    bool ta = false;
    for (const GemmSeg<T>& g : segs) ta = ta || g.ta;
    if (prefix.back() <= (ta ? 1023 : 64) * (long long)tasks.size()) prefix.clear();
  }
  const bool runs = prefix.empty();
  for (size_t t = 0; t < tasks.size() && runs; t++) {
    const GemmTask<T>& g = tasks[t];
    if (g.m <= 0 || g.n <= 0) continue;
    const Tiling c = bf16 ? Tiling{(g.m + BM - 1) / BM, (g.n + BN - 1) / BN, 4, 0} : tiling(g.m, g.n, cap);
    MXG_REQUIRE(tiles.size() + c.nf * c.ns < (1ull << 31), "gemm grid too large");
    for (long long y = 0; y < c.ns; y++)
      for (long long x = 0; x < c.nf; x++)
        tiles.push_back(GemmTile{(int)t, (int)(x * 16 * c.mi), (int)(y * 64), (short)c.mi, (short)c.swap});
  }
  const size_t total = runs ? tiles.size() : (size_t)prefix.back();
  if (total == 0) return;
  DevBuf<GemmTask<T>> dt;
  DevBuf<GemmSeg<T>> ds;
  DevBuf<GemmTile> dp;
  DevBuf<long long> dx;
  const GemmTask<T>* pt;
  const GemmSeg<T>* ps;
  const GemmTile* pp;
  const long long* px;
  if (st) {
    pt = st->put(tasks);
    ps = st->put(segs);
    pp = st->put(tiles);
    px = st->put(prefix);
  } else {
    dt.upload(tasks, s);
    ds.upload(segs, s);
    dp.upload(tiles, s);
    dx.upload(prefix, s);
    pt = dt.p;
    ps = ds.p;
    pp = dp.p;
    px = dx.p;
  }
  const dim3 grid((unsigned)total);
  const int ntasks = (int)tasks.size();
  auto launch = [=] {
    auto go = [&](auto k, auto... more) {
      hipLaunchKernelGGL(k, grid, dim3(256), 0, s, pt, ps, pp, more...);
      MXG_HIP(hipGetLastError());
    };
    if constexpr (std::is_same<T, float>::value)
      if (bf16) return runs ? go(k_bgemm_bf16<true>, px, ntasks) : go(k_bgemm_bf16<false>, px, ntasks);
    // slabs of 32 rows where a short FP32 tile's products would not cover its
    // loads (the FP32 sums over segments with 1 and 2 blocks: 25.0 and 28.1 us
    // against 29.0 and 33.1 with 16); in FP64 they gain nothing
    constexpr int KH = sizeof(T) == 4 ? 2 : 1;
    if (wide) go(k_bgemm<T, 4, 1, unsigned long long>);
    else if (cap == 8) go(k_bgemm<T, 8, 1, unsigned>);
    else if (cap == 4) go(k_bgemm<T, 4, 1, unsigned>);
    else if (cap == 2) go(k_bgemm<T, 2, KH, unsigned>);
    else go(k_bgemm<T, 1, KH, unsigned>);
  };
  if (st) {
    st->later(launch);
  } else {
    launch();
    MXG_HIP(hipStreamSynchronize(s));  // descriptor arrays are freed on return
  }
}

template void gemm_batched<double>(const std::vector<GemmTask<double>>&, const std::vector<GemmSeg<double>>&, hipStream_t,
                                   bool, Stage*);
template void gemm_batched<float>(const std::vector<GemmTask<float>>&, const std::vector<GemmSeg<float>>&, hipStream_t, bool,
                                  Stage*);

}  // namespace mxg

using namespace mxg;

namespace {
template <class T>
void one_gemm(mxg_ctx_t ctx, int ta, int tb, long long m, long long n, long long k, double alpha, const void* A, long long lda,
              const void* B, long long ldb, double beta, void* C, long long ldc, bool bf16 = false) {
  std::vector<GemmSeg<T>> segs{GemmSeg<T>{static_cast<const T*>(A), static_cast<const T*>(B), (int)lda, (int)ldb, (int)k,
                                          (unsigned char)(ta != 0), (unsigned char)(tb != 0), 0, 0}};
  std::vector<GemmTask<T>> tasks{GemmTask<T>{static_cast<T*>(C), (int)ldc, (int)m, (int)n, 0, k > 0 ? 1 : 0, alpha, beta}};
  gemm_batched<T>(tasks, segs, ctx->stream, bf16);
}
}  // namespace

extern "C" int mxg_gemm(mxg_ctx_t ctx, int precision, int ta, int tb, long long m, long long n, long long k, double alpha,
                        const void* d_A, long long lda, const void* d_B, long long ldb, double beta, void* d_C, long long ldc) {
  return guarded([&] {
    MXG_REQUIRE(ctx, "ctx is null");
    MXG_REQUIRE(m >= 0 && n >= 0 && k >= 0, "negative size");
    MXG_REQUIRE(m < (1ll << 31) && n < (1ll << 31) && k < (1ll << 31) && lda < (1ll << 31) && ldb < (1ll << 31) &&
                    ldc < (1ll << 31), "size exceeds 2^31");
    MXG_REQUIRE(ldc >= std::max<long long>(m, 1), "ldc < m");
    MXG_REQUIRE(lda >= std::max<long long>(ta ? k : m, 1) && ldb >= std::max<long long>(tb ? n : k, 1), "lda/ldb too small");
    if (m == 0 || n == 0) return;
    MXG_REQUIRE(d_C && (k == 0 || (d_A && d_B)), "null pointer");
    PoolScope pool(ctx->pool);
    if (precision == MXG_FP64)
      one_gemm<double>(ctx, ta, tb, m, n, k, alpha, d_A, lda, d_B, ldb, beta, d_C, ldc);
    else if (precision == MXG_FP32)
      one_gemm<float>(ctx, ta, tb, m, n, k, alpha, d_A, lda, d_B, ldb, beta, d_C, ldc);
    else if (precision == MXG_BF16)
      one_gemm<float>(ctx, ta, tb, m, n, k, alpha, d_A, lda, d_B, ldb, beta, d_C, ldc, true);
    else
      throw Error(MXG_ERR_ARG, "unknown precision");
  });
}
