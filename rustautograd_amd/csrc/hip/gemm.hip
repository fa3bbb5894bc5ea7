// Dense products for MatMul / MatMulT (reference src/plan.rs:1453-1493, flags from
// src/optimize.rs:338-350).
//
// fp32: most products run on the bf16 matrix cores, every operand value split exactly into three
// bf16 values (gemm_split.h: block tiles of 128x128, 128x64 and 64x64). Products of too few tiles
// for that take fp32 MFMA tiles (gemm_mfma.h), of four wave64s, each owning a grid of 16x16 MFMA
// tiles (v_mfma_f32_16x16x4_f32). There global loads run two K steps ahead through two register
// stages, and operands are staged through double-buffered LDS in their own global layout, so no
// operand is transposed while staging:
//  - a K-contiguous operand (A, or B when transposed) sits in LDS as [rows][BK + 4]; one 16-byte
//    LDS read gives a lane four consecutive k of one tile row, feeding four MFMA k-steps;
//  - an M- or N-contiguous operand sits as [BK][cols]; one read gives a lane T consecutive
//    columns at one k, one for each of the wave's T tiles (tile t holds columns t, t + T, ...).
// Global loads are 16-byte vectors without branches: a vector lies wholly inside or outside the
// operand (leading dimensions are multiples of 4), and an outside vector reads a valid address
// and is replaced by zeros; products whose tiles divide M, N and K skip even that check. Unaligned
// operands take the same kernel with scalar loads. The tile is chosen per product to fill 256 CUs
// with little padding; products whose output has too few tiles split K and combine the partial
// sums in a fixed order (deterministic).
// fp32 products with at most 16 rows and a long K, or a K of at most 16, stream through the
// skinny kernels below (HBM-bound shapes); fp64 products run on fp64
// MFMA tiles; what remains is a wave per output where K is long, a thread per output otherwise.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <stdexcept>
#include <string>
#include <type_traits>

#include "gemm_mfma.h"
#include "gemm_split.h"
#include "kernels.h"
#include "ops.h"

namespace rgk {

namespace {

using namespace rgg;

template <int BM, int BN, int BK, int WM, int WN, bool TA, bool TB, int MODE>
__global__ void __launch_bounds__(64 * WM * WN) k_gemm_f32(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C,
                                                           int M, int N, int K, const int64_t* a_off, const int64_t* b_off,
                                                           uint64_t a_stride, uint64_t b_stride, int splits, int k_per_split,
                                                           float* __restrict__ partial, const float* __restrict__ bias, uint32_t tiles_m,
                                                           uint32_t tiles_n) {
  rgg::StoreC epi{C, partial, splits, (uint64_t)M * N};
  rgg::gemm_f32_block<BM, BN, BK, WM, WN, TA, TB, MODE>(A, B, M, N, K, a_off, b_off, a_stride, b_stride, splits, k_per_split, bias, tiles_m,
                                                        tiles_n, epi);
}

// Waves per SIMD the registers must leave room for: two 128x128 blocks of eight waves per CU (one
// with two steps in LDS), three 128x64 or 64x64 blocks of four.
constexpr int split_waves(int bm, int bn, int u) { return bm * bn >= 128 * 128 ? (u == 1 ? 4 : 2) : 3; }

template <int BM, int BN, int WM, int WN, int U, bool TA, bool TB, bool TAIL>
__global__ void __launch_bounds__(64 * WM * WN, split_waves(BM, BN, U)) k_gemm_mfma(const float* __restrict__ A, const float* __restrict__ B,
                                                                                  float* __restrict__ C, int M, int N, int K,
                                                                                  const int64_t* a_off, const int64_t* b_off, uint64_t a_stride,
                                                                                  uint64_t b_stride, int splits, int k_per_split,
                                                                                  float* __restrict__ partial, const float* __restrict__ bias,
                                                                                  uint32_t tiles_m, uint32_t tiles_n) {
  rgg::StoreC epi{C, partial, splits, (uint64_t)M * N};
  rgg::gemm_mfma_block<BM, BN, WM, WN, U, TA, TB, TAIL>(A, B, M, N, K, a_off, b_off, a_stride, b_stride, splits, k_per_split, bias, tiles_m,
                                                        tiles_n, epi);
}

// One unbatched product's share of a grouped launch (k_gemm_mfma_group).
struct GroupPart {
  const float *a, *b;
  float *c, *part;
  const float* bias;
  int m, n, k, splits, kps;
  uint32_t tm, tn, blocks;
};
constexpr int GROUP_MAX = 3;
struct GroupParts {
  GroupPart p[GROUP_MAX];
};

// Part I of a grouped launch: flags bits 2I (TB) and 2I + 1 (TA).
template <int BM, int BN, int WM, int WN, int U, int FLAGS, int I>
__device__ __forceinline__ void group_part(const GroupPart& p, uint32_t bid, cell* smem) {
  constexpr bool TA = (FLAGS >> (2 * I + 1)) & 1, TB = (FLAGS >> (2 * I)) & 1;
  StoreC epi{p.c, p.part, p.splits, (uint64_t)p.m * p.n};
  gemm_split_tile<BM, BN, WM, WN, U, TA, TB, false>(p.a, p.b, p.m, p.n, p.k, nullptr, nullptr, 0, 0, p.splits, p.kps, p.bias, p.tm, p.tn, epi, bid,
                                                 p.blocks, smem);
}

template <int BM, int BN, int WM, int WN, int U, int FLAGS, int I>
constexpr int part_lds() {
  return SplitLds<BM, BN, WM, WN, U, ((FLAGS >> (2 * I + 1)) & 1) != 0, ((FLAGS >> (2 * I)) & 1) != 0>::CELLS;
}

// N independent unbatched products on one tile shape in one launch: part i takes the next
// p[i].blocks blocks, all staging through the same LDS. Each block runs the code of a single
// product's launch, so every output gets the same bits; the launch's fixed cost is paid once,
// and the parts' grids (each one or two blocks per CU) run side by side.
template <int BM, int BN, int WM, int WN, int U, int N, int FLAGS>
__global__ void __launch_bounds__(64 * WM * WN, split_waves(BM, BN, U)) k_gemm_mfma_group(GroupParts g) {
  constexpr int F0 = part_lds<BM, BN, WM, WN, U, FLAGS, 0>(), F1 = part_lds<BM, BN, WM, WN, U, FLAGS, 1>();
  constexpr int F2 = N > 2 ? part_lds<BM, BN, WM, WN, U, FLAGS, 2>() : 0;
  constexpr int F01 = F0 > F1 ? F0 : F1;
  __shared__ cell smem[F01 > F2 ? F01 : F2];
  uint32_t bid = blockIdx.x;
  if (bid < g.p[0].blocks) return group_part<BM, BN, WM, WN, U, FLAGS, 0>(g.p[0], bid, smem);
  bid -= g.p[0].blocks;
  if (N == 2 || bid < g.p[1].blocks) return group_part<BM, BN, WM, WN, U, FLAGS, 1>(g.p[1], bid, smem);
  if constexpr (N > 2) group_part<BM, BN, WM, WN, U, FLAGS, 2>(g.p[2], bid - g.p[1].blocks, smem);
}

// The same on 32x32 fp32 MFMA tiles: products too small to fill the chip alone (C3's input and weight
// gradients, 256 to 512 blocks of 8-10 us, run side by side).
template <int FLAGS, int I>
__device__ __forceinline__ void small_part(const GroupPart& p, uint32_t bid, float* smem) {
  constexpr bool TA = (FLAGS >> (2 * I + 1)) & 1, TB = (FLAGS >> (2 * I)) & 1;
  StoreC epi{p.c, p.part, p.splits, (uint64_t)p.m * p.n};
  gemm_f32_tile<32, 32, 32, 2, 2, TA, TB, LOAD_EVEN>(p.a, p.b, p.m, p.n, p.k, nullptr, nullptr, 0, 0, p.splits, p.kps, p.bias, p.tm, p.tn, epi,
                                                     bid, p.blocks, smem);
}

template <int N, int FLAGS>
__global__ void __launch_bounds__(256) k_gemm_f32_group(GroupParts g) {
  __shared__ float smem[TileLds<32, 32, 32, false, true>::FLOATS];  // both operands K-contiguous: the largest
  uint32_t bid = blockIdx.x;
  if (bid < g.p[0].blocks) return small_part<FLAGS, 0>(g.p[0], bid, smem);
  bid -= g.p[0].blocks;
  if (N == 2 || bid < g.p[1].blocks) return small_part<FLAGS, 1>(g.p[1], bid, smem);
  if constexpr (N > 2) small_part<FLAGS, 2>(g.p[2], bid - g.p[1].blocks, smem);
}

// Sums the K-split partial products in split order. Four outputs per thread (16-byte loads when
// M N is a multiple of 4), all splits' loads issued before the adds.
__global__ void __launch_bounds__(256) k_split_sum(const float* __restrict__ partial, float* __restrict__ C, uint64_t mn, int splits,
                                                   const float* __restrict__ bias, uint64_t n) {
  const uint64_t i = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  const uint32_t b = blockIdx.y;
  if (i >= mn) return;
  const float* p = partial + (uint64_t)b * splits * mn + i;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  if (mn % 4 == 0) {
    float4 v[16];
#pragma unroll
    for (int s = 0; s < 16; s++)
      if (s < splits) v[s] = *(const float4*)(p + (uint64_t)s * mn);
    acc = v[0];
#pragma unroll
    for (int s = 1; s < 16; s++)
      if (s < splits) acc = make_float4(acc.x + v[s].x, acc.y + v[s].y, acc.z + v[s].z, acc.w + v[s].w);
    if (bias) acc = make_float4(acc.x + bias[i % n], acc.y + bias[(i + 1) % n], acc.z + bias[(i + 2) % n], acc.w + bias[(i + 3) % n]);
    *(float4*)(C + (uint64_t)b * mn + i) = acc;
    return;
  }
  for (uint64_t e = i; e < i + 4 && e < mn; e++) {
    float x = partial[(uint64_t)b * splits * mn + e];
    for (int s = 1; s < splits; s++) x += partial[((uint64_t)b * splits + s) * mn + e];
    if (bias) x += bias[e % n];
    C[(uint64_t)b * mn + e] = x;
  }
}

// C[e] += bias[e mod n]: the bias of a product that does not run on the matrix cores.
__global__ void __launch_bounds__(256) k_add_bias(float* __restrict__ C, const float* __restrict__ bias, uint64_t total, uint64_t n) {
  const uint64_t e = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (e < total) C[e] = C[e] + bias[e % n];
}

// One output element per thread; k ascending, eight loads of each operand in flight.
template <class T>
__global__ void __launch_bounds__(256) k_gemm_plain(const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ C, uint32_t M,
                                                    uint32_t N, uint32_t K, bool ta, bool tb, const int64_t* a_off, const int64_t* b_off,
                                                    uint64_t a_stride, uint64_t b_stride) {
  uint32_t b = blockIdx.y;
  uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= (uint64_t)M * N) return;
  uint32_t i = (uint32_t)(t / N), j = (uint32_t)(t % N);
  const T* a = A + batch_offset(a_off, a_stride, b) + (ta ? (uint64_t)i : (uint64_t)i * K);
  const T* bb = B + batch_offset(b_off, b_stride, b) + (tb ? (uint64_t)j * K : (uint64_t)j);
  const uint64_t sa = ta ? M : 1, sb = tb ? 1 : N;
  T acc = (T)0;
  uint32_t p = 0;
  for (; p + 8 <= K; p += 8) {
    T x[8], y[8];
#pragma unroll
    for (int u = 0; u < 8; u++) x[u] = a[(p + u) * sa], y[u] = bb[(p + u) * sb];
#pragma unroll
    for (int u = 0; u < 8; u++) acc = acc + x[u] * y[u];
  }
  for (; p < K; p++) acc = acc + a[p * sa] * bb[p * sb];
  C[(uint64_t)b * M * N + t] = acc;
}

// Few outputs over a longer K, any type, flags and batch: W waves per output, four outputs per block
// of W = 1 and one otherwise. Lanes take k 64 W apart in increasing order (eight loads of each
// operand in flight), a wave's sum by a fixed butterfly, the wave sums added in order. One thread per
// output walked K alone: 256 x 1 x 8 transposed (linear regression's gradient) took 25 us, 3 here;
// 1000 x 1 x 500 132 us, 4 here.
template <class T, int W>
__global__ void __launch_bounds__(W == 1 ? 256 : 64 * W) k_gemm_dots(const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ C,
                                                                    uint32_t M, uint32_t N, uint32_t K, bool ta, bool tb,
                                                                    const int64_t* a_off, const int64_t* b_off, uint64_t a_stride,
                                                                    uint64_t b_stride) {
  constexpr int PER = W == 1 ? 4 : 1;
  __shared__ T wsum[W];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, w = W == 1 ? 0 : wave;
  const uint32_t b = blockIdx.y;
  const uint64_t e = (uint64_t)blockIdx.x * PER + (W == 1 ? wave : 0);
  if (e >= (uint64_t)M * N) return;  // whole waves; blocks of several waves have one output
  const uint32_t i = (uint32_t)(e / N), j = (uint32_t)(e % N);
  const T* a = A + batch_offset(a_off, a_stride, b) + (ta ? (uint64_t)i : (uint64_t)i * K);
  const T* bb = B + batch_offset(b_off, b_stride, b) + (tb ? (uint64_t)j * K : (uint64_t)j);
  const uint64_t sa = ta ? M : 1, sb = tb ? 1 : N;
  T acc = (T)0;
  uint64_t k = (uint64_t)w * 64 + lane;
  for (; k + 7 * 64 * W < K; k += 8 * 64 * W) {
    T x[8], y[8];
#pragma unroll
    for (int u = 0; u < 8; u++) x[u] = a[(k + u * 64 * W) * sa], y[u] = bb[(k + u * 64 * W) * sb];
#pragma unroll
    for (int u = 0; u < 8; u++) acc = fma(x[u], y[u], acc);
  }
  for (; k < K; k += 64 * W) acc = fma(a[k * sa], bb[k * sb], acc);
  T sum = rg_wave_sum(acc);
  if constexpr (W > 1) {
    if (lane == 0) wsum[w] = sum;
    __syncthreads();
    if (w != 0) return;
    sum = wsum[0];
#pragma unroll
    for (int q = 1; q < W; q++) sum += wsum[q];
  }
  if (lane == 0) C[(uint64_t)b * M * N + e] = sum;
}

// fp64 products on v_mfma_f64_16x16x4_f64: four wave64s per block, WM x WN over the BM x BN tile and
// WK over each step of KW WK k (their sums added in order at the end). Operands are staged through
// LDS as [k][row], one step ahead in registers, zeros outside M, N and K. The instruction takes 64
// cycles; with one staging buffer what bounds a tile is the loads and barriers of its steps, so the
// steps are long (T 512 x 512 x 1024 on 32x32 tiles: 46 us with 16 k a step, 30 with 64). 1024 x 512
// products of K = 512 take 22 us (24.8 of 78.6 TFLOP/s), where a thread per output took 560.
template <int BM, int BN, int WM, int WN, int WK, int KW, bool TA, bool TB>
__global__ void __launch_bounds__(256) k_gemm_f64(const double* __restrict__ A, const double* __restrict__ B, double* __restrict__ C, int M, int N,
                                                  int K, const int64_t* a_off, const int64_t* b_off, uint64_t a_stride, uint64_t b_stride,
                                                  uint32_t tiles_m, uint32_t tiles_n) {
  static_assert(WM * WN * WK == 4, "four waves");
  typedef double doublex4 __attribute__((ext_vector_type(4)));
  constexpr int BK = KW * WK, TM = BM / WM / 16, TN = BN / WN / 16, PA = BM * BK / 256, PB = BN * BK / 256;
  constexpr int LDA = BM + 1, LDB = BN + 1;
  __shared__ double as[BK * LDA], bs[BK * LDB];
  __shared__ double part[WK > 1 ? (WK - 1) * BM * BN : 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lo = lane >> 4;
  const int wk = wave / (WM * WN), wm = wave / WN % WM, wn = wave % WN;
  const TileIndex ti = tile_of(blockIdx.x, gridDim.x, tiles_m, tiles_n);
  const int m0 = ti.tm * BM, n0 = ti.tn * BN;
  const double* a = A + batch_offset(a_off, a_stride, ti.z);
  const double* b = B + batch_offset(b_off, b_stride, ti.z);
  double va[PA], vb[PB];
  // Element e of a step: along k where the operand is K-contiguous, along its rows otherwise.
  auto load = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < PA; q++) {
      const int e = q * 256 + tid, r = TA ? e % BM : e / BK, k = k0 + (TA ? e / BM : e % BK), row = m0 + r;
      const bool ok = row < M && k < K;
      const double x = a[ok ? (TA ? (int64_t)k * M + row : (int64_t)row * K + k) : 0];
      va[q] = ok ? x : 0.0;
    }
#pragma unroll
    for (int q = 0; q < PB; q++) {
      const int e = q * 256 + tid, r = TB ? e / BK : e % BN, k = k0 + (TB ? e % BK : e / BN), col = n0 + r;
      const bool ok = col < N && k < K;
      const double x = b[ok ? (TB ? (int64_t)col * K + k : (int64_t)k * N + col) : 0];
      vb[q] = ok ? x : 0.0;
    }
  };
  auto store = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < PA; q++) {
      const int e = q * 256 + tid;
      as[(TA ? e / BM : e % BK) * LDA + (TA ? e % BM : e / BK)] = va[q];
    }
#pragma unroll
    for (int q = 0; q < PB; q++) {
      const int e = q * 256 + tid;
      bs[(TB ? e % BK : e / BN) * LDB + (TB ? e / BK : e % BN)] = vb[q];
    }
  };
  doublex4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int n = 0; n < TN; n++) acc[i][n] = doublex4{0.0, 0.0, 0.0, 0.0};
  load(0);
  store();
  __syncthreads();
  for (int k0 = 0; k0 < K; k0 += BK) {
    if (k0 + BK < K) load(k0 + BK);
#pragma unroll
    for (int kk = 0; kk < KW; kk += 4) {
      const int k = wk * KW + kk + lo;
      double x[TM], y[TN];
#pragma unroll
      for (int i = 0; i < TM; i++) x[i] = as[k * LDA + (wm * TM + i) * 16 + li];
#pragma unroll
      for (int n = 0; n < TN; n++) y[n] = bs[k * LDB + (wn * TN + n) * 16 + li];
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int n = 0; n < TN; n++) acc[i][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i], y[n], acc[i][n], 0, 0, 0);
    }
    __syncthreads();
    if (k0 + BK < K) {
      store();
      __syncthreads();
    }
  }
  // Register r of lane l holds row 4 r + l / 16, column l % 16 of its 16x16 tile.
  if constexpr (WK > 1) {
    if (wk > 0)
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int n = 0; n < TN; n++)
#pragma unroll
          for (int r = 0; r < 4; r++) part[((wk - 1) * BM + i * 16 + 4 * r + lo) * BN + n * 16 + li] = acc[i][n][r];
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int n = 0; n < TN; n++)
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
          for (int q = 0; q < WK - 1; q++) acc[i][n][r] += part[(q * BM + i * 16 + 4 * r + lo) * BN + n * 16 + li];
  }
  double* c = C + (uint64_t)ti.z * M * N;
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int n = 0; n < TN; n++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int row = m0 + (wm * TM + i) * 16 + 4 * r + lo, col = n0 + (wn * TN + n) * 16 + li;
        if (row < M && col < N) c[(uint64_t)row * N + col] = acc[i][n][r];
      }
}

// ---- skinny fp32 products: HBM-bound shapes streamed at full bandwidth -------------------------
//
// Products with at most 16 rows and a long K (a few vectors against a large matrix), or with a
// K of at most 16 (outer products), do about 4 flops per byte they move: the matrix cores cannot
// speed them up, the number of bytes in flight can. Each kernel reads its large operand exactly
// once with 16-byte loads and fixes the order of every sum, so results are deterministic.

// A lane's four columns of these kernels start at a multiple of four, the last ones moved back to
// N - 4 where N is no multiple of four: the columns two lanes then share get the same sums from both.
// Rows need only 4-byte alignment (rowx4).

// C (M <= MR rows) = op(A) B with B row-major K x N (N >= 4). A block of
// four waves owns 256 columns (a float4 per lane) and one K split; its waves take consecutive
// quarters of the split and combine in wave order through LDS. With several splits, split s writes
// partials [s][M N], summed in split order afterwards. Rows m >= M read row M - 1 and are not stored.
// Bound by the latency of its loads (a wave or two per SIMD): B's next eight rows are loaded while
// these are multiplied, and op(A)'s values of 64 k go through the wave's own part of LDS. (Read as
// scalars, one load each, they took longer than B: 16 x 4096 x 4096 35 us, 25.6 here; 8 x 1024 x 4096
// 16.8 and 14.6.) The products of 16 k are summed by themselves and then added, so that a wave's sum
// meets one rounding of its own size per 16 k: 1.2e-7 against 64-bit sums at K = 4096, 1.7e-7 when
// each was added to it.
__device__ __forceinline__ float4 row4(const float* p) {
  const rowx4 x = *(const rowx4*)p;
  return make_float4(x[0], x[1], x[2], x[3]);
}
// The first `left` of four values, zeros after them.
__device__ __forceinline__ float4 row4(const float* p, int left) {
  if (left >= 4) return row4(p);
  return make_float4(left > 0 ? p[0] : 0.f, left > 1 ? p[1] : 0.f, left > 2 ? p[2] : 0.f, 0.f);
}

template <int MR>
struct RowsLds {
  static constexpr int SUMS = 3 * MR * 64;  // float4s: the sums of waves 1..3; wave 0 keeps its own
  static constexpr int PANEL = 64 * MR / 4;  // a wave's op(A) values of 64 k; waves 1..3 have theirs where their sums go
  static constexpr int FLOAT4S = SUMS + PANEL;
};

// op(A) of the streaming kernels, read through the constant address space: the launch never
// writes it, and so its wave-uniform loads are scalar loads also where the block code runs inside
// a grouped launch, whose operand pointers come from a struct and carry no __restrict__.
typedef const __attribute__((address_space(4))) float* ConstOperand;

// Block (bx, by) of k_gemm_skinny_rows, its wave sums combined through `lds`.
// AHEAD: B's next eight rows wait in registers of their own (3x2050x8192 35.3 us against 36.3, 8x8192x2048
// 28.3 and 28.8; 154 registers for 8 rows, 120 without).
template <int MR, bool AHEAD = true>
__device__ __forceinline__ void skinny_rows_block(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ out, int M,
                                                  int N, int K, bool ta, int kps, uint32_t bx, uint32_t by, float4* lds) {
  float4(*red)[MR][64] = (float4(*)[MR][64])lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  float4(*panel)[MR / 4] = (float4(*)[MR / 4])(wave == 0 ? lds + RowsLds<MR>::SUMS : &red[wave - 1][0][0]);
  const int col = (bx * 64 + lane) * 4;
  const int colr = min(col, N - 4);
  const int k0 = by * kps, k1 = min(K, k0 + kps);
  const int quarter = (k1 - k0 + 3) / 4;
  const int kw0 = min(k1, k0 + wave * quarter), kw1 = min(k1, kw0 + quarter);
  const uint64_t sm = ta ? 1 : (uint64_t)K, sk = ta ? (uint64_t)M : 1;  // op(A)[m][k] = A[m * sm + k * sk]
  float4 acc[MR], run[MR];
#pragma unroll
  for (int m = 0; m < MR; m++) acc[m] = run[m] = make_float4(0.f, 0.f, 0.f, 0.f);
  // The wave's op(A) values of 64 k from kc on, a k to a lane.
  auto stage = [&](int kc) __attribute__((always_inline)) {
    const int k = min(kc + lane, kw1 - 1);
    float a[MR];
#pragma unroll
    for (int m = 0; m < MR; m++) a[m] = A[(uint64_t)min(m, M - 1) * sm + (uint64_t)k * sk];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < MR / 4; q++) panel[lane][q] = make_float4(a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  auto load = [&](float4* b, int k) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 8; u++) b[u] = row4(B + (uint64_t)(k + u) * N + colr);
  };
  auto row = [&](int i, const float4& b) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < MR / 4; q++) {
      const float4 t = panel[i][q];
      const float a[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
      for (int m = 0; m < 4; m++) {
        float4& r = run[4 * q + m];
        r = make_float4(fmaf(a[m], b.x, r.x), fmaf(a[m], b.y, r.y), fmaf(a[m], b.z, r.z), fmaf(a[m], b.w, r.w));
      }
    }
  };
  auto add = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < MR; m++) {
      acc[m] = make_float4(acc[m].x + run[m].x, acc[m].y + run[m].y, acc[m].z + run[m].z, acc[m].w + run[m].w);
      run[m] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  const int whole = kw0 + (kw1 - kw0) / 8 * 8;
  float4 b0[8], b1[AHEAD ? 8 : 1];
  if (kw0 < whole) load(b0, kw0);
  int kc = kw0;
  if (kw0 < kw1) stage(kw0);
#pragma unroll 1
  for (int k = kw0; k < whole; k += 16) {
    if (k - kc == 64) stage(kc = k);
    const bool second = k + 8 < whole;
    if constexpr (AHEAD) {
      if (second) load(b1, k + 8);
#pragma unroll
      for (int u = 0; u < 8; u++) row(k - kc + u, b0[u]);
      if (second) {
        if (k + 16 < whole) load(b0, k + 16);
#pragma unroll
        for (int u = 0; u < 8; u++) row(k - kc + 8 + u, b1[u]);
      }
    } else {
#pragma unroll
      for (int u = 0; u < 8; u++) row(k - kc + u, b0[u]);
      if (second) {
        load(b0, k + 8);
#pragma unroll
        for (int u = 0; u < 8; u++) row(k - kc + 8 + u, b0[u]);
      }
      if (k + 16 < whole) load(b0, k + 16);
    }
    add();
  }
  if (whole < kw1) {
    if (whole - kc == 64) stage(kc = whole);
    for (int k = whole; k < kw1; k++) row(k - kc, row4(B + (uint64_t)k * N + colr));
    add();
  }
  if (wave > 0)
#pragma unroll
    for (int m = 0; m < MR; m++) red[wave - 1][m][lane] = acc[m];
  __syncthreads();
  if (wave != 0 || col >= N) return;
  float* dst = out + (uint64_t)by * M * N;
#pragma unroll
  for (int m = 0; m < MR; m++)
    if (m < M) {
      float4 v = acc[m];
#pragma unroll
      for (int w = 0; w < 3; w++) {
        const float4 x = red[w][m][lane];
        v = make_float4(v.x + x.x, v.y + x.y, v.z + x.z, v.w + x.w);
      }
      *(rowx4*)(dst + (uint64_t)m * N + colr) = rowx4{v.x, v.y, v.z, v.w};
    }
}

// C (M <= MR rows) = A B^T with A row-major M x K and B stored N x K (N >= NC): every output is the dot product of two contiguous rows. A block owns
// 4 NC consecutive columns of C (NC per wave) and one K split of `kps` (a multiple of 256, at
// most DOT_KPS); it copies its A panel to LDS while its first B rows load, so the loop's only
// global loads are the B rows, four float4 steps deep. Lanes take k in float4 steps 256 apart, each lane summing its
// share in increasing k, four at a time; the 64 lane sums combine by a fixed xor butterfly, and with several
// splits, split s writes partials [s][M N], summed in split order afterwards. Rows m >= M read
// row M - 1 and are not stored. (For 16 rows the split is at most DOT_KPS / 2.)
constexpr int DOT_KPS = 1024;
template <int MR>
struct DotLds {
  static constexpr int KPS_MAX = MR <= 8 ? DOT_KPS : DOT_KPS / 2;  // a 32 KiB panel either way
  static constexpr int FLOAT4S = MR * KPS_MAX / 4;
};

// Block (bx, by) of a k_gemm_skinny_dot grid of ny splits, its A panel in `lds`.
template <int MR, int NC>
__device__ __forceinline__ void skinny_dot_block(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ out, int M,
                                                 int N, int K, int kps, uint32_t bx, uint32_t by, uint32_t ny, float4* lds) {
  constexpr int KPS_MAX = DotLds<MR>::KPS_MAX;
  float4(*panel)[KPS_MAX / 4] = (float4(*)[KPS_MAX / 4])lds;
  const int lane = threadIdx.x & 63;
  // Blocks side by side take different K chunks (rotated by the column tile), so concurrent
  // blocks read B at addresses spread over the rows rather than one column range of every row.
  const int split = (by + bx) % ny;
  const int k0 = split * kps, len = min(K - k0, kps);
  const int n0 = (bx * 4 + (threadIdx.x >> 6)) * NC;
  const bool active = n0 < N;
  const int nr = min(n0, N - NC);  // an idle wave reads valid rows and stores nothing
  // The first four steps of B rows are issued before the panel copy, so their latency overlaps it.
  auto load = [&](float4 (&b)[4][NC], int kk) {
#pragma unroll
    for (int h = 0; h < 4; h++)
#pragma unroll
      for (int c = 0; c < NC; c++)
        b[h][c] = row4(B + (uint64_t)(nr + c) * K + k0 + kk + h * 256, len - kk - h * 256);
  };
  float4 b[4][NC];
  load(b, lane * 4);
  const int len4 = (len + 3) / 4;
  for (int q = threadIdx.x; q < MR * len4; q += 256) {
    const int m = q / len4, c = q % len4;
    panel[m][c] = row4(A + (uint64_t)min(m, M - 1) * K + k0 + 4 * c, len - 4 * c);
  }
  __syncthreads();
  if (!active) return;
  float acc[MR][NC];
#pragma unroll
  for (int m = 0; m < MR; m++)
#pragma unroll
    for (int c = 0; c < NC; c++) acc[m][c] = 0.f;
  for (int kk = lane * 4; kk < len; kk += 1024) {
#pragma unroll
    for (int h = 0; h < 4; h++)
      if (kk + h * 256 < len)
#pragma unroll
        for (int m = 0; m < MR; m++) {
          const float4 a = panel[m][(kk + h * 256) / 4];
#pragma unroll
          for (int c = 0; c < NC; c++)
            acc[m][c] += fmaf(a.w, b[h][c].w, fmaf(a.z, b[h][c].z, fmaf(a.y, b[h][c].y, a.x * b[h][c].x)));
        }
    if (kk + 1024 < len) load(b, kk + 1024);
  }
  float* dst = out + (uint64_t)split * M * N;
#pragma unroll
  for (int m = 0; m < MR; m++)
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const float v = rg_wave_sum(acc[m][c]);
      if (m < M && lane == 0) dst[(uint64_t)m * N + nr + c] = v;
    }
}

// C (M x N, N >= 4) = op(A) op(B) with K <= KR (an outer product of a few vectors): write
// bound. A block of four waves owns 256 columns; each lane keeps its float4 of every op(B) row in
// registers and walks the wave's rows, reading op(A)'s row values as wave-uniform scalars. The
// output is written with non-temporal stores: it is large (a full matrix from a few vectors) and
// streaming it past the caches leaves them to the operands of the kernels that follow (4 % off a
// C5 pass on MI355X).
// Block (bx, by) of k_gemm_outer.
template <int KR, bool TA, bool TB>
__device__ __forceinline__ void outer_block(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C, int M, int N,
                                            int K, int rows_per_wave, uint32_t bx, uint32_t by) {
  const ConstOperand Ac = (ConstOperand)A;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if ((bx * 64 + lane) * 4 >= N) return;
  const int col = min((int)(bx * 64 + lane) * 4, N - 4);
  // Rows k >= K are zeros: the extra terms add exact zeros, so the sums are unchanged.
  float4 b[KR];
#pragma unroll
  for (int k = 0; k < KR; k++) {
    if (k < K) {
      if (TB) b[k] = make_float4(B[(uint64_t)col * K + k], B[(uint64_t)(col + 1) * K + k], B[(uint64_t)(col + 2) * K + k], B[(uint64_t)(col + 3) * K + k]);
      else b[k] = row4(B + (uint64_t)k * N + col);
    } else {
      b[k] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  const int r0 = (by * 4 + wave) * rows_per_wave, r1 = min(M, r0 + rows_per_wave);
  for (int i = r0; i < r1; i++) {
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int k = 0; k < KR; k++) {
      const float a = k < K ? (TA ? Ac[(uint64_t)k * M + i] : Ac[(uint64_t)i * K + k]) : 0.f;
      acc = make_float4(fmaf(a, b[k].x, acc.x), fmaf(a, b[k].y, acc.y), fmaf(a, b[k].z, acc.z), fmaf(a, b[k].w, acc.w));
    }
    __builtin_nontemporal_store(rowx4{acc.x, acc.y, acc.z, acc.w}, (rowx4*)(C + (uint64_t)i * N + col));
  }
}

template <int MR>
__global__ void __launch_bounds__(256) k_gemm_skinny_rows(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ out,
                                                          int M, int N, int K, bool ta, int kps) {
  __shared__ float4 lds[RowsLds<MR>::FLOAT4S];
  skinny_rows_block<MR>(A, B, out, M, N, K, ta, kps, blockIdx.x, blockIdx.y, lds);
}

template <int MR, int NC>
__global__ void __launch_bounds__(256) k_gemm_skinny_dot(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ out,
                                                         int M, int N, int K, int kps) {
  __shared__ float4 lds[DotLds<MR>::FLOAT4S];
  skinny_dot_block<MR, NC>(A, B, out, M, N, K, kps, blockIdx.x, blockIdx.y, gridDim.y, lds);
}

template <int KR, bool TA, bool TB>
__global__ void __launch_bounds__(256) k_gemm_outer(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C, int M,
                                                    int N, int K, int rows_per_wave) {
  outer_block<KR, TA, TB>(A, B, C, M, N, K, rows_per_wave, blockIdx.x, blockIdx.y);
}

// One streamed product's share of a grouped launch (k_stream_group): which kernel's block code it
// runs, its arguments (`arg`: K split length of the rows and dot kernels, rows per wave of the
// outer product) and its 2-D grid, gx blocks wide.
// A few outputs with a long K (at most 16384 outputs): one block of W waves per output, its
// threads taking k 64 W apart in increasing order (eight loads of each operand in flight), each
// wave's sum by a fixed butterfly, and the W wave sums added in wave order. Any flags, any
// alignment.
//
// Output e of k_gemm_tiny_out<W>, computed by 64 W / V threads: thread t also runs threads
// t + 64 W / V, t + 128 W / V, ... of the W-wave block (V of them in all), with the same loads,
// sums and order, so that a grouped launch of 256-thread blocks gives the single kernel's bits.
template <int W, int V>
__device__ __forceinline__ void tiny_block(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C, int M, int N,
                                           int K, bool ta, bool tb, uint32_t e, float* wsum) {
  constexpr int NT = 64 * W, RT = NT / V;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = e / N, j = e % N;
  float sum[V];
#pragma unroll
  for (int v = 0; v < V; v++) {
    float acc = 0.f;
    int k = threadIdx.x + v * RT;
    for (; k + 7 * NT < K; k += 8 * NT) {
      float a[8], b[8];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const uint64_t kk = (uint64_t)(k + u * NT);
        a[u] = ta ? A[kk * M + i] : A[(uint64_t)i * K + kk];
        b[u] = tb ? B[(uint64_t)j * K + kk] : B[kk * N + j];
      }
#pragma unroll
      for (int u = 0; u < 8; u++) acc = fmaf(a[u], b[u], acc);
    }
    for (; k < K; k += NT) {
      const float a = ta ? A[(uint64_t)k * M + i] : A[(uint64_t)i * K + k];
      const float b = tb ? B[(uint64_t)j * K + k] : B[(uint64_t)k * N + j];
      acc = fmaf(a, b, acc);
    }
    sum[v] = rg_wave_sum(acc);
  }
  if (W == 1) {
    if (lane == 0) C[e] = sum[0];
    return;
  }
  if (lane == 0)
#pragma unroll
    for (int v = 0; v < V; v++) wsum[w + v * (W / V)] = sum[v];
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = wsum[0];
#pragma unroll
    for (int q = 1; q < W; q++) t += wsum[q];
    C[e] = t;
  }
}

template <int W>
__global__ void __launch_bounds__(64 * W) k_gemm_tiny_out(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C, int M,
                                                          int N, int K, bool ta, bool tb) {
  __shared__ float wsum[W];
  tiny_block<W, 1>(A, B, C, M, N, K, ta, tb, blockIdx.x, wsum);
}

enum StreamKind { STREAM_ROWS8 = 0, STREAM_DOT8, STREAM_OUTER8_TN, STREAM_OUTER8_NT, STREAM_OUTER8_NN, STREAM_TINY4, STREAM_TINY8, STREAM_TINY16 };
struct StreamPart {
  const float *a, *b;
  float* out;
  int m, n, k, arg, kind;
  bool ta, tb;
  uint32_t gx, gy, blocks;
};
struct StreamParts {
  StreamPart p[3];
};

__device__ __forceinline__ void stream_part(const StreamPart& p, uint32_t bid, float4* lds) {
  const uint32_t bx = bid % p.gx, by = bid / p.gx;
  switch (p.kind) {
    case STREAM_ROWS8: skinny_rows_block<8, false>(p.a, p.b, p.out, p.m, p.n, p.k, p.ta, p.arg, bx, by, lds); break;
    case STREAM_DOT8: skinny_dot_block<8, 4>(p.a, p.b, p.out, p.m, p.n, p.k, p.arg, bx, by, p.gy, lds); break;
    case STREAM_OUTER8_TN: outer_block<8, true, false>(p.a, p.b, p.out, p.m, p.n, p.k, p.arg, bx, by); break;
    case STREAM_OUTER8_NT: outer_block<8, false, true>(p.a, p.b, p.out, p.m, p.n, p.k, p.arg, bx, by); break;
    case STREAM_TINY4: tiny_block<4, 1>(p.a, p.b, p.out, p.m, p.n, p.k, p.ta, p.tb, bid, (float*)lds); break;
    case STREAM_TINY8: tiny_block<8, 2>(p.a, p.b, p.out, p.m, p.n, p.k, p.ta, p.tb, bid, (float*)lds); break;
    case STREAM_TINY16: tiny_block<16, 4>(p.a, p.b, p.out, p.m, p.n, p.k, p.ta, p.tb, bid, (float*)lds); break;
    default: outer_block<8, false, false>(p.a, p.b, p.out, p.m, p.n, p.k, p.arg, bx, by); break;
  }
}

// Up to three independent streamed products of at most 8 rows (or K at most 8), or of a few
// outputs with a long K, in one launch: part i takes the next p[i].blocks blocks and runs its own
// kernel's block code, with one LDS buffer. The reads of one product and the writes of another share HBM in the same launch, and
// the launch's fixed cost is paid once.
// At most 128 registers, four waves per SIMD: the row kernel's blocks load B's next rows into the
// registers of the last ones, the same sums (the chain of 4096 x 4096 by 8 rows, three such launches a
// pass: 71.5 us, 75.0 with rows loaded ahead at 156 registers).
__global__ void __launch_bounds__(256, 4) k_stream_group(StreamParts g) {
  constexpr int F = RowsLds<8>::FLOAT4S > DotLds<8>::FLOAT4S ? RowsLds<8>::FLOAT4S : DotLds<8>::FLOAT4S;
  __shared__ float4 lds[F];
  uint32_t bid = blockIdx.x;
  if (bid < g.p[0].blocks) return stream_part(g.p[0], bid, lds);
  bid -= g.p[0].blocks;
  if (bid < g.p[1].blocks) return stream_part(g.p[1], bid, lds);
  stream_part(g.p[2], bid - g.p[1].blocks, lds);
}

enum SkinnyKind { SKINNY_NONE = 0, SKINNY_ROWS, SKINNY_DOT, SKINNY_OUTER, SKINNY_TINY };

// A skinny product as one of the kernels sees it. A matrix-vector product (n == 1) is run as its
// transpose, C^T = op(B)^T op(A)^T: with one column, C and C^T are the same memory, and the
// streamed matrix becomes the kernels' right operand.
struct Skinny {
  SkinnyKind kind = SKINNY_NONE;
  bool swapped = false;  // roles of A and B exchanged (n == 1)
  uint64_t m = 0, n = 0, k = 0;
  bool ta = false;
};

// fp32 products on matrix cores: both sides at least 32, or at least 16 at a K under 512 (attention
// heads of 16 or 24). With a longer K, 16 columns or rows stream, and sides of 17 to 31 take a block per
// output (k_gemm_tiny_out) up to 16384 outputs and a thread per output above.
bool use_mfma(int dtype, uint64_t m, uint64_t n, uint64_t k) {
  const uint64_t side = k < 512 ? 16 : 32;
  return dtype == RG_F32 && m >= side && n >= side && k >= 8 && m * n * k >= (1u << 18);
}

// Products up to which a block per output (k_gemm_tiny_out) is faster than the row kernel, or than
// the dot kernel where each output is a product of two contiguous rows. Its time grows with their
// number, the others' hardly does (us, M x N x K): rows 1x66x513 6 against 15, 8x66x2050 10 and 14,
// 3x515x2050 19 and 18; 16x66x513 6 and 20, 16x515x513 21 and 20; dots 1x2050x4096 9 and 18,
// 3x1001x4096 12 and 14, 8x1001x1000 11 and 10; 16x1001x513 11 and 15, 16x1024x2050 28 and 16. Its sums are also the more
// exact, the lanes each taking a few k (1x1001x1000: 0.9e-7 against 64-bit sums, rows 1.0e-7).
// A dot product of more than DOT_KPS takes a second launch.
uint64_t tiny_products(uint64_t rows, uint64_t k, bool dots) {
  if (dots) return rows <= 8 && k <= DOT_KPS ? 8u << 20 : 12u << 20;
  return rows <= 8 ? 2u << 20 : 4u << 20;
}

// Which skinny kernel a product takes, from shapes and flags alone. Every size goes: a chain of
// 8 x 2050 x 2050 products on the plain kernel instead took 10 times as long.
Skinny skinny_plan(int dtype, uint64_t m, uint64_t n, uint64_t k, uint64_t batch, bool ta, bool tb) {
  Skinny sk;
  if (dtype != RG_F32 || batch != 1 || m == 0 || n == 0 || k == 0) return sk;
  sk.m = m;
  sk.n = n;
  sk.k = k;
  sk.ta = ta;
  if (k <= 16 && n >= 4 && m * n >= (1ull << 14)) {
    sk.kind = SKINNY_OUTER;
    return sk;
  }
  // Few enough products for a block per output (skinny_plan's last rule) to take them all in the
  // time the row and dot kernels take to start up (us on MI355X).
  const bool tiny = m * n <= 16384 && k >= 512 && m * n * k <= tiny_products(std::min(m, n), k, n == 1 ? !ta : tb);
  if (m <= 16 && k >= 512 && n >= 64 && !tiny) {
    if (!tb) sk.kind = SKINNY_ROWS;
    else if (!ta) sk.kind = SKINNY_DOT;
    if (sk.kind != SKINNY_NONE) return sk;
  }
  if (n == 1 && k >= 512 && m >= 64 && !tiny) {
    // op(A) x with A stored K x M (ta): rows kernel over A; stored M x K: dot kernel over A's rows.
    sk.swapped = true;
    sk.m = 1;
    sk.n = m;
    sk.ta = false;
    sk.kind = ta ? SKINNY_ROWS : SKINNY_DOT;
    return sk;
  }
  // Outputs with both sides at least 32 (a tied embedding's gradient, 96 x 128 over 4096 rows)
  // go to the MFMA tiles, which read both operands in coalesced tiles.
  if (m * n <= 16384 && k >= 512 && !use_mfma(dtype, m, n, k)) {
    sk = Skinny{};
    sk.kind = SKINNY_TINY;
    sk.m = m;
    sk.n = n;
    sk.k = k;
    sk.ta = ta;
  }
  return sk;
}

// K split length of SKINNY_DOT: the whole K in chunks of at most DOT_KPS (1024, or 512 for 16
// rows, whose panel would not fit), each a multiple of 256.
int skinny_dot_kps(uint64_t m, uint64_t k) {
  const uint64_t cap = m <= 8 ? DOT_KPS : DOT_KPS / 2;
  const uint64_t splits = (k + cap - 1) / cap;
  return (int)(((k + splits - 1) / splits + 255) / 256 * 256);
}

// K splits of SKINNY_ROWS: about 1024 waves, each at least 64 rows of K deep, at most 16.
int skinny_rows_splits(uint64_t n, uint64_t k) {
  const uint64_t blocks = (n + 255) / 256;
  uint64_t want = (256 + blocks - 1) / blocks;
  const uint64_t most = std::max<uint64_t>(1, k / 256);
  return (int)std::max<uint64_t>(1, std::min<uint64_t>(std::min(want, most), 16));
}

struct TileCfg {
  int bm, bn, bk, wm, wn;
  int split;  // steps in LDS of the bf16 terms' tile (gemm_split.h); 0: fp32 MFMA (gemm_mfma.h)
};
constexpr TileCfg SPLIT_128x128 = {128, 128, SPLIT_BK, 2, 4, 1}, SPLIT_128x128_2 = {128, 128, SPLIT_BK, 2, 4, 2},
                  SPLIT_128x64 = {128, 64, SPLIT_BK, 2, 2, 1}, SPLIT_64x64 = {64, 64, SPLIT_BK, 2, 2, 2};

uint64_t tile_count(const TileCfg& t, uint64_t m, uint64_t n, uint64_t batch) { return ((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn) * batch; }

// K splits for products with too few tiles: about 512 blocks of 128x128 (two per CU), 768 of the
// smaller tiles, each split at least 512 deep, at most 16.
int split_count(const TileCfg& t, uint64_t m, uint64_t n, uint64_t k, uint64_t batch) {
  uint64_t tiles = tile_count(t, m, n, batch);
  if (tiles >= 256 || k < 1024) return 1;
  uint64_t target = t.bm * t.bn >= 128 * 128 ? 512 : 768;
  uint64_t want = (target + tiles - 1) / tiles;
  uint64_t most = k / 512;
  return (int)std::max<uint64_t>(1, std::min<uint64_t>(std::min(want, most), 16));
}

// Block tile, from measurements on MI355X (us; M x N x K, T: that operand transposed).
// Products whose 64x64 tiles, split over K where K allows, come to a block per CU run on the bf16
// terms:
//  - 128x128 at two blocks per CU (4096x2048x2048: 179 against 214 on 128x64; 8192x1024x256: 26.9
//    and 30.7), or a K of 2048 and more whose splits give most CUs a block, then with two steps in
//    LDS (T 256x1024x8192: 29.4 against 33.1 with one and 35.6 on 64x64; T 2048x2048x4096: 200
//    against 232 and 252);
//  - 128x64 at three blocks per CU (8192x768x256: 24.4 against 27.4 on 64x64);
//  - 64x64 otherwise (8192x256x1024: 35.7 against 41 on 128x64; 8192x256x256: 11.5 and 12.9).
// Below that a block runs alone on its CU and fp32 MFMA tiles are faster: 32-wide ones for outputs
// 32..96 wide or 32 tall (attention heads, the vocabulary), 32x32 otherwise (256x768x256: 4.3
// against 7.1 on bf16 terms; 4096x128x512: 8.6 and 13), or 64x64 where a side under 64 keeps a
// large output off the tiles above. (Figures of single launches before the operands were scaled, which
// adds up to 4 % to each of the bf16 tiles alike.)
TileCfg pick_tile(uint64_t m, uint64_t n, uint64_t k, uint64_t batch) {
  auto filled = [&](const TileCfg& t) { return tile_count(t, m, n, batch) * (uint64_t)split_count(t, m, n, k, batch); };
  // A column-contiguous operand's offsets within 24 rows are 32-bit: sides of less than 2^25.
  if (m >= 64 && n >= 64 && m < (1u << 25) && n < (1u << 25) && filled(SPLIT_64x64) >= 256) {
    if (m >= 128 && n >= 128) {
      const uint64_t blocks = filled(SPLIT_128x128);
      if (tile_count(SPLIT_128x128, m, n, batch) >= 512 || (k >= 2048 && blocks > 256)) return SPLIT_128x128;
      if (k >= 2048 && blocks >= 192) return SPLIT_128x128_2;
    }
    if (m >= 128 && tile_count(SPLIT_128x64, m, n, batch) >= 768) return SPLIT_128x64;
    return SPLIT_64x64;
  }
  if ((n <= 96 && n % 32 == 0) || n < 32) return {128, 32, 32, 4, 1, 0};
  if (m <= 32) return {32, 128, 32, 1, 4, 0};
  const TileCfg t64 = {64, 64, 32, 2, 2, 0};
  return filled(t64) < 256 ? TileCfg{32, 32, 32, 2, 2, 0} : t64;
}

struct Launch {
  dim3 grid;
  const float *a, *b;
  float* c;
  int m, n, k;
  const int64_t *a_off, *b_off;
  uint64_t as, bs;
  int splits, kps;
  float* part;
  const float* bias;
  uint32_t tm, tn;
};

// `mode`: the fp32 tile's load mode, or whether some K range of the split tile is no multiple of 32.
template <int BM, int BN, int WM, int WN, bool TA, bool TB, int U>
void launch_mode(hipStream_t s, int mode, const Launch& l) {
  const dim3 block(64 * WM * WN);
  if constexpr (U > 0) {
#define RG_GEMM(TAIL_)                                                                                                              \
  hipLaunchKernelGGL((k_gemm_mfma<BM, BN, WM, WN, U, TA, TB, TAIL_>), l.grid, block, 0, s, l.a, l.b, l.c, l.m, l.n, l.k, l.a_off, l.b_off, \
                     l.as, l.bs, l.splits, l.kps, l.part, l.bias, l.tm, l.tn)
    if (mode) RG_GEMM(true);
    else RG_GEMM(false);
#undef RG_GEMM
  } else {
#define RG_GEMM(MODE_)                                                                                                                \
  hipLaunchKernelGGL((k_gemm_f32<BM, BN, 32, WM, WN, TA, TB, MODE_>), l.grid, block, 0, s, l.a, l.b, l.c, l.m, l.n, l.k, l.a_off, l.b_off, \
                     l.as, l.bs, l.splits, l.kps, l.part, l.bias, l.tm, l.tn)
    if (mode == LOAD_EVEN) RG_GEMM(LOAD_EVEN);
    else if (mode == LOAD_VEC) RG_GEMM(LOAD_VEC);
    else RG_GEMM(LOAD_SCALAR);
#undef RG_GEMM
  }
}

template <int BM, int BN, int WM, int WN, int U>
void launch_flags(hipStream_t s, bool ta, bool tb, int mode, const Launch& l) {
  if (!ta && !tb) launch_mode<BM, BN, WM, WN, false, false, U>(s, mode, l);
  else if (ta && !tb) launch_mode<BM, BN, WM, WN, true, false, U>(s, mode, l);
  else if (!ta && tb) launch_mode<BM, BN, WM, WN, false, true, U>(s, mode, l);
  else launch_mode<BM, BN, WM, WN, true, true, U>(s, mode, l);
}

// Instantiates the tile shapes pick_tile can return.
void launch_mfma(hipStream_t s, const TileCfg& t, bool ta, bool tb, int mode, const Launch& l) {
#define RG_TILE(BM_, BN_, WM_, WN_, U_)                                                    \
  if (t.bm == BM_ && t.bn == BN_ && t.wm == WM_ && t.wn == WN_ && t.bk == 32 && t.split == U_) \
  return launch_flags<BM_, BN_, WM_, WN_, U_>(s, ta, tb, mode, l)
  RG_TILE(128, 128, 2, 4, 1);
  RG_TILE(128, 128, 2, 4, 2);
  RG_TILE(128, 64, 2, 2, 1);
  RG_TILE(64, 64, 2, 2, 2);
  RG_TILE(64, 64, 2, 2, 0);
  RG_TILE(128, 32, 4, 1, 0);
  RG_TILE(32, 128, 1, 4, 0);
  RG_TILE(32, 32, 2, 2, 0);
#undef RG_TILE
  throw std::runtime_error("product tile without a kernel");
}

}  // namespace

// Products priced by bytes: the streamed ones, but for dot products over a K that is no multiple of
// 256, whose price stays the operations'.
bool gemm_streamed(int dtype, uint64_t m, uint64_t n, uint64_t k, uint64_t batch, bool ta, bool tb) {
  const Skinny sk = skinny_plan(dtype, m, n, k, batch, ta, tb);
  return sk.kind != SKINNY_NONE && !(sk.kind == SKINNY_DOT && k % 256 != 0);
}

bool gemm_on_bf16_terms(int dtype, uint64_t m, uint64_t n, uint64_t k, uint64_t batch, bool ta, bool tb) {
  return skinny_plan(dtype, m, n, k, batch, ta, tb).kind == SKINNY_NONE && use_mfma(dtype, m, n, k) && pick_tile(m, n, k, batch).split != 0;
}

int gemm_splits(int dtype, uint64_t m, uint64_t n, uint64_t k, uint64_t batch, bool ta, bool tb) {
  if (m == 0 || n == 0 || batch == 0) return 1;
  const Skinny sk = skinny_plan(dtype, m, n, k, batch, ta, tb);
  if (sk.kind == SKINNY_ROWS) {
    const int splits = skinny_rows_splits(sk.n, sk.k);
    const uint64_t kps = (sk.k + splits - 1) / splits;
    return (int)((sk.k + kps - 1) / kps);
  }
  if (sk.kind == SKINNY_DOT) {
    const uint64_t kps = (uint64_t)skinny_dot_kps(sk.m, sk.k);
    return (int)((sk.k + kps - 1) / kps);
  }
  if (sk.kind != SKINNY_NONE || !use_mfma(dtype, m, n, k)) return 1;
  TileCfg t = pick_tile(m, n, k, batch);
  int splits = split_count(t, m, n, k, batch);
  uint64_t kps = ((k + splits - 1) / splits + t.bk - 1) / t.bk * t.bk;
  return (int)((k + kps - 1) / kps);
}

bool gemm_outer_product(uint64_t m, uint64_t n, uint64_t k, bool ta, bool tb) {
  return skinny_plan(RG_F32, m, n, k, 1, ta, tb).kind == SKINNY_OUTER;
}

bool gemm_epilogue_tile(int dtype, uint64_t m, uint64_t n, uint64_t k, bool ta, bool tb, GemmTile* out) {
  if (m == 0 || n == 0 || m >= (1ull << 31) || n >= (1ull << 31) || k >= (1ull << 31)) return false;
  if (skinny_plan(dtype, m, n, k, 1, ta, tb).kind != SKINNY_NONE || !use_mfma(dtype, m, n, k)) return false;
  TileCfg t = pick_tile(m, n, k, 1);
  if (!t.split || split_count(t, m, n, k, 1) != 1) return false;
  // The epilogue's loads and stores are aligned vectors of four columns.
  if (n % 4 != 0) return false;
  *out = GemmTile{t.bm, t.bn, t.wm, t.wn, t.split, k % SPLIT_BK != 0, m % t.bm == 0 && n % t.bn == 0,
                  (int)((k + t.bk - 1) / t.bk * t.bk), (uint32_t)((m + t.bm - 1) / t.bm), (uint32_t)((n + t.bn - 1) / t.bn)};
  return true;
}

uint64_t gemm_workspace(int dtype, uint64_t m, uint64_t n, uint64_t k, uint64_t batch, bool ta, bool tb) {
  int s = gemm_splits(dtype, m, n, k, batch, ta, tb);
  return s > 1 ? (uint64_t)s * batch * m * n * sizeof(float) : 0;
}

// Launches the skinny kernel of `sk`; false for a product with a bias.
bool gemm_skinny(hipStream_t s, const GemmArgs& g, const Skinny& sk) {
  if (g.bias || g.a_off || g.b_off) return false;
  // With the roles exchanged (n == 1) the vector is the left operand of one row.
  const float* A = (const float*)(sk.swapped ? g.b : g.a);
  const float* B = (const float*)(sk.swapped ? g.a : g.b);
  float* C = (float*)g.c;
  const int M = (int)sk.m, N = (int)sk.n, K = (int)sk.k;
  const SkinnyKind kind = sk.kind;
  if (g.defer_split && (kind == SKINNY_TINY || kind == SKINNY_OUTER))
    throw std::runtime_error("deferred K-split product on a kernel that does not split K");
  if (kind == SKINNY_TINY) {
    // Waves per output: enough that each thread's share of K is one batch of eight loads.
    const dim3 grid((uint32_t)(M * N));
    const int w = std::min(16, std::max(1, (K + 511) / 512));
    if (w <= 1) hipLaunchKernelGGL(k_gemm_tiny_out<1>, grid, dim3(64), 0, s, A, B, C, M, N, K, g.ta, g.tb);
    else if (w <= 2) hipLaunchKernelGGL(k_gemm_tiny_out<2>, grid, dim3(128), 0, s, A, B, C, M, N, K, g.ta, g.tb);
    else if (w <= 4) hipLaunchKernelGGL(k_gemm_tiny_out<4>, grid, dim3(256), 0, s, A, B, C, M, N, K, g.ta, g.tb);
    else if (w <= 8) hipLaunchKernelGGL(k_gemm_tiny_out<8>, grid, dim3(512), 0, s, A, B, C, M, N, K, g.ta, g.tb);
    else hipLaunchKernelGGL(k_gemm_tiny_out<16>, grid, dim3(1024), 0, s, A, B, C, M, N, K, g.ta, g.tb);
    return true;
  }
  if (kind == SKINNY_OUTER) {
    // 16 rows per wave for tall outputs; fewer for short ones, so more waves share the work.
    const int rows = std::max(1, std::min(16, M / 256));
    dim3 grid((uint32_t)((N + 255) / 256), (uint32_t)((M + 4 * rows - 1) / (4 * rows)));
#define RG_OUTER_K(KR_, TA_, TB_) hipLaunchKernelGGL((k_gemm_outer<KR_, TA_, TB_>), grid, dim3(256), 0, s, A, B, C, M, N, K, rows)
#define RG_OUTER(TA_, TB_)                   \
  do {                                       \
    if (K <= 1) RG_OUTER_K(1, TA_, TB_);     \
    else if (K <= 4) RG_OUTER_K(4, TA_, TB_); \
    else if (K <= 8) RG_OUTER_K(8, TA_, TB_); \
    else RG_OUTER_K(16, TA_, TB_);           \
  } while (0)
    if (g.ta && g.tb) RG_OUTER(true, true);
    else if (g.ta) RG_OUTER(true, false);
    else if (g.tb) RG_OUTER(false, true);
    else RG_OUTER(false, false);
#undef RG_OUTER
#undef RG_OUTER_K
    return true;
  }
  // Both K-split kernels leave split s's partials at [s][M N] of the workspace; the split sum (or
  // the deferred fold_wide) adds them in split order.
  auto sum_splits = [&](const float* part, int splits) {
    if (g.defer_split && splits != g.planned_splits)
      throw std::runtime_error("deferred K-split product: " + std::to_string(splits) + " streamed partial products, the fold expects " +
                               std::to_string(g.planned_splits));
    if (splits > 1 && !g.defer_split) {
      const uint64_t mn = g.m * g.n;
      hipLaunchKernelGGL(k_split_sum, dim3((uint32_t)((mn + 1023) / 1024), 1), dim3(256), 0, s, part, C, mn, splits, (const float*)nullptr, g.n);
    }
  };
  if (kind == SKINNY_DOT) {
    constexpr int NC = 4;
    const int kps = skinny_dot_kps(sk.m, sk.k);
    const int splits = (K + kps - 1) / kps;
    float* out = splits > 1 ? (float*)g.workspace : C;
    dim3 grid((uint32_t)((N + 4 * NC - 1) / (4 * NC)), (uint32_t)splits);
    if (M <= 8) hipLaunchKernelGGL((k_gemm_skinny_dot<8, NC>), grid, dim3(256), 0, s, A, B, out, M, N, K, kps);
    else hipLaunchKernelGGL((k_gemm_skinny_dot<16, NC>), grid, dim3(256), 0, s, A, B, out, M, N, K, kps);
    sum_splits(out, splits);
    return true;
  }
  const int splits0 = skinny_rows_splits(sk.n, sk.k);
  const int kps = (K + splits0 - 1) / splits0;
  const int splits = (K + kps - 1) / kps;
  float* out = splits > 1 ? (float*)g.workspace : C;
  dim3 grid((uint32_t)((N + 255) / 256), (uint32_t)splits);
  if (M <= 8) hipLaunchKernelGGL((k_gemm_skinny_rows<8>), grid, dim3(256), 0, s, A, B, out, M, N, K, sk.ta, kps);
  else hipLaunchKernelGGL((k_gemm_skinny_rows<16>), grid, dim3(256), 0, s, A, B, out, M, N, K, sk.ta, kps);
  sum_splits(out, splits);
  return true;
}

namespace {

// The MFMA tile launch of product `g` on tile `t` with `splits` K splits: its load mode and launch arguments.
void mfma_launch(const GemmArgs& g, const TileCfg& t, int splits, int* load_mode, Launch* launch) {
  int kps = (int)(((g.k + splits - 1) / splits + t.bk - 1) / t.bk * t.bk);
  splits = (int)((g.k + kps - 1) / kps);
  if (g.defer_split && splits != g.planned_splits)
    throw std::runtime_error("deferred K-split product: " + std::to_string(splits) + " partial products, the fold expects " +
                             std::to_string(g.planned_splits));
  // 16-byte vector loads need 16-byte aligned operand rows: aligned bases, leading dimensions
  // (K, or M / N for the contiguous-column layouts) and batch offsets that are multiples of 4.
  auto aligned = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  bool vec = aligned(g.a) && aligned(g.b) && g.k % 4 == 0 && (!g.ta || g.m % 4 == 0) && (g.tb || g.n % 4 == 0) &&
             (g.a_off ? g.a_off4 : g.a_stride % 4 == 0) && (g.b_off ? g.b_off4 : g.b_stride % 4 == 0);
  bool even = g.m % t.bm == 0 && g.n % t.bn == 0 && g.k % t.bk == 0 && kps % t.bk == 0;
  int mode = t.split ? (g.k % SPLIT_BK != 0) : !vec ? LOAD_SCALAR : even ? LOAD_EVEN : LOAD_VEC;
  Launch l;
  l.tm = (uint32_t)((g.m + t.bm - 1) / t.bm);
  l.tn = (uint32_t)((g.n + t.bn - 1) / t.bn);
  l.grid = dim3((uint32_t)(l.tm * l.tn * g.batch * splits));
  l.a = (const float*)g.a;
  l.b = (const float*)g.b;
  l.c = (float*)g.c;
  l.m = (int)g.m;
  l.n = (int)g.n;
  l.k = (int)g.k;
  l.a_off = g.a_off;
  l.b_off = g.b_off;
  l.as = g.a_stride;
  l.bs = g.b_stride;
  l.splits = splits;
  l.kps = kps;
  l.part = splits > 1 ? (float*)g.workspace : nullptr;
  l.bias = splits > 1 ? nullptr : (const float*)g.bias;
  *load_mode = mode;
  *launch = l;
}

// Whether product `g` goes to the MFMA tiles (not a streaming kernel, not the plain kernel).
bool on_mfma_tiles(const GemmArgs& g) {
  return g.m && g.n && g.batch && skinny_plan(g.dtype, g.m, g.n, g.k, g.batch, g.ta, g.tb).kind == SKINNY_NONE &&
         use_mfma(g.dtype, g.m, g.n, g.k);
}

}  // namespace

namespace {

// fp64 tiles: 64x64 at a block and a half per CU, 32x32 at one, else 16x16 with the four waves sharing
// each step of K (T 128 x 512 x 1024, 256 such tiles: 14 us, where a 32x32 tile walks that K in 30);
// none that both sides fill by less than half (2048 products of 20 x 20 x 8: 15.3 us on 32x32 tiles,
// 20.7 on 64x64).
// False for sides under 16, which waste the tile.
bool gemm_f64(hipStream_t s, const GemmArgs& g) {
  if (g.m < 16 || g.n < 16 || g.k < 4) return false;
  auto tiles = [&](uint64_t t) { return ((g.m + t - 1) / t) * ((g.n + t - 1) / t) * g.batch; };
  const uint64_t least = std::min(g.m, g.n);
  const int side = tiles(64) >= 384 && least > 32 ? 64 : tiles(32) >= 256 && least > 16 ? 32 : 16;
  if (tiles(side) >= (1ull << 31)) return false;
  const uint32_t tm = (uint32_t)((g.m + side - 1) / side), tn = (uint32_t)((g.n + side - 1) / side);
  const dim3 grid((uint32_t)tiles(side));
#define RG_F64(S_, WM_, WK_, KW_, TA_, TB_)                                                                                                \
  hipLaunchKernelGGL((k_gemm_f64<S_, S_, WM_, WM_, WK_, KW_, TA_, TB_>), grid, dim3(256), 0, s, (const double*)g.a, (const double*)g.b, (double*)g.c, \
                     (int)g.m, (int)g.n, (int)g.k, g.a_off, g.b_off, g.a_stride, g.b_stride, tm, tn)
#define RG_F64_FLAGS(S_, WM_, WK_, KW_)                    \
  do {                                                \
    if (g.ta && g.tb) RG_F64(S_, WM_, WK_, KW_, true, true); \
    else if (g.ta) RG_F64(S_, WM_, WK_, KW_, true, false); \
    else if (g.tb) RG_F64(S_, WM_, WK_, KW_, false, true); \
    else RG_F64(S_, WM_, WK_, KW_, false, false);          \
  } while (0)
  if (side == 64) RG_F64_FLAGS(64, 2, 1, 32);
  else if (side == 32) RG_F64_FLAGS(32, 2, 1, 64);
  else RG_F64_FLAGS(16, 1, 4, 32);
#undef RG_F64_FLAGS
#undef RG_F64
  return true;
}

// Products off the fp32 tiles and the streaming kernels.
template <class T>
void gemm_small(hipStream_t s, const GemmArgs& g) {
  if (std::is_same<T, double>::value && gemm_f64(s, g)) return;
  const uint64_t outputs = g.m * g.n;
  const bool rows = g.n == 1 && !g.ta;  // every output a contiguous row against one vector
  // A wave per output where K gives its lanes work and the outputs alone do not fill the chip.
  // (A launch has fewer than 2^32 threads in x: fewer than 2^24 blocks of four outputs.)
  if (g.k >= 32 && (outputs * g.batch <= 16384 || rows) && (outputs + 3) / 4 < (1ull << 24)) {
    const int w = outputs * g.batch >= 2048 ? 1 : g.k <= 512 ? 1 : g.k <= 2048 ? 4 : 16;
    const dim3 grid((uint32_t)(w == 1 ? (outputs + 3) / 4 : outputs), (uint32_t)g.batch);
#define RG_DOTS(W_)                                                                                                                        \
  hipLaunchKernelGGL((k_gemm_dots<T, W_>), grid, dim3(W_ == 1 ? 256 : 64 * W_), 0, s, (const T*)g.a, (const T*)g.b, (T*)g.c, (uint32_t)g.m, \
                     (uint32_t)g.n, (uint32_t)g.k, g.ta, g.tb, g.a_off, g.b_off, g.a_stride, g.b_stride)
    if (w == 1) RG_DOTS(1);
    else if (w == 4) RG_DOTS(4);
    else RG_DOTS(16);
#undef RG_DOTS
    return;
  }
  hipLaunchKernelGGL(k_gemm_plain<T>, dim3((uint32_t)((outputs + 255) / 256), (uint32_t)g.batch), dim3(256), 0, s, (const T*)g.a, (const T*)g.b,
                     (T*)g.c, (uint32_t)g.m, (uint32_t)g.n, (uint32_t)g.k, g.ta, g.tb, g.a_off, g.b_off, g.a_stride, g.b_stride);
}

}  // namespace

// A product whose K-split partials are deferred to the fold area must leave exactly
// the planned number of partial products there: a launch that would take another path (the
// streaming kernel refusing its operands, another split count) throws instead, and the error is
// latched like any failed launch, rather than letting the fold overwrite C with stale partials.
void gemm(hipStream_t s, const GemmArgs& g) {
  if (g.m == 0 || g.n == 0 || g.batch == 0) return;
  const Skinny sk = skinny_plan(g.dtype, g.m, g.n, g.k, g.batch, g.ta, g.tb);
  if (sk.kind != SKINNY_NONE) {
    if (gemm_skinny(s, g, sk)) return;
    if (g.defer_split) throw std::runtime_error("deferred K-split product: the streaming kernel refused its operands");
  }
  if (use_mfma(g.dtype, g.m, g.n, g.k)) {
    const TileCfg t = pick_tile(g.m, g.n, g.k, g.batch);
    int mode;
    Launch l;
    mfma_launch(g, t, split_count(t, g.m, g.n, g.k, g.batch), &mode, &l);
    const int splits = l.splits;
    launch_mfma(s, t, g.ta, g.tb, mode, l);
    if (splits > 1 && !g.defer_split) {
      uint64_t mn = g.m * g.n;
      hipLaunchKernelGGL(k_split_sum, dim3((uint32_t)((mn + 1023) / 1024), (uint32_t)g.batch), dim3(256), 0, s, (const float*)l.part,
                         (float*)g.c, mn, splits, (const float*)g.bias, g.n);
    }
    return;
  }
  if (g.defer_split) throw std::runtime_error("deferred K-split product on the plain kernel, which does not split K");
  if (g.dtype == RG_F32) gemm_small<float>(s, g);
  else gemm_small<double>(s, g);
  if (g.bias && g.dtype == RG_F32) {
    const uint64_t total = g.m * g.n * g.batch;
    hipLaunchKernelGGL(k_add_bias, dim3((uint32_t)((total + 255) / 256)), dim3(256), 0, s, (float*)g.c, (const float*)g.bias, total, g.n);
  }
}

namespace {

// Product `g` as a part of a grouped streaming launch: the kernel gemm_skinny would launch for
// it, when that is the row, dot or outer-product kernel for at most 8 rows (or K), or the
// tiny-output kernel of 4, 8 or 16 waves, and its K splits, if any,
// deferred to the fold area.
bool stream_part_of(const GemmArgs& g, StreamPart* p) {
  if (g.m == 0 || g.n == 0 || g.batch != 1 || g.bias || g.a_off || g.b_off) return false;
  const Skinny sk = skinny_plan(g.dtype, g.m, g.n, g.k, g.batch, g.ta, g.tb);
  const float* A = (const float*)(sk.swapped ? g.b : g.a);
  const float* B = (const float*)(sk.swapped ? g.a : g.b);
  const int M = (int)sk.m, N = (int)sk.n, K = (int)sk.k;
  auto split_ok = [&](int splits) {
    if (splits > 1 && !g.defer_split) return false;
    return !g.defer_split || splits == g.planned_splits;
  };
  StreamPart q{A, B, (float*)g.c, M, N, K, 0, 0, sk.ta, g.tb, 0, 0, 0};
  if (sk.kind == SKINNY_TINY) {
    // k_gemm_tiny_out of 4, 8 or 16 waves (fewer do not fill a 256-thread block).
    const int w = std::min(16, std::max(1, (K + 511) / 512));
    if (w < 3 || g.defer_split) return false;
    q.kind = w <= 4 ? STREAM_TINY4 : w <= 8 ? STREAM_TINY8 : STREAM_TINY16;
    q.ta = g.ta;
    q.gx = (uint32_t)(M * N);
    q.gy = 1;
  } else if (sk.kind == SKINNY_OUTER) {
    if (K > 8 || (g.ta && g.tb) || g.defer_split) return false;
    q.kind = g.ta ? STREAM_OUTER8_TN : g.tb ? STREAM_OUTER8_NT : STREAM_OUTER8_NN;
    // Half the single kernel's rows per wave, so twice its blocks: 8 rows for C5's 4096-row
    // outputs measured 3 us (4 %) faster per pass on MI355X than 16, and 6 alike, 4 or 32 slower.
    // Each output is one sum either way, so the results do not change.
    q.arg = std::max(1, std::min(8, M / 512));
    q.gx = (uint32_t)((N + 255) / 256);
    q.gy = (uint32_t)((M + 4 * q.arg - 1) / (4 * q.arg));
  } else if (sk.kind == SKINNY_DOT) {
    if (M > 8) return false;
    const int kps = skinny_dot_kps(sk.m, sk.k), splits = (K + kps - 1) / kps;
    if (!split_ok(splits)) return false;
    q.kind = STREAM_DOT8;
    q.arg = kps;
    q.out = splits > 1 ? (float*)g.workspace : (float*)g.c;
    q.gx = (uint32_t)((N + 15) / 16);
    q.gy = (uint32_t)splits;
  } else if (sk.kind == SKINNY_ROWS) {
    if (M > 8) return false;
    const int splits0 = skinny_rows_splits(sk.n, sk.k);
    const int kps = (K + splits0 - 1) / splits0, splits = (K + kps - 1) / kps;
    if (!split_ok(splits)) return false;
    q.kind = STREAM_ROWS8;
    q.arg = kps;
    q.out = splits > 1 ? (float*)g.workspace : (float*)g.c;
    q.gx = (uint32_t)((N + 255) / 256);
    q.gy = (uint32_t)splits;
  } else {
    return false;
  }
  q.blocks = q.gx * q.gy;
  *p = q;
  return true;
}

}  // namespace

bool gemm_group(hipStream_t s, const GemmArgs* g, int count, bool launch) {
  if (count < 2 || count > GROUP_MAX) return false;
  {
    // Streamed products (C5's chain): any mix of the row, dot, outer-product and tiny-output kernels.
    StreamParts parts{};
    uint32_t blocks = 0;
    bool all = true;
    for (int i = 0; i < count && all; i++) {
      all = stream_part_of(g[i], &parts.p[i]);
      blocks += all ? parts.p[i].blocks : 0;
    }
    if (all) {
      if (launch) hipLaunchKernelGGL(k_stream_group, dim3(blocks), dim3(256), 0, s, parts);
      return true;
    }
  }
  // One tile for all. Split tiles: 128x128, since every split tile sums a K range's terms in the same
  // order, so a product picked for a smaller one keeps its bits, and its K splits; one step in LDS, two
  // blocks per CU (the 4096 x 512 x 2048 MLP's pair of 512 blocks each, 96 steps: 99.9 ms, 104.6 with two
  // steps and a block per CU, 101.5 as single launches; the GPT of 8192 tokens, d = 256, 120 steps: 375,
  // 375 and 394 ms, two steps for its pair of 256 blocks alone no faster). fp32 tiles: 32x32 whole ones.
  // K-split partials, if any, must be the deferred kind: a split sum after the grouped launch would be a
  // second launch anyway.
  const TileCfg first = pick_tile(g[0].m, g[0].n, g[0].k, 1);
  const bool split = first.split;
  const TileCfg t = split ? SPLIT_128x128 : TileCfg{32, 32, 32, 2, 2, 0};
  int mode;
  Launch l[GROUP_MAX];
  int flags = 0;
  bool small = false, large = false;  // weight gradients of fewer than 256 blocks, and of more
  for (int i = 0; i < count; i++) {
    if (!on_mfma_tiles(g[i]) || g[i].batch != 1 || g[i].m % t.bm || g[i].n % t.bn) return false;
    const TileCfg own = pick_tile(g[i].m, g[i].n, g[i].k, 1);
    const int own_splits = split_count(own, g[i].m, g[i].n, g[i].k, 1);
    if ((own.split != 0) != split || (!split && (own.bm != 32 || own.bn != 32)) || (own_splits > 1 && !g[i].defer_split)) return false;
    mfma_launch(g[i], t, own_splits, &mode, &l[i]);
    if (mode != 0 || (i + 1 < count && l[i].grid.x % 8 != 0)) return false;
    flags |= ((g[i].ta ? 2 : 0) | (g[i].tb ? 1 : 0)) << (2 * i);
    (g[i].ta && !g[i].tb && l[i].grid.x < 256 ? small : large) |= g[i].ta;
  }
  // The flag sequences instantiated, from C4's backward pass: fc1's input and weight gradients as a
  // pair, with fc2's weight gradient ahead of them as a triple; and the attention projection's
  // weight gradient with the q, k, v projection's, which do not fill the chip alone (64 and 192
  // blocks) and so go together rather than each with its input gradient.
  if (split && small && (large || flags != (2 | 2 << 2))) return false;
  constexpr int T = 2, N = 1;  // (ta, tb) = (true, false) and (false, true)
  GroupParts parts{};
  uint32_t blocks = 0;
  for (int i = 0; i < count; i++) {
    parts.p[i] = GroupPart{l[i].a, l[i].b, l[i].c, l[i].part, l[i].bias, l[i].m, l[i].n, l[i].k, l[i].splits, l[i].kps, l[i].tm, l[i].tn,
                           l[i].grid.x};
    blocks += l[i].grid.x;
  }
#define RG_GROUP(COUNT_, FLAGS_)                                                                                                   \
  if (count == COUNT_ && flags == (FLAGS_)) {                                                                                      \
    if (launch && split) hipLaunchKernelGGL((k_gemm_mfma_group<128, 128, 2, 4, 1, COUNT_, FLAGS_>), dim3(blocks), dim3(512), 0, s, parts); \
    else if (launch) hipLaunchKernelGGL((k_gemm_f32_group<COUNT_, FLAGS_>), dim3(blocks), dim3(256), 0, s, parts);                  \
    return true;                                                                                                                   \
  }
  RG_GROUP(2, N | T << 2)
  RG_GROUP(2, T | N << 2)
  RG_GROUP(2, T | T << 2)
  RG_GROUP(3, T | N << 2 | T << 4)
#undef RG_GROUP
  return false;
}

}  // namespace rgk
