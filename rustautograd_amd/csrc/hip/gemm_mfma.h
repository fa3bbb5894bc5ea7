// The fp32 MFMA product tile (`gemm_f32_tile`), for products of too few tiles to fill the chip: a
// block is then alone on its CU, and the split tile's (gemm_split.h) conversions and second barrier
// lengthen each of its K steps (256 x 768 x 256: 4.3 us on 32x32 tiles here, 7.1 there).
#pragma once

#include "gemm_split.h"

namespace rgg {

// Load modes: every vector inside the operand (no checks), checked 16-byte vectors, or checked
// scalar loads (operands whose rows are not 16-byte aligned).
enum LoadMode { LOAD_EVEN = 0, LOAD_VEC = 1, LOAD_SCALAR = 2 };

// Stages an R x W tile (W contiguous floats per row, W % 4 == 0) of a row-major operand with
// leading dimension `ld`, rows r0.. (valid below `rows`) and columns c0.. (valid below `cols`),
// through registers: NT threads, one 4-float vector per thread and pass.
template <int R, int W, int NT, int MODE>
struct Stager {
  static constexpr int NVEC = R * W / 4;
  static constexpr int PER = (NVEC + NT - 1) / NT;
  float4 v[PER];
  __device__ __forceinline__ void load(const float* base, int64_t ld, int r0, int c0, int rows, int cols, int tid) {
#pragma unroll
    for (int q = 0; q < PER; q++) {
      const int idx = q * NT + tid;
      const int r = idx / (W / 4), c = (idx % (W / 4)) * 4;
      const bool live = NVEC % NT == 0 || idx < NVEC;
      const int gr = r0 + r, gc = c0 + c;
      if constexpr (MODE == LOAD_SCALAR) {
        const float* p = base + (int64_t)gr * ld + gc;
        float t[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          bool ok = live && gr < rows && gc + e < cols;
          t[e] = ok ? p[e] : 0.0f;
        }
        v[q] = make_float4(t[0], t[1], t[2], t[3]);
      } else {
        const bool ok = live && (MODE == LOAD_EVEN || (gr < rows && gc < cols));
        const float4 x = *(const float4*)(ok ? base + (int64_t)gr * ld + gc : base);
        v[q] = ok ? x : make_float4(0.f, 0.f, 0.f, 0.f);
      }
    }
  }
  __device__ __forceinline__ void store(float* lds, int ldl, int tid) const {
#pragma unroll
    for (int q = 0; q < PER; q++) {
      const int idx = q * NT + tid;
      if (NVEC % NT == 0 || idx < NVEC) *(float4*)(lds + (idx / (W / 4)) * ldl + (idx % (W / 4)) * 4) = v[q];
    }
  }
};

template <int T>
__device__ __forceinline__ void lds_read(const float* p, float* v) {
  if constexpr (T == 1) {
    v[0] = *p;
  } else if constexpr (T == 2) {
    float2 x = *(const float2*)p;
    v[0] = x.x; v[1] = x.y;
  } else {
    float4 x = *(const float4*)p;
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
  }
}

// C = op(A) op(B) for one BM x BN block tile; WM x WN wave64s, each owning (BM/WM) x (BN/WN) as
// TM x TN MFMA tiles of 16x16. The grid is one-dimensional: tiles_m * tiles_n * batch * splits
// blocks (tile_of); split `sp` covers K range [sp * k_per_split, (sp + 1) * k_per_split).

// LDS of one tile: two buffers of each operand's K step, in the operand's own layout (rows padded
// by 4 floats where K is contiguous).
template <int BM, int BN, int BK, bool TA, bool TB>
struct TileLds {
  static constexpr int LDA = !TA ? BK + 4 : BM, LDB = TB ? BK + 4 : BN;
  static constexpr int SA = !TA ? BM * LDA : BK * LDA, SB = TB ? BN * LDB : BK * LDB;
  static constexpr int FLOATS = 2 * (SA + SB);
};

// The tile of block `bid` of a product launched as `nb` blocks, staging through `smem` (at least
// TileLds<...>::FLOATS floats of LDS): a kernel that runs two products side by side gives each
// its share of the grid and the same LDS.
template <int BM, int BN, int BK, int WM, int WN, bool TA, bool TB, int MODE, class Epi>
__device__ __forceinline__ void gemm_f32_tile(const float* __restrict__ A, const float* __restrict__ B, int M, int N, int K,
                                               const int64_t* a_off, const int64_t* b_off, uint64_t a_stride, uint64_t b_stride, int splits,
                                               int k_per_split, const float* __restrict__ bias, uint32_t tiles_m, uint32_t tiles_n,
                                               Epi& epi, uint32_t bid, uint32_t nb, float* smem) {
  constexpr int NT = 64 * WM * WN;
  constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / 16, TN = WTN / 16;
  static_assert(TM >= 1 && TN >= 1 && TM <= 2 && TN <= 2, "wave tiles");
  // A group of 16 k: four MFMA steps, lane l taking k = 4 (l / 16) + j at step j in both operands.
  // v_mfma_f32_16x16x4_f32: lane l supplies row (A) / column (B) l % 16, and register r of its
  // accumulator holds row 4 (l / 16) + r, column l % 16.
  static_assert(BK % 16 == 0, "K step");
  constexpr bool AK = !TA, BKC = TB;  // K-contiguous operands
  typedef TileLds<BM, BN, BK, TA, TB> L;
  constexpr int LDA = L::LDA, LDB = L::LDB, SA = L::SA, SB = L::SB;
  float(*As)[SA] = (float(*)[SA])smem;
  float(*Bs)[SB] = (float(*)[SB])(smem + 2 * SA);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const TileIndex ti = tile_of(bid, nb, tiles_m, tiles_n);
  const uint32_t b = ti.z / splits, sp = ti.z % splits;
  const int m0 = ti.tm * BM, n0 = ti.tn * BN;
  const float* Ab = A + batch_offset(a_off, a_stride, b);
  const float* Bb = B + batch_offset(b_off, b_stride, b);
  const int kbeg = sp * k_per_split, kend = min(K, kbeg + k_per_split);
  const int nk = (kend - kbeg + BK - 1) / BK;

  // Two register stages: the global loads of tile t + 2 are issued while tile t is multiplied
  // out of LDS and tile t + 1 waits in registers, so each load has two iterations to arrive.
  Stager<AK ? BM : BK, AK ? BK : BM, NT, MODE> sa0, sa1;
  Stager<BKC ? BN : BK, BKC ? BK : BN, NT, MODE> sb0, sb1;
  // The register stage SET (a constant): two variables rather than an array, so that no stage is
  // ever indexed and both stay in registers.
  auto stage_a = [&](auto set) -> auto& {
    if constexpr (decltype(set)::value == 0) return sa0;
    else return sa1;
  };
  auto stage_b = [&](auto set) -> auto& {
    if constexpr (decltype(set)::value == 0) return sb0;
    else return sb1;
  };
  // Tile t of this block's K range into register stage `stage`.
  auto load_tiles = [&](int t, auto stage) __attribute__((always_inline)) {
    auto& xa = stage_a(stage);
    auto& xb = stage_b(stage);
    const int k0 = kbeg + t * BK;
    if (AK) xa.load(Ab, K, m0, k0, M, kend, tid);
    else xa.load(Ab, M, k0, m0, kend, M, tid);
    if (BKC) xb.load(Bb, K, n0, k0, N, kend, tid);
    else xb.load(Bb, N, k0, n0, kend, N, tid);
  };

  floatx4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) acc[i][j][r] = 0.0f;

  if (nk > 0) {
    load_tiles(0, IC<0>());
    load_tiles(min(1, nk - 1), IC<1>());
    sa0.store(As[0], LDA, tid);
    sb0.store(Bs[0], LDB, tid);
  }
  __syncthreads();
  const int li = lane % 16, q4 = (lane / 16) * 4;
  auto multiply = [&](const float* as, const float* bs) __attribute__((always_inline)) {
#pragma unroll
    for (int kg = 0; kg < BK; kg += 16) {
      float a[4][TM], bv[4][TN];  // [k-step][tile]
      if (AK) {
#pragma unroll
        for (int i = 0; i < TM; i++) {
          float v[4];
          lds_read<4>(as + (wm * WTM + i * 16 + li) * LDA + kg + q4, v);
#pragma unroll
          for (int j = 0; j < 4; j++) a[j][i] = v[j];
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; j++) lds_read<TM>(as + (kg + q4 + j) * LDA + wm * WTM + TM * li, a[j]);
      }
      if (BKC) {
#pragma unroll
        for (int i = 0; i < TN; i++) {
          float v[4];
          lds_read<4>(bs + (wn * WTN + i * 16 + li) * LDB + kg + q4, v);
#pragma unroll
          for (int j = 0; j < 4; j++) bv[j][i] = v[j];
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; j++) lds_read<TN>(bs + (kg + q4 + j) * LDB + wn * WTN + TN * li, bv[j]);
      }
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int n = 0; n < TN; n++) {
            // With a K-contiguous B the product is formed transposed (B supplies the MFMA rows), so
            // that each lane ends up with four adjacent output columns.
            if constexpr (BKC) acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[j][n], a[j][i], acc[i][n], 0, 0, 0);
            else acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j][i], bv[j][n], acc[i][n], 0, 0, 0);
          }
    }
  };
  // Iteration t multiplies LDS buffer t % 2, whose register stage t % 2 is then free for tile
  // t + 2; tile t + 1 goes from register stage (t + 1) % 2 into the other LDS buffer, which every
  // wave finished reading before the previous barrier. The body has no branches, so the compiler
  // can interleave the loads and address arithmetic with the MFMAs: past the end of the range the
  // last tile is loaded again and stored into the idle buffer, and never read.
  auto iteration = [&](int t, auto parity) __attribute__((always_inline)) {
    constexpr int P = decltype(parity)::value;
    load_tiles(min(t + 2, nk - 1), parity);
    multiply(As[P], Bs[P]);
    stage_a(IC<P ^ 1>()).store(As[P ^ 1], LDA, tid);
    stage_b(IC<P ^ 1>()).store(Bs[P ^ 1], LDB, tid);
    __syncthreads();
  };
  int t = 0;
  for (; t + 1 < nk; t += 2) {
    iteration(t, IC<0>());
    iteration(t + 1, IC<1>());
  }
  if (t < nk) iteration(t, IC<0>());
  // Accumulator register r of lane l holds MFMA row rho = 4 (l / 16) + r, column l % 16 (for the
  // transposed form: output row l % 16, column rho). MFMA tile i row rho is block row 16 i + rho
  // (K-contiguous A) or TM rho + i (M-contiguous A); tile n column gamma is block column
  // 16 n + gamma (K-contiguous B) or TN gamma + n (N-contiguous B). Either way a lane holds adjacent
  // output columns: four in one tile (K-contiguous B) or one in each of its TN tiles.
  epi.begin(b, sp);
  const bool vec_out = MODE != LOAD_SCALAR && N % 4 == 0;
  // A per-column bias (unsplit products only) added to the finished sums, as one fp32 addition.
  if (bias) {
    if constexpr (BKC) {
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int n = 0; n < TN; n++) {
          const int col = n0 + wn * WTN + n * 16 + q4;
#pragma unroll
          for (int r = 0; r < 4; r++)
            if (col + r < N) acc[i][n][r] += bias[col + r];
        }
    } else {
      const int col = n0 + wn * WTN + TN * li;
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
          for (int n = 0; n < TN; n++)
            if (col + n < N) acc[i][n][r] += bias[col + n];
    }
  }
  if constexpr (BKC) {
#pragma unroll
    for (int i = 0; i < TM; i++) {
      const int row = m0 + wm * WTM + (AK ? i * 16 + li : TM * li + i);
      if (row >= M) continue;
      const uint64_t erow = (uint64_t)row * N;
#pragma unroll
      for (int n = 0; n < TN; n++) {
        const int col = n0 + wn * WTN + n * 16 + q4;
        const floatx4 c = acc[i][n];
        if (vec_out && col + 4 <= N) {
          epi.put4(erow + col, make_float4(c[0], c[1], c[2], c[3]));
        } else {
#pragma unroll
          for (int r = 0; r < 4; r++)
            if (col + r < N) epi.put1(erow + col + r, c[r]);
        }
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int rho = q4 + r;
        const int row = m0 + wm * WTM + (AK ? i * 16 + rho : TM * rho + i);
        if (row >= M) continue;
        const uint64_t erow = (uint64_t)row * N;
        const int col = n0 + wn * WTN + TN * li;
        if (TN > 1 && vec_out && col + TN <= N) {
          if constexpr (TN == 2) epi.put2(erow + col, make_float2(acc[i][0][r], acc[i][1][r]));
        } else {
#pragma unroll
          for (int n = 0; n < TN; n++)
            if (col + n < N) epi.put1(erow + col + n, acc[i][n][r]);
        }
      }
  }
}

// One product over the whole grid, with its own LDS.
template <int BM, int BN, int BK, int WM, int WN, bool TA, bool TB, int MODE, class Epi>
__device__ __forceinline__ void gemm_f32_block(const float* __restrict__ A, const float* __restrict__ B, int M, int N, int K,
                                                const int64_t* a_off, const int64_t* b_off, uint64_t a_stride, uint64_t b_stride, int splits,
                                                int k_per_split, const float* __restrict__ bias, uint32_t tiles_m, uint32_t tiles_n,
                                                Epi& epi) {
  __shared__ float smem[TileLds<BM, BN, BK, TA, TB>::FLOATS];
  gemm_f32_tile<BM, BN, BK, WM, WN, TA, TB, MODE>(A, B, M, N, K, a_off, b_off, a_stride, b_stride, splits, k_per_split, bias, tiles_m, tiles_n,
                                                  epi, blockIdx.x, gridDim.x, smem);
}

}  // namespace rgg
