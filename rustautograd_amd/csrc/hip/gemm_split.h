// The fp32 product tile on the bf16 matrix cores (`gemm_mfma_block`), shared by the precompiled
// product kernels (gemm.hip) and by the JIT-compiled products whose epilogue applies the
// elementwise group that reads the product (jit.cpp). Self-contained device code: no includes, so
// that hiprtc can compile it from its text (rg_gemm_split_source).
//
// Every fp32 operand value is split exactly into three bf16 values, each the rounding of what the
// ones before it left (8 bits of the 24 each): x = x1 + x2 + x3. A product is the sum of the six
// terms a1 b1, a1 b2, a2 b1, a2 b2, a1 b3 and a3 b1; what is left out, a2 b3 + a3 b2 + a3 b3, is at
// most 2^-24 of it, one fp32 rounding (a2 up to 2^-8 and a3 up to 2^-17 of a, two such terms).
// v_mfma_f32_16x16x32_bf16 sums a lane's eight exact terms on the largest one's scale (bits below 2^-24
// of it cut off) and adds the four lanes' sums to the accumulator one after the other, each addition
// rounded, with a small bias downwards. So the terms of one K step of 32 are summed from zero, small terms
// first, and the step's sum is added to the running one by an ordinary addition: the MFMA's roundings are
// then on the scale of one step. Odd steps form the sum of a (-b) and subtract it, which turns their bias
// the other way (without that it made up a quarter of the error at K = 5000 and showed in sums over a
// gradient's rows). Against
// 64-bit sums the relative error is 0.40 of the fp32 MFMA tile's at K = 24, 0.24 at 256 and 0.13 from
// 2048 on (normal operands, 4096: 1.0e-7 against 8.1e-7). Only where a sum has few terms that are not
// zero is it larger: a single product errs by 3.5e-8 in the mean and 1.6e-7 at most (fp32: one rounding,
// 2.5e-8 and 6e-8), sums of four by 5.0e-8 (4.0e-8). (With the a1 b1 sums formed apart from the small
// terms' and added by fp32 additions, 2.6e-8 and 4.4e-8; but the 128x128 tile, at its 128 registers,
// spills: 4096 x 512 x 2048 MLP steps 20 % slower.)
// A value that is not finite, or that rounds past the largest bf16 value (scaled: see SPLIT_SCALE),
// leaves NaN in every sum it enters. Sums that end not finite are formed again with fp32 MFMAs
// straight from memory: such outputs are the fp32 tile's, all others are not touched.
//
// What bounds it: six bf16 terms at 2.5 PFLOP/s are 417 TFLOP/s of fp32 products against 157 on the
// fp32 MFMA; a large bf16 product of the vendor library reaches 1.2 PFLOP/s on this chip, a sixth of
// which is 199. Replayed back to back, at the clock that the chip's power leaves, this tile reaches 164 at
// 4096 x 2048 x 2048 (171 within a training step; 127 for the fp32 tile) and 77-135 at K = 256 to 1024 over
// 8192 rows, where the launch, the first loads and the stores weigh (the fp32 tile: 77-107). Multiplying
// the operands by SPLIT_SCALE and looking at each 16 rows' finiteness cost up to 4 % of it (4096 x 2048 x
// 2048 209 us either way, T 2048 x 2048 x 4096 228.7 and 237.8, 8192 x 256 x 1024 44.3 and 45.3).
#pragma once

namespace rgg {

#if defined(__HIPCC_RTC__)
// hiprtc declares the fixed-width integer types in its own namespace.
typedef __hip_internal::int64_t int64_t;
typedef __hip_internal::uint64_t uint64_t;
typedef __hip_internal::uint32_t uint32_t;
#endif

template <int V>
struct IC {
  static constexpr int value = V;
};

typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float rowx2 __attribute__((ext_vector_type(2), aligned(4)));
typedef float rowx4 __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ int64_t batch_offset(const int64_t* offs, uint64_t stride, uint32_t b) {
  return offs ? offs[b] : (int64_t)(stride * b);
}

// Which output tile a block computes. The dispatcher deals consecutive blocks round-robin over
// the 8 XCDs, each with its own L2; so XCD x is to receive the contiguous run
// x*nb/8 ... (x+1)*nb/8 - 1 of tiles, and within a batch the tiles run in groups of 8 M-panels
// per N sweep, so blocks resident on one XCD share their A and B panels in its L2.
struct TileIndex {
  uint32_t tm, tn, z;
};

// Block `bid` of a product launched as `nb` blocks (its share of the grid).
__device__ __forceinline__ TileIndex tile_of(uint32_t bid, uint32_t nb, uint32_t tiles_m, uint32_t tiles_n) {
  uint32_t per_batch = tiles_m * tiles_n;
  uint32_t lid = (nb % 8 == 0) ? (bid % 8) * (nb / 8) + bid / 8 : bid;
  uint32_t z = lid / per_batch, t = lid % per_batch;
  constexpr uint32_t GROUP = 8;
  uint32_t span = GROUP * tiles_n;
  uint32_t first = (t / span) * GROUP;
  uint32_t rows = min(tiles_m - first, GROUP);
  uint32_t in = t % span;
  return {first + in % rows, in / rows, z};
}

// The plain epilogue: each finished output (flat index `e` within the block's output matrix) is
// stored into C, or into the block's split of the K-split partials. Non-temporal stores: every
// block writes its whole tile at the end, all at once; written past the L2 they leave less for the
// end of the kernel to write back (4-10 % off C4's products with 1024- and 768-wide outputs on
// MI355X, results unchanged). Rows of C need only 4-byte alignment.
struct StoreC {
  float* C;
  float* partial;
  int splits;
  uint64_t mn;
  float* out = nullptr;
  __device__ __forceinline__ void begin(uint32_t b, uint32_t sp) {
    out = splits > 1 ? partial + ((uint64_t)b * splits + sp) * mn : C + (uint64_t)b * mn;
  }
  __device__ __forceinline__ void put4(uint64_t e, float4 v) { __builtin_nontemporal_store(rowx4{v.x, v.y, v.z, v.w}, (rowx4*)(out + e)); }
  __device__ __forceinline__ void put2(uint64_t e, float2 v) { __builtin_nontemporal_store(floatx2{v.x, v.y}, (floatx2*)(out + e)); }
  __device__ __forceinline__ void put1(uint64_t e, float v) { __builtin_nontemporal_store(v, out + e); }
};

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t cell __attribute__((ext_vector_type(4)));  // eight bf16 values: one row's or column's next 8 k

// Two values' three bf16 parts, packed in pairs.
__device__ __forceinline__ uint32_t pack_bf16(float x0, float x1) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2{x0, x1}), bf16x2));
}
__device__ __forceinline__ void split_bf16(float x0, float x1, uint32_t& p1, uint32_t& p2, uint32_t& p3) {
  p1 = pack_bf16(x0, x1);
  const float r0 = x0 - __builtin_bit_cast(float, p1 << 16), r1 = x1 - __builtin_bit_cast(float, p1 & 0xffff0000u);
  p2 = pack_bf16(r0, r1);
  const float s0 = r0 - __builtin_bit_cast(float, p2 << 16), s1 = r1 - __builtin_bit_cast(float, p2 & 0xffff0000u);
  p3 = pack_bf16(s0, s1);
}

constexpr int SPLIT_BK = 32;  // K step

// Operands are split after multiplication by 2^23, and a step's sums, 2^46 too large, are multiplied
// by 2^-46 as they are added: both are exact. So any fp32 value, 2^-149 at the least, has a first part
// in bf16's normal range and loses none of the others (unscaled, values of 2^-120 kept 15 bits and
// those below 2^-134 none; with 2^16 a part below 2^-126 is held, but the MFMA cuts off what it is
// added to on the scale of 2^-126: 8.5e-7 for values of a few 2^-149). The price is at the other end:
// outputs of values from 2^104 or step sums from 2^82 on are formed by the fp32 MFMAs.
constexpr float SPLIT_SCALE = 8388608.0f, SPLIT_UNSCALE = 1.0f / (8388608.0f * 8388608.0f);

// Layout of R rows (or columns) x 32 k of one operand in LDS: three planes of cells (16 bytes,
// eight consecutive k), [k / 8][row], the k / 8 groups two cells further apart than R so that the
// stores of a K-contiguous operand (four lanes per row) spread over all banks; the MFMA's reads are
// 16 consecutive rows of one group. NT threads stage it, each thread taking units of 8 k for VN
// adjacent columns (K-contiguous: one row), VN chosen so that every thread has one.
template <int R, bool KC, int NT>
struct SplitGeo {
  static constexpr int VN = KC ? 1 : (R * 4 / NT >= 2 ? 2 : 1);
  static constexpr int UNITS = R / VN * 4, PER = UNITS / NT;
  static_assert(UNITS % NT == 0, "whole units per thread");
  static constexpr int GROUP = R + 2, PLANE = 4 * GROUP, CELLS = 3 * PLANE;
  // Two adjacent columns of one thread trade places in every second eight, so that eight lanes'
  // stores of their first (or second) column reach eight different banks.
  static __device__ __forceinline__ int place(int r) { return VN == 1 ? r : r ^ ((r >> 3) & 1); }
};

template <int R, bool KC, int NT>
struct SplitStage {
  typedef SplitGeo<R, KC, NT> G;
  float v[G::PER][G::VN][8];
  // The R x 32 tile at `base` (its first row or column, k = 0) and k0. Every row or column lies
  // inside the operand; with `partial` the tile's k reach past `kend` and are zeros there. Loads
  // need only 4-byte alignment. A column's eight k share one 32-bit offset (rows of the operand
  // have less than 2^25 columns), each k its own scalar base.
  __device__ __forceinline__ void load(const float* base, int64_t ld, int k0, int kend, bool partial, int tid) {
#pragma unroll
    for (int q = 0; q < G::PER; q++) {
      const int u = q * NT + tid;
      if constexpr (KC) {
        const int64_t off = (int64_t)(u >> 2) * ld + (u & 3) * 8;
        if (!partial) {
          const float* p = base + off + k0;
          const rowx4 x = *(const rowx4*)p, y = *(const rowx4*)(p + 4);
#pragma unroll
          for (int e = 0; e < 4; e++) v[q][0][e] = x[e], v[q][0][4 + e] = y[e];
        } else {
          const int k = k0 + (u & 3) * 8;
          const float* row = base + (int64_t)(u >> 2) * ld;
#pragma unroll
          for (int e = 0; e < 8; e++) {
            const float x = row[min(k + e, kend - 1)];
            v[q][0][e] = k + e < kend ? x : 0.0f;
          }
        }
      } else {
        constexpr int W = R / G::VN;
        const int g = u / W, c = (u % W) * G::VN;
        if (!partial) {
          const uint32_t off = ((uint32_t)g * 8 * (uint32_t)ld + (uint32_t)c) * 4;
#pragma unroll
          for (int e = 0; e < 8; e++) {
            const char* p = (const char*)(base + (int64_t)(k0 + e) * ld) + off;
            if constexpr (G::VN == 1) {
              v[q][0][e] = *(const float*)p;
            } else {
              const rowx2 x = *(const rowx2*)p;
              v[q][0][e] = x[0], v[q][1][e] = x[1];
            }
          }
        } else {
#pragma unroll
          for (int e = 0; e < 8; e++) {
            const int k = k0 + g * 8 + e;
            const float* p = base + (int64_t)min(k, kend - 1) * ld + c;
#pragma unroll
            for (int j = 0; j < G::VN; j++) {
              const float x = p[j];
              v[q][j][e] = k < kend ? x : 0.0f;
            }
          }
        }
      }
    }
  }
  // `factor` times the staged values, split, into LDS.
  __device__ __forceinline__ void store(cell* lds, int tid, float factor) const {
#pragma unroll
    for (int q = 0; q < G::PER; q++) {
      const int u = q * NT + tid;
      constexpr int W = R / G::VN;
      const int g = KC ? u & 3 : u / W, r = KC ? u >> 2 : (u % W) * G::VN;
#pragma unroll
      for (int j = 0; j < G::VN; j++) {
        cell p1, p2, p3;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          uint32_t x1, x2, x3;
          split_bf16(v[q][j][2 * e] * factor, v[q][j][2 * e + 1] * factor, x1, x2, x3);
          p1[e] = x1, p2[e] = x2, p3[e] = x3;
        }
        cell* d = lds + g * G::GROUP + G::place(r + j);
        d[0] = p1, d[G::PLANE] = p2, d[2 * G::PLANE] = p3;
      }
    }
  }
};

template <int BM, int BN, int WM, int WN, int U, bool TA, bool TB>
struct SplitLds {
  static constexpr int STEP = SplitGeo<BM, !TA, 64 * WM * WN>::CELLS + SplitGeo<BN, TB, 64 * WM * WN>::CELLS;
  static constexpr int CELLS = U * STEP;
};

// C = op(A) op(B), the BM x BN tile of block `bid` of a product launched as `nb` blocks, staged
// through `smem` (SplitLds<...>::CELLS cells): WM x WN wave64s, each owning (BM/WM) x (BN/WN) as
// 16x16 MFMA tiles. M >= BM and N >= BN: the last tile along an edge that BM or BN does not divide
// is moved inwards, so that no load of a row or column is out of range, and stores only what the
// tile before it does not. Split `sp` covers K range [sp * k_per_split, (sp + 1) * k_per_split), a
// multiple of 32 long except the last; TAIL: some range is not a multiple of 32.
//
// One LDS buffer of U steps: the next U steps' values wait in registers while these are multiplied,
// are converted and stored between two barriers, and the loads after them go out at once. Where
// several blocks share a CU, one's conversions run beside another's MFMAs and U is 1 (two LDS buffers
// and one barrier per step, at half the blocks per CU, measured 3-6 % slower at 4096 x 2048 x 2048);
// a block with few or no others beside it takes U = 2, half the barriers and waits (T 256x1024x8192
// on 128x128 tiles, a block per CU: 33.1 -> 29.4 us; 8192x256x1024 on 64x64: 39 -> 35.7). The sums
// do not depend on U or on the tile's size.
// The product is formed transposed (B supplies the MFMA rows), so that each lane holds runs of
// four adjacent output columns. Every put4 of a lane is of the same four columns, so that an
// epilogue can keep per-column sums in registers.
template <int BM, int BN, int WM, int WN, int U, bool TA, bool TB, bool TAIL, class Epi>
__device__ __forceinline__ void gemm_split_tile(const float* __restrict__ A, const float* __restrict__ B, int M, int N, int K,
                                                const int64_t* a_off, const int64_t* b_off, uint64_t a_stride, uint64_t b_stride, int splits,
                                                int k_per_split, const float* __restrict__ bias, uint32_t tiles_m, uint32_t tiles_n, Epi& epi,
                                                uint32_t bid, uint32_t nb, cell* smem) {
  constexpr int NT = 64 * WM * WN;
  constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / 16, TN = WTN / 16;
  typedef SplitGeo<BM, !TA, NT> GA;
  typedef SplitGeo<BN, TB, NT> GB;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN, li = lane & 15, lo = lane >> 4;
  const TileIndex ti = tile_of(bid, nb, tiles_m, tiles_n);
  const uint32_t b = ti.z / splits, sp = ti.z % splits;
  const int m_first = ti.tm * BM, n_first = ti.tn * BN, m0 = min(m_first, M - BM), n0 = min(n_first, N - BN);
  const int64_t lda = TA ? M : K, ldb = TB ? K : N;
  const float* Ab = A + batch_offset(a_off, a_stride, b) + (TA ? (int64_t)m0 : (int64_t)m0 * K);
  const float* Bb = B + batch_offset(b_off, b_stride, b) + (TB ? (int64_t)n0 * K : (int64_t)n0);
  const int kbeg = sp * k_per_split, kend = min(K, kbeg + k_per_split);
  const int nk = (kend - kbeg + SPLIT_BK - 1) / SPLIT_BK;
  constexpr int STEP = SplitLds<BM, BN, WM, WN, U, TA, TB>::STEP;
  SplitStage<BM, !TA, NT> sa[U];
  SplitStage<BN, TB, NT> sb[U];
  // Rounds of U steps; the last may have fewer.
  const int rounds = (nk + U - 1) / U;
  auto load = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (U > 1 && t * U + u >= nk) break;
      const int k0 = kbeg + (t * U + u) * SPLIT_BK;
      const bool partial = TAIL && k0 + SPLIT_BK > kend;
      sa[u].load(Ab, lda, k0, kend, partial, tid);
      sb[u].load(Bb, ldb, k0, kend, partial, tid);
    }
  };
  // Odd steps' B is stored negated, and their sums subtracted (multiply's sign).
  auto store = [&](float sign) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      sa[u].store(smem + u * STEP, tid, SPLIT_SCALE);
      sb[u].store(smem + u * STEP + GA::CELLS, tid, u % 2 ? -sign * SPLIT_SCALE : sign * SPLIT_SCALE);
    }
  };
  floatx4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int n = 0; n < TN; n++) acc[i][n] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  auto multiply_step = [&](float sign, int u) __attribute__((always_inline)) {
    const cell* as = smem + u * STEP + lo * GA::GROUP;
    const cell* bs = smem + u * STEP + GA::CELLS + lo * GB::GROUP;
    bf16x8 y[3][TN];
#pragma unroll
    for (int p = 0; p < 3; p++)
#pragma unroll
      for (int n = 0; n < TN; n++) y[p][n] = __builtin_bit_cast(bf16x8, bs[p * GB::PLANE + GB::place(wn * WTN + n * 16 + li)]);
#pragma unroll
    for (int i = 0; i < TM; i++) {
      bf16x8 x[3];
#pragma unroll
      for (int p = 0; p < 3; p++) x[p] = __builtin_bit_cast(bf16x8, as[p * GA::PLANE + GA::place(wm * WTM + i * 16 + li)]);
      constexpr int PX[6] = {0, 2, 1, 0, 1, 0}, PY[6] = {2, 0, 1, 1, 0, 0};
      floatx4 step[TN];
#pragma unroll
      for (int n = 0; n < TN; n++) step[n] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int q = 0; q < 6; q++)
#pragma unroll
        for (int n = 0; n < TN; n++) step[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(y[PY[q]][n], x[PX[q]], step[n], 0, 0, 0);
#pragma unroll
      for (int n = 0; n < TN; n++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[i][n][r] = __builtin_fmaf(step[n][r], sign * SPLIT_UNSCALE, acc[i][n][r]);
    }
  };
  auto multiply = [&](float sign, int t, bool last) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (last && U > 1 && t * U + u >= nk) break;
      multiply_step(u % 2 ? -sign : sign, u);
    }
  };
  load(0);
  float sign = 1.0f;  // of the first step in LDS
  store(sign);
  if (rounds > 1) load(1);
  __syncthreads();
  for (int t = 0; t < rounds - 1; t++) {
    multiply(sign, t, false);
    __syncthreads();
    if (U % 2 == 1) sign = -sign;
    store(sign);
    if (t + 2 < rounds) load(t + 2);
    __syncthreads();
  }
  multiply(sign, rounds - 1, true);
  // Lane l of the wave's tile (i, n) holds output row 16 i + l % 16, columns 16 n + 4 (l / 16) .. + 3.
  // Sums that are not finite again, in fp32: those alone, so that an output depends on its own row and
  // column and on no neighbour, whatever the tile.
#pragma unroll
  for (int i = 0; i < TM; i++) {
    float finite = 0.0f;  // NaN once any sum of these 16 rows is infinite or NaN
#pragma unroll
    for (int n = 0; n < TN; n++)
#pragma unroll
      for (int r = 0; r < 4; r++) finite = __builtin_fmaf(acc[i][n][r], 0.0f, finite);
    if (__ballot(!(finite == 0.0f)) == 0) continue;
    floatx4 again[TN];
#pragma unroll
    for (int n = 0; n < TN; n++) again[n] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
    for (int k0 = kbeg; k0 < kend; k0 += 4) {
      const int k = min(k0 + lo, kend - 1);
      const bool live = k0 + lo < kend;
      const int64_t r = wm * WTM + i * 16 + li;
      const float v = Ab[TA ? (int64_t)k * M + r : r * K + k];
      const float x = live ? v : 0.0f;
#pragma unroll
      for (int n = 0; n < TN; n++) {
        const int64_t c = wn * WTN + n * 16 + li;
        const float w = Bb[TB ? c * K + k : (int64_t)k * N + c];
        again[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(live ? w : 0.0f, x, again[n], 0, 0, 0);
      }
    }
#pragma unroll
    for (int n = 0; n < TN; n++)
#pragma unroll
      for (int r = 0; r < 4; r++) acc[i][n][r] = acc[i][n][r] * 0.0f == 0.0f ? acc[i][n][r] : again[n][r];
  }
  // The outputs leave through LDS, 32 rows x 32 columns of a wave at a time, so that a lane stores
  // the same four columns of every eighth row and a store covers whole 128-byte runs of eight rows
  // (from the accumulators it would cover 64 bytes of sixteen). Each wave has its own part.
  static_assert(WTN == 32 && TM % 2 == 0 && WM * WN * 32 * 9 <= STEP, "wave tiles");
  epi.begin(b, sp);
  const int c4 = lane & 7, col = n0 + wn * 32 + 4 * c4;
  floatx4 add = {0.0f, 0.0f, 0.0f, 0.0f};
  if (bias) add = *(const rowx4*)(bias + col);
  floatx4* out = (floatx4*)smem + wave * 32 * 9;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TM; i += 2) {
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int n = 0; n < TN; n++) out[(16 * h + li) * 9 + 4 * n + lo] = acc[i + h][n];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int r = 8 * q + (lane >> 3), row = m0 + wm * WTM + 16 * i + r;
      floatx4 c = out[r * 9 + c4];
      // A per-column bias (unsplit products only) added to the finished sums, as one fp32 addition.
      if (bias) c = c + add;
      if (row < m_first) continue;
      const uint64_t e = (uint64_t)row * N + col;
      if (col >= n_first) {
        epi.put4(e, make_float4(c[0], c[1], c[2], c[3]));
      } else {
#pragma unroll
        for (int x = 0; x < 4; x++)
          if (col + x >= n_first) epi.put1(e + x, c[x]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// One product over the whole grid, with its own LDS.
template <int BM, int BN, int WM, int WN, int U, bool TA, bool TB, bool TAIL, class Epi>
__device__ __forceinline__ void gemm_mfma_block(const float* __restrict__ A, const float* __restrict__ B, int M, int N, int K,
                                                const int64_t* a_off, const int64_t* b_off, uint64_t a_stride, uint64_t b_stride, int splits,
                                                int k_per_split, const float* __restrict__ bias, uint32_t tiles_m, uint32_t tiles_n, Epi& epi) {
  __shared__ cell smem[SplitLds<BM, BN, WM, WN, U, TA, TB>::CELLS];
  gemm_split_tile<BM, BN, WM, WN, U, TA, TB, TAIL>(A, B, M, N, K, a_off, b_off, a_stride, b_stride, splits, k_per_split, bias, tiles_m, tiles_n,
                                                epi, blockIdx.x, gridDim.x, smem);
}

}  // namespace rgg
