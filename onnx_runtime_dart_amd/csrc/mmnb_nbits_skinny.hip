// MatMulNBits for a few rows (2 <= M <= 32, and more rows of a small weight)
// on the matrix cores, in one launch.
//
// The work of these calls is the weight stream, a round trip to memory and
// the launch; a separate pass that prepares the activations costs more than
// the product.  So a workgroup stages its own activations: it owns 32 * CW
// columns of up to 32 rows and a range of K, walks the range in chunks of 512
// k, and per chunk
//
//   - reads the rows' 512 activations (8 per lane, one row piece per wave),
//     scales each piece by a power of two (its largest magnitude lands in
//     [2^13, 2^14)) and splits it into fp16 terms in LDS, in the operand
//     order of v_mfma_f32_32x32x16_f16;
//   - takes the weights straight from memory into registers (every weight is
//     used by one wave only), one contiguous 1 KB operand unit per load, a
//     chunk ahead (read from the column-major pack, 64 lines of 16 bytes per
//     load, a chunk took 3.3 us instead of 2.3 with 128 columns);
//   - multiplies: CW column waves x KW k waves, each 32 rows x 32 columns x
//     512 / KW k, the exact integers q - zp in fp16 as the prefill GEMM forms
//     them, one scale FMA per quantisation block.
//
// Row layout V of the 32-row operand tile.  With few rows the tile's free
// rows hold the other terms of the split, so one MFMA multiplies all of them:
//   0: M <= 8,  three terms at rows 8p + m, each times a power of two of its
//      own (kSkGain1, kSkGain2): the activations exactly as fp32 holds them,
//      down to 2^-39 of the piece's largest.  What the terms miss of smaller
//      ones is multiplied at the end, in passes with a power of two of their
//      own until nothing is left (9 at most, over the whole range of fp32):
//      7.3e-8 .. 9e-8 off the 64-bit product where the fp32 FMA kernel is
//      1.0e-7 .. 1.3e-7 (K = 1024 .. 4096, 2-norm);
//   1: M <= 16, two terms at rows 16p + m;
//   2: M <= 32, two MFMAs (hi, lo) per step.
// Two terms are what the prefill GEMM uses (they leave 2^-22); with a power of
// two per 512 k instead of per row, 0.95e-7 .. 1.1e-7 against its 0.95e-7 ..
// 1.2e-7.
//
// The k waves meet in LDS.  With K cut over several workgroups (nsl slices)
// each stores its partial tile and the last to arrive adds them in slice
// order, so the bits do not depend on the arrival order (protocol and memory
// order as the prefill GEMM's K slices).  The partials live in a buffer of
// the context, so a call never grows scratch and can be captured first.
//
// Bound: the launch, one pass of the weights and then latency: a chunk is a
// serial chain of staging, barrier, LDS reads and MFMAs of two waves per
// SIMD, 1.3 (M <= 8) to 2.6 us (M <= 32) long; the slice exchange ~2.5 us.
// us per call back to back, block 128, before (k_gemv_lds for M <= 8, else
// k_prep_a and the GEMM) and now: M = 8, K = N = 4096 12.4 -> 8.6; N = 14336
// 45.9 -> 13.4; (1024, 6144) 6.8 -> 4.3; M = 12, 4096^2 19.3 -> 9.3; M = 24
// 19.6 -> 11.4; M = 32 and 256, 1024^2 12.5 -> 6.3 and 14.1 -> 6.9.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "mmnb_device.h"
#include "mmnb_internal.h"

namespace mmnb {

constexpr int kSkChunk = 512;          // k per staged chunk
constexpr int kSkSegs = kSkChunk / 64;  // 64-k segments per chunk
constexpr int kSkThreads = 512;
constexpr int kSkRows = 32;             // rows per row group

// Nibbles of w as 8 fp16 values q - zp in the order {0,4,1,5,2,6,3,7} (see
// dequant8).  Plain C with opaque masks (m0 = 0x000F000F, m1 = 0x00F000F0,
// still one v_and_or_b32 each): part of this kernel's MFMA results are dead
// (row layout 0), and the compiler does not guard an inline-asm write of a
// register that such an MFMA is still going to write.
__device__ __forceinline__ half8_t sk_dequant(uint32_t w, int zp, uint32_t m0, uint32_t m1,
                                              uint32_t magic) {
  const uint32_t w8 = w >> 8;
  const half2_t zz = __builtin_bit_cast(half2_t, (uint32_t)(0x6400 + zp) * 0x10001u);
  const half2_t zs = __builtin_bit_cast(half2_t, (uint32_t)(0x5400 + (zp << 4)) * 0x10001u);
  const half2_t sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f};
  const half2_t h0 = __builtin_bit_cast(half2_t, (w & m0) | magic) - zz;
  const half2_t h1 = __builtin_bit_cast(half2_t, (w & m1) | magic) * sixteenth - zs;
  const half2_t h2 = __builtin_bit_cast(half2_t, (w8 & m0) | magic) - zz;
  const half2_t h3 = __builtin_bit_cast(half2_t, (w8 & m1) | magic) * sixteenth - zs;
  half8_t r = {h0.x, h0.y, h1.x, h1.y, h2.x, h2.y, h3.x, h3.y};
  return r;
}

// Workgroup barrier that orders LDS accesses only: __syncthreads() also
// drains every outstanding load, i.e. the prefetched chunk.
__device__ __forceinline__ void sk_lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ uint32_t sk_move(uint32_t v) {
  uint32_t r;
  asm volatile("v_mov_b32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}

typedef float f2vec __attribute__((ext_vector_type(2)));
typedef float f4vec __attribute__((ext_vector_type(4)));

// max over the 64 lanes, wave-uniform.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_max_u32(uint32_t v) {
  return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  v = dpp_max_u32<0xB1>(v);   // quad_perm [1,0,3,2]
  v = dpp_max_u32<0x4E>(v);   // quad_perm [2,3,0,1]
  v = dpp_max_u32<0x141>(v);  // row_half_mirror
  v = dpp_max_u32<0x140>(v);  // row_mirror
  const uint32_t a = max((uint32_t)__builtin_amdgcn_readlane((int)v, 0),
                         (uint32_t)__builtin_amdgcn_readlane((int)v, 16));
  const uint32_t b = max((uint32_t)__builtin_amdgcn_readlane((int)v, 32),
                         (uint32_t)__builtin_amdgcn_readlane((int)v, 48));
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)max(a, b));
}
// The power of two that takes a finite magnitude's bits to [2^13, 2^14) (subnormal
// ones, and 0, as far as the smallest normal one), in scalar integers.
__device__ __forceinline__ int sk_exponent(uint32_t bits) {
  return 140 - (int)max(bits >> 23, 1u);
}

template <int V>
struct SkRows {
  static constexpr int kParts = V == 0 ? 3 : 2;          // terms of the split
  static constexpr int kMax = V == 0 ? 8 : V == 1 ? 16 : kSkRows;
  static constexpr int kMfma = V == 2 ? 2 : 1;           // MFMAs per 16-k step
  static constexpr int kOut = V == 0 ? 4 : V == 1 ? 8 : 16;  // outputs per lane
  static constexpr int kPer = kMax / 8;                  // row pieces per wave
  static constexpr int kUnits = 32 * kMfma;        // 1 KB operand units per chunk
};

// Layout 0: log2 of the second and third term's powers of two.  A scaled
// activation x is below 2^14, so the first fp16 term misses at most 4 of it and
// the second, of that times 2^13, 8: every term stays below 2^16.  The third has
// a resolution of 2^-48, the ulp of the binary32 numbers from 2^-25 on: from there
// up the three terms add up to x.
constexpr int kSkGain1 = 13, kSkGain2 = 24;
constexpr int kSkWindow = -25;

template <int V, int CW, int KW, int NBPS>
__global__ __launch_bounds__(kSkThreads) void k_nbits_skinny(
    const float *__restrict__ Aall, int64_t lda, const uint8_t *__restrict__ Wt,
    const float *__restrict__ ST, int ldsz, int nb, int bs_log2, int segs, int K, int kwrap,
    int Mall, int N, float *__restrict__ Yall, const float *__restrict__ bias, int nchunks, int cps,
    int nsl, int gy, float *__restrict__ part, int *__restrict__ tile_cnt) {
  using R = SkRows<V>;
  static_assert(CW * KW == 8, "eight waves");
  constexpr int kWS = kSkSegs / KW;   // segments of a chunk per k wave
  constexpr int kBN = 32 * CW;        // columns per workgroup
  constexpr int kJB = 4 / NBPS;       // 16-k steps per quantisation block
  extern __shared__ u4vec sk_smem[];  // operand units, then (reused) the k waves' tiles
  __shared__ int sex[R::kMax];        // piece exponents of the staged chunk
  __shared__ int srest[8];            // waves whose terms miss something (layout 0)
  kernarg_fence(Aall, lda, Wt, ST, ldsz, nb, bs_log2, segs, K, kwrap, Mall, N, Yall, bias, nchunks,
                cps, nsl, gy, part, tile_cnt);
  const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63, cl = lane & 31, g = lane >> 5;
  const int cw = wid % CW, kw = wid / CW;
  // slices of one tile are consecutive workgroups: they spread over the XCDs,
  // and with 8 slices an XCD's workgroups share one K range of A in its L2
  const int slice = blockIdx.x, n0 = blockIdx.y * kBN;
  const int m0 = blockIdx.z * R::kMax;  // a group of kMax rows
  const int M = min(Mall - m0, R::kMax);
  const float *A = Aall + (int64_t)m0 * lda;
  float *Y = Yall + (int64_t)m0 * N;
  const int c0 = slice * cps, c1 = min(c0 + cps, nchunks);
  // loads go through buffer resources: a fixed lane offset plus a scalar one
  const __amdgpu_buffer_rsrc_t w_rs =
      buf_rsrc(Wt + (int64_t)min((n0 >> 5) + cw, (N - 1) >> 5) * segs * 1024);
  const uint32_t soff = 4u * (uint32_t)min(n0 + 32 * cw + cl, N - 1);

  // ---- loads of one chunk (clamped addresses, nothing conditional per lane)
  struct Weights {
    u4vec w[kWS];
    float s[kWS][NBPS];
    uint32_t z[kWS][NBPS];
  };
  auto block_of = [&](int c, int i, int q) __attribute__((always_inline)) {
    return ((c * kSkSegs + kw * kWS + i) * kSegK + q * (kSegK / NBPS)) >> bs_log2;
  };
  auto load_w = [&](Weights &x, int c) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kWS; i++) {
      const int seg = min(c * kSkSegs + kw * kWS + i, segs - 1);
#pragma unroll
      for (int q = 0; q < NBPS; q++) {
        const __amdgpu_buffer_rsrc_t rs =
            buf_rsrc(ST + (int64_t)min(block_of(c, i, q), nb - 1) * 2 * ldsz);
        x.s[i][q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, soff, 0, 0));
        x.z[i][q] = __builtin_amdgcn_raw_buffer_load_b32(rs, soff, 4u * (uint32_t)ldsz, 0);
      }
      // non-temporal (aux 2), as ld_weights16
      x.w[i] = __builtin_bit_cast(u4vec, __builtin_amdgcn_raw_buffer_load_b128(
                                             w_rs, 16u * (uint32_t)lane, (uint32_t)seg * 1024u, 2));
    }
  };
  float av[R::kPer][8];
  // the column of A under row k of the weight (8-bit weights: two planes of kwrap
  // rows, a multiple of 64, over the same A)
  auto col_of = [&](int k) __attribute__((always_inline)) { return k < kwrap ? k : k - kwrap; };
  auto load_a = [&](int c) __attribute__((always_inline)) {
    const int kc = c * kSkChunk, k0 = col_of(kc + 8 * lane);
    // (buffer loads of four dwords need no more than dword alignment: rows of any
    // length and start.  Value by value where K % 8 or a row's alignment forbade the
    // aligned form, M = 54, (1999, 4083) took 36.3 us, M = 3, (859, 2142) 6.7; now
    // 15.2 and 4.7.)
    // four values that end past the row's end are read from its last four, and
    // moved to their places in trim(), which also drops those past the end (K >= 4)
    const uint32_t off0 = 4u * (uint32_t)min(k0, K - 4);
    const uint32_t off1 = 4u * (uint32_t)min(k0 + 4, K - 4);
#pragma unroll
    for (int i = 0; i < R::kPer; i++) {
      const __amdgpu_buffer_rsrc_t rs = buf_rsrc(A + (int64_t)min(wid + 8 * i, M - 1) * lda);
      const f4vec x0 =
          __builtin_bit_cast(f4vec, __builtin_amdgcn_raw_buffer_load_b128(rs, off0, 0, 0));
      const f4vec x1 =
          __builtin_bit_cast(f4vec, __builtin_amdgcn_raw_buffer_load_b128(rs, off1, 0, 0));
      av[i][0] = x0.x; av[i][1] = x0.y; av[i][2] = x0.z; av[i][3] = x0.w;
      av[i][4] = x1.x; av[i][5] = x1.y; av[i][6] = x1.z; av[i][7] = x1.w;
    }
  };
  // A chunk's pieces to LDS: lane l holds k = 8l .. 8l + 7, i.e. half l & 1 of
  // 16-k step u = l >> 1 (unit u of a part).  A unit's 32 rows are stored at
  // row ^ u: the 64 lanes of a piece write one row of 32 units, which without
  // it all fall on the same banks.
  // (Values that end past the row's end to their places, those past it dropped.)
  auto trim = [&](int c) __attribute__((always_inline)) {
    const int left = K - col_of(c * kSkChunk + 8 * lane);  // values of the lane inside K
    if (c * kSkChunk + kSkChunk > K) {                // uniform
#pragma unroll
      for (int i = 0; i < R::kPer; i++) {
        if (K & 3) {  // uniform: else no four values straddle the end
#pragma unroll
          for (int q = 0; q < 8; q += 4) {  // values q .. q + 3 were read 4 - n further on
            const int n = left - q;
            const float x0 = av[i][q], x1 = av[i][q + 1], x2 = av[i][q + 2], x3 = av[i][q + 3];
            av[i][q] = n == 1 ? x3 : n == 2 ? x2 : n == 3 ? x1 : x0;
            av[i][q + 1] = n == 2 ? x3 : n == 3 ? x2 : x1;
            av[i][q + 2] = n == 3 ? x3 : x2;
          }
        }
#pragma unroll
        for (int e = 0; e < 8; e++) av[i][e] = e < left ? av[i][e] : 0.0f;
      }
    }
  };
  // STORE: to LDS.  REST: av becomes what the terms miss (layout 0).
  auto stage = [&](auto STORE, auto REST) __attribute__((always_inline)) {
    const int u = lane >> 1, gg = lane & 1;
#pragma unroll
    for (int i = 0; i < R::kPer; i++) {
      const int row = wid + 8 * i;  // wave-uniform
      if (row >= M) break;
      // largest and (layout 0) smallest magnitude, NaN from a NaN; then the largest of
      // the wave's 64 lanes as an integer (NaN and infinities above every finite value)
      float mxa = fabsf(av[i][0]), mna = mxa;
#pragma unroll
      for (int e = 1; e < 8; e++) {
        mxa = __builtin_elementwise_maximum(mxa, fabsf(av[i][e]));
        if constexpr (V == 0 && !REST) mna = __builtin_elementwise_minimum(mna, fabsf(av[i][e]));
      }
      if constexpr (V == 0 && !REST) asm volatile("" : "+v"(mna));  // here, not where it is used
      uint32_t mu = __builtin_bit_cast(uint32_t, mxa);
      bool fin = true;
      mu = wave_max_u32(mu);
      if (mu >= 0x7F800000u) {  // uniform: scale by the largest finite magnitude
        fin = false;
        mu = 0;
#pragma unroll
        for (int e = 0; e < 8; e++)
          mu = max(mu, __builtin_bit_cast(uint32_t, finite_abs(av[i][e])));
        mu = wave_max_u32(mu);
      }
      const int ex = sk_exponent(mu);
      half2_t t[R::kParts][4];  // pairs (e, e + 4): the operand's k order
      constexpr int kUp[3] = {0, V == 0 ? kSkGain1 : 0, V == 0 ? kSkGain2 - kSkGain1 : 0};
#pragma unroll
      for (int e = 0; e < 4; e++) {
        f2vec x = {ldexpf(av[i][e], ex), ldexpf(av[i][e + 4], ex)};
        t[0][e] = __builtin_convertvector(x, half2_t);
#pragma unroll
        for (int p = 1; p < R::kParts; p++) {
          const float up = 1 << kUp[p];
          x.x = fmaf((float)t[p - 1][e].x, -up, x.x * up);
          x.y = fmaf((float)t[p - 1][e].y, -up, x.y * up);
          t[p][e] = __builtin_convertvector(x, half2_t);
        }
        if constexpr (REST) {
          // (below 2^-50 all terms are 0, and x may be subnormal and rounded; a row
          // with an infinity or NaN is one or the other in every column)
          const float tiny = ldexpf(1.0f, -50 - ex);
          x.x -= (float)t[2][e].x;
          x.y -= (float)t[2][e].y;
          av[i][e] = fabsf(av[i][e]) < tiny ? av[i][e] : ldexpf(x.x, -kSkGain2 - ex);
          av[i][e + 4] = fabsf(av[i][e + 4]) < tiny ? av[i][e + 4] : ldexpf(x.y, -kSkGain2 - ex);
          av[i][e] = fin ? av[i][e] : 0.0f;
          av[i][e + 4] = fin ? av[i][e + 4] : 0.0f;
        }
      }
      // of an infinity or NaN the first term alone, so that the sums follow IEEE (the
      // others, formed with it, are NaN)
      if (__builtin_expect(!fin, 0)) {  // uniform
        asm volatile("");  // a branch, not two selects a term in every piece
#pragma unroll
        for (int p = 1; p < R::kParts; p++)
#pragma unroll
          for (int e = 0; e < 4; e++) {
            t[p][e].x = t[p][e].x == t[p][e].x ? t[p][e].x : (_Float16)0.0f;
            t[p][e].y = t[p][e].y == t[p][e].y ? t[p][e].y : (_Float16)0.0f;
          }
      }
      if (STORE) {
        if (lane == 0) sex[row] = ex;
#pragma unroll
        for (int p = 0; p < R::kParts; p++) {
          const half8_t h = {t[p][0].x, t[p][0].y, t[p][1].x, t[p][1].y,
                             t[p][2].x, t[p][2].y, t[p][3].x, t[p][3].y};
          const int trow = V == 0 ? 8 * p + row : V == 1 ? 16 * p + row : row;
          const int unit = V == 2 ? u * 2 + p : u;
          sk_smem[unit * 64 + 32 * gg + (trow ^ u)] = __builtin_bit_cast(u4vec, h);
        }
      }
      if constexpr (V == 0 && !REST) {
        // whether the terms miss anything: a value other than 0 below the window (looked
        // at while the stores are under way)
        const float lim = ldexpf(1.0f, kSkWindow - ex);
        // (lanes past the row's end hold zeros only)
        if (fin && __builtin_amdgcn_ballot_w64((mna < lim) & (mxa > 0.0f)) != 0) {  // wave-uniform
          bool miss = false;
#pragma unroll
          for (int e = 0; e < 8; e++) miss |= fabsf(av[i][e]) < lim && av[i][e] != 0.0f;
          if (__builtin_amdgcn_ballot_w64(miss) != 0 && lane == 0) srest[wid] = 1;
        }
      }
    }
  };

  float tot[R::kOut];
#pragma unroll
  for (int i = 0; i < R::kOut; i++) tot[i] = 0.0f;
  uint32_t k0f = 0x000F000Fu, kf0 = 0x00F000F0u, magic = 0x64006400u;
  asm volatile("" : "+s"(k0f), "+s"(kf0));
  asm volatile("" : "+v"(magic));
  const float16_t zero16 = {};

  // segments multiplied together: independent accumulators, so that a step's
  // MFMA does not wait for the one before it
  constexpr int kG = kWS < 2 ? 1 : 2;
  auto multiply = [&](const int c, const Weights &wc) __attribute__((always_inline)) {
    float acc[16];
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
#pragma unroll
    for (int i0 = 0; i0 < kWS; i0 += kG) {
      half8_t a[kG][4][R::kMfma];
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int ii = 0; ii < kG; ii++)
#pragma unroll
          for (int p = 0; p < R::kMfma; p++) {
            const int u = (kw * kWS + i0 + ii) * 4 + j;
            const int unit = V == 2 ? u * 2 + p : u;
            a[ii][j][p] = __builtin_bit_cast(half8_t, sk_smem[unit * 64 + 32 * g + (cl ^ u)]);
          }
      float16_t D[kG];
#pragma unroll
      for (int j = 0; j < 4; j++) {
#pragma unroll
        for (int ii = 0; ii < kG; ii++) {
          const half8_t b = sk_dequant(wc.w[i0 + ii][j], (int)wc.z[i0 + ii][j / kJB], k0f, kf0,
                                      magic);
#pragma unroll
          for (int p = 0; p < R::kMfma; p++)
            D[ii] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                a[ii][j][p], b, j % kJB == 0 && p == 0 ? zero16 : D[ii], 0, 0, 0);
        }
        if ((j + 1) % kJB == 0) {
#pragma unroll
          for (int ii = 0; ii < kG; ii++) {
            // blocks past the last hold zero activations; their (clamped)
            // scale is dropped, so that whatever it is cannot matter
            const int q = j / kJB;
            const float s = block_of(c, i0 + ii, q) < nb ? wc.s[i0 + ii][q] : 0.0f;
#pragma unroll
            for (int r = 0; r < (V == 0 ? 12 : 16); r++) acc[r] = fmaf(s, D[ii][r], acc[r]);
          }
        }
      }
    }
    // parts (smallest first) and the piece's power of two: row of output i of
    // lane group g is 8 (i / 4) + 4 g + i % 4 of the wave's tile
#pragma unroll
    for (int i = 0; i < R::kOut; i++) {
      const int row = (i >> 2) * 8 + g * 4 + (i & 3);
      float v = acc[i];
      if constexpr (V == 0) v = fmaf(fmaf(acc[8 + i], 0x1p-11f, acc[4 + i]), 0x1p-13f, acc[i]);
      if constexpr (V == 1) v = acc[8 + i] + acc[i];
      tot[i] += ldexpf(v, -sex[row]);
    }
  };
  const std::true_type yes;
  const std::false_type no;
  if (V == 0 && lane == 0) srest[wid] = 0;
  int rest = 0;  // srest of wave lane % 8
  Weights w0;
  load_a(c0);
  load_w(w0, c0);
  for (int c = c0; c < c1; c++) {
    trim(c);
    stage(yes, no);
    // the next chunk's loads go out before this one is multiplied, the
    // activations first: the next stage() waits for them alone.  (The weights are
    // moved, not alternated between two copies of the loop's code: M = 8, (4096,
    // 14336) 16.4 -> 14.6 us, (1024, 1024) 4.75 -> 4.6.)
    Weights wc;
    // (explicit moves, before the loads: the compiler puts its own behind them, with a
    // wait for them)
    auto move_w = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < kWS; i++) {
#pragma unroll
        for (int d = 0; d < 4; d++) wc.w[i][d] = sk_move(w0.w[i][d]);
#pragma unroll
        for (int q = 0; q < NBPS; q++) {
          wc.s[i][q] =
              __builtin_bit_cast(float, sk_move(__builtin_bit_cast(uint32_t, w0.s[i][q])));
          wc.z[i][q] = sk_move(w0.z[i][q]);
        }
      }
    };
    if (c + 1 < c1) {  // uniform
      load_a(c + 1);
      move_w();
      load_w(w0, c + 1);
    } else {
      move_w();
    }
    sk_lds_barrier();
    if constexpr (V == 0) {  // (read here, needed after the last chunk)
      rest = srest[lane & 7];
    }
    multiply(c, wc);
    sk_lds_barrier();  // every wave is done with the staged chunk
  }
  if constexpr (V == 0) {
    auto any_rest = [&]() __attribute__((always_inline)) {  // of the workgroup
      return __builtin_amdgcn_ballot_w64(rest != 0) != 0;
    };
    if (__builtin_expect(any_rest(), 0)) {
      for (int c = c0; c < c1; c++) {
        load_a(c);
        trim(c);
        stage(no, yes);
        while (true) {
          int nz = 0;
#pragma unroll
          for (int e = 0; e < 8; e++) nz |= av[0][e] != 0.0f;
          nz = __any(nz) && wid < M;
          sk_lds_barrier();  // every wave has read srest
          if (lane == 0) srest[wid] = nz;
          sk_lds_barrier();
          rest = srest[lane & 7];
          if (!any_rest()) break;
          stage(yes, yes);  // (zeros in the rows with nothing left)
          load_w(w0, c);
          sk_lds_barrier();
          multiply(c, w0);
          sk_lds_barrier();
        }
      }
    }
  }

  // ---- the k waves' tiles -> LDS [kw][row][kBN], summed by all threads
  float *red = (float *)sk_smem;
#pragma unroll
  for (int i = 0; i < R::kOut; i++) {
    const int row = (i >> 2) * 8 + g * 4 + (i & 3);
    red[(kw * R::kMax + row) * kBN + 32 * cw + cl] = tot[i];
  }
  __syncthreads();
  const int total = M * kBN;
  const int tile = blockIdx.z * gy + blockIdx.y;  // its partials and counter
  float *pt = part + (int64_t)tile * nsl * (R::kMax * kBN);
  for (int e = threadIdx.x; e < total; e += kSkThreads) {
    // in double: a k wave of 32-column workgroups rounds every block's scaled
    // partial by itself, and the sum in binary32 on top made the result 4%
    // less accurate than the GEMM's (K = 1024: 9.9e-8 against 9.5e-8)
    double sum = red[e];
#pragma unroll
    for (int q = 1; q < KW; q++) sum += (double)red[q * R::kMax * kBN + e];
    const float v = (float)sum;
    if (nsl == 1) {
      const int cc = n0 + e % kBN;
      if (cc < N) Y[(int64_t)(e / kBN) * N + cc] = bias ? v + bias[cc] : v;
    } else {
      st_act<true>(pt + slice * (R::kMax * kBN) + e, v);
    }
  }
  if (nsl == 1) return;
  // every thread's partial stores complete before thread 0 counts in
  // (release); the last slice acquires what the others released
  __shared__ int s_last;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) {
    const int prev =
        __hip_atomic_fetch_add(&tile_cnt[tile], 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    s_last = prev == nsl - 1;
    if (s_last) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
  if (!s_last) return;  // whole workgroup
  for (int e = threadIdx.x; e < total; e += kSkThreads) {
    float t[kSkMaxSlices];
#pragma unroll
    for (int q = 0; q < kSkMaxSlices; q++)
      t[q] = ld_act<true>(pt + min(q, nsl - 1) * (R::kMax * kBN) + e);
    double sum = t[0];
#pragma unroll
    for (int q = 1; q < kSkMaxSlices; q++) sum += q < nsl ? (double)t[q] : 0.0;
    const float v = (float)sum;
    const int cc = n0 + e % kBN;
    if (cc < N) Y[(int64_t)(e / kBN) * N + cc] = bias ? v + bias[cc] : v;
  }
  if (threadIdx.x == 0)
    __hip_atomic_store(&tile_cnt[tile], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int V, int CW, int KW>
static int launch_skinny(mmnb_ctx *ctx, const mmnb_pack *p, const float *d_a, int64_t lda,
                         int64_t m, float *d_y, int nsl, bool wrap) {
  using R = SkRows<V>;
  const int64_t n = p->n;
  const int tiles = (int)((n + 32 * CW - 1) / (32 * CW));
  const int nchunks = (int)((p->k + kSkChunk - 1) / kSkChunk);
  // whole chunks per slice, no slice empty
  const int cps = (nchunks + nsl - 1) / nsl;
  nsl = (nchunks + cps - 1) / cps;
  const int k = (int)(wrap ? p->k_in : p->k), kwrap = (int)(wrap ? p->k / 2 : INT32_MAX);
  const size_t red = (size_t)KW * R::kMax * 32 * CW * 4;
  const size_t shmem = std::max<size_t>((size_t)R::kUnits * 1024, red);  // 64 KB at most
  int bs_log2 = 0;
  while ((int64_t(1) << (bs_log2 + 1)) <= p->block) bs_log2++;
  const dim3 grid((unsigned)nsl, (unsigned)tiles, (unsigned)((m + R::kMax - 1) / R::kMax));
#define MMNB_SKINNY(Q)                                                                        \
  {                                                                                           \
    auto kern = k_nbits_skinny<V, CW, KW, Q>;                                                 \
    return launch(ctx, kKernSkinny, kern, grid, dim3(kSkThreads), shmem, d_a, lda,            \
                  (const uint8_t *)p->d_wt,                                                   \
                  (const float *)p->d_st, (int)p->ldsz, (int)p->n_blocks, bs_log2,            \
                  (int)(p->k64 / kSegK), k, kwrap, (int)m, (int)n,                             \
                  d_y, p->direct_bias(), nchunks, cps, nsl, tiles, ctx->d_sk_part,            \
                  ctx->d_gemm_cnt);                                                           \
  }
  if (p->block >= 64) MMNB_SKINNY(1);
  if (p->block == 32) MMNB_SKINNY(2);
  MMNB_SKINNY(4);
#undef MMNB_SKINNY
}

// Column waves and K slices of a call, and whether it should take this path.
//   - up to two chunks of K: 32-column workgroups without slices (every k wave
//     one segment) while they fit the CUs, else 64-column ones (us at M = 16,
//     (1024, 4096): 5.4 against 7.3; M = 256, (1024, 2048), 512 and 256
//     workgroups: 14.0 against 9.2);
//   - three or four chunks: 64 columns with a slice per chunk when all of it
//     stays below one round of the CUs (M = 2, (2048, 2048): 5.6 against 6.6; M = 5,
//     (1999, 4083), 256 workgroups: 7.8 against 7.2; with more than 16 rows in short
//     blocks also where it is the round, M = 33, 2048^2, block 32: 10.3 against 11.0),
//     else as above;
//   - longer K: 64 columns and the slices that fill the CUs (M = 24, 4096^2:
//     12.6 with 4 slices, 17.5 with 2, 19.3 with 8; 128-column workgroups 21
//     and more, their registers spill).
// It takes all calls of up to 16 rows that the multi-row GEMV does not (M = 12, (4096,
// 28672): 37.5 against the GEMM's 39.5; M = 16, (28672, 8192) 63 against 64).  Up to
// 32 rows while one round of the CUs holds the columns (M = 20, N = 14336 26.7 against
// 29.2, but M = 17, N = 28672 49.6 against 40.0) and a workgroup has at most 8 chunks,
// 10 where its columns fill three quarters of the CUs (M = 32, (4608, 13824) 26.8 against
// 29.0, (5120, 13824) 29.4 against 30.4, but (5120, 10240) 28.8 against 27.3, (16384,
// 16384), 32 chunks, 92 against 77), or, of four slices and more, whose columns the GEMM's
// tiles leave CUs idle for, 14 ((28672, 4096), block 16 54 against 59).  With more rows,
// i.e. several row groups, for at most 4 chunks of one round (M = 64, 4096^2: 17.9
// against 19.9; 28 with the 8 chunks of one slice) or one chunk, more than three eighths
// filled, of two (M = 2048, 512^2: 10.8 against 20.4; M = 256, N = 4096, K = 256 9.8
// against 10.0, K = 128 9.8 against 8.7; four rounds, M = 100, (512, 14336): 19.6 against
// 13.2).  Blocks of 16 fill the registers of the two-pass layout: of more than 32 rows
// two chunks at most in 64-column workgroups (M = 64, 4096^2, four: 30.2 against 23.6; but
// (2048, 4096), four in 32-column ones, 12.0 against 17.9; M = 32, (4096, 14336), eight,
// 29.6 against 32.5).
bool nbits_skinny_plan(const mmnb_ctx *ctx, const mmnb_pack *p, int64_t m, int *cw, int *nsl) {
  if (p->generic || m < 2 || !p->few_rows()) return false;
  const int64_t cus = ctx->cu_count, chunks = (p->k + kSkChunk - 1) / kSkChunk;
  const int64_t rows = (m + kSkRows - 1) / kSkRows;
  const int64_t g1 = (p->n + 31) / 32 * rows, g2 = (p->n + 63) / 64 * rows;
  const bool round = m <= 16 || p->block >= 64 ? g2 * chunks >= cus : g2 * chunks > cus;
  *cw = chunks <= 4 && g1 <= cus && (chunks <= 2 || round) ? 1 : 2;
  *nsl = *cw == 1 || g2 > cus
             ? 1
             : (int)std::min<int64_t>({cus / g2, chunks, (int64_t)kSkMaxSlices});
  if (m <= 16) return true;
  const int64_t cps = (chunks + *nsl - 1) / *nsl;
  if (g2 > cus) return g2 <= 2 * cus && cps == 1 && p->k > 3 * kSkChunk / 8;
  if (m > kSkRows) return cps <= (p->block == 16 && *cw == 2 ? 2 : 4);
  return cps <= (*nsl >= 4 ? 14 : 4 * g2 > 3 * cus ? 10 : 8);
}

bool nbits_skinny_sizes(const mmnb_pack *p) {
  // 31-bit column offsets, 32-bit unit offsets, grid.y
  return p->n <= ((int64_t)1 << 21) && p->k64 <= ((int64_t)1 << 26);
}

int launch_nbits_skinny(mmnb_ctx *ctx, const mmnb_pack *p, const float *d_a, int64_t lda,
                        int64_t m, float *d_y, int cw, int nsl, bool wrap) {
  if (cw == 1) {
    if (m <= 8) return launch_skinny<0, 1, 8>(ctx, p, d_a, lda, m, d_y, nsl, wrap);
    if (m <= 16) return launch_skinny<1, 1, 8>(ctx, p, d_a, lda, m, d_y, nsl, wrap);
    return launch_skinny<2, 1, 8>(ctx, p, d_a, lda, m, d_y, nsl, wrap);
  }
  if (m <= 8) return launch_skinny<0, 2, 4>(ctx, p, d_a, lda, m, d_y, nsl, wrap);
  if (m <= 16) return launch_skinny<1, 2, 4>(ctx, p, d_a, lda, m, d_y, nsl, wrap);
  return launch_skinny<2, 2, 4>(ctx, p, d_a, lda, m, d_y, nsl, wrap);
}

}  // namespace mmnb
