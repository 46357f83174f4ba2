// MatMulNBits beyond the reference's 4-bit form: bits = 8, g_idx
// (act-order groups), bias, floating-point zero points, fp16 scales and
// bias, and ORT's per-column zero-point layout.
//
// Everything is mapped onto the 4-bit kernels at pack time ("virtual"
// 4-bit weight of Kv rows), plus an optional A gather before and one
// correction pass after the product:
//
//   bits = 8:  q8 = 16 hi + lo.  The virtual weight stacks the hi plane (scale
//              16 s, exact) over the lo plane (scale s), over Kv = 2 * kp rows (kp:
//              K padded to whole blocks and 64-k segments).  Without zero points
//              (q8 - 128) s = (hi - 8)(16 s) + lo s: the planes have zero points 8
//              and 0, the kernels read A again from row kp on, and no correction is
//              left.  Otherwise both planes have zero point 8, A is gathered as
//              [A | A], and (136 - z) s is the correction below (zero points z / 16
//              and z % 16 in the planes need none, but the larger terms left the GEMM
//              5% further from the 64-bit product).  One row with integer zero points
//              takes k_gemv8, on the joined bytes.
//   float zp:  (q - z) s = q s - z s: the kernels run with zero point 0 and
//              the correction adds -z s per block.
//   g_idx:     the rows are sorted by group (stable), so every group is one
//              block of the virtual weight; A is gathered in the same order.
//              Each group must hold exactly block_size rows.
//   bias:      added where the kernels store a result, or in the correction pass
//              where there is one.
//
// Correction: y[m, n] += bias[n] + sum_b c[b][n] * asum[m][b], with asum the
// block sums of the (gathered) A over the first corr_nb blocks.  c is built
// in double and rounded once to fp32.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "mmnb_device.h"
#include "mmnb_host.h"
#include "mmnb_internal.h"

using namespace mmnb;

namespace mmnb {

// out[m, j] = A[m, src[j]] for j < kv (src[j] < 0: 0), zero for kv <= j < ldo.
__global__ __launch_bounds__(256) void k_gather_a(const float *__restrict__ A, int64_t lda,
                                                  int64_t M, const int32_t *__restrict__ src,
                                                  int64_t kv, int64_t ldo,
                                                  float *__restrict__ out) {
  const int64_t total = M * ldo;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t m = i / ldo, j = i % ldo;
    const int s = src[j < kv ? j : 0];
    const bool ok = j < kv && s >= 0;
    const float v = A[m * lda + (ok ? s : 0)];
    out[i] = ok ? v : 0.0f;
  }
}

// asum[m][b] = sum of A[m, b*bs .. min((b+1)*bs, ka) - 1]; one wave per (b, m).
__global__ __launch_bounds__(64) void k_block_sums(const float *__restrict__ A, int64_t lda,
                                                   int64_t ka, int64_t bs, int64_t nb,
                                                   float *__restrict__ asum) {
  const int64_t b = blockIdx.x, m = blockIdx.y;
  const int64_t k0 = b * bs, k1 = std::min(ka, k0 + bs);
  float s = 0.0f;
  for (int64_t kk = k0 + threadIdx.x; kk < k1; kk += 64) s += A[m * lda + kk];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (threadIdx.x == 0) asum[m * nb + b] = s;
}

// y[m, n] += bias[n] + sum_b corr[b][n] * asum[m][b]
__global__ __launch_bounds__(256) void k_nbits_correct(float *__restrict__ Y, int64_t N,
                                                       const float *__restrict__ bias,
                                                       const float *__restrict__ corr,
                                                       int64_t nb,
                                                       const float *__restrict__ asum) {
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, m = blockIdx.y;
  if (n >= N) return;
  float v = bias ? bias[n] : 0.0f;
  if (corr) {
    const float *as = asum + m * nb;
    for (int64_t b = 0; b < nb; b++) v = fmaf(corr[b * N + n], as[b], v);
  }
  Y[m * N + n] += v;
}

// The same correction for few rows, with the block sums of row m formed in
// LDS by the workgroup itself (one launch instead of two; every column
// workgroup re-reads its row, which is cheap for M <= 8).  A workgroup takes
// 64 columns; its 4 waves split the blocks (wave w: b = w, w + 4, ...) with
// eight loads of corr in flight per lane, then add their partial sums in a
// fixed order through LDS (a single chain over all blocks waited on every
// load in turn).
constexpr int kFusedMaxBlocks = 8192;
constexpr int kCorrCols = 64;

__global__ __launch_bounds__(256) void k_nbits_correct_rows(
    float *__restrict__ Y, int64_t N, const float *__restrict__ bias,
    const float *__restrict__ corr, int64_t nb, const float *__restrict__ A, int64_t lda,
    int64_t ka, int64_t bs) {
  __shared__ float sas[kFusedMaxBlocks];
  __shared__ float spart[4][kCorrCols];
  const int64_t m = blockIdx.y;
  const int w = threadIdx.x >> 6, ln = threadIdx.x & 63;
  if (corr) {
    for (int64_t b = w; b < nb; b += 4) {
      const int64_t k0 = b * bs, k1 = std::min(ka, k0 + bs);
      float s = 0.0f;
      for (int64_t kk = k0 + ln; kk < k1; kk += 64) s += A[m * lda + kk];
      for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
      if (ln == 0) sas[b] = s;
    }
    __syncthreads();
  }
  const int64_t n = (int64_t)blockIdx.x * kCorrCols + ln;
  const int64_t nc = n < N ? n : N - 1;
  float v = 0.0f;
  if (corr) {
    int64_t b = w;
    for (; b + 28 < nb; b += 32) {
      float c[8];
#pragma unroll
      for (int u = 0; u < 8; u++) c[u] = corr[(b + 4 * u) * N + nc];
#pragma unroll
      for (int u = 0; u < 8; u++) v = fmaf(c[u], sas[b + 4 * u], v);
    }
    for (; b < nb; b += 4) v = fmaf(corr[b * N + nc], sas[b], v);
  }
  spart[w][ln] = v;
  __syncthreads();
  if (w == 0 && n < N) {
    float t = bias ? bias[n] : 0.0f;
    t += ((spart[0][ln] + spart[1][ln]) + spart[2][ln]) + spart[3][ln];
    Y[m * N + n] += t;
  }
}

// ---------------------------------------------------------------------------
// One row of 8-bit weights with integer zero points, in one launch: the GEMV of
// k_gemv_valu on the virtual weight's two planes at once.  A lane reads the
// high and the low nibbles of the same 32 k of a column (one 16-byte chunk
// each), joins them into bytes and multiplies the exact q - z, so A is neither
// gathered nor corrected for, and the bias is added where the column is stored.
//
// Bound by the weight stream once K * N fills the chip, by the launch below
// that.  R columns per lane as in k_gemv_valu, each of two chunks: R = 2.
// K = N = 4096, block 128, bias: 14.8 us (gather of A, GEMV of the virtual weight,
// correction) -> 5.1 us back to back, 3.4 TB/s of weights and scales.
// ---------------------------------------------------------------------------
constexpr int kGemv8Waves = 4;
typedef float gemv8_f4 __attribute__((ext_vector_type(4), aligned(4)));

template <int R, int NBPC, bool HAS_ZP, bool FAST>
__global__ __launch_bounds__(64 * kGemv8Waves) void k_gemv8(
    const float *__restrict__ A, const uint8_t *__restrict__ W, int64_t col_bytes,
    const float *__restrict__ S, const uint8_t *__restrict__ Z, const float *__restrict__ bias,
    int nb, int bs_log2, int K, int N, float *__restrict__ Y, int C, int iters, int nbv) {
  __shared__ float red[kGemv8Waves][2 * R];
  kernarg_fence(A, W, col_bytes, S, Z, bias, nb, bs_log2, K, N, Y, C, iters, nbv, blockDim.x);
  const int nw = blockDim.x >> 6;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int h = l >> 5, t = l & 31;
  const int col0 = blockIdx.x * (2 * R);
  int colr[R];
#pragma unroll
  for (int r = 0; r < R; r++) colr[r] = min(col0 + 2 * r + h, N - 1);
  // without a bias its pointer is the scales': read and not used
  const float bv = bias[min(col0 + (int)threadIdx.x, N - 1)];
  float acc[R];
#pragma unroll
  for (int r = 0; r < R; r++) acc[r] = 0.0f;
  for (int it = 0; it < iters; it++) {
    const int c = 32 * w + t + it * 32 * nw;
    const bool cv = c < C;
    const int cc = cv ? c : 0;
    const int s = cc >> 1, g = cc & 1;
    float av[32];
    const float *ar = A + s * kSegK + 8 * g;
    if constexpr (FAST) {
      load_chunk32_paired(ar, h, av);
    } else {
      // rows that do not fill the plane or start off 16 bytes: four values at a time
      // (dword-aligned loads); those that end past the row are its last four, moved to
      // their places below.  (Value by value, 32 loads a lane, block 128: K = 1000, N =
      // 14336 15.1 us and the former gather, GEMV and correction 10.6; now 5.9.  K =
      // 4000, N = 14336 56.4 and 22.5; now 15.2.  K = 1000, N = 4096 5.8 and 8.6; 3.8.)
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int k = s * kSegK + 8 * g + 16 * (i >> 1) + 4 * (i & 1);
        if (K >= 4) {  // uniform
          const gemv8_f4 x = *(const gemv8_f4 *)(A + min(k, K - 4));
#pragma unroll
          for (int e = 0; e < 4; e++) av[4 * i + e] = x[e];
        } else {
#pragma unroll
          for (int e = 0; e < 4; e++) av[4 * i + e] = A[max(K - 4 + e, 0)];
        }
      }
    }
    float sraw[R][NBPC], zraw[R][NBPC];
    bool inb[NBPC];
#pragma unroll
    for (int q = 0; q < NBPC; q++) {
      const int kq = s * kSegK + 16 * (q * (4 / NBPC)) + (NBPC == 4 ? 8 * g : 0);
      int blk = kq >> bs_log2;
      inb[q] = cv && blk < nb;
      blk = blk < nb ? blk : nb - 1;
#pragma unroll
      for (int r = 0; r < R; r++) {
        sraw[r][q] = S[(int64_t)colr[r] * nbv + (nbv >> 1) + blk];
        zraw[r][q] = HAS_ZP ? (float)Z[(int64_t)colr[r] * nb + blk] : 128.0f;
      }
    }
    u4vec wh[R], wl[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
      const uint8_t *wc = W + (int64_t)colr[r] * col_bytes + (int64_t)cc * 16;
      wh[r] = ld_weights16(wc);
      wl[r] = ld_weights16(wc + (col_bytes >> 1));
    }
    // every load in flight before any arithmetic, column by column after it
    // (as k_gemv_valu)
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!FAST) {
#pragma unroll
      for (int i = 0; i < 32; i += 4) {
        // n values inside the row, read 4 - n further on where n < 4
        const int n = cv ? K - (s * kSegK + 8 * g + 16 * (i >> 3) + (i & 4)) : 0;
        const float x0 = av[i], x1 = av[i + 1], x2 = av[i + 2], x3 = av[i + 3];
        const float y0 = n == 1 ? x3 : n == 2 ? x2 : n == 3 ? x1 : x0;
        const float y1 = n == 2 ? x3 : n == 3 ? x2 : x1, y2 = n == 3 ? x3 : x2;
        av[i] = n > 0 ? y0 : 0.0f;
        av[i + 1] = n > 1 ? y1 : 0.0f;
        av[i + 2] = n > 2 ? y2 : 0.0f;
        av[i + 3] = n > 3 ? x3 : 0.0f;
      }
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
#pragma unroll
      for (int q = 0; q < NBPC; q++) {
        float d = 0.0f;
#pragma unroll
        for (int jj = 0; jj < 4 / NBPC; jj++) {
          const int j = q * (4 / NBPC) + jj;
          const uint32_t hi = wh[r][j], lo = wl[r][j];
          uint32_t ev = ((hi << 4) & 0xF0F0F0F0u) | (lo & 0x0F0F0F0Fu);
          uint32_t od = (hi & 0xF0F0F0F0u) | ((lo >> 4) & 0x0F0F0F0Fu);
          float qv[8];
          if constexpr (HAS_ZP) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
              qv[2 * e] = (float)((ev >> (8 * e)) & 255u) - zraw[r][q];
              qv[2 * e + 1] = (float)((od >> (8 * e)) & 255u) - zraw[r][q];
            }
          } else {
            ev ^= 0x80808080u;
            od ^= 0x80808080u;
            qv[0] = sbyte_f32<0>(ev); qv[1] = sbyte_f32<0>(od);
            qv[2] = sbyte_f32<1>(ev); qv[3] = sbyte_f32<1>(od);
            qv[4] = sbyte_f32<2>(ev); qv[5] = sbyte_f32<2>(od);
            qv[6] = sbyte_f32<3>(ev); qv[7] = sbyte_f32<3>(od);
          }
#pragma unroll
          for (int e = 0; e < 8; e++) d = fmaf(av[8 * j + e], qv[e], d);
        }
        acc[r] = inb[q] ? fmaf(sraw[r][q], d, acc[r]) : acc[r];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int r = 0; r < R; r++) {
    const float v = half_wave_sum(acc[r]);
    if (t == 0) red[w][2 * r + h] = v;
  }
  __syncthreads();
  if ((int)threadIdx.x < 2 * R) {
    float v = 0.0f;
    for (int ww = 0; ww < nw; ww++) v += red[ww][threadIdx.x];
    const int col = col0 + threadIdx.x;
    if (col < N) Y[col] = bias != S ? v + bv : v;
  }
}

template <int R, int NBPC>
static int launch_gemv8_r(mmnb_ctx *ctx, const mmnb_pack *p, const float *d_a, bool fast,
                          float *d_y) {
  const int C = (int)(p->col_bytes / 32);  // chunks of a plane
  int nw = (C + 31) / 32, iters = 1;
  if (nw > kGemv8Waves) {
    iters = (nw + kGemv8Waves - 1) / kGemv8Waves;
    nw = (C + 32 * iters - 1) / (32 * iters);
  }
  const int64_t n = p->n;
  const dim3 grid((unsigned)((n + 2 * R - 1) / (2 * R))), block((unsigned)(64 * nw));
  int bs_log2 = 0;
  while ((int64_t(1) << bs_log2) < p->block) bs_log2++;
  const float *bias = p->d_bias ? p->d_bias : p->d_scales;
#define MMNB_GEMV8(ZP, F)                                                                     \
  return launch(ctx, kKernGemv8, k_gemv8<R, NBPC, ZP, F>, grid, block, 0, d_a, p->d_w,         \
                p->col_bytes, p->d_scales, p->d_z8, bias, (int)p->nb8, bs_log2,               \
                (int)p->k_in, (int)n, d_y, C, iters, (int)p->n_blocks)
  if (p->d_z8) {
    if (fast) MMNB_GEMV8(true, true);
    MMNB_GEMV8(true, false);
  }
  if (fast) MMNB_GEMV8(false, true);
  MMNB_GEMV8(false, false);
#undef MMNB_GEMV8
}

static int launch_gemv8(mmnb_ctx *ctx, const mmnb_pack *p, const float *d_a, int64_t lda,
                        float *d_y) {
  // float4 loads of whole chunks where the row fills the plane (col_bytes rows
  // of the virtual weight); past K the joined bytes are not the zero point, so
  // there the kernel zeroes the activations
  const bool fast = lda % 4 == 0 && ((uintptr_t)d_a & 15) == 0 && p->k_in == p->col_bytes;
  if (p->block >= 64) return launch_gemv8_r<2, 1>(ctx, p, d_a, fast, d_y);
  if (p->block == 32) return launch_gemv8_r<2, 2>(ctx, p, d_a, fast, d_y);
  return launch_gemv8_r<2, 4>(ctx, p, d_a, fast, d_y);
}

int run_matmul_nbits(mmnb_ctx *ctx, const mmnb_pack *p, const float *d_a, int64_t lda,
                     int64_t m, float *d_y) {
  if (!p->ext) return launch_matmul_nbits(ctx, p, d_a, lda, m, d_y);
  // (several rows one by one where there is no few-row kernel)
  if (p->bytes8 && (m == 1 || (m <= 8 && !p->few_rows()))) {
    int rc = MMNB_OK;
    for (int64_t r = 0; r < m && rc == MMNB_OK; r++)
      rc = launch_gemv8(ctx, p, d_a + r * lda, lda, d_y + r * p->n);
    return rc;
  }
  // without gather and correction the kernels take A and the bias themselves (us a
  // call with the passes and without, block 128: 8 bits, bias, M = 8, 4096^2 34.2 and
  // 12.0; M = 24 39.2 and 18.4; M = 512 120 and 78; M = 24, 1024^2 21.2 and 8.9; 4
  // bits, bias, M = 8, (1000, 3001) 8.8 and 4.8)
  if (p->direct())
    return m > 1 ? launch_matmul_nbits(ctx, p, d_a, lda, m, d_y)
                 : launch_gemv_bias(ctx, p, d_a, lda, d_y);
  int rc;
  const float *a2 = d_a;
  int64_t lda2 = lda, ka = p->k_in;
  // the few-row kernel reads the planes' A twice by itself (block 128, M = 8, (1000,
  // 4096): 14.1 us with the gather, 11.3 without)
  const bool planes = p->bytes8 && launch_nbits_planes(ctx, p, d_a, lda, m, d_y, &rc);
  if (planes && rc) return rc;
  if (p->d_asrc && !planes) {
    void *buf = nullptr;
    if ((rc = scratch_get(ctx, 9, (size_t)(m * p->k64) * 4, &buf))) return rc;
    int64_t blocks = (m * p->k64 + 255) / 256;
    blocks = std::max<int64_t>(1, std::min<int64_t>(blocks, 16384));
    if ((rc = launch(ctx, kKernNbitsEx, k_gather_a, dim3((unsigned)blocks), dim3(256), 0, d_a, lda,
                     m, (const int32_t *)p->d_asrc, p->k, p->k64, (float *)buf)))
      return rc;
    a2 = (const float *)buf;
    lda2 = p->k64;
    ka = p->k;
  }
  if (!planes && (rc = launch_matmul_nbits(ctx, p, a2, lda2, m, d_y))) return rc;
  if (m <= 8 && p->corr_nb <= kFusedMaxBlocks)
    return launch(ctx, kKernNbitsEx, k_nbits_correct_rows,
                  dim3((unsigned)((p->n + kCorrCols - 1) / kCorrCols), (unsigned)m), dim3(256), 0,
                  d_y, p->n,
                  (const float *)p->d_bias, (const float *)p->d_corr, p->corr_nb, a2, lda2, ka,
                  p->block);
  const float *d_asum = nullptr;
  if (p->d_corr) {
    void *buf = nullptr;
    if ((rc = scratch_get(ctx, 7, (size_t)(m * p->corr_nb) * 4, &buf))) return rc;
    if ((rc = launch(ctx, kKernNbitsEx, k_block_sums, dim3((unsigned)p->corr_nb, (unsigned)m),
                     dim3(64), 0, a2, lda2, ka, p->block, p->corr_nb, (float *)buf)))
      return rc;
    d_asum = (const float *)buf;
  }
  return launch(ctx, kKernNbitsEx, k_nbits_correct,
                dim3((unsigned)((p->n + 255) / 256), (unsigned)m), dim3(256), 0, d_y, p->n,
                (const float *)p->d_bias, (const float *)p->d_corr, p->corr_nb, d_asum);
}

}  // namespace mmnb

namespace {

template <typename T>
int upload(mmnb_pack *p, const std::vector<T> &v, T **dst) {
  int rc = device_alloc(v.size() * sizeof(T), (void **)dst);
  if (rc) return rc;
  MMNB_HIP(hipMemcpy(*dst, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  p->bytes += (int64_t)(v.size() * sizeof(T));
  return MMNB_OK;
}

}  // namespace

int mmnb_pack_nbits_ex(mmnb_ctx *ctx, const mmnb_nbits_desc *d, mmnb_pack **out) {
  MMNB_GUARD_CTX(ctx);
  if (!out || !d) return fail(MMNB_ERR_ARG, "mmnb_pack_nbits_ex: null argument");
  *out = nullptr;
  // validation and the virtual 4-bit weight: host code (mmnb_host.cpp)
  NbitsHost h;
  int rc = nbits_prepare(d, &h);
  if (rc) return rc;
  mmnb_pack *p = nullptr;
  int urc = MMNB_OK;
  {
    CtxLock lk(ctx);
    if ((rc = set_device(ctx))) return rc;
    // the reference's own form takes any even block size (pack_nbits_any);
    // the extensions run on power-of-two blocks (nbits_prepare checks)
    const bool plain = h.asrc.empty() && h.corr.empty() && h.bias.empty() && !h.planes;
    const uint8_t *vz = h.vz.empty() ? nullptr : h.vz.data();
    rc = plain ? pack_nbits_any(ctx, h.vb.data(), h.vs.data(), vz, h.zfill, h.kv, h.n, h.block, &p)
               : pack_nbits_core(ctx, h.vb.data(), h.vs.data(), vz, h.zfill, h.kv, h.n, h.block,
                                 &p);
    if (rc) return rc;
    p->k_in = h.k;
    p->ext = !plain;
    if (!h.asrc.empty()) urc = upload(p, h.asrc, &p->d_asrc);
    if (!urc && !h.corr.empty()) {
      std::vector<float> c32(h.corr.begin(), h.corr.end());
      urc = upload(p, c32, &p->d_corr);
      p->corr_nb = h.n_blocks;
    }
    if (!urc && !h.bias.empty()) urc = upload(p, h.bias, &p->d_bias);
    p->bytes8 = h.bytes8;
    p->nb8 = h.n_blocks;
    if (!urc && !h.z8.empty()) urc = upload(p, h.z8, &p->d_z8);
  }
  if (urc) {
    (void)mmnb_pack_free(p);  // takes the context lock itself
    return urc;
  }
  *out = p;
  return MMNB_OK;
}
