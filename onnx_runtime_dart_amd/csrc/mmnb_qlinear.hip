// QLinearMatMul, ConvInteger and QLinearConv.
//
// QLinearMatMul (onnx_qlinear_ops.dart:83-106) is MatMulInteger with an
// 8-bit requantising epilogue, on its kernels.  A convolution (:157-308) is the
// product A[p][kc] * w^T per image and group (p an output position, kc =
// (c*kh + ky)*kw + kx, out-of-image taps set to the input zero point so that
// (x - x_zp) = 0 there, which is the reference's skipping of them), in one
// launch of k_conv (matrix cores) or k_conv_taps (few channels), or a few
// where the grid would pass its limits: the weight w[m][c/g][kh][kw] is a MatMulInteger pack of B^T per
// group (batch = group), and the epilogue stores channel-major y[m][oy][ox],
// requantising per output channel for QLinearConv.
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "mmnb_conv_plan.h"
#include "mmnb_internal.h"

using namespace mmnb;

namespace mmnb {

// ---------------------------------------------------------------------------
// One convolution launch: PT output positions x 16 CW output channels of one
// (image, group) per workgroup, as a matrix product whose A rows are gathered
// from the image on the way into LDS.
//
// The products of an image layer are small (56 x 56 x 64 channels of 3 x 3: 0.05
// us of the matrix cores); what such a call spends is launches, round trips and
// the byte gather.  So there is one launch: A never goes to memory, and the
// per-channel requantisation parameters ride in the kernel's arguments (INL, up
// to kConvInline channels), which saves the upload and the wait for it.
//
// K (kc = (c*kh + ky)*kw + kx, the weight's order) moves in chunks of 32 KB of A.
// Per chunk a table of every kc's source offset and window position is built
// (two divisions per entry instead of per byte), then thread t gathers the bytes
// of position t % PT -- neighbouring lanes read neighbouring image bytes -- with 16
// loads in flight, out-of-image taps taking the input zero point.  16-byte piece c of row r lies at c ^ (r & 15), so the 16 rows
// of an operand read spread over the banks.  The weights go straight to
// registers, four 64-k steps ahead.
//
// 16 waves, all of which gather: CW of them (a power of two) take 16 channels
// each, the other factor KW = 16 / CW splits the chunk's 64-k steps and meets in LDS
// at the end (integer adds: exact in any order).  A workgroup covers the group's
// channels up to 256, so that few bytes are gathered twice, and fewer where the
// positions alone leave the chip idle (conv_run).
//
// Against an im2col launch and the MatMulInteger kernel (ConvInteger, us per call, u8
// x i8, back to back; QLinearConv took 13 us more there for the parameters): 64
// channels of 56 x 56, 3 x 3 to 64 11.5 -> 6.6; 256 of 14 x 14 to 256 12.8 -> 10.7; 512
// of 7 x 7 to 512 18.9 -> 16.7; 512 of 28 x 28 to 512 28.9 -> 27.4; 256 of 112 x 112 to
// 256 103 -> 35.0; 512 of 112 x 112 to 512 234 -> 125.
// ---------------------------------------------------------------------------
typedef int conv_i4 __attribute__((ext_vector_type(4)));
typedef uint32_t conv_u4 __attribute__((ext_vector_type(4)));

constexpr int kConvInline = 256;  // channels whose parameters fit the arguments
struct ConvChan {
  double mult[kConvInline];
  int32_t bias[kConvInline];
};
struct ConvNoChan {};

struct ConvArgs {
  const uint8_t *x;       // [images][groups * cg][H][W]
  const int8_t *bt;       // [groups][N][kpad]
  const int32_t *colsum;  // [groups][N]
  const int32_t *ecol;    // [N], or [groups][N] with ecol_bstride = N
  int H, W, cg, kh, kw, ow, sh, sw, ph, pw, dh, dw;
  int P, K, kpad, N, groups, ecol_bstride;
  int p0;                 // first position of the launch (k_conv)
  uint32_t mkhw, mkw;     // floor(2^32 / d) + 1 of kh * kw and kw
  int cw;                 // channel waves of a workgroup: a power of two <= 16
  uint32_t flip;          // 0x80808080: unsigned input
  int32_t azp;            // input zero point
  int32_t *y;             // int32 output, or
  uint8_t *yq;            // requantised bytes
  const double *mult;     // [groups * N] (without INL)
  const int32_t *bias;    // [groups * N]
  int32_t yzp, lo, hi;
  int vec;                // P % 4 == 0 and an aligned output
};

// A table entry: source offset, and the window position (ky * dh, kx * dw) in 16
// bits each or, WIDE (images whose padded coordinates need more), 32.
struct ConvTap {
  uint32_t off, pos;
};
typedef unsigned short conv_h2 __attribute__((ext_vector_type(2)));  // (x, y)
struct ConvTapWide {
  uint32_t off, dy, dx;
};

// double, as the reference: (acc + bias) * mult, half to even, saturated
__device__ __forceinline__ uint32_t conv_requant(uint32_t v, double mult, int32_t bias,
                                                 const ConvArgs &c) {
  const double f = rint(((double)(int32_t)v + (double)bias) * mult) + (double)c.yzp;
  return (uint32_t)(uint8_t)(int32_t)fmin(fmax(f, (double)c.lo), (double)c.hi);
}

template <bool WIDE>
using ConvTapOf = std::conditional_t<WIDE, ConvTapWide, ConvTap>;

// An output position: its window's first input coordinates (y, x) and offset.
struct ConvPos {
  int iy0, ix0;
  unsigned base;
  __device__ ConvPos(const ConvArgs &c, int p) {
    const int oy = p / c.ow, ox = p - oy * c.ow;
    iy0 = oy * c.sh - c.ph;
    ix0 = ox * c.sw - c.pw;
    base = (unsigned)iy0 * (unsigned)c.W + (unsigned)ix0;
  }
  // whether the tap lies inside the image
  template <typename TAP>
  __device__ bool inside(const ConvArgs &c, const TAP &t) const {
    if constexpr (std::is_same<TAP, ConvTapWide>::value) {
      return ((unsigned)iy0 + t.dy < (unsigned)c.H) & ((unsigned)ix0 + t.dx < (unsigned)c.W);
    } else {
      const conv_h2 pos0 = {(unsigned short)ix0, (unsigned short)iy0};
      const conv_h2 last = {(unsigned short)(c.W - 1), (unsigned short)(c.H - 1)};
      const conv_h2 at = pos0 + __builtin_bit_cast(conv_h2, t.pos);
      return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(at, last)) ==
             __builtin_bit_cast(uint32_t, at);
    }
  }
};
template <bool WIDE>
__host__ __device__ __forceinline__ ConvTapOf<WIDE> conv_tap(const ConvArgs &c, unsigned ci,
                                                             unsigned ky, unsigned kx) {
  const unsigned dy = ky * (unsigned)c.dh, dx = kx * (unsigned)c.dw;
  const unsigned off = (ci * (unsigned)c.H + dy) * (unsigned)c.W + dx;
  if constexpr (WIDE)
    return {off, dy, dx};
  else
    return {off, dy << 16 | (dx & 65535u)};
}

template <int PT, typename CHAN, bool WIDE>
__global__ __launch_bounds__(kConvThreads) void k_conv(ConvArgs c, CHAN chan) {
  constexpr int KC = kConvLds / PT;         // k per chunk
  constexpr int TP = PT / 16;               // 16-position tiles
  constexpr int WQ = kConvThreads / PT;     // words per position and gather pass
  __shared__ conv_u4 sA[kConvLds / 16];  // the chunk; at the end the sums' tile
  __shared__ __align__(16) ConvTapOf<WIDE> tab[KC];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cw = wave & (c.cw - 1), kw = wave / c.cw, nkw = 16 / c.cw;
  const int r16 = lane & 15, q = lane >> 4;
  const int g = blockIdx.z % c.groups;
  const int p0 = c.p0 + (int)blockIdx.x * PT, left = c.P - p0;

  // this lane's output channel and its constants
  const int n = (blockIdx.y * c.cw + cw) * 16 + r16;
  const int col = n < c.N ? n : c.N - 1;
  const uint32_t ce = (uint32_t)c.ecol[g * c.ecol_bstride + col];
  const uint32_t cs = (uint32_t)c.colsum[(int64_t)g * c.N + col];
  const int ch = g * c.N + col;
  double cm;
  int32_t cb;
  if constexpr (std::is_same<CHAN, ConvChan>::value) {
    cm = chan.mult[ch];
    cb = chan.bias[ch];
  } else {
    // (the int32 output has no parameters: both point at a zero page)
    cm = c.mult[c.y ? 0 : ch];
    cb = c.bias[c.y ? 0 : ch];
  }
  const int8_t *bp = c.bt + ((int64_t)g * c.N + col) * c.kpad + q * 16;

  // this thread's position of the gather
  const int row = tid % PT, wq = tid / PT;
  const int pc = row < left ? p0 + row : c.P - 1;
  const ConvPos at(c, pc);
  const uint8_t *xg = c.x + (int64_t)blockIdx.z * c.cg * c.H * c.W;
  const int khw = c.kh * c.kw;
  const uint32_t zb = (uint32_t)c.azp & 255u;

  conv_i4 acc[TP];
  int rsum[TP];
#pragma unroll
  for (int t = 0; t < TP; t++) {
    rsum[t] = 0;
    acc[t] = (conv_i4){0, 0, 0, 0};
  }

  for (int k0 = 0; k0 < c.kpad; k0 += KC) {
    const int kn = c.kpad - k0 < KC ? c.kpad - k0 : KC;  // a multiple of 64
    const int nst = kn >> 6, words = kn >> 2;
    // weights of this wave's steps s, s + nkw, ... (clamped to the chunk)
    conv_i4 bw[4];
    auto load_b = [&](int s) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < 4; u++)
        bw[u] = *(const conv_i4 *)(bp + k0 + (s + u * nkw < nst ? s + u * nkw : nst - 1) * 64);
    };
    load_b(kw);
    for (int i = tid; i < kn; i += kConvThreads) {
      const int kk = k0 + i < c.K ? k0 + i : c.K - 1;
      // (kk < 2^16, so the multiplications give the quotients)
      const int ci = khw == 1 ? kk : (int)__umulhi((uint32_t)kk, c.mkhw), r = kk - ci * khw;
      const int ky = c.kw == 1 ? r : (int)__umulhi((uint32_t)r, c.mkw), kx = r - ky * c.kw;
      tab[i] = conv_tap<WIDE>(c, (unsigned)ci, (unsigned)ky, (unsigned)kx);
    }
    __syncthreads();  // the table, and every wave past the last chunk's products
    // gather: words wq, wq + WQ, ... of the position's row (clamped: repeated).  No
    // conditional around a load or in its use that the compiler could turn into a
    // branch: as conditional expressions every byte was a basic block of its own
    // and waited for its table entry alone (512 channels of 7 x 7, 3 x 3: 21.6 us
    // instead of 16.3; of 112 x 112 264 instead of 126)
    auto gather = [&](auto count, int u0) __attribute__((always_inline)) {
      constexpr int NP = decltype(count)::value;
      uint32_t v[NP][4];
      bool in[NP][4];
#pragma unroll
      for (int u = 0; u < NP; u++) {
        const int word = min(wq + WQ * (u0 + u), words - 1);
        ConvTapOf<WIDE> t4[4];
        if constexpr (WIDE) {
#pragma unroll
          for (int e = 0; e < 4; e++) t4[e] = tab[4 * word + e];
        } else {
          const conv_u4 *tp = (const conv_u4 *)&tab[4 * word];
          const conv_u4 lo = tp[0], hi = tp[1];
          t4[0] = {lo.x, lo.y}, t4[1] = {lo.z, lo.w}, t4[2] = {hi.x, hi.y}, t4[3] = {hi.z, hi.w};
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
          in[u][e] = at.inside(c, t4[e]);
          v[u][e] = xg[(at.base + t4[e].off) & (0u - (uint32_t)in[u][e])];
        }
      }
#pragma unroll
      for (int u = 0; u < NP; u++) {
        const int word = min(wq + WQ * (u0 + u), words - 1);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const uint32_t m = 0u - (uint32_t)in[u][e];
          v[u][e] = (v[u][e] & m) | (zb & ~m);
        }
        ((uint32_t *)sA)[row * (KC / 4) + (((word >> 2) ^ (row & 15)) << 2) + (word & 3)] =
            v[u][0] | v[u][1] << 8 | v[u][2] << 16 | v[u][3] << 24;
      }
    };
    const int passes = (words + WQ - 1) / WQ;  // 1 .. 8
    if (passes == 1) {
      gather(std::integral_constant<int, 1>(), 0);
    } else if (passes == 2) {
      gather(std::integral_constant<int, 2>(), 0);
    } else if (passes <= 4) {
      gather(std::integral_constant<int, 4>(), 0);
    } else {
      gather(std::integral_constant<int, 4>(), 0);
      gather(std::integral_constant<int, 4>(), 4);
    }
    __syncthreads();
    for (int s = kw; s < nst; s += 4 * nkw) {
      conv_i4 b[4];
#pragma unroll
      for (int u = 0; u < 4; u++) b[u] = bw[u];
      if (s + 4 * nkw < nst) load_b(s + 4 * nkw);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (s + u * nkw < nst) {
          // row sums over k < K only (the weights past K are 0, A's bytes there are not)
          int ones[4] = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
          const int k1 = k0 + (s + u * nkw) * 64;
          if (k1 + 64 > c.K) {  // uniform
#pragma unroll
            for (int d = 0; d < 4; d++) {
              const int in4 = min(max(c.K - k1 - 16 * q - 4 * d, 0), 4);
              ones[d] = (int)(0x01010101ull >> (8 * (4 - in4)));
            }
          }
#pragma unroll
          for (int t = 0; t < TP; t++) {
            const int ra = t * 16 + r16;
            const conv_u4 x =
                sA[ra * (KC / 16) + (((s + u * nkw) * 4 + q) ^ (ra & 15))] ^ c.flip;
            const conv_i4 a = __builtin_bit_cast(conv_i4, x);
#pragma unroll
            for (int d = 0; d < 4; d++)
              rsum[t] = __builtin_amdgcn_sdot4(a[d], ones[d], rsum[t], false);
            acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b[u], acc[t], 0, 0, 0);
          }
        }
      }
    }
  }

  // acc += e * (row sum), per k wave; then the k waves' sums through LDS
#pragma unroll
  for (int t = 0; t < TP; t++) {
    rsum[t] += __shfl_xor(rsum[t], 16, 64);
    rsum[t] += __shfl_xor(rsum[t], 32, 64);
#pragma unroll
    for (int r = 0; r < 4; r++)
      acc[t][r] = (int)((uint32_t)acc[t][r] + ce * (uint32_t)__shfl(rsum[t], q * 4 + r, 64));
  }
  if (nkw > 1) {
    // [CW <= 8 channel waves][PT / 16][4][64] dwords fit the chunk's LDS
    uint32_t *red = (uint32_t *)sA + cw * (TP * 256);
    __syncthreads();
    if (kw == 0) {
#pragma unroll
      for (int t = 0; t < TP; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) red[(t * 4 + r) * 64 + lane] = (uint32_t)acc[t][r];
    }
    __syncthreads();
    if (kw > 0) {
#pragma unroll
      for (int t = 0; t < TP; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) atomicAdd(&red[(t * 4 + r) * 64 + lane], (uint32_t)acc[t][r]);
    }
    __syncthreads();
    if (kw > 0) return;
#pragma unroll
    for (int t = 0; t < TP; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) acc[t][r] = (int)red[(t * 4 + r) * 64 + lane];
  }

  // exact zero-point corrections, in wrapping 32 bits, and the stores
  if (n >= c.N) return;
  const uint32_t azc = (uint32_t)((c.flip ? 128 : 0) - c.azp);
  const uint32_t fix = azc * cs + (uint32_t)c.K * azc * ce;
#pragma unroll
  for (int t = 0; t < TP; t++) {
    const int pt = t * 16 + q * 4;  // of the workgroup's positions
    if (pt >= left) continue;
    uint32_t v[4];
#pragma unroll
    for (int r = 0; r < 4; r++) v[r] = (uint32_t)acc[t][r] + fix;
    const int64_t o0 = ((int64_t)blockIdx.z * c.N + col) * c.P + p0 + pt;
    if (c.y) {
      if (c.vec) {
        *(conv_u4 *)(c.y + o0) = (conv_u4){v[0], v[1], v[2], v[3]};
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (pt + r < left) c.y[o0 + r] = (int32_t)v[r];
      }
    } else {
      uint32_t o[4];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        o[r] = conv_requant(v[r], cm, cb, c);
      }
      if (c.vec) {
        *(uint32_t *)(c.yq + o0) = o[0] | o[1] << 8 | o[2] << 16 | o[3] << 24;
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (pt + r < left) c.yq[o0 + r] = (uint8_t)o[r];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Few taps (K <= 4 NW) and few output channels per group, depthwise above all: a
// lane per output position.  It gathers its K bytes into NW registers and
// multiplies them by each channel's weights, four at a time (v_dot4); taps (a table
// in the arguments) and weights are the same for all lanes, so both are scalars.
// No LDS and no barrier, and a wave goes over several blocks of 64 positions.
//
// k_conv pads such a product to 64 taps, 16 channels and 16 waves, and what it then
// takes is the launch of its waves (300 000 for 384 channels of 56 x 56).  Bound
// here by the gather's instructions, about 8 a byte; few positions, by the launch.
//
// ConvInteger, us per call by im2col and MatMulInteger launches, k_conv and here: 384
// channels of 56 x 56, 3 x 3 depthwise 103, 342 and 9.2; four images of 960 of 28 x
// 28, 5 x 5 depthwise 470, 941 and 33.7; 1 of 512 x 512, 3 x 3 to 8 27.7, 75.5 and
// 6.0; 16 of 160000 samples, 3 taps, to 16 35.7, 139 and 15.8.
// ---------------------------------------------------------------------------
typedef __attribute__((address_space(4))) int conv_const_int;

template <int NW, bool WIDE>
struct ConvTaps {
  ConvTapOf<WIDE> t[4 * NW];
};

template <int NW, bool WIDE, typename CHAN>
__global__ __launch_bounds__(256) void k_conv_taps(ConvArgs c, ConvTaps<NW, WIDE> taps, CHAN chan,
                                                   int nper) {
  const int g = blockIdx.z % c.groups;
  const int n0 = blockIdx.y * nper, n1 = min(n0 + nper, c.N);
  const uint8_t *xg = c.x + (int64_t)blockIdx.z * c.cg * c.H * c.W;
  const int8_t *bt = c.bt + (int64_t)g * c.N * c.kpad;
  const uint32_t zb = (uint32_t)c.azp & 255u;
  const uint32_t azc = (uint32_t)((c.flip ? 128 : 0) - c.azp);
  for (unsigned p = blockIdx.x * blockDim.x + threadIdx.x; p < (unsigned)c.P;
       p += gridDim.x * blockDim.x) {
    const ConvPos at(c, (int)p);
    int a[NW];
    int rs = 0;  // sum over k < K
#pragma unroll
    for (int w = 0; w < NW; w++) {
      uint32_t v[4];
      bool in[4];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const ConvTapOf<WIDE> t = taps.t[4 * w + e];
        in[e] = at.inside(c, t);
        v[e] = xg[(at.base + t.off) & (0u - (uint32_t)in[e])];
      }
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const uint32_t m = 0u - (uint32_t)in[e];
        v[e] = (v[e] & m) | (zb & ~m);
      }
      a[w] = (int)((v[0] | v[1] << 8 | v[2] << 16 | v[3] << 24) ^ c.flip);
      const int left = min(max(c.K - 4 * w, 0), 4);
      rs = __builtin_amdgcn_sdot4(a[w], (int)(0x01010101ull >> (8 * (4 - left))), rs, false);
    }
    const int64_t o0 = ((int64_t)blockIdx.z * c.N + n0) * c.P + p;
    // (scalar loads: left to itself the compiler reads them per lane, for the stores
    // between them could alias)
#pragma unroll NW > 8 ? 2 : 4
    for (int n = n0; n < n1; n++) {
      const conv_const_int *wp = (const conv_const_int *)(uintptr_t)(bt + (int64_t)n * c.kpad);
      int acc = 0;
#pragma unroll
      for (int w = 0; w < NW; w++) acc = __builtin_amdgcn_sdot4(a[w], wp[w], acc, false);
      const uint32_t ce =
          (uint32_t)((const conv_const_int *)(uintptr_t)c.ecol)[g * c.ecol_bstride + n];
      const uint32_t cs =
          (uint32_t)((const conv_const_int *)(uintptr_t)c.colsum)[(int64_t)g * c.N + n];
      // exact zero-point corrections, in wrapping 32 bits
      const uint32_t v = (uint32_t)acc + ce * (uint32_t)rs + azc * cs + (uint32_t)c.K * azc * ce;
      const int64_t o = o0 + (int64_t)(n - n0) * c.P;
      if (c.y) {
        c.y[o] = (int32_t)v;
      } else {
        const int ch = g * c.N + n;
        double cm;
        int32_t cb;
        if constexpr (std::is_same<CHAN, ConvChan>::value) {
          cm = chan.mult[ch];
          cb = chan.bias[ch];
        } else {
          cm = c.mult[ch];
          cb = c.bias[ch];
        }
        c.yq[o] = (uint8_t)conv_requant(v, cm, cb, c);
      }
    }
  }
}

// More channels than the arguments hold: 256 channels' parameters per launch,
// written where k_conv reads them.
__global__ __launch_bounds__(256) void k_conv_params(ConvChan chan, int n, double *mult,
                                                     int32_t *bias) {
  const int i = threadIdx.x;
  if (i < n) {
    mult[i] = chan.mult[i];
    bias[i] = chan.bias[i];
  }
}

}  // namespace mmnb

namespace {

struct ConvShape {
  int64_t n, c, h, w, oh, ow;
  int sh, sw, ph, pw, dh, dw;
};

// Output size per axis, `(in + pad_begin + pad_end - window) ~/ stride + 1`
// (onnx_qlinear_ops.dart:222-231); strides, dilations >= 1, pads >= 0.
int conv_shape(const mmnb_pack *p, int64_t n, int64_t c, int64_t h, int64_t w,
               const mmnb_conv_params *prm, ConvShape *s) {
  if (!p || p->kind != kPackConv) return fail(MMNB_ERR_ARG, "conv: not a convolution pack");
  if (!prm) return fail(MMNB_ERR_ARG, "conv: null parameters");
  if (n < 0 || h < 1 || w < 1) return fail(MMNB_ERR_ARG, "conv: bad input shape");
  if (c != p->conv_cg * p->conv_group)
    return fail(MMNB_ERR_ARG, "conv: input channels != weight channels * group");
  for (int a = 0; a < 2; a++)
    if (prm->strides[a] < 1 || prm->dilations[a] < 1)
      return fail(MMNB_ERR_ARG, "conv: strides and dilations must be >= 1");
  for (int a = 0; a < 4; a++)
    if (prm->pads[a] < 0) return fail(MMNB_ERR_ARG, "conv: negative pad");
  const int64_t kdim[2] = {p->conv_kh, p->conv_kw}, in[2] = {h, w};
  int64_t out[2];
  for (int a = 0; a < 2; a++) {
    const int64_t window = prm->dilations[a] * (kdim[a] - 1) + 1;
    const int64_t span = in[a] + prm->pads[a] + prm->pads[2 + a] - window;
    if (span < 0) return fail(MMNB_ERR_ARG, "conv: kernel window larger than the padded input");
    out[a] = span / prm->strides[a] + 1;
  }
  if (prm->strides[0] > INT32_MAX || prm->strides[1] > INT32_MAX ||
      prm->pads[0] > INT32_MAX || prm->pads[1] > INT32_MAX ||
      prm->dilations[0] > INT32_MAX || prm->dilations[1] > INT32_MAX)
    return fail(MMNB_ERR_UNSUPPORTED, "conv: parameter beyond int32");
  *s = ConvShape{n, c, h, w, out[0], out[1], (int)prm->strides[0], (int)prm->strides[1],
                 (int)prm->pads[0], (int)prm->pads[1], (int)prm->dilations[0],
                 (int)prm->dilations[1]};
  return MMNB_OK;
}

int check_zp(int64_t v, int is_signed, const char *what) {
  const int64_t lo = is_signed ? -128 : 0, hi = is_signed ? 127 : 255;
  if (v < lo || v > hi) return fail(MMNB_ERR_ARG, std::string(what) + " out of range");
  return MMNB_OK;
}

// Where a convolution's results go: int32 y, or bytes yq requantised with the
// channels' parameters (in the arguments up to kConvInline channels, else in
// scratch slot 8).
struct ConvOut {
  int32_t *y = nullptr;
  uint8_t *yq = nullptr;
  int32_t yzp = 0, lo = 0, hi = 255;
  bool inl = false;
  ConvChan chan;
  const double *d_mult = nullptr;
  const int32_t *d_bias = nullptr;
};

template <int PT, bool WIDE>
int conv_launch(mmnb_ctx *ctx, ConvArgs &c, const ConvOut &o, int64_t z, const ConvPlan &pl) {
  for (int64_t p0 = 0; p0 < c.P; p0 += pl.step) {
    c.p0 = (int)p0;
    const int64_t np = c.P - p0 < pl.step ? c.P - p0 : pl.step;
    const dim3 grid((unsigned)((np + PT - 1) / PT), (unsigned)pl.gy, (unsigned)z);
    const dim3 block((unsigned)pl.threads);
    const int rc =
        o.inl ? launch(ctx, kKernConv, k_conv<PT, ConvChan, WIDE>, grid, block, 0, c, o.chan)
              : launch(ctx, kKernConv, k_conv<PT, ConvNoChan, WIDE>, grid, block, 0, c,
                       ConvNoChan{});
    if (rc) return rc;
  }
  return MMNB_OK;
}

template <int NW, bool WIDE>
int conv_taps_launch(mmnb_ctx *ctx, const ConvArgs &c, const ConvOut &o, int64_t z,
                     const ConvPlan &pl) {
  ConvTaps<NW, WIDE> taps;
  for (int i = 0; i < 4 * NW; i++) {
    // (past the last tap: the last one again, times weights of 0)
    const int k = i < c.K ? i : c.K - 1, r = k % (c.kh * c.kw);
    taps.t[i] = conv_tap<WIDE>(c, (unsigned)(k / (c.kh * c.kw)), (unsigned)(r / c.kw),
                               (unsigned)(r % c.kw));
  }
  const dim3 grid((unsigned)pl.gx, (unsigned)pl.gy, (unsigned)z), block((unsigned)pl.threads);
  if (o.inl)
    return launch(ctx, kKernConv, k_conv_taps<NW, WIDE, ConvChan>, grid, block, 0, c, taps,
                  o.chan, (int)pl.nper);
  return launch(ctx, kKernConv, k_conv_taps<NW, WIDE, ConvNoChan>, grid, block, 0, c, taps,
                ConvNoChan{}, (int)pl.nper);
}

template <bool WIDE>
int conv_dispatch(mmnb_ctx *ctx, ConvArgs &c, const ConvOut &o, int64_t z) {
  const ConvPlan pl = conv_plan(c.P, c.K, c.N, z, ctx->cu_count);
  if (pl.taps)
    return pl.nw == 3   ? conv_taps_launch<3, WIDE>(ctx, c, o, z, pl)
           : pl.nw == 7 ? conv_taps_launch<7, WIDE>(ctx, c, o, z, pl)
                        : conv_taps_launch<16, WIDE>(ctx, c, o, z, pl);
  c.cw = pl.cw;
  return pl.pt == 64   ? conv_launch<64, WIDE>(ctx, c, o, z, pl)
         : pl.pt == 32 ? conv_launch<32, WIDE>(ctx, c, o, z, pl)
                       : conv_launch<16, WIDE>(ctx, c, o, z, pl);
}

// Device side of a convolution: all images and groups in one launch (grid.z,
// at most 65535 of them at a time).
int conv_run(mmnb_ctx *ctx, const mmnb_pack *p, const uint8_t *d_x, int x_signed,
             const ConvShape &s, int64_t x_zp, const ConvOut &o) {
  const int64_t P = s.oh * s.ow, kcn = p->k, g = p->conv_group, n = p->n;
  if (s.n == 0 || P == 0) return MMNB_OK;
  if (kcn > 65535 * 256 || g > 65535 || g * P * kcn > INT32_MAX ||
      s.c * s.h * s.w > INT32_MAX)
    return fail(MMNB_ERR_UNSUPPORTED, "conv: image too large for one launch");
  const int64_t esz = o.y ? 4 : 1;
  ConvArgs c{};
  c.bt = p->d_bt;
  c.colsum = p->d_colsum;
  c.ecol = p->d_ecol;
  c.H = (int)s.h; c.W = (int)s.w; c.cg = (int)p->conv_cg;
  c.kh = (int)p->conv_kh; c.kw = (int)p->conv_kw; c.ow = (int)s.ow;
  c.sh = s.sh; c.sw = s.sw; c.ph = s.ph; c.pw = s.pw; c.dh = s.dh; c.dw = s.dw;
  c.P = (int)P; c.K = (int)kcn; c.kpad = (int)p->kpad; c.N = (int)n; c.groups = (int)g;
  c.ecol_bstride = (int)p->ecol_bstride;
  c.flip = x_signed ? 0u : 0x80808080u;
  c.azp = (int32_t)x_zp;
  c.mult = o.d_mult ? o.d_mult : (const double *)ctx->d_pad;
  c.bias = o.d_bias ? o.d_bias : (const int32_t *)ctx->d_pad;
  c.yzp = o.yzp; c.lo = o.lo; c.hi = o.hi;
  auto magic = [](int64_t d) { return (uint32_t)((int64_t(1) << 32) / d + 1); };
  c.mkhw = magic(p->conv_kh * p->conv_kw);
  c.mkw = magic(p->conv_kw);
  // 16-bit window positions: every input coordinate of a tap, from -pad to the
  // last window's end, is told apart from those inside the image modulo 2^16
  const int64_t ymax = (s.oh - 1) * s.sh - s.ph + (p->conv_kh - 1) * s.dh;
  const int64_t xmax = (s.ow - 1) * s.sw - s.pw + (p->conv_kw - 1) * s.dw;
  const bool wide = s.h + s.ph > 65536 || s.w + s.pw > 65536 || ymax > 65535 || xmax > 65535;
  const int64_t zmax = 65535 / g * g;  // whole images per launch
  for (int64_t z0 = 0; z0 < s.n * g; z0 += zmax) {
    const int64_t z = s.n * g - z0 < zmax ? s.n * g - z0 : zmax;
    c.x = d_x + z0 * p->conv_cg * s.h * s.w;
    c.y = o.y ? o.y + z0 * n * P : nullptr;
    c.yq = o.y ? nullptr : o.yq + z0 * n * P;
    const uintptr_t out = o.y ? (uintptr_t)c.y : (uintptr_t)c.yq;
    c.vec = P % 4 == 0 && out % (4 * esz) == 0;
    const int rc = wide ? conv_dispatch<true>(ctx, c, o, z) : conv_dispatch<false>(ctx, c, o, z);
    if (rc) return rc;
  }
  return MMNB_OK;
}

}  // namespace

// -------------------------------------------------------------- QLinearMatMul

// mult = fl32(fl32(a_scale * b_scale) / y_scale), the reference's two
// binary32 roundings (onnx_qlinear_ops.dart:93-96).
static int qmm_mult(float a_scale, float b_scale, float y_scale, float *mult) {
  if (!std::isfinite(a_scale) || !std::isfinite(b_scale) || !std::isfinite(y_scale) ||
      y_scale == 0.0f)
    return fail(MMNB_ERR_ARG, "QLinearMatMul: scales must be finite and y_scale non-zero");
  const float ab = (float)((double)a_scale * (double)b_scale);
  *mult = (float)((double)ab / (double)y_scale);
  if (!std::isfinite(*mult)) return fail(MMNB_ERR_ARG, "QLinearMatMul: multiplier overflows");
  return MMNB_OK;
}

static int qmm_check(mmnb_ctx *ctx, const mmnb_pack *p, int64_t a_batch, int64_t m,
                     int64_t azl) {
  if (!p || p->kind != kPackInteger)
    return fail(MMNB_ERR_ARG, "QLinearMatMul: not a MatMulInteger pack");
  if (p->ctx != ctx) return fail(MMNB_ERR_ARG, "pack belongs to another context");
  if (a_batch < 1 || m < 0) return fail(MMNB_ERR_ARG, "QLinearMatMul: bad A shape");
  if (azl != 0 && azl != 1 && azl != m)
    return fail(MMNB_ERR_UNSUPPORTED,
                "MatMulInteger: zero points must be scalar, per-row [M] for A or "
                "per-column [N] for B");
  const int64_t batch = a_batch > p->batch ? a_batch : p->batch;
  if ((a_batch != batch && a_batch != 1) || (p->batch != batch && p->batch != 1))
    return fail(MMNB_ERR_ARG, "MatMulInteger batch mismatch");
  return MMNB_OK;
}

int mmnb_qlinear_matmul_dev(mmnb_ctx *ctx, const mmnb_pack *pack, const void *d_a,
                            int a_is_signed, int64_t a_batch, int64_t m,
                            const int32_t *d_a_zero_point, int64_t a_zero_point_len,
                            float a_scale, float b_scale, float y_scale, int64_t y_zero_point,
                            int y_is_signed, void *d_y) {
  MMNB_GUARD_CTX(ctx);
  const int64_t azl = d_a_zero_point ? a_zero_point_len : 0;
  int rc = qmm_check(ctx, pack, a_batch, m, azl);
  if (rc) return rc;
  float mult;
  if ((rc = qmm_mult(a_scale, b_scale, y_scale, &mult))) return rc;
  if ((rc = check_zp(y_zero_point, y_is_signed, "QLinearMatMul: y zero point"))) return rc;
  if (m == 0) return MMNB_OK;
  if (!d_y || (!d_a && pack->k > 0)) return fail(MMNB_ERR_ARG, "QLinearMatMul: null buffer");
  CtxLock lk(ctx);
  if ((rc = set_device(ctx))) return rc;
  MmiEpi o;
  o.yq = (uint8_t *)d_y;
  o.rq_mult = mult;
  o.yzp = (int32_t)y_zero_point;
  o.lo = y_is_signed ? -128 : 0;
  o.hi = y_is_signed ? 127 : 255;
  return launch_matmul_integer(ctx, pack, d_a, a_is_signed ? 1 : 0, a_batch, m, d_a_zero_point,
                               azl, o);
}

int mmnb_qlinear_matmul(mmnb_ctx *ctx, const mmnb_pack *pack, const void *a, int a_is_signed,
                        int64_t a_batch, int64_t m, const int64_t *a_zero_point,
                        int64_t a_zero_point_len, float a_scale, float b_scale, float y_scale,
                        int64_t y_zero_point, int y_is_signed, void *y) {
  MMNB_GUARD_CTX(ctx);
  if (ctx->capturing) return fail(MMNB_ERR_ARG, "host entry point during graph capture");
  const int64_t azl = a_zero_point ? a_zero_point_len : 0;
  int rc = qmm_check(ctx, pack, a_batch, m, azl);
  if (rc) return rc;
  float mult;
  if ((rc = qmm_mult(a_scale, b_scale, y_scale, &mult))) return rc;
  if ((rc = check_zp(y_zero_point, y_is_signed, "QLinearMatMul: y zero point"))) return rc;
  if (m == 0) return MMNB_OK;
  if (!y || (!a && pack->k > 0)) return fail(MMNB_ERR_ARG, "QLinearMatMul: null buffer");
  std::vector<int32_t> az((size_t)(azl ? azl : 1));
  for (int64_t i = 0; i < azl; i++) {
    if ((rc = check_zp(a_zero_point[i], a_is_signed, "QLinearMatMul: A zero point"))) return rc;
    az[(size_t)i] = (int32_t)a_zero_point[i];
  }
  CtxLock lk(ctx);
  if ((rc = set_device(ctx))) return rc;
  const int64_t k = pack->k, n = pack->n;
  const int64_t batch = a_batch > pack->batch ? a_batch : pack->batch;
  void *d_a = nullptr, *d_y = nullptr, *d_az = nullptr;
  if ((rc = scratch_get(ctx, 0, (size_t)(a_batch * m * k) + 256, &d_a))) return rc;
  if ((rc = scratch_get(ctx, 1, (size_t)(batch * m * n), &d_y))) return rc;
  if ((rc = scratch_get(ctx, 5, az.size() * 4, &d_az))) return rc;
  if (a_batch * m * k)
    MMNB_HIP(hipMemcpyAsync(d_a, a, (size_t)(a_batch * m * k), hipMemcpyHostToDevice,
                            ctx->stream));
  if (azl)
    MMNB_HIP(hipMemcpyAsync(d_az, az.data(), (size_t)azl * 4, hipMemcpyHostToDevice,
                            ctx->stream));
  MmiEpi o;
  o.yq = (uint8_t *)d_y;
  o.rq_mult = mult;
  o.yzp = (int32_t)y_zero_point;
  o.lo = y_is_signed ? -128 : 0;
  o.hi = y_is_signed ? 127 : 255;
  if ((rc = launch_matmul_integer(ctx, pack, d_a, a_is_signed ? 1 : 0, a_batch, m,
                                  azl ? (const int32_t *)d_az : nullptr, azl, o)))
    return rc;
  MMNB_HIP(hipMemcpyAsync(y, d_y, (size_t)(batch * m * n), hipMemcpyDeviceToHost, ctx->stream));
  MMNB_HIP(hipStreamSynchronize(ctx->stream));
  return MMNB_OK;
}

// ------------------------------------------------------------- convolutions

int mmnb_pack_conv(mmnb_ctx *ctx, const void *w, int w_is_signed, int64_t m,
                   int64_t c_per_group, int64_t kh, int64_t kw, int64_t group,
                   const int64_t *w_zero_point, int64_t w_zero_point_len, mmnb_pack **out) {
  MMNB_GUARD_CTX(ctx);
  if (!out) return fail(MMNB_ERR_ARG, "mmnb_pack_conv: out is null");
  *out = nullptr;
  if (m < 1 || c_per_group < 1 || kh < 1 || kw < 1 || group < 1)
    return fail(MMNB_ERR_ARG, "conv: bad weight shape");
  if (m % group) return fail(MMNB_ERR_ARG, "conv: output channels not divisible by group");
  if (!w) return fail(MMNB_ERR_ARG, "conv: weight is null");
  const int64_t wzl = w_zero_point ? w_zero_point_len : 0;
  if (wzl != 0 && wzl != 1 && wzl != m)
    return fail(MMNB_ERR_UNSUPPORTED,
                "ConvInteger: weight zero point must be scalar or per-output-channel");
  const int64_t k = c_per_group * kh * kw, n = m / group;
  if (k > 33025) return fail(MMNB_ERR_UNSUPPORTED, "conv: c/group*kh*kw > 33025 may overflow int32");
  std::vector<int32_t> zp((size_t)(wzl ? wzl : 1));
  int rc;
  for (int64_t i = 0; i < wzl; i++) {
    if ((rc = check_zp(w_zero_point[i], w_is_signed, "conv: weight zero point"))) return rc;
    zp[(size_t)i] = (int32_t)w_zero_point[i];
  }
  CtxLock lk(ctx);
  if ((rc = set_device(ctx))) return rc;
  mmnb_pack *p = new (std::nothrow) mmnb_pack();
  if (!p) return fail(MMNB_ERR_OOM, "out of host memory");
  p->ctx = ctx;
  p->kind = kPackConv;
  p->batch = group;
  p->k = k;
  p->n = n;
  p->kpad = (k + 63) / 64 * 64;
  p->b_signed = w_is_signed ? 1 : 0;
  p->conv_m = m;
  p->conv_cg = c_per_group;
  p->conv_kh = kh;
  p->conv_kw = kw;
  p->conv_group = group;
  // per-channel zero points differ between groups: one offset per (group, column)
  const bool per_batch = wzl == m && m != 1 && group > 1;
  p->ecol_bstride = per_batch ? n : 0;
  auto cleanup = [&](int code) {
    if (p->d_bt) (void)hipFree(p->d_bt);
    if (p->d_colsum) (void)hipFree(p->d_colsum);
    if (p->d_ecol) (void)hipFree(p->d_ecol);
    delete p;
    return code;
  };
  const size_t bt_bytes = (size_t)(group * n * p->kpad);
  if ((rc = device_alloc(bt_bytes, (void **)&p->d_bt))) return cleanup(rc);
  if ((rc = device_alloc((size_t)(group * n) * 4, (void **)&p->d_colsum))) return cleanup(rc);
  if ((rc = device_alloc((size_t)(per_batch ? m : n) * 4, (void **)&p->d_ecol)))
    return cleanup(rc);
  const size_t raw_bytes = (size_t)(m * k);
  void *d_raw = nullptr, *d_zp = nullptr;
  if ((rc = scratch_get(ctx, 4, raw_bytes + 256, &d_raw))) return cleanup(rc);
  if ((rc = scratch_get(ctx, 5, zp.size() * 4, &d_zp))) return cleanup(rc);
  hipError_t e;
  if ((e = hipMemcpyAsync(d_raw, w, raw_bytes, hipMemcpyHostToDevice, ctx->stream)) !=
      hipSuccess)
    return cleanup(check_hip(e, "hipMemcpyAsync(w)"));
  if (wzl && (e = hipMemcpyAsync(d_zp, zp.data(), (size_t)wzl * 4, hipMemcpyHostToDevice,
                                 ctx->stream)) != hipSuccess)
    return cleanup(check_hip(e, "hipMemcpyAsync(w_zp)"));
  // zero points per (group, column) are the flat per-channel list
  if ((rc = prepare_integer_b(ctx, (const uint8_t *)d_raw, p->b_signed, 1, group, k, n, p->kpad,
                              (const int32_t *)d_zp, wzl,
                              p->d_bt, p->d_colsum, p->d_ecol)))
    return cleanup(rc);
  if ((e = hipStreamSynchronize(ctx->stream)) != hipSuccess)
    return cleanup(check_hip(e, "hipStreamSynchronize(pack)"));
  p->bytes = (int64_t)bt_bytes + group * n * 4 + (per_batch ? m : n) * 4;
  ctx->live_packs++;
  *out = p;
  return MMNB_OK;
}

int mmnb_conv_output_shape(const mmnb_pack *w, int64_t n, int64_t c, int64_t h, int64_t wd,
                           const mmnb_conv_params *prm, int64_t *oh, int64_t *ow) {
  ConvShape s;
  int rc = conv_shape(w, n, c, h, wd, prm, &s);
  if (rc) return rc;
  if (oh) *oh = s.oh;
  if (ow) *ow = s.ow;
  return MMNB_OK;
}

int mmnb_conv_integer_dev(mmnb_ctx *ctx, const mmnb_pack *w, const void *d_x, int x_is_signed,
                          int64_t n, int64_t c, int64_t h, int64_t wd, int64_t x_zero_point,
                          const mmnb_conv_params *prm, int32_t *d_y) {
  MMNB_GUARD_CTX(ctx);
  ConvShape s;
  int rc = conv_shape(w, n, c, h, wd, prm, &s);
  if (rc) return rc;
  if (w->ctx != ctx) return fail(MMNB_ERR_ARG, "pack belongs to another context");
  if ((rc = check_zp(x_zero_point, x_is_signed, "ConvInteger: x zero point"))) return rc;
  if (!d_x || !d_y) return fail(MMNB_ERR_ARG, "ConvInteger: null buffer");
  CtxLock lk(ctx);
  if ((rc = set_device(ctx))) return rc;
  ConvOut o;
  o.y = d_y;
  return conv_run(ctx, w, (const uint8_t *)d_x, x_is_signed ? 1 : 0, s, x_zero_point, o);
}

int mmnb_conv_integer(mmnb_ctx *ctx, const mmnb_pack *w, const void *x, int x_is_signed,
                      int64_t n, int64_t c, int64_t h, int64_t wd, int64_t x_zero_point,
                      const mmnb_conv_params *prm, int32_t *y) {
  MMNB_GUARD_CTX(ctx);
  if (ctx->capturing) return fail(MMNB_ERR_ARG, "host entry point during graph capture");
  ConvShape s;
  int rc = conv_shape(w, n, c, h, wd, prm, &s);
  if (rc) return rc;
  if (w->ctx != ctx) return fail(MMNB_ERR_ARG, "pack belongs to another context");
  if ((rc = check_zp(x_zero_point, x_is_signed, "ConvInteger: x zero point"))) return rc;
  if (!x || !y) return fail(MMNB_ERR_ARG, "ConvInteger: null buffer");
  CtxLock lk(ctx);
  if ((rc = set_device(ctx))) return rc;
  const size_t xb = (size_t)(n * c * h * wd), yn = (size_t)(n * w->conv_m * s.oh * s.ow);
  void *d_x = nullptr, *d_y = nullptr;
  if ((rc = scratch_get(ctx, 0, xb + 256, &d_x))) return rc;
  if ((rc = scratch_get(ctx, 1, yn * 4, &d_y))) return rc;
  if (xb) MMNB_HIP(hipMemcpyAsync(d_x, x, xb, hipMemcpyHostToDevice, ctx->stream));
  ConvOut o;
  o.y = (int32_t *)d_y;
  if ((rc = conv_run(ctx, w, (const uint8_t *)d_x, x_is_signed ? 1 : 0, s, x_zero_point, o)))
    return rc;
  if (yn) MMNB_HIP(hipMemcpyAsync(y, d_y, yn * 4, hipMemcpyDeviceToHost, ctx->stream));
  MMNB_HIP(hipStreamSynchronize(ctx->stream));
  return MMNB_OK;
}

// Per-channel requantisation parameters of QLinearConv, in double as the
// reference computes them (onnx_qlinear_ops.dart:295-305): mult[c] =
// x_scale * w_scale[c] / y_scale, bias[c] (int32, optional).  Up to kConvInline
// channels stay in o->chan; more go to scratch slot 8, [m doubles][m int32]: by way
// of kernel arguments, without a copy from host memory to wait for, up to three
// launches (3.6 us each on the host), beyond by one copy and the wait (about 13 us;
// 512 channels of 7 x 7, 1 x 1 to 2048: 38.3 us by eight launches, 26.6 by the copy).
static int qconv_params(mmnb_ctx *ctx, int64_t m, float x_scale, const float *w_scale,
                        int64_t w_scale_len, float y_scale, const int32_t *bias, ConvOut *o) {
  if (!w_scale || (w_scale_len != 1 && w_scale_len != m))
    return fail(MMNB_ERR_ARG, "QLinearConv: w_scale must have 1 or M values");
  if (!std::isfinite(x_scale) || !std::isfinite(y_scale) || y_scale == 0.0f)
    return fail(MMNB_ERR_ARG, "QLinearConv: scales must be finite and y_scale non-zero");
  auto mult = [&](int64_t c) {
    return (double)x_scale * (double)w_scale[w_scale_len == 1 ? 0 : c] / (double)y_scale;
  };
  for (int64_t c = 0; c < m; c++)
    if (!std::isfinite(mult(c))) return fail(MMNB_ERR_ARG, "QLinearConv: non-finite scale");
  o->inl = m <= kConvInline;
  double *d_mult = nullptr;
  int32_t *d_bias = nullptr;
  if (!o->inl) {
    void *d = nullptr;
    int rc = scratch_get(ctx, 8, (size_t)m * 12, &d);
    if (rc) return rc;
    d_mult = (double *)d;
    d_bias = (int32_t *)((char *)d + m * 8);
    o->d_mult = d_mult;
    o->d_bias = d_bias;
  }
  if (m > 3 * kConvInline) {
    std::vector<char> buf((size_t)m * 12);
    double *hm = (double *)buf.data();
    int32_t *hb = (int32_t *)(buf.data() + m * 8);
    for (int64_t c = 0; c < m; c++) {
      hm[c] = mult(c);
      hb[c] = bias ? bias[c] : 0;
    }
    MMNB_HIP(hipMemcpyAsync(d_mult, buf.data(), buf.size(), hipMemcpyHostToDevice, ctx->stream));
    MMNB_HIP(hipStreamSynchronize(ctx->stream));  // `buf` is about to go away
    return MMNB_OK;
  }
  for (int64_t c0 = 0; c0 < m; c0 += kConvInline) {
    const int cnt = (int)(m - c0 < kConvInline ? m - c0 : kConvInline);
    std::memset(&o->chan, 0, sizeof(o->chan));
    for (int i = 0; i < cnt; i++) {
      o->chan.mult[i] = mult(c0 + i);
      o->chan.bias[i] = bias ? bias[c0 + i] : 0;
    }
    if (o->inl) break;
    int rc = launch(ctx, kKernConv, k_conv_params, dim3(1), dim3(kConvInline), 0, o->chan, cnt,
                    d_mult + c0, d_bias + c0);
    if (rc) return rc;
  }
  return MMNB_OK;
}

int mmnb_qlinear_conv_dev(mmnb_ctx *ctx, const mmnb_pack *w, const void *d_x, int x_is_signed,
                          int64_t n, int64_t c, int64_t h, int64_t wd, int64_t x_zero_point,
                          float x_scale, const float *w_scale, int64_t w_scale_len,
                          float y_scale, int64_t y_zero_point, int y_is_signed,
                          const int32_t *bias, const mmnb_conv_params *prm, void *d_y) {
  MMNB_GUARD_CTX(ctx);
  if (ctx->capturing) return fail(MMNB_ERR_ARG, "QLinearConv reads host arrays at the call: not capturable");
  ConvShape s;
  int rc = conv_shape(w, n, c, h, wd, prm, &s);
  if (rc) return rc;
  if (w->ctx != ctx) return fail(MMNB_ERR_ARG, "pack belongs to another context");
  if ((rc = check_zp(x_zero_point, x_is_signed, "QLinearConv: x zero point"))) return rc;
  if ((rc = check_zp(y_zero_point, y_is_signed, "QLinearConv: y zero point"))) return rc;
  if (!d_x || !d_y) return fail(MMNB_ERR_ARG, "QLinearConv: null buffer");
  CtxLock lk(ctx);
  if ((rc = set_device(ctx))) return rc;
  ConvOut o;
  if ((rc = qconv_params(ctx, w->conv_m, x_scale, w_scale, w_scale_len, y_scale, bias, &o)))
    return rc;
  o.yq = (uint8_t *)d_y;
  o.yzp = (int32_t)y_zero_point;
  o.lo = y_is_signed ? -128 : 0;
  o.hi = y_is_signed ? 127 : 255;
  return conv_run(ctx, w, (const uint8_t *)d_x, x_is_signed ? 1 : 0, s, x_zero_point, o);
}

int mmnb_qlinear_conv(mmnb_ctx *ctx, const mmnb_pack *w, const void *x, int x_is_signed,
                      int64_t n, int64_t c, int64_t h, int64_t wd, int64_t x_zero_point,
                      float x_scale, const float *w_scale, int64_t w_scale_len, float y_scale,
                      int64_t y_zero_point, int y_is_signed, const int32_t *bias,
                      const mmnb_conv_params *prm, void *y) {
  MMNB_GUARD_CTX(ctx);
  if (ctx->capturing) return fail(MMNB_ERR_ARG, "host entry point during graph capture");
  ConvShape s;
  int rc = conv_shape(w, n, c, h, wd, prm, &s);
  if (rc) return rc;
  if (w->ctx != ctx) return fail(MMNB_ERR_ARG, "pack belongs to another context");
  if ((rc = check_zp(x_zero_point, x_is_signed, "QLinearConv: x zero point"))) return rc;
  if ((rc = check_zp(y_zero_point, y_is_signed, "QLinearConv: y zero point"))) return rc;
  if (!x || !y) return fail(MMNB_ERR_ARG, "QLinearConv: null buffer");
  CtxLock lk(ctx);
  if ((rc = set_device(ctx))) return rc;
  const size_t xb = (size_t)(n * c * h * wd), yn = (size_t)(n * w->conv_m * s.oh * s.ow);
  void *d_x = nullptr, *d_y = nullptr;
  if ((rc = scratch_get(ctx, 0, xb + 256, &d_x))) return rc;
  if ((rc = scratch_get(ctx, 1, yn + 256, &d_y))) return rc;
  ConvOut o;
  if ((rc = qconv_params(ctx, w->conv_m, x_scale, w_scale, w_scale_len, y_scale, bias, &o)))
    return rc;
  if (xb) MMNB_HIP(hipMemcpyAsync(d_x, x, xb, hipMemcpyHostToDevice, ctx->stream));
  o.yq = (uint8_t *)d_y;
  o.yzp = (int32_t)y_zero_point;
  o.lo = y_is_signed ? -128 : 0;
  o.hi = y_is_signed ? 127 : 255;
  if ((rc = conv_run(ctx, w, (const uint8_t *)d_x, x_is_signed ? 1 : 0, s, x_zero_point, o)))
    return rc;
  if (yn) MMNB_HIP(hipMemcpyAsync(y, d_y, yn, hipMemcpyDeviceToHost, ctx->stream));
  MMNB_HIP(hipStreamSynchronize(ctx->stream));
  return MMNB_OK;
}
