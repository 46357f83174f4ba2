// Which kernel a convolution takes and how it is cut into launches.  Plain C++, so
// that the arithmetic can be checked on the CPU.
#pragma once

#include <cstdint>

namespace mmnb {

constexpr int kConvThreads = 1024;  // of a k_conv workgroup
constexpr int kConvLds = 32768;     // bytes of A per chunk of k_conv

struct ConvPlan {
  bool taps = false;   // k_conv_taps, else k_conv
  int nw = 0;          // taps: words of K per lane (3, 7 or 16)
  int64_t nper = 0;    // taps: channels per workgroup
  int pt = 0, cw = 0;  // k_conv: positions and channel waves per workgroup
  int threads = 0;     // per workgroup
  int64_t gx = 0, gy = 0;  // grid of a launch of `step` positions (the last one: fewer)
  int64_t step = 0;        // positions per launch
};

// P output positions, K taps and N channels per group, z (image, group) pairs.
inline ConvPlan conv_plan(int64_t P, int64_t K, int64_t N, int64_t z, int64_t cus) {
  ConvPlan pl;
  const int64_t blocks = (P + 63) / 64;  // of 64 positions
  // Few taps: k_conv_taps for as many channels per group as it is the faster one (us
  // here and in k_conv, ConvInteger; from two rounds of k_conv's workgroups on their
  // launch counts):
  //   K <= 12: 128 channels, 112 x 112 6.6 and 7.5; 256 channels 10.2 and 8.4;
  //   K <= 28: 64 channels, 112 x 112 6.0 and 6.6, 128 channels 7.9 and 7.5, but 224 x
  //     224 18.9 and 25.1, 256 channels 43.6 and 26.0;
  //   K <= 64: 32 channels, 112 x 112 8.6 and 6.2, but 64 channels, 224 x 224 15.9 and
  //     22.4, 128 channels as bytes 26.8 and 23.8.
  const bool many = blocks * z > 2 * cus;
  if (N <= (K <= 12 ? 128 : K <= 28 ? (many ? 128 : 64) : K <= 64 && many ? 64 : 0)) {
    pl.taps = true;
    pl.nw = K <= 12 ? 3 : K <= 28 ? 7 : 16;
    // a wave per SIMD at least, with fewer channels each and the bytes gathered again;
    // more than 8 per SIMD go over several blocks of positions
    pl.nper = N;
    while (pl.nper > 4 && blocks * z * ((N + pl.nper - 1) / pl.nper) < 4 * cus)
      pl.nper = (pl.nper + 1) / 2;
    pl.gy = (N + pl.nper - 1) / pl.nper;
    const int64_t waves = blocks < 4 ? blocks : 4;
    pl.threads = (int)(64 * waves);
    pl.gx = (blocks + waves - 1) / waves;
    const int64_t most = 32 * cus / (waves * pl.gy * z);
    if (pl.gx > most) pl.gx = most > 1 ? most : 1;
    pl.step = P;
    return pl;
  }
  // the most positions per read of the weights that leave a workgroup on three
  // quarters of the CUs; then, while half of them are idle, fewer channels per
  // workgroup: the gather is repeated, but a workgroup reads less of the weights
  // (256 channels of 14 x 14, 3 x 3 to 256: 13.3 us, with all 256 in one workgroup
  // 25.8)
  pl.cw = 1;
  while (pl.cw < 16 && 16 * pl.cw < N) pl.cw *= 2;
  auto groups = [&](int64_t pt) {
    return (P + pt - 1) / pt * ((N + 16 * pl.cw - 1) / (16 * pl.cw)) * z;
  };
  const int64_t enough = 3 * cus / 4;
  while (pl.cw > 1 && groups(16) < cus / 2) pl.cw /= 2;
  pl.pt = groups(64) >= enough ? 64 : groups(32) >= enough ? 32 : 16;
  pl.threads = kConvThreads;
  pl.gy = (N + 16 * pl.cw - 1) / (16 * pl.cw);
  // a launch holds less than 2^32 threads along x
  pl.gx = (P + pl.pt - 1) / pl.pt;
  const int64_t most = (int64_t)(UINT32_MAX / kConvThreads);
  if (pl.gx > most) pl.gx = most;
  pl.step = pl.gx * pl.pt;
  return pl;
}

}  // namespace mmnb
