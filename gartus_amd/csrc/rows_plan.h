// rows_plan.h — which convolution layers the row kernel (denoise.hip) takes, and how it splits them. Host code only.
#pragma once
#include <algorithm>
#include <cstdint>

namespace gdn {

// The 16-channel output fragments a block of k_conv makes of a layer of `tiles` tiles of 4 x 64 pixels: levels with few
// tiles take narrower groups (more blocks, each staging the same halo for fewer channels), so that the launch still has
// blocks for most CUs.
inline int conv_frags(int64_t tiles) { return tiles >= 1024 ? 4 : tiles >= 256 ? 2 : 1; }

// The 16-channel output fragments a wave of the row kernel's instance makes for a layer from ca channels at half
// resolution and cb at full resolution to cout; 0: the layer takes k_conv, which sums its forward outputs in the same
// order. grad: the data gradient, whose input is the layer's output gradient.
//
// Two things make the row kernel the slower one on small images. A wave of a wide instance loads many weights for a few
// rows. And output channels beyond a multiple of two fragments need a second launch, which is about 5 us whatever its
// size. So such layers take k_conv while it has few blocks. On one MI355X, k_conv and the row kernel in us, below and
// at or above the line:
//   16 -> 112 (a second launch): 160 to 448 blocks 5.6 to 7.0 and 6.0 to 7.2; 1400 blocks 15.1 and 11.3
//   32 -> 80: 160 blocks 5.8 and 6.2; 320 blocks 7.2 and 6.6
//   32 -> 112, 48 -> 80, 96 -> 80 (second launches): 320 to 448 blocks 7.5, 9.0, 11.7 and 9.6, 9.8, 14.2; 1000 to 1400
//     blocks 16.5, 15.9, 21.4 and 14.1, 14.8, 20.2
//   64 -> 128: 512 blocks 10.3 and 10.8. 64 -> 64: 800 blocks 16.5 and 14.1. Gradient 64 -> 160: 640 blocks 16.6 and 12.8
//   64 -> 16, whose wave holds half the weights: 64 blocks 7.5 and 6.5; 384 blocks 9.6 and 14.4; 2025 blocks 35 and 31
//   64 -> 80 and 64 -> 112 (second launches): 1152 and 1400 blocks 31.9, 21.6 and 35.2, 29.0; 2700 blocks (80) 70 and 54
// Data gradients of 64 channels whose outputs are whole groups take the row kernel at every size: alone k_conv is the
// faster one there too (64 -> 64, 256 blocks: 8.3 and 9.0), but a training step on two 119x140 images took 576 us with it
// and 565 with the row kernel.
// 48 channels are one group of three fragments: in groups of two and one, 64 -> 48 and 96 -> 48 read their input twice
// and lost on large images (1920x1080: k_conv 215 and 294 us, 269 and 348 in two launches, 132 and 174 so).
inline int rows_frags(int ca, int cb, int cout, bool grad, int64_t tiles) {
  const int frags = cout / 16;
  const int per = conv_frags(tiles);
  const int64_t blocks = tiles * ((frags + per - 1) / per);  // k_conv's
  const bool rest = frags > 2 && frags % 2 != 0;  // of an instance of two fragments
  switch (ca * 1000 + cb) {
    case 16:
      if (cout == 48) return 3;
      return rest && blocks < 300 ? 0 : 2;
    case 32:
      if (cout == 48) return 3;
      if (frags % 5 == 0) return blocks < 300 ? 0 : 5;
      return rest && blocks < 500 ? 0 : 2;
    case 48:
      if (cout == 48) return 3;
      return rest && blocks < 500 ? 0 : 2;
    case 64:
      if (grad && !rest && cout != 48) return 2;
      if (cout == 16) return blocks >= 100 && blocks < 900 ? 0 : 2;
      if (cout == 48) return blocks < 620 ? 0 : 3;
      return blocks < (rest ? 1500 : 620) ? 0 : 2;
    case 80: return cout == 32 && !grad ? 2 : 0;
    case 96:
      if (cout == 48) return blocks < 500 ? 0 : 3;
      return rest && blocks < 500 ? 0 : 2;
    case 48032: return cout == 32 ? 2 : 0;
    case 64032: return cout == 32 ? 2 : 0;
    case 64048: return cout == 48 ? 3 : 0;
    case 96064: return cout == 64 ? 2 : 0;
    default: return 0;
  }
}

// A launch of the row kernel: n images of h x w in segments of `rows` rows (the last one shorter) by strips of 16
// columns, for `groups` groups of output channels, on a chip that holds `waves` waves.
struct RowsSplit {
  int rows, segs, strips;
  int blocks;  // of each of the 8 XCDs, a multiple of groups; a block's four waves take a tile (segment x strip) each
};
inline RowsSplit rows_split(int n, int h, int w, int groups, int waves) {
  RowsSplit s{0, 0, (w + 15) / 16, 0};
  // the fewest rows in sequence, each segment costing two rows more than it makes
  int64_t best = INT64_MAX;
  for (int r : {64, 48, 32, 24, 16, 12, 8, 6, 4, 2}) {
    const int64_t jobs = int64_t(n) * ((h + r - 1) / r) * s.strips * groups;
    const int64_t cost = (jobs + waves - 1) / waves * (std::min(r, h) + 2);
    if (cost < best) s.rows = r, best = cost;
  }
  s.segs = (h + s.rows - 1) / s.rows;
  const int64_t quads = (int64_t(n) * s.segs * s.strips + 31) / 32 * groups;  // blocks an XCD could use
  const int bpx = int(std::min<int64_t>(quads, std::max(waves / 32, groups)));
  s.blocks = std::max(bpx / groups, 1) * groups;
  return s;
}

}  // namespace gdn
