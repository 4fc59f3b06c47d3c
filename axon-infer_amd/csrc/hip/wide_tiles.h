// Which tile a many-row quantized matmul takes: plain host code, without a device.
//
// A tile's workgroups run in rounds of one per CU, two to four of which share the CU, and the last
// round costs nearly a whole one however few workgroups it holds. So the tile is the one of the least
// estimated time: rounds times blocks per row times the time of a block, plus what a round costs
// whatever its blocks. With fixed numbers of workgroups as lines (512 for the largest and the 32 x 64
// tiles, 320 for 64 x 64), Q8_0 174 x 4168 x 1984 ran 786 workgroups of 32 x 32 in 21.5 us where 198 of
// 64 x 64 take 20.1 and 396 of 32 x 64 19.2; Q4_0 300 x 3606 x 5760 570 of 32 x 64 in 72 us where 285 of
// 64 x 64 take 55.5.
// Fitted to 655 shapes (33 to 512 rows, 400 to 32768 outputs, 64 to 8192 inputs) on an MI355X: 0.5 % off
// the best tile in the mean, 3.2 % faster than the fixed lines and over 3 % slower at one shape.
#pragma once
#include <cstdint>

namespace axon_hip {

// Activation rows x weight rows of a tile.
enum WideTile { kTile64x128, kTile64x64, kTile32x64, kTile32x32, kWideTiles };
enum WideType { kWideQ4_0, kWideQ8_0, kWideQ4_1 };

constexpr uint32_t kWideMinBlocks = 48;  // blocks per row from which the largest tiles pay (896 x 9728 at 512 rows 31 / 25 us)

inline WideTile wide_tile(WideType type, uint32_t nb, const uint64_t (&workgroups)[kWideTiles], uint32_t cus,
                          bool largest_fits) {
  // ns of a block of 32 elements for one to four rounds side by side.
  static constexpr float kBlock[3][kWideTiles][4] = {
      {{364, 470, 900, 1000}, {234, 299, 417, 560}, {147, 203, 360, 440}, {94, 135, 172, 240}},
      {{397, 540, 1000, 1120}, {232, 305, 590, 620}, {168, 230, 390, 545}, {92, 134, 193, 280}},
      {{552, 715, 1400, 1500}, {302, 405, 690, 830}, {185, 258, 420, 560}, {113, 159, 225, 336}}};
  // ns of a launch and of each round in it.
  static constexpr float kFixed[kWideTiles][2] = {{3600, 600}, {4200, 600}, {3800, 600}, {3600, 400}};
  WideTile best = kWideTiles;
  float least = 0;
  for (int t = 0; t < kWideTiles; ++t) {
    if (t == kTile64x128 && (nb < kWideMinBlocks || !largest_fits)) continue;
    const uint64_t rounds = (workgroups[t] + cus - 1) / cus;
    const float* side = kBlock[type][t];
    const float block = static_cast<float>(rounds / 4) * side[3] + (rounds % 4 != 0 ? side[rounds % 4 - 1] : 0);
    const float time = kFixed[t][0] + kFixed[t][1] * static_cast<float>(rounds) + block * static_cast<float>(nb);
    if (best == kWideTiles || time < least) {
      best = static_cast<WideTile>(t);
      least = time;
    }
  }
  return best;
}

}  // namespace axon_hip
