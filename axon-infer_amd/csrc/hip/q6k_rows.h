// Which kernels run the activation rows of a planar Q6_K matmul: plain host code, without a device.
//
// q6k_planar_mfma_kernel takes chunks of 32 or 16 activation rows, a partial one at the price of a
// whole, q6k_planar_kernel up to 8 rows a lane. Each runs its waves of 64 output rows in rounds of
// one wave per SIMD, and a round that is hardly begun costs nearly what a full one does, so neither
// the rows nor the outputs alone say which is faster: 10 rows take 116 us in q6k_planar_kernel and
// 177 in one 16-row chunk at 80000 x 2048 (two rounds either way), 164 and 178 at 106305 x 2048 (four
// and two). So the plan is the one of the least estimated time. The times below, in ns per element
// of the weight row, are the slopes between n_in 512 and 2048 over 19 output sizes from 4000 to
// 128256 on an MI355X; over 1767 points (rows 2 to 64, n_in 512, 1024, 2048) the plan is nowhere over
// 2 % slower than q6k_planar_kernel for all rows, 5 % faster in the mean, and 0.1 % off the best plan.
#pragma once
#include <algorithm>
#include <cstdint>

namespace axon_hip {

constexpr uint32_t kQ6MaxRows = 8;  // activation rows per lane of q6k_planar_kernel

// q6k_planar_kernel's launch for m activation rows: rows per lane, chunks of them, and 256 (wide) or
// 64 output rows per workgroup.
//  * Up to kQ6MaxRows rows per lane (each then runs that many chains, and every weight slice is read
//    once per that many rows), but fewer while that leaves under 1024 waves of 64 output rows: a
//    lane's chains run one element after another, so a short matrix needs the rows spread over more
//    waves more than it needs fewer weight reads.
//  * Chunks of equal size (20 rows: 7, 7 and 6 rather than 8, 8 and 4, whose last chunk would run eight
//    chains per lane for four rows).
//  * 256 rows per workgroup when that still gives a workgroup per CU, else 64.
struct Q6kLaneRows {
  uint32_t mm, chunks;
  bool wide;
};

inline Q6kLaneRows q6k_lane_rows(uint32_t m, uint32_t n_out) {
  auto div_up = [](uint64_t a, uint64_t b) { return (a + b - 1) / b; };
  uint32_t mm = 1;
  while (mm < kQ6MaxRows && mm < m) mm *= 2;
  while (mm > 1 && div_up(m, mm) * div_up(n_out, 64) < 1024) mm /= 2;
  mm = static_cast<uint32_t>(div_up(m, div_up(m, mm)));
  const uint32_t chunks = static_cast<uint32_t>(div_up(m, mm));
  return {mm, chunks, div_up(n_out, 256) * chunks >= 256};
}

// ns per element for a number of rounds: `batch` of them run side by side in `full`, what is left of
// a batch in `part`; a launch of one round alone takes `one`.
struct Q6kRounds {
  float base, full;
  uint32_t batch;
  float part[3];
  float one;
  float time(uint64_t rounds) const {
    return rounds == 1 ? one : base + full * static_cast<float>(rounds / batch) + part[rounds % batch];
  }
};

inline float q6k_lane_time(uint32_t m, uint32_t n_out, uint32_t simds) {
  if (m == 0) return 0;
  static constexpr Q6kRounds kTimes[kQ6MaxRows] = {
      {0, 17, 2, {0, 14}, 14},   {0, 22, 2, {0, 13}, 13}, {0, 30, 2, {0, 18}, 18}, {0, 34.8f, 2, {0, 22}, 22},
      {0, 38, 2, {0, 19}, 19},   {1, 43, 2, {0, 33}, 34}, {1, 49, 2, {0, 36}, 37}, {8, 71, 3, {0, 32, 47}, 40}};
  const Q6kLaneRows l = q6k_lane_rows(m, n_out);
  const uint64_t waves = (l.wide ? (n_out + 255ull) / 256 * 4 : (n_out + 63ull) / 64) * l.chunks;
  return kTimes[l.mm - 1].time((waves + simds - 1) / simds);
}

// Chunks of 32 and of 16 rows that run on the matrix cores; the rows past them run in
// q6k_planar_kernel. Four chunks of 16 are as fast as two of 32 or faster where rounds are few;
// beyond that 32 always wins.
struct Q6kRowsPlan {
  uint32_t c32, c16;
};

inline Q6kRowsPlan q6k_rows_plan(uint32_t m, uint32_t n_out, uint32_t cus) {
  static constexpr Q6kRounds k32 = {3, 139.5f, 2, {0, 85}, 88}, k16 = {6, 39.2f, 1, {0}, 51.5f};
  constexpr float kLaunch = 2;  // a further launch
  const uint32_t simds = 4 * cus;
  const uint64_t blocks = (n_out + 255ull) / 256;  // workgroups of four waves
  Q6kRowsPlan plan = {0, 0};
  if (m <= kQ6MaxRows || blocks > 65535) return plan;
  auto rounds = [&](uint64_t chunks) { return (4 * blocks * chunks + simds - 1) / simds; };
  float best = q6k_lane_time(m, n_out, simds) / 1.01f;  // (an even estimate stays there)
  for (uint32_t c32 = 0; c32 <= (m + 31ull) / 32; ++c32) {
    const uint32_t after32 = m - std::min<uint64_t>(m, 32ull * c32);
    for (uint32_t c16 = c32 == 0 ? 1 : 0; c16 <= std::min(4u, (after32 + 15) / 16); ++c16) {
      const uint32_t rest = after32 - std::min(after32, 16 * c16);
      const float t = (c32 != 0 ? k32.time(rounds(c32)) + kLaunch : 0) + (c16 != 0 ? k16.time(rounds(c16)) + kLaunch : 0) +
                      (rest != 0 ? q6k_lane_time(rest, n_out, simds) + kLaunch : 0) - kLaunch;
      if (t < best) {
        best = t;
        plan = {c32, c16};
      }
    }
  }
  return plan;
}

}  // namespace axon_hip
