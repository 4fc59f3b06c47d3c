"""The rule that chooses the tile of a many-row quantized matmul (csrc/hip/wide_tiles.h, plain host
code), against times measured on an MI355X."""
import subprocess
from pathlib import Path

import pytest

HIP = Path(__file__).resolve().parents[1] / "axon-infer_amd" / "csrc" / "hip"

# (type, rows, outputs, inputs): us with tiles of 64 x 128, 64 x 64, 32 x 64 and 32 x 32
TIMES = {
    ("q4_0", 111, 701, 448): (9.1, 6.7, 5.9, 6.2),
    ("q4_0", 229, 639, 960): (14.9, 10.4, 7.9, 6.2),
    ("q4_0", 82, 662, 2688): (34.1, 22.9, 16.5, 11.9),
    ("q4_0", 150, 1312, 960): (14.9, 10.4, 8.0, 6.4),
    ("q4_0", 258, 3603, 320): (8.5, 6.8, 8.4, 6.6),
    ("q4_0", 70, 7269, 768): (11.9, 8.5, 9.0, 8.4),
    ("q4_0", 74, 3770, 1664): (22.6, 15.8, 11.7, 10.9),
    ("q4_0", 263, 3646, 704): (12.3, 9.7, 12.7, 11.3),
    ("q4_0", 109, 8213, 1344): (19.8, 15.5, 20.0, 17.2),
    ("q4_0", 125, 5503, 1984): (26.2, 18.4, 17.1, 15.3),
    ("q4_0", 216, 8109, 1280): (18.9, 16.1, 24.4, 22.2),
    ("q4_0", 127, 8410, 2496): (34.3, 26.7, 32.7, 28.6),
    ("q4_0", 227, 15272, 832): (18.2, 22.1, 32.8, 29.5),
    ("q4_0", 153, 6666, 3520): (49.9, 35.9, 45.8, 38.7),
    ("q4_0", 300, 3606, 5760): (79.1, 55.5, 72.0, 62.1),
    ("q4_0", 269, 11660, 2048): (34.3, 42.0, 54.5, 51.8),
    ("q4_0", 361, 12692, 2048): (73.7, 57.5, 85.4, 79.1),
    ("q4_0", 284, 13967, 2944): (83.6, 66.4, 90.1, 89.1),
    ("q4_1", 66, 2207, 832): (19.0, 11.3, 8.4, 6.4),
    ("q4_1", 478, 771, 1088): (23.6, 14.2, 10.8, 10.0),
    ("q4_1", 182, 4076, 768): (17.2, 10.4, 10.6, 9.7),
    ("q4_1", 90, 10694, 768): (17.5, 12.7, 10.9, 12.6),
    ("q4_1", 121, 1238, 4992): (87.8, 49.9, 33.6, 22.8),
    ("q4_1", 285, 2327, 2112): (41.2, 24.1, 22.4, 20.0),
    ("q4_1", 100, 2309, 7488): (140.9, 76.8, 53.0, 44.6),
    ("q4_1", 119, 15463, 1152): (27.8, 20.1, 27.9, 28.6),
    ("q4_1", 366, 1667, 3712): (71.3, 42.0, 35.8, 31.8),
    ("q4_1", 236, 10201, 1792): (43.4, 40.8, 44.9, 50.0),
    ("q4_1", 362, 7813, 2304): (56.7, 54.3, 68.2, 71.8),
    ("q4_1", 286, 3025, 7552): (137.9, 78.6, 65.9, 82.6),
    ("q4_1", 455, 9481, 2752): (123.7, 99.2, 118.4, 125.0),
    ("q8_0", 68, 1682, 2112): (28.8, 19.0, 15.2, 10.6),
    ("q8_0", 158, 5325, 768): (12.8, 9.1, 9.9, 10.9),
    ("q8_0", 216, 2049, 1536): (21.2, 13.6, 11.0, 9.8),
    ("q8_0", 233, 4647, 832): (15.1, 12.3, 16.5, 13.4),
    ("q8_0", 229, 4777, 832): (15.0, 12.3, 16.6, 13.3),
    ("q8_0", 414, 1240, 2496): (32.8, 21.7, 20.6, 15.6),
    ("q8_0", 175, 6347, 1408): (23.8, 17.2, 21.7, 20.4),
    ("q8_0", 490, 2143, 1600): (27.5, 19.0, 25.2, 22.6),
    ("q8_0", 170, 6544, 1728): (26.4, 21.8, 29.5, 25.1),
    ("q8_0", 227, 4172, 2112): (34.8, 25.3, 32.5, 28.6),
    ("q8_0", 370, 3172, 1792): (29.1, 20.3, 27.7, 22.9),
    ("q8_0", 468, 3024, 2112): (30.3, 24.4, 31.0, 33.1),
    ("q8_0", 281, 7560, 1408): (25.6, 31.4, 36.7, 30.9),
    ("q8_0", 247, 4948, 3008): (46.9, 34.7, 44.6, 38.1),
    ("q8_0", 266, 7297, 3328): (60.6, 74.0, 86.8, 72.7),
    ("q8_0", 166, 16361, 2496): (47.5, 58.0, 70.2, 68.9),
    ("q8_0", 351, 7938, 2944): (55.9, 61.8, 75.9, 70.2),
}


@pytest.fixture(scope="module")
def tile(tmp_path_factory):
    d = tmp_path_factory.mktemp("tile")
    (d / "tile.cpp").write_text("""#include <cstdio>
#include "wide_tiles.h"
using namespace axon_hip;
int main() {
  int type, fits;
  unsigned long long m, n, nb;
  while (scanf("%d %llu %llu %llu %d", &type, &m, &n, &nb, &fits) == 5) {
    auto count = [&](uint64_t tm, uint64_t tn) { return (m + tm - 1) / tm * ((n + tn - 1) / tn); };
    const uint64_t w[kWideTiles] = {count(64, 128), count(64, 64), count(32, 64), count(32, 32)};
    printf("%d\\n", static_cast<int>(wide_tile(static_cast<WideType>(type), static_cast<uint32_t>(nb), w, 256, fits)));
  }
}
""")
    subprocess.run(["g++", "-std=c++20", "-O1", "-Wall", "-Werror", "-I", str(HIP), str(d / "tile.cpp"), "-o", str(d / "tile")], check=True)

    def ask(cases):
        text = "".join("%d %d %d %d %d\n" % c for c in cases)
        out = subprocess.run([str(d / "tile")], input=text, check=True, capture_output=True, text=True).stdout
        return [int(line) for line in out.splitlines()]
    return ask


def test_the_tile_is_near_the_best_one(tile):
    kinds = {"q4_0": 0, "q8_0": 1, "q4_1": 2}
    cases = [(kinds[t], m, n, k // 32, 1) for t, m, n, k in TIMES]
    total = 1.0
    for (shape, times), t in zip(TIMES.items(), tile(cases)):
        best = min(times if shape[3] >= 48 * 32 else times[1:])
        assert times[t] <= 1.1 * best, (shape, t)
        total *= times[t] / best
    assert total ** (1 / len(TIMES)) < 1.02


def test_the_largest_tile_only_where_it_fits_and_rows_are_long(tile):
    shapes = [(t, m, n, nb) for t in range(3) for m in (33, 512, 4096) for n in (1, 8192, 1 << 20) for nb in (2, 46, 48, 1 << 17)]
    assert 0 not in tile([s + (0,) for s in shapes])
    assert all(t != 0 or s[3] >= 48 for s, t in zip(shapes, tile([s + (1,) for s in shapes])))
    assert set(tile([s + (1,) for s in shapes + [(0, 319, 2906, 84)]])) == {0, 1, 2, 3}
