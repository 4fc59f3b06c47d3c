"""The rule that splits the activation rows of a planar Q6_K matmul between the matrix-core chunks and
the vector-ALU kernel (csrc/hip/q6k_rows.h, plain host code), against times measured on an MI355X: no
plan is slower than all rows in the vector-ALU kernel by more than the runs differ, and none is far
from the best plan."""
import subprocess
from pathlib import Path

import pytest

HIP = Path(__file__).resolve().parents[1] / "axon-infer_amd" / "csrc" / "hip"

ROWS = (1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 14, 15, 16, 20, 21, 22, 24, 25, 28, 31)
# us at n_in 2048, by output rows: one and two chunks of 32, one to four of 16, and ROWS in the
# vector-ALU kernel.
TIMES = {
    16000: ((192, 198), (108, 113, 114, 116), (15, 34, 32, 40, 43, 43, 45, 41, 53, 52, 52, 52, 52, 48, 49, 74, 75, 75, 75, 76, 76, 76)),
    32000: ((192, 205), (109, 116, 179, 180), (19, 39, 43, 40, 54, 52, 47, 51, 64, 74, 74, 74, 77, 76, 76, 106, 107, 128, 130, 110, 108, 129)),
    56000: ((197, 299), (109, 180, 259, 347), (39, 40, 50, 49, 63, 62, 74, 74, 81, 81, 92, 93, 105, 125, 126, 184, 184, 175, 174, 203, 203, 238)),
    64000: ((198, 302), (109, 183, 270, 354), (39, 42, 52, 52, 70, 69, 80, 78, 86, 85, 95, 95, 107, 129, 128, 189, 187, 180, 177, 210, 215, 240)),
    66000: ((293, 458), (173, 255, 341, 421), (39, 46, 59, 70, 78, 90, 102, 120, 115, 114, 163, 164, 180, 171, 171, 202, 204, 232, 234, 269, 269, 268)),
    80000: ((299, 463), (177, 261, 345, 431), (39, 46, 60, 72, 79, 91, 104, 123, 118, 116, 166, 164, 182, 173, 173, 210, 208, 239, 238, 271, 273, 270)),
    99000: ((299, 586), (176, 346, 433, 576), (40, 47, 62, 74, 82, 92, 106, 126, 157, 159, 180, 177, 200, 236, 234, 274, 276, 272, 272, 360, 360, 366)),
    112000: ((301, 588), (177, 340, 508, 582), (40, 46, 62, 74, 82, 93, 106, 125, 159, 164, 188, 181, 204, 239, 238, 302, 302, 314, 316, 362, 364, 378)),
    128256: ((310, 591), (178, 345, 519, 670), (40, 47, 67, 78, 85, 96, 109, 127, 158, 165, 189, 186, 209, 240, 241, 310, 308, 321, 322, 402, 400, 415)),
}


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text("""#include <cstdio>
#include "q6k_rows.h"
int main() {
  unsigned m, n, cus;
  while (scanf("%u %u %u", &m, &n, &cus) == 3) {
    const auto p = axon_hip::q6k_rows_plan(m, n, cus);
    printf("%u %u\\n", p.c32, p.c16);
  }
}
""")
    subprocess.run(["g++", "-std=c++20", "-O1", "-Wall", "-Werror", "-I", str(HIP), str(d / "plan.cpp"), "-o", str(d / "plan")], check=True)

    def ask(cases):
        text = "".join("%d %d %d\n" % c for c in cases)
        out = subprocess.run([str(d / "plan")], input=text, check=True, capture_output=True, text=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]
    return ask


def cost(n_out, m, c32, c16):
    """The measured parts one after another; None where one of them was not measured."""
    chunks32, chunks16, lanes = TIMES[n_out]
    rest = max(0, max(0, m - 32 * c32) - 16 * c16)
    if c32 > len(chunks32) or c16 > len(chunks16) or (rest and rest not in ROWS):
        return None
    return (chunks32[c32 - 1] if c32 else 0) + (chunks16[c16 - 1] if c16 else 0) + (lanes[ROWS.index(rest)] if rest else 0)


def test_no_plan_is_slower_than_the_vector_kernel(plan):
    cases = [(m, n, 256) for n in TIMES for m in ROWS]
    for (m, n, _), (c32, c16) in zip(cases, plan(cases)):
        t = cost(n, m, c32, c16)
        assert t is not None and t <= 1.02 * cost(n, m, 0, 0) + 1, (m, n, c32, c16)
        best = min(v for v in (cost(n, m, a, b) for a in range(3) for b in range(5)) if v is not None)
        assert t <= 1.06 * best + 1, (m, n, c32, c16)


def test_plans_hold_the_rows(plan):
    """Chunks never outnumber what the rows need, up to the largest calls and on other chips."""
    cases = [(m, n, cus) for m in (1, 2, 8, 9, 16, 17, 31, 32, 33, 64, 65, 200, 512, 2048) for n in
             (1, 64, 300, 16384, 65473, 65536, 65537, 128256, 262144, 4194305, 16776961) for cus in (64, 256, 304)]
    for (m, n, cus), (c32, c16) in zip(cases, plan(cases)):
        assert 32 * c32 < m + 32 and (c16 == 0 or 32 * c32 + 16 * c16 < m + 16), (m, n, cus, c32, c16)
        if m <= 8 or n > 65535 * 256:
            assert (c32, c16) == (0, 0)
