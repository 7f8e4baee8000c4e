"""The points per device batch and the choice to keep the first pass's products (csrc/qt_plan.h, compiled for
the host): a call that fits the memory without the kept products fits with the plan, and blocks that take
more than 128 points leave the rest of the device alone."""
import itertools
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "quantum_transport_amd", "csrc")
MAIN = r"""
#include <cstdio>
#include "qt_plan.h"
// lines "npts nmax avail total extra fixed per": per bytes a point, half as much again with kept products
int main() {
    int npts, nmax, fixed;
    unsigned long long avail, total, extra, per;
    while (scanf("%d %d %llu %llu %llu %d %llu", &npts, &nmax, &avail, &total, &extra, &fixed, &per) == 7) {
        const qt::BatchPlan p = qt::plan_batch(npts, nmax, avail, total, extra, fixed, [&](int B, bool keep) {
            return (size_t)B * per * (keep ? 3 : 2) / 2;
        });
        printf("%d %d\n", p.B, (int)p.keep);
    }
}
"""
GB = 1 << 30
TOTAL = 288 * GB


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC}", "-o", str(d / "plan"), str(d / "main.cpp")], check=True)

    def run(rows):
        text = "\n".join(" ".join(str(int(v)) for v in r) for r in rows)
        out = subprocess.run([str(d / "plan")], input=text, capture_output=True, text=True, check=True).stdout
        return [(int(a), bool(int(b))) for a, b in (line.split() for line in out.splitlines())]

    return run


def _workspace(per, B, keep):
    return B * per * (3 if keep else 2) // 2


@pytest.mark.parametrize("row,want", [
    # npts, nmax, avail, total, extra, fixed, per
    ((64, 512, TOTAL, TOTAL, 0, 0, GB), (64, True)),             # room for all
    ((1000, 64, TOTAL, TOTAL, 0, 0, 8 << 20), (1000, True)),     # small blocks: up to 1024 points
    ((200, 64, TOTAL, TOTAL, 0, 0, 8 << 20), (200, True)),
    ((300, 96, TOTAL, TOTAL, 0, 0, 8 << 20), (150, True)),       # 256 points at most, dealt evenly
    ((1000, 64, TOTAL, TOTAL, 0, 0, 256 << 20), (125, True)),    # ... but a sixteenth of the memory at most
    ((64, 512, 36 * GB, TOTAL, 0, 0, GB), (22, False)),          # short of memory: 22 points a batch, 16 with X and V
    ((64, 512, GB, TOTAL, 0, 0, 9 * GB // 10), (1, False)),      # one point fits without them only
    ((64, 512, 36 * GB, TOTAL, 0, 28, GB), (28, False)),         # fixed points fit without them only
    ((64, 512, 36 * GB, TOTAL, 0, 16, GB), (16, True)),
    ((200, 64, TOTAL, TOTAL, 1, 0, 8 << 20), (100, False)),      # extra memory refused
    ((64, 512, TOTAL, TOTAL, 0, 0, 8 * GB), (22, False)),        # 32 points with them exceed the device
    ((3, 512, TOTAL, 0, 0, 0, GB), (3, False)),                  # memory unknown
    ((1, 1, TOTAL, TOTAL, 0, 0, 1), (1, True)),
])
def test_plan(plan, row, want):
    assert plan([row]) == [want]


def test_plan_fits_where_the_plain_sweep_does(plan):
    grid = list(itertools.product((1, 7, 64, 128, 129, 500, 4096), (1, 33, 64, 65, 129, 512, 1024),
                                  (GB // 2, 3 * GB, 17 * GB, 120 * GB, TOTAL), (TOTAL,), (0, 1, 5 * GB),
                                  (0, 1, 16, 300), (1 << 10, 3 << 20, 700 << 20, 5 * GB)))
    for (npts, nmax, avail, total, extra, fixed, per), (B, keep) in zip(grid, plan(grid)):
        row = (npts, nmax, avail, total, extra, fixed, per)
        budget = int(0.8 * avail)
        assert 1 <= B <= npts, row
        if fixed:
            assert B == min(npts, fixed), row
        else:
            assert _workspace(per, B, keep) <= budget or (B, keep) == (1, False), row
            assert B <= 128 or _workspace(per, B, keep) <= total // 16, row
            assert -(-npts // B) * B - npts < -(-npts // B), row  # padding: less than a point a batch
        if keep:
            assert _workspace(per, B, True) <= min(extra or budget, budget), row
