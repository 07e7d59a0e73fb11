"""How columns are cut among workgroups: the launch rule alone, compiled for the host."""
import random
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).parent.parent / "scaffold_amd" / "csrc"
MAIN = """
#include <cstdio>
#include "column_cut.hpp"
int main() {
  long long n, cols, steps, wgs;
  int records;
  while (std::scanf("%lld %lld %lld %lld %d", &n, &cols, &steps, &wgs, &records) == 5) {
    const sfh::BatchCut b = sfh::cut_batch(n, cols, steps, wgs, records != 0);
    std::printf("%d %d %d %d %d %d %lld\\n", b.parts, b.cut.segs, b.cut.seg_steps, b.cut.items, b.cut.items_per_wg, b.cut.wgs, (long long)b.cut.cost);
  }
}
"""


@pytest.fixture(scope="module")
def cut(tmp_path_factory):
    compiler = shutil.which("g++") or shutil.which("c++")
    if compiler is None:
        pytest.skip("no host compiler")
    where = tmp_path_factory.mktemp("cut")
    (where / "main.cpp").write_text(MAIN)
    subprocess.run([compiler, "-std=c++17", "-O1", f"-I{CSRC}", str(where / "main.cpp"), "-o", str(where / "cut")], check=True)

    def run(problems):
        text = "".join("%d %d %d %d %d\n" % p for p in problems)
        out = subprocess.run([str(where / "cut")], input=text, capture_output=True, text=True, check=True).stdout
        return [tuple(int(v) for v in line.split()) for line in out.splitlines()]
    return run


def _reference(cols, steps, wgs):
    """(busiest workgroup's time, segments, segment length, items, items per workgroup, workgroups), the first of the least time."""
    best = None
    for want in range(1, min(-(-4 * wgs // cols), steps) + 1):
        length = -(-steps // want)
        segs = -(-steps // length)
        per_wg = -(-cols * segs // wgs)
        if best is None or per_wg * (length + 1) < best[0]:
            best = (per_wg * (length + 1), segs, length, cols * segs, per_wg, -(-cols * segs // per_wg))
    return best


def _problems():
    rng = random.Random(5)
    log = lambda hi: round(hi ** rng.random())
    drawn = [(rng.choice((1, 2, 3, 5, 6, 7, 8)), log(4000), log(200), rng.choice((256, 128, 85, 64, 32, 4, 1))) for _ in range(1500)]
    return drawn + [(2, 900_000, 40, 256), (1, 50, 5000, 256), (1, 1, 1 << 20, 256), (1, 1, 1023, 256), (3, 1 << 20, 1, 7)]  # past 32-bit arithmetic, and the last within it


def test_batch_without_records_ends_soonest(cut):
    """Nobody takes the sums: the samples share the workgroups, whatever walking them apart would cost."""
    problems = _problems() + [(3, 16 * 2, 26, 128)]  # three samples of 51 x 126 x 40, 32 -> 64 channels: 24 steps, 27 apart
    for (n, cols, steps, wgs), got in zip(problems, cut([(*p, 0) for p in problems])):
        cost, *rest = _reference(n * cols, steps, wgs)
        assert got == (1, *rest, cost), (n, cols, steps, wgs)


def test_one_sample_with_records_keeps_the_order_of_its_sums(cut):
    """Until every workgroup has an item, and no further."""
    problems = [(1, *p[1:]) for p in _problems()] + [(1, 54 // 4 * 27, 53, 256), (1, 64, 32, 256), (1, 700, 3, 256)]
    for (n, cols, steps, wgs), got in zip(problems, cut([(*p, 1) for p in problems])):
        want = 1 if cols >= wgs else min(-(-wgs // cols), steps)
        length = -(-steps // want)
        segs = -(-steps // length)
        per_wg = -(-cols * segs // wgs)
        assert got == (1, segs, length, cols * segs, per_wg, -(-cols * segs // per_wg), per_wg * (length + 1)), (n, cols, steps, wgs)


def test_batch_with_records_is_walked_apart_where_that_costs_an_eighth_at_most(cut):
    problems = [p for p in _problems() if p[0] > 1]
    apart = 0
    for (n, cols, steps, wgs), got in zip(problems, cut([(*p, 1) for p in problems])):
        line = _reference(n * cols, steps, wgs)
        want = (1, *line[1:], line[0])
        if wgs // n >= 8:
            one = _reference(cols, steps, wgs // n)
            if 8 * one[0] <= 9 * line[0] and one[5] >= 8:
                want = (n, *one[1:], one[0])
                apart += 1
        assert got == want, (n, cols, steps, wgs)
    assert apart > 100
