"""How calls are cut into workgroups (``csrc/*_plan.h``, host code): what the
plans launch fits a launch, and every size they refuse has another path.
Compiled with g++ and run here; no GPU."""
import os
import random
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "tensorly_amd", "csrc")
MAX_THREADS = 2 ** 32 - 1  # of one launch's x dimension

TTM = r"""
#include <cstdio>
#include "ttm_plan.h"
int main() {
  long long f64, Pa, Im, Pb, J;
  while (std::scanf("%lld %lld %lld %lld %lld", &f64, &Pa, &Im, &Pb, &J) == 5) {
    tla::TtmPlan p;
    const bool ok = tla::ttm_any_plan(f64, Pa, Im, Pb, J, &p);
    std::printf("%d %d %d %lld %d %lld %lld %d\n", ok, p.JT, p.TN, (long long)p.tiles, p.split, (long long)p.gx, (long long)p.gy, p.vector);
  }
}
"""


ANY = r"""
#include <cstdio>
#include "mttkrp_any_plan.h"
int main() {
  long long f64, R, mode, weights, n;
  while (std::scanf("%lld %lld %lld %lld %lld", &f64, &R, &mode, &weights, &n) == 5) {
    int64_t shape[8];
    for (int m = 0; m < n; ++m) {
      long long s = 0;
      if (std::scanf("%lld", &s) != 1) return 1;
      shape[m] = s;
    }
    tla::AnyPlan p;
    const bool ok = tla::any_plan(f64, n, shape, R, mode, weights, &p);
    std::printf("%d %d %d %d %lld %lld %lld %lld %d %d %zu %d\n", ok, p.last, p.TN, p.RT, (long long)p.groups,
                (long long)p.slices, (long long)p.nblk, (long long)p.nchunks, p.build_g, p.direct_g, p.ws_bytes, p.vector);
  }
}
"""


def compiled(tmp_path_factory, name, text):
    d = tmp_path_factory.mktemp(name)
    src, exe = d / "main.cpp", d / "main"
    src.write_text(text)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)

    def ask(rows):
        out = subprocess.run([str(exe)], input="\n".join(" ".join(str(int(v)) for v in r) for r in rows), text=True,
                             capture_output=True, check=True).stdout
        return [[int(v) for v in line.split()] for line in out.splitlines()]
    return ask


@pytest.fixture(scope="module")
def ttm_plan(tmp_path_factory):
    ask = compiled(tmp_path_factory, "ttm", TTM)
    keys = ("ok", "JT", "TN", "tiles", "split", "gx", "gy", "vector")
    return lambda rows: [dict(zip(keys, r)) for r in ask(rows)]


def test_mode_dot_grids_fit_a_launch(ttm_plan):
    """Many short runs: a tile of 64 columns each.  Sizes past a launch are
    left to the vector kernel (fewer than 2^32 outputs here)."""
    edge = [(0, 70_000_000, 2, 4, 2), (0, 67_108_864, 4, 4, 1), (0, 67_108_860, 4, 4, 1), (1, 67_108_868, 3, 2, 1),
            (0, 2 ** 30, 5, 1, 1), (0, 2 ** 33, 2, 1, 1), (0, 2 ** 36, 2, 1, 1), (0, 2 ** 40, 2, 4, 1)]
    rng = random.Random(1)
    rows = edge + [(rng.random() < 0.5, int(2 ** rng.uniform(0, 36)), int(2 ** rng.uniform(0, 12)),
                    rng.choice([1, 2, 3, 4, 5, 8, 63, 64, 65, 1000, 10 ** 6]), int(2 ** rng.uniform(0, 12)))
                   for _ in range(4000)]
    plans = ttm_plan(rows)
    for row, p in zip(rows, plans):
        if p["ok"]:
            assert 0 < p["gx"] * 256 <= MAX_THREADS and 0 < p["gy"] <= 65535, (row, p)
    assert [p["ok"] for p in plans[:4]] == [0, 0, 1, 0]


def test_mode_dot_plans_cover_every_output(ttm_plan):
    rng = random.Random(2)
    rows = [(rng.random() < 0.5, int(2 ** rng.uniform(0, 16)), int(2 ** rng.uniform(0, 10)),
             rng.choice([1, 4, 5, 31, 32, 33, 64, 65, 129, 1000]), int(2 ** rng.uniform(0, 9))) for _ in range(4000)]
    for (f64, Pa, Im, Pb, J), p in zip(rows, ttm_plan(rows)):
        assert p["ok"] and 1 <= p["JT"] <= 4 and p["gy"] * 16 * p["JT"] >= J
        if Pb == 1:
            assert p["TN"] in ((1, 4) if p["JT"] <= 2 else (1, 2)) and p["gx"] * 4 * 16 * p["TN"] >= Pa
        else:
            assert p["TN"] in ((1, 2) if p["JT"] <= 2 else (1,))
            assert p["tiles"] * 16 * (2 if f64 else 4) * p["TN"] >= Pb
            assert p["gx"] * (1 if p["split"] else 4) >= Pa * p["tiles"]


@pytest.fixture(scope="module")
def any_plan(tmp_path_factory):
    ask = compiled(tmp_path_factory, "any", ANY)
    keys = ("ok", "last", "TN", "RT", "groups", "slices", "nblk", "nchunks", "build_g", "direct_g", "ws", "vector")
    return lambda rows: [dict(zip(keys, r)) for r in ask([(f, R, m, w, len(s), *s) for f, s, R, m, w in rows])]


def _shapes(rng, count, most):
    for _ in range(count):
        nd = rng.choice([2, 3, 3, 4, 4, 5, 6])
        side = 2 ** (rng.uniform(3, most) / nd)
        s = [max(1, int(side * 2 ** rng.uniform(-most / 4, most / 4))) for _ in range(nd)]
        for m in range(nd):
            yield rng.random() < 0.5, s, rng.choice([1, 7, 16, 33, 64, 65, 200]), m, rng.random() < 0.5


def test_mttkrp_scratch_is_bounded(any_plan):
    """Scale rows: at most 256 MiB; partial sums: 32 MiB, or one set of a rank
    slab for each slice of the scale rows (past rank 64, for one); and a call
    without weights needs no more than the query said."""
    rng = random.Random(3)
    rows = [(0, s, 64, 0, 1) for s in ((2, 8192, 8192, 2), (6, 4096, 682, 8))]
    rows += [(0, (4096, 4096, 4, 6), 64, 2, 1), (0, (2000, 4096, 4, 6), 64, 3, 1)]
    rows += list(_shapes(rng, 1500, 38))
    plans = any_plan(rows)
    bare = any_plan([(f, s, R, m, 0) for f, s, R, m, _ in rows])
    full = any_plan([(f, s, R, m, 1) for f, s, R, m, _ in rows])
    for (f, s, R, m, _), p, b, w in zip(rows, plans, bare, full):
        if p["ok"]:
            assert p["ws"] <= (256 << 20) + max(32 << 20, p["slices"] * s[m] * 64 * (8 if f else 4)) + 512, (f, s, R, m, p)
        assert b["ok"] == w["ok"] and b["ws"] <= w["ws"], (f, s, R, m)
    assert [p["slices"] for p in plans[2:4]] == [16, 8]


def test_mttkrp_grids_fit_a_launch(any_plan):
    rng = random.Random(4)
    rows = [(0, (500_000_000, 2, 2), 1, 0, 1), (0, (2 ** 28, 4), 1, 0, 1)] + list(_shapes(rng, 1500, 50))
    for row, p in zip(rows, any_plan(rows)):
        if p["ok"]:
            rows_out = row[1][row[3]]
            assert 0 < p["groups"] * p["nblk"] * 256 <= MAX_THREADS, (row, p)
            assert (rows_out * min(row[2], 64) + 31) // 32 * 256 + 256 <= MAX_THREADS, (row, p)
            assert p["groups"] * p["TN"] * (16 * (2 if row[0] else 4) if p["last"] else 16) >= rows_out


def test_mttkrp_tiles_of_long_modes(any_plan):
    """With more groups than waves fit the GPU, several tiles per wave share
    the rows of the Khatri-Rao product."""
    rows = [(0, (200_000, 30, 41), 16, 0, 0), (0, (1_000_000, 7, 9), 16, 0, 1), (1, (100_000, 33, 35), 20, 0, 0),
            (0, (5, 9, 500_001), 8, 2, 0), (0, (9, 70_001, 31), 33, 1, 1)]
    assert all(p["TN"] >= 2 for p in any_plan(rows))


def test_mode_dot_short_runs_keep_the_vector_kernel(ttm_plan):
    """Tiles that would be mostly padding: short contiguous runs, few rows,
    short sums; and not where the tiles are full."""
    vector = [(0, 2_000_000, 4, 4, 1), (1, 2_000_000, 4, 4, 1), (0, 100_000, 2, 4, 2), (1, 100_000, 2, 4, 2),
              (0, 1, 2, 3_000_000, 1), (0, 1_000_000, 5, 1, 1), (0, 262_144, 16, 4, 4)]
    tiles = [(0, 1, 256, 65536, 32), (0, 256, 256, 256, 32), (0, 65536, 256, 1, 32), (0, 250, 30, 20, 331),
             (1, 25, 331, 190, 30), (0, 82_750, 190, 1, 20), (0, 82_750, 20, 1, 190), (0, 100, 100, 100, 16)]
    assert all(p["vector"] for p in ttm_plan(vector))
    assert not any(p["vector"] for p in ttm_plan(tiles))


def test_mode_dot_narrow_runs_take_one_tile(ttm_plan):
    rows = [(0, 100_000, 64, 64, 16), (0, 100_000, 64, 4, 16), (1, 100_000, 64, 32, 16), (0, 100_000, 64, 130, 16)]
    assert all(p["TN"] == 1 for p in ttm_plan(rows))
    assert ttm_plan([(0, 100_000, 64, 128, 16)])[0]["TN"] == 2


def test_mttkrp_of_little_work_keeps_the_vector_kernel(any_plan):
    """Few contracted indices, many short modes, ranks above 64; and not
    where a launch or two of the matrix kernels do more."""
    vector = [(0, (4, 2, 2, 2, 2, 7), 100, 3, 1), (0, (16, 50, 3), 65, 1, 1), (1, (2, 8, 9, 2), 100, 2, 1),
              (0, (6, 4), 100, 1, 1), (0, (8, 26, 15, 6), 17, 1, 1), (1, (13, 14, 13), 100, 1, 1)]
    matrix = [(0, (32, 12, 10, 30), 3, m, 0) for m in range(4)] + [(0, (257, 301, 203), 20, m, 0) for m in range(3)]
    matrix += [(0, (149, 120, 90), 10, m, 1) for m in range(3)] + [(0, (14, 27, 5, 5), 64, 2, 1), (1, (40, 50, 60), 70, 0, 1)]
    assert all(p["vector"] for p in any_plan(vector))
    assert not any(p["vector"] for p in any_plan(matrix))


def test_the_shapes_of_the_gpu_tests_reach_every_tile_count(any_plan, ttm_plan):
    from any_shape_cases import MODE_DOT, MTTKRP
    plans = any_plan([(f, s, R, m, w) for f, s, R, m, w, _ in MTTKRP])
    reached = set()
    for (f, s, R, m, w, TN), p in zip(MTTKRP, plans):
        assert p["ok"] and not p["vector"], (s, R, m)
        assert TN is None or p["TN"] == TN, (s, R, m, p["TN"])
        reached.add((f, p["last"], p["TN"]))
    assert {(f, 0, t) for f in (False, True) for t in (2, 3, 4)} <= reached
    assert {(f, 1, t) for f in (False, True) for t in (2, 3)} <= reached
    rows = []
    for f, s, m, J, _, _ in MODE_DOT:
        before, after = 1, 1
        for i, v in enumerate(s):
            before, after = (before * v if i < m else before), (after * v if i > m else after)
        rows.append((f, before, s[m], after, J))
    for (f, s, m, J, TN, split), p in zip(MODE_DOT, ttm_plan(rows)):
        assert p["ok"] and not p["vector"] and p["TN"] == TN and p["split"] == split, (s, m, J, p)
