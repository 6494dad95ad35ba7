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
    std::printf("%d %d %d %lld %d %lld %lld\n", ok, p.JT, p.TN, (long long)p.tiles, p.split, (long long)p.gx, (long long)p.gy);
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
    keys = ("ok", "JT", "TN", "tiles", "split", "gx", "gy")
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
