"""The logits launch's work-groups (logits_plan.h, compiled here for the host):
every (key split, query group) pair is dealt once, each XCD gets as many as the
others, and so it is for any run of splits and groups - what a causal bound, a
call over a part of its keys or windows leave of them."""

import ctypes
import shutil
import subprocess

import numpy as np
import pytest

from cxldsagr_amd.csrc import build

SOURCE = """
#include "logits_plan.h"
extern "C" void plan(int64_t rows, int64_t ldo, int64_t cus, int64_t* out) {
  const auto p = dsa::split_plan(rows, ldo, 16, 128, 0, cus);
  out[0] = p.qgroups; out[1] = p.splits; out[2] = p.per; out[3] = p.live; out[4] = p.grid();
}
extern "C" void deal(uint32_t grid, uint32_t qgroups, uint32_t live, uint32_t* out) {
  for (uint32_t id = 0; id < grid; ++id) {
    const auto p = dsa::dealt_pair(id, qgroups, live);
    out[2 * id] = p.split; out[2 * id + 1] = p.group;
  }
}
"""


@pytest.fixture(scope="module")
def plan_library(tmp_path_factory):
    compiler = shutil.which("g++")
    if compiler is None:
        pytest.skip("needs g++")
    path = tmp_path_factory.mktemp("plan")
    (path / "plan.cpp").write_text(SOURCE)
    subprocess.run([compiler, "-O1", "-std=c++17", "-shared", "-fPIC", f"-I{build.HERE}",
                    str(path / "plan.cpp"), "-o", str(path / "plan.so")], check=True)
    return ctypes.CDLL(str(path / "plan.so"))


SHAPES = [(1, 256), (1, 65792), (16, 50176), (17, 131584), (40, 20224), (100, 50176), (129, 4352),
          (340, 9216), (700, 100096), (1000, 2048), (2048, 2048), (2048, 65792), (4100, 4352),
          (8192, 8192), (6000, 12032)]


@pytest.mark.parametrize("rows,ldo", SHAPES)
def test_pairs_are_dealt_once_and_evenly(plan_library, rows, ldo):
    out = (ctypes.c_int64 * 5)()
    plan_library.plan(ctypes.c_int64(rows), ctypes.c_int64(ldo), ctypes.c_int64(256), out)
    qgroups, splits, per, live, grid = out
    assert qgroups == (rows + 15) // 16 and (live - 1) * per < ldo <= live * per
    assert splits == (live if live < 8 else (live + 7) // 8 * 8) and grid % 8 == 0
    ids = np.zeros((grid, 2), dtype=np.uint32)
    plan_library.deal(ctypes.c_uint32(grid), ctypes.c_uint32(qgroups), ctypes.c_uint32(live),
                      ids.ctypes.data_as(ctypes.c_void_p))
    xcd = np.arange(grid) % 8
    used = ids[:, 0] < live
    assert grid - used.sum() < 8  # at most one idle slot an XCD
    # (XCD, split, group): each pair on exactly one XCD.
    on = np.zeros((8, live, qgroups), dtype=np.int64)
    np.add.at(on, (xcd[used], ids[used, 0], ids[used, 1]), 1)
    assert (on.sum(0) == 1).all()
    # Runs of splits and of groups: the XCDs' shares differ by one split's at most.
    rng = np.random.default_rng(rows)
    sums = on.cumsum(1).cumsum(2)
    sums = np.pad(sums, ((0, 0), (1, 0), (1, 0)))
    for _ in range(200):
        a, b = sorted(rng.integers(0, live + 1, 2))
        c, d = sorted(rng.integers(0, qgroups + 1, 2))
        share = sums[:, b, d] - sums[:, a, d] - sums[:, b, c] + sums[:, a, c]
        # (The last live % 8 splits go round by pairs: up to one pair each.)
        bound = (d - c if live >= 8 else 0) + 1 + live % 8
        assert share.max() - share.min() <= bound, (a, b, c, d, share)
    # The causal triangle, in keys seen: within one split's share of the mean.
    first = ldo - rows
    ends = np.minimum(first + 16 * np.arange(1, qgroups + 1), ldo)
    seen = np.clip(ends[None, :] - per * np.arange(live)[:, None], 0, per)
    work = (on * seen).sum((1, 2))
    assert work.max() <= 1.1 * work.mean() + per * (qgroups if live >= 8 else 1), work


@pytest.mark.parametrize("cus", [256, 304, 7])
def test_the_plan_is_the_cheapest_of_all_split_counts(plan_library, cus):
    """Each split length is looked at once; the result is that of every count in
    turn, the first of those that cost the same."""
    rng = np.random.default_rng(cus)
    ldos = np.concatenate([256 * np.arange(1, 40), 256 * rng.integers(40, 4200, 60)])
    out = (ctypes.c_int64 * 5)()
    for ldo in ldos.tolist():
        rows = int(rng.choice([1, 16, 17, 100, 128, 700, 2048, 9000]))
        stages, qgroups = (ldo + 127) // 128, (rows + 15) // 16
        s = np.arange(1, min(stages, cus) + 1)
        per = -(-stages // s)
        rounds = -(-(-(-stages // per) * qgroups) // cus)
        best = per[np.argmin(rounds * (8.0 + 3.0 * per))] * 128
        plan_library.plan(ctypes.c_int64(rows), ctypes.c_int64(ldo), ctypes.c_int64(cus), out)
        assert out[2] == best, (rows, ldo)
