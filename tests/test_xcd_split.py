"""CPU test: the split of a launch's units over the eight XCDs (csrc/cq_split.h).

Every unit belongs to one XCD, in order, and no XCD has more than its eighth of
the work by more than one unit at each end and what the 64ths leave open (for
several products, two 64ths of the largest). A split by counts fails the second
for the skewed works here: few heavy units among many light ones, triangles (as
in symmetric-result plans), units without work.
"""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "conquest-release_amd", "csrc")


@pytest.fixture(scope="module")
def split(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    exe = tmp_path_factory.mktemp("xcd") / "split"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", CSRC, os.path.join(ROOT, "tests", "xcd_split_driver.cpp"),
                    "-o", str(exe)], check=True, timeout=120)

    def run(works, at_once=0, brief=0):
        lines = [f"{len(works)} {at_once} {brief}"]
        for w in works:
            before = np.concatenate(([0], np.cumsum(w)))
            at = [int(np.searchsorted(before, before[-1] / 64 * k)) for k in range(64)] + [len(w)]
            lines.append(f"{before[-1]} " + " ".join(map(str, at)))
        out = subprocess.run([str(exe)], input="\n".join(lines), capture_output=True, text=True, check=True,
                             timeout=60).stdout
        return np.array(out.split(), np.int64)

    return run


def _works(kind, n, rng):
    if kind == "equal":
        return np.full(n, 7)
    if kind == "triangle":
        return np.arange(n) * 3
    if kind == "heavy":
        return np.where(rng.random(n) < 0.02, 4000, 1 + rng.integers(0, 5, n))
    return np.where(rng.random(n) < 0.5, 0, rng.integers(0, 100, n))


@pytest.mark.parametrize("kind", ["equal", "triangle", "heavy", "empty"])
@pytest.mark.parametrize("sizes", [(1,), (2,), (7,), (9,), (300,), (100003,), (5, 3000, 40), (1,) * 16,
                                   tuple(50 * k + 1 for k in range(16))])
def test_every_xcd_has_its_eighth_of_the_work(split, kind, sizes):
    rng = np.random.default_rng(len(sizes) * 1000 + sizes[-1])
    works = [_works(kind, n, rng).astype(np.int64) for n in sizes]
    xcd = split(works)
    unit = np.concatenate(works)
    assert xcd[0] == 0 and xcd[-1] == len(unit) and (np.diff(xcd) >= 0).all()
    before = np.concatenate(([0], np.cumsum(unit)))
    have = np.diff(before[xcd])
    slack = 2 * unit.max() + (0 if len(works) == 1 else 2 * max(w.sum() for w in works) / 64)
    assert have.max() <= before[-1] / 8 + slack + 1, (have, before[-1] / 8)


@pytest.mark.parametrize("sizes", [(1,), (7,), (300,), (5, 3000, 40)])
def test_brief_units_that_run_at_once_are_split_by_count(split, sizes):
    works = [_works("heavy", n, np.random.default_rng(n)).astype(np.int64) for n in sizes]
    total = sum(sizes)
    each, mean = -(-total // 8), -(-sum(int(w.sum()) for w in works) // total)
    by_count = np.minimum(np.arange(9) * each, total)
    np.testing.assert_array_equal(split(works, total, mean), by_count)
    by_work = split(works)
    np.testing.assert_array_equal(split(works, total - 1, mean), by_work)
    np.testing.assert_array_equal(split(works, total, mean - 1), by_work)


def test_no_work_at_all(split):
    xcd = split([np.zeros(20, np.int64), np.zeros(3, np.int64)])
    assert xcd[0] == 0 and xcd[-1] == 23 and (np.diff(xcd) >= 0).all()
