"""The passes of a batched start (q3h_passes.h), compiled for the host."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
#include "q3h_passes.h"
extern "C" void passes(const int *rows, int n, int limit, int *pass_of, int *place) {
  const auto p = q3h::start_passes(rows, n, limit);
  for (int i = 0; i < (int)p.size(); i++)
    for (int j = 0; j < (int)p[i].size(); j++) pass_of[p[i][j]] = i, place[p[i][j]] = j;
}
"""


@pytest.fixture(scope="module")
def passes(tmp_path_factory):
    d = tmp_path_factory.mktemp("passes")
    src, lib = str(d / "passes.cpp"), str(d / "libpasses.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-I",
                    os.path.join(ROOT, "mormot2-qwen-tts_amd", "csrc"), src, "-o", lib], check=True)
    so = ctypes.CDLL(lib)

    def run(rows, limit):
        p = ctypes.POINTER(ctypes.c_int)
        a = [np.ascontiguousarray(v, np.int32) for v in (rows, np.full(len(rows), -1),
                                                         np.full(len(rows), -1))]
        so.passes(a[0].ctypes.data_as(p), len(rows), limit, a[1].ctypes.data_as(p),
                  a[2].ctypes.data_as(p))
        return a[1].tolist(), a[2].tolist()
    return run


@pytest.mark.parametrize("rows, expect", [
    ([], []),
    ([8192], [0]),
    ([5000, 4000, 100, 100, 100], [0, 1, 0, 0, 0]),      # one too long to join the first
    ([8192, 500, 500, 500], [0, 1, 1, 1]),               # one that fills a pass by itself
    ([8000, 500, 500, 192, 1], [0, 1, 1, 0, 1]),
    ([4096, 4096, 4096, 4096, 1], [0, 0, 1, 1, 2]),
])
def test_start_passes(passes, rows, expect):
    assert passes(rows, 8192)[0] == expect


def test_start_passes_random(passes):
    """Every prompt in one pass, in order, no pass over the limit, and no two
    passes of which all of the later one fitted the earlier."""
    rng = np.random.default_rng(1)
    for _ in range(200):
        rows = rng.integers(1, rng.choice([60, 300, 1000]) + 1, rng.integers(1, 40))
        of, place = passes(rows, 1000)
        assert min(of) == 0 and set(of) == set(range(max(of) + 1))
        for k in range(max(of) + 1):
            mine = [i for i in range(len(rows)) if of[i] == k]
            assert [place[i] for i in mine] == list(range(len(mine)))
            total = int(rows[mine].sum())
            assert total <= 1000
            later = [int(rows[i]) for i in range(len(rows)) if of[i] > k]
            assert all(total + r > 1000 for r in later)
