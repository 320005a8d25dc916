"""Scalar math of the kernels (q3h_math.h), compiled for the host: the same
sources and operations, run on the CPU."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"

SOURCE = """
#include "q3h_math.h"
extern "C" void sin_squared_rows(const float *x, int n, float *y) {
  for (int i = 0; i < n; i++) y[i] = q3h::sin_squared(x[i]);
}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("math")
    src, lib = str(d / "math.hip"), str(d / "libmath.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-fPIC", "-shared", "--offload-host-only", "-I",
                    os.path.join(ROOT, "mormot2-qwen-tts_amd", "csrc"), src, "-o", lib],
                   check=True)
    return ctypes.CDLL(lib)


def _sin_squared(host, x):
    x = np.ascontiguousarray(x, np.float32)
    y = np.empty_like(x)
    p = ctypes.POINTER(ctypes.c_float)
    host.sin_squared_rows(x.ctypes.data_as(p), x.size, y.ctypes.data_as(p))
    return y


def _arguments(name):
    rng = np.random.default_rng(2)
    if name == "multiples_of_pi":  # the floats around k pi, where the reduction cancels
        c = (np.arange(1, 127400) * np.pi).astype(np.float32)
        return np.concatenate([c, np.nextafter(c, np.float32(0)), np.nextafter(c, np.float32(1e9))])
    if name == "switch":  # both sides of the change to sinf
        c = np.float32(4e5)
        x = c + np.arange(-2000, 2000, dtype=np.float32) * np.float32(0.03125)
        return np.concatenate([x, rng.uniform(4e5, 1e8, 20000)])
    lo, hi = {"small": (1e-30, 1.0), "ordinary": (1.0, 100.0), "large": (100.0, 4e5)}[name]
    return np.exp(rng.uniform(np.log(lo), np.log(hi), 200000))


@pytest.mark.parametrize("name", ["small", "ordinary", "large", "multiples_of_pi", "switch"])
def test_sin_squared(host, name):
    """Against float64. The reduced argument is rounded twice and the series' last
    step once, so sin x is within 3 units of 2^-24 of itself and its square,
    rounded once more, within 7."""
    x = np.asarray(_arguments(name), np.float32)
    x = np.concatenate([x, -x])
    ref = np.sin(x.astype(np.float64)) ** 2
    y = _sin_squared(host, x).astype(np.float64)
    normal = ref > 2.0 ** -126
    err = np.abs(y - ref)[normal] / ref[normal]
    print(f"{name}: {err.max() * 2 ** 24:.2f} units of 2^-24 at {x[normal][err.argmax()]!r}")
    assert err.max() <= 7 * 2.0 ** -24


def test_sin_squared_not_finite(host):
    y = _sin_squared(host, [np.inf, -np.inf, np.nan, 0.0, 1e-45])
    assert np.isnan(y[:3]).all() and (y[3:] == 0).all()
