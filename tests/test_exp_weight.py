"""The bilateral filter's weight (exp_weight in kinectfusion_amd/csrc/
kf_exp.hpp), compiled from the same header for the host with g++: the float
that math.exp rounds to wherever that is normal, within one denormal step
below, and 0 far below and for a NaN."""
import ctypes as C
import math
import subprocess
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parents[1]
SRC = r"""
#include "kf_exp.hpp"
static const double kTable[64] = KF_EXP2_J64_TABLE;
extern "C" void weights(const float* x, float* y, long n) {
  for (long i = 0; i < n; ++i) y[i] = kf::exp_weight(x[i], kTable);
}
"""


@pytest.fixture(scope="module")
def weights(tmp_path_factory):
    d = tmp_path_factory.mktemp("weight")
    (d / "w.cpp").write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC",
                    f"-I{ROOT / 'kinectfusion_amd' / 'csrc'}", str(d / "w.cpp"), "-o", str(d / "libw.so")], check=True)
    so = C.CDLL(str(d / "libw.so"))

    def run(x):
        x = np.ascontiguousarray(x, np.float32)
        y = np.empty_like(x)
        so.weights(x.ctypes.data_as(C.c_void_p), y.ctypes.data_as(C.c_void_p), C.c_long(x.size))
        return x, y

    return run


@pytest.mark.parametrize("kind", ["filter", "uniform", "tiny", "steps"])
def test_weight_is_the_rounded_exponential(weights, kind):
    rng = np.random.default_rng(7)
    n = 200_000
    if kind == "filter":
        x = -rng.exponential(2.0, n)
    elif kind == "uniform":
        x = -rng.uniform(0.0, 87.3, n)
    elif kind == "tiny":
        x = -rng.uniform(0.0, 1.0, n) * 10.0 ** -rng.uniform(0, 40, n)
    else:  # around the halves and wholes of ln2/64, where the reduction changes step
        x = -(rng.integers(0, 16000, n) * 0.5 * math.log(2.0) / 64 * (1 + rng.uniform(-1, 1, n) * 1e-6))
        x = x[x > -87.3]
    x, y = weights(x)
    ref = np.array([math.exp(float(v)) for v in x]).astype(np.float32)
    assert np.array_equal(y, ref)


def test_far_below(weights):
    x, y = weights(-np.concatenate([np.linspace(87.4, 110, 5000), [200.0, 1e6, 1e30, np.inf]]))
    ref = np.array([math.exp(float(v)) for v in x])
    assert np.abs(y.astype(np.float64) - ref).max() <= 2.0 ** -149
    assert np.all(y[x < -104] == 0)
    assert weights([np.nan])[1][0] == 0 and weights([0.0, -0.0])[1].tolist() == [1.0, 1.0]
