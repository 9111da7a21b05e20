"""The bilateral filter's weight (exp_weight in kinectfusion_amd/csrc/
kf_exp.hpp), compiled from the same header for the host with g++, where its
float is denormal or 0: every float argument there gives the FP64 exponential
rounded once."""
import ctypes as C
import subprocess
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parents[1]
SRC = r"""
#include "kf_exp.hpp"
static const double kTable[64] = KF_EXP2_J64_TABLE;
extern "C" void weights(const float* x, float* y, long n) {
  for (long i = 0; i < n; ++i) y[i] = kf::exp_weight(x[i], kTable);
}
"""


def test_denormal_weights_are_rounded_once(tmp_path):
    (tmp_path / "w.cpp").write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC",
                    f"-I{ROOT / 'kinectfusion_amd' / 'csrc'}", str(tmp_path / "w.cpp"), "-o",
                    str(tmp_path / "libw.so")], check=True)
    so = C.CDLL(str(tmp_path / "libw.so"))
    first, last = (int(np.float32(v).view(np.uint32)) for v in (-87.0, -105.0))
    x = np.arange(first, last + 1, dtype=np.uint32).view(np.float32)  # every float from -87 down to -105
    y = np.empty_like(x)
    so.weights(x.ctypes.data_as(C.c_void_p), y.ctypes.data_as(C.c_void_p), C.c_long(x.size))
    with np.errstate(under="ignore"):
        ref = np.exp(x.astype(np.float64)).astype(np.float32)
    assert (ref == 0).any() and ((ref > 0) & (ref < 2.0 ** -126)).any()
    assert np.array_equal(y, ref)
