"""The figures of csrc/row_bounds.h on the CPU: what the rounding of a squared distance can come to, in the orders the
kernels add in."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "h2o4gpu_amd", "csrc")

SOURCE = r"""
#include "row_bounds.h"
#include <algorithm>
static float norm(const float *x, int d) {
  float s = 0;
  for (int j = 0; j < d; j++) { volatile float p = x[j] * x[j]; s = s + p; }
  return s;
}
extern "C" float noise(int d, int long_rows) { return kmhip::bound_noise<float>(d, long_rows != 0); }
// the float32 instructions: half a distance, one multiply-add per feature
extern "C" float chain(const float *x, const float *c, int d) {
  float a = fmaf(-0.5f, norm(c, d), -0.5f * norm(x, d));
  for (int j = 0; j < d; j++) a = fmaf(x[j], c[j], a);
  return 2 * fabsf(a);
}
// the long-row kernel: a lane's features, four at a time, then six exchanges
extern "C" float lanes(const float *x, const float *c, int d) {
  float v[64] = {};
  for (int j = 0; j < d; j++) v[j / 4 % 64] = fmaf(x[j], c[j], v[j / 4 % 64]);
  for (int m = 32; m; m /= 2)
    for (int l = 0; l < m; l++) v[l] = v[l] + v[l + m];
  return fabsf(norm(x, d) + norm(c, d) - 2 * v[0]);
}
"""


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    where = tmp_path_factory.mktemp("row_bounds")
    src, so = where / "model.cpp", where / "model.so"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-w", "-I" + CSRC,
                           "-I/opt/rocm/include", "-o", str(so), str(src)])
    lib = ctypes.CDLL(str(so))
    for name in ("noise", "chain", "lanes"):
        getattr(lib, name).restype = ctypes.c_float
    return lib


def ptr(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_float))


@pytest.mark.parametrize("form,d", [("chain", d) for d in (5, 16, 61, 64, 101, 298, 784, 1024, 3000, 8000)] +
                         [("lanes", d) for d in (68, 132, 300, 784, 1024)])
def test_noise_covers_the_rounding(model, form, d):
    """Random features, and equal ones, whose roundings all go the same way."""
    rng = np.random.default_rng(d)
    bound, worst = model.noise(d, form == "lanes"), 0.0
    for trial in range(2000):
        if trial % 2:
            x, c = rng.uniform(1, 4, 2).astype(np.float32)[:, None] * np.ones((2, d), np.float32)
        else:
            x, c = rng.standard_normal((2, d)).astype(np.float32) + np.float32(trial % 3)
        x, c = np.ascontiguousarray(x), np.ascontiguousarray(c)
        x64, c64 = x.astype(np.float64), c.astype(np.float64)
        want = ((x64 - c64) ** 2).sum()
        off = abs(getattr(model, form)(ptr(x), ptr(c), d) - want) / ((x64 ** 2).sum() + (c64 ** 2).sum())
        worst = max(worst, off)
    assert worst <= bound, (worst * 2 ** 23, bound * 2 ** 23)
    assert worst > bound / 50  # (what equal features show)
