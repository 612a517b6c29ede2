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
extern "C" float noise(int d, int long_rows) {
  const kmhip::Rounding r = kmhip::bound_noise<float>(d, long_rows != 0);
  return r.products + r.norms;
}
extern "C" float limit(float best, float second, float xx, int d, int long_rows, float share) {
  kmhip::Rounding r = kmhip::bound_noise<float>(d, long_rows != 0);
  r.products *= share;
  r.norms *= share;
  return kmhip::row_limit(best, second, xx, 0.0f, r, 0.0f);
}
extern "C" float square(const float *x, int d) { return norm(x, d); }
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
    for name in ("noise", "chain", "lanes", "limit", "square"):
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


def labels_that_change(model, form, d, share):
    """How many rows with a limit change sides although the two centroids have not used it up: one moves away from the
    row or towards it, the other towards the row. Rows and centroids of equal features, on which roundings add up, and
    of any, far from the origin and near, near their centroid and not, the centroids at all but the same distance."""
    f, rng, changed, limits = getattr(model, form), np.random.default_rng(d), 0, 0
    for trial in range(3000):
        away = 10.0 ** rng.uniform(-3, 0.5)
        if trial % 3:
            x = np.full(d, rng.uniform(1, 2))
            side, other = np.full(d, 1.0), np.full(d, -1.0)
        else:
            x = rng.standard_normal(d) + rng.uniform(0, 3)
            side, other = rng.standard_normal((2, d))
        x = x.astype(np.float32)
        x64 = x.astype(np.float64)
        scale = away * np.sqrt((x64 ** 2).mean() * d)
        side, other = (v / np.sqrt((v ** 2).sum()) * scale for v in (side, other))
        more = 1 + 10.0 ** rng.uniform(-5, 0)
        a, b = (x64 + side).astype(np.float32), (x64 + other * more).astype(np.float32)
        best, second = f(ptr(x), ptr(a), d), f(ptr(x), ptr(b), d)
        if best > second:
            a, b, side, other, best, second = b, a, other, side, second, best
        lim = model.limit(ctypes.c_float(best), ctypes.c_float(second), ctypes.c_float(model.square(ptr(x), d)), d,
                          form == "lanes", ctypes.c_float(share))
        if not lim > 0:
            continue
        limits += 1
        for part in (0.0, 0.3, 1.0, -0.3, -1.0):  # of the limit, the row's own centroid
            to = side / np.sqrt((side ** 2).sum()) * lim * 0.9999
            fro = other / np.sqrt((other ** 2).sum()) * lim * 0.9999
            a2 = (a + part * to).astype(np.float32)
            b2 = (b - (1 - abs(part)) * fro).astype(np.float32)
            used = sum(np.sqrt(((p.astype(np.float64) - q) ** 2).sum()) for p, q in ((a, a2), (b, b2)))
            if used <= lim:
                changed += not f(ptr(x), ptr(a2), d) < f(ptr(x), ptr(b2), d)
    assert limits > 300
    return changed


@pytest.mark.parametrize("form,d", [("chain", d) for d in (5, 61, 298, 1024)] + [("lanes", d) for d in (68, 300, 784)])
def test_rows_within_their_limit_keep_their_label(model, form, d):
    assert labels_that_change(model, form, d, 1.0) == 0
    if d >= 298:  # (and the rows above are such that it matters)
        assert labels_that_change(model, form, d, 0.03) > 0
