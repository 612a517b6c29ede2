"""Fits that measure only the rows whose label may have changed: labels, centroids, counts and minimum
distances are those of fits that measure every row in every step, after any number of steps, in each
kernel that has the form, whatever the data."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (rows, features, centroids): one and several blocks of centroids, rows of whole stages and 16-byte vectors
# and not, fewer rows than a workgroup takes, a last stretch of rows that is not whole
TILED = [("float32", 20003, 70, 260), ("float32", 9001, 101, 300), ("float32", 30000, 132, 130), ("float32", 12345, 298, 90),
         ("float32", 5000, 160, 257), ("float32", 300, 67, 230), ("float32", 20000, 780, 66), ("float64", 20003, 80, 700),
         ("float64", 9001, 101, 130), ("float64", 12345, 96, 300), ("float64", 300, 75, 70)]

# lists long enough for the centroids' neighbours to be asked in later steps too: models staged in LDS and not,
# rows of whole 16-byte vectors and not, each number of lanes and pieces a row is dealt to
TILED += [("float32", 100003, 68, 260), ("float32", 70001, 101, 300), ("float32", 70001, 130, 300), ("float32", 70001, 298, 100),
          ("float32", 70001, 260, 100), ("float32", 36001, 601, 66), ("float64", 70001, 70, 300), ("float64", 70001, 33, 900),
          ("float64", 70001, 129, 100), ("float64", 40001, 300, 70), ("float64", 36001, 601, 66)]

# rows of whole 16-byte vectors and not, a model of one and several tiles, two wavefronts' layouts (d > 32),
# the smallest k, sums with and without copies, less than a tile of rows
FUSED = [("float32", 20003, 16, 140), ("float32", 30001, 32, 256), ("float32", 9001, 13, 300), ("float32", 12345, 30, 70),
         ("float32", 5000, 64, 100), ("float32", 5003, 61, 65), ("float32", 140000, 9, 66), ("float32", 140, 40, 100)]

# rows of one to four vectors a lane, each number of sums a launch is made for, less than a workgroup's rows
FUSED += [("float32", 20003, 784, 10), ("float32", 9001, 68, 3), ("float32", 5003, 132, 16), ("float32", 12345, 516, 8),
          ("float32", 6001, 772, 2), ("float32", 40, 200, 5)]

# rows ordered in space: one and several windows and workgroups' worth of blocks, a last block and window
# that are not whole, less than a block, models whose blocks are measured against all and against a few
CELLS = [("float32", 300007, 3, 27), ("float32", 70001, 3, 40), ("float32", 20000, 3, 100), ("float32", 4096, 3, 17),
         ("float32", 60, 3, 20), ("float32", 100100, 3, 128)]


def blobs(n, d, k, dtype, seed=0, offset=0.0):
    rng = np.random.default_rng(1000 * seed + n + 7 * d + k)
    centers = rng.uniform(-10, 10, size=(k, d))
    X = centers[rng.integers(0, k, size=n)] + 2 * rng.standard_normal((n, d)) + offset
    if dtype == "float32":  # (sums of such values are exact, in whatever order they are made)
        X = np.round(X * 1024) / 1024
    return X.astype(dtype), X[rng.permutation(n)[:k]].astype(dtype)


def fit(hip, X, C, steps, bounds, tol=0.0):
    with hip.Handle(X.shape[0], X.shape[1], C.shape[0], X.dtype) as h:
        h.set_data(X)
        h.set_option("bounds", bounds)
        h.set_centroids(C)
        it = h.fit(steps, tol)
        return dict(it=it, labels=h.labels(), centers=h.centroids(), mind=h.min_distances(), counts=h.counts(),
                    inertia=h.inertia(), measured=h.rows_measured())


def same(got, want, X, exact=True):
    """Minimum distances: where only some rows were measured they are made from the differences, where all were
    from norms and products, which are off by at most (8 + 2 sqrt(d)) eps (xx + cc) in float32 (a centroid's cc
    is at most 2 xx + 2 dist) and have 4 bits less where they are compared as keys.
    exact False: float64 sums made in LDS, in the order their rows arrive: a sum of m rows is off by up to
    m eps of its terms, a mean by m eps of the largest value (m < 1000 here), and a distance, of norms of
    that size, by as much of the largest norm."""
    assert got["it"] == want["it"]
    assert np.array_equal(got["labels"], want["labels"])
    assert np.array_equal(got["counts"], want["counts"])
    if exact:
        assert np.array_equal(got["centers"], want["centers"], equal_nan=True)
        d, xx = X.shape[1], (X.astype(np.float64) ** 2).sum(1)
        g, w = got["mind"].astype(np.float64), want["mind"].astype(np.float64)
        fine = np.isfinite(xx) & (w < 3e38)
        tol = (8 + 2 * np.sqrt(d)) * 2.0 ** -23 * (3 * xx + 2 * w) + 2e-6 * w + 1e-36
        assert (np.abs(g - w)[fine] <= tol[fine]).all()
        assert not (g[~fine] < 3e38).any()
        return
    finite = np.isfinite(want["centers"]).all(1)
    big = np.abs(want["centers"][finite]).max()
    eps = 1000 * np.finfo(np.float64).eps
    assert np.allclose(got["centers"], want["centers"], rtol=0, atol=eps * big, equal_nan=True)
    d = want["centers"].shape[1]
    assert np.allclose(got["mind"], want["mind"], rtol=0, atol=4 * d * eps * big ** 2, equal_nan=True)


@pytest.mark.parametrize("dtype,n,d,k", TILED + FUSED + CELLS)
def test_fits_of_any_length(hip, dtype, n, d, k):
    X, C = blobs(n, d, k, dtype)
    few = n
    for steps in (3, 4, 5, 6, 8, 11, 20, 40):
        got, want = fit(hip, X, C, steps, 2), fit(hip, X, C, steps, 0)
        assert want["measured"] == -1 and got["measured"] >= 0
        same(got, want, X, dtype == "float32")
        few = min(few, got["measured"])
    assert few < n / 2 or k < 8 or d < 8  # rows were left alone (a few centroids may share one cluster throughout)


@pytest.mark.parametrize("dtype,n,d,k", TILED + FUSED + CELLS)
def test_fits_that_converge(hip, dtype, n, d, k):
    X, C = blobs(n, d, k, dtype, seed=1)
    got, want = fit(hip, X, C, 300, 2, tol=1e-8), fit(hip, X, C, 300, 0, tol=1e-8)
    assert got["it"] > 3 or n < 1000 or k <= 16
    same(got, want, X, dtype == "float32")
    got, want = fit(hip, X, C, 5, 2, tol=1e-8), fit(hip, X, C, 5, 0, tol=1e-8)  # (the limit ends it)
    same(got, want, X, dtype == "float32")


@pytest.mark.parametrize("dtype,n,d,k", TILED + FUSED + CELLS)
@pytest.mark.parametrize("what", ["noise", "far", "twins", "not finite", "small", "large", "empty", "tiny"])
def test_whatever_the_data(hip, dtype, n, d, k, what):
    X, C = blobs(n, d, k, dtype, seed=2, offset=3000.0 if what == "far" else 0.0)
    rng = np.random.default_rng(5)
    if what == "noise":
        X = (np.round(rng.standard_normal(X.shape) * 1024) / 1024).astype(dtype)
        C = X[:k].copy()
    elif what == "twins":  # equal centroids, and ones a hair apart
        C[1::3] = C[0::3][:len(C[1::3])]
        C[2::3] = (C[0::3][:len(C[2::3])] * (1 + 1e-6)).astype(dtype)
        X[::2] = X[0]
    elif what == "not finite":
        X[5, 2], X[17, 0], X[n - 1, d - 1] = np.nan, np.inf, -np.inf
    elif what == "small":
        X, C = (X * 2.0 ** -50).astype(dtype), (C * 2.0 ** -50).astype(dtype)
    elif what == "tiny" and dtype == "float64":  # moves that no float holds
        X, C = X * 2.0 ** -200, C * 2.0 ** -200
    elif what == "large":
        X, C = (X * 2.0 ** 53).astype(dtype), (C * 2.0 ** 53).astype(dtype)
    elif what == "empty":  # centroids that never get a row, one of them at infinity
        C[k // 2:] += 1e5
        C[-1] = np.inf
    for steps in (4, 9):
        same(fit(hip, X, C, steps, 2), fit(hip, X, C, steps, 0), X, dtype == "float32")


def test_short_fits_and_asked_for_kernels_measure_every_row(hip):
    X, C = blobs(20000, 132, 130, "float32")
    assert fit(hip, X, C, 7, 1)["measured"] == -1 and fit(hip, X, C, 20, 1)["measured"] == -1  # (too little to do)
    for name, value in (("assign", 3), ("exact_argmin", 1), ("fp32_split", 6)):
        with hip.Handle(20000, 132, 130, np.float32) as h:
            h.set_data(X)
            h.set_option("bounds", 2)
            h.set_option(name, value)
            h.set_centroids(C)
            h.fit(10, 0.0)
            assert h.rows_measured() == -1


@pytest.mark.parametrize("d,k", [(96, 256), (24, 80)])
def test_limits_are_the_triangle_inequalitys(hip, d, k):
    """Rows on a line between two centroids that drift: a row is measured again before it can change sides."""
    n = 4096
    rng = np.random.default_rng(3)
    C = np.zeros((k, d))
    C[:, 0] = np.arange(k) * 10.0
    X = np.zeros((n, d))
    X[:, 0] = np.round(rng.uniform(0, 10.0 * k, size=n) ** 1.01 * 64) / 64
    X, C = X.astype(np.float32), C.astype(np.float32)
    for steps in (3, 6, 12, 50, 200):
        same(fit(hip, X, C, steps, 2), fit(hip, X, C, steps, 0), X)
