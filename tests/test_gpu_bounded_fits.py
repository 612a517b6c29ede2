"""Fits that measure only the rows whose label may have changed, where their parts meet: rows that no pass
has given a limit, steps that go without limits and begin anew, sums carried from step to step, handles that
are used again, the rule that makes fits bounded by themselves, and what they need memory for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(h, X, C, steps, bounds=None, tol=0.0):
    if bounds is not None:
        h.set_option("bounds", bounds)
    h.set_centroids(C)
    it = h.fit(steps, tol)
    return dict(it=it, labels=h.labels(), centers=h.centroids(), mind=h.min_distances(), counts=h.counts(),
                measured=h.rows_measured())


def fit(hip, X, C, steps, bounds=None, tol=0.0):
    with hip.Handle(X.shape[0], X.shape[1], C.shape[0], X.dtype) as h:
        h.set_data(X)
        return run(h, X, C, steps, bounds, tol)


def same(got, want, exact=True):
    """exact False: float64 sums made in LDS, in the order their rows arrive (off by up to the rows' number in
    eps of the largest value)."""
    assert got["it"] == want["it"]
    assert np.array_equal(got["labels"], want["labels"])
    assert np.array_equal(got["counts"], want["counts"])
    if exact:
        assert np.array_equal(got["centers"], want["centers"], equal_nan=True)
    else:
        big = np.abs(want["centers"]).max()
        assert np.allclose(got["centers"], want["centers"], rtol=0, atol=1000 * np.finfo(np.float64).eps * big)


def border_after_two_steps(q, tied, z):
    """Between two centroids of the rows z and of so many rows at q."""
    z, w = np.concatenate([[q], z]), np.concatenate([[tied], np.ones(len(z))])
    c = np.array([0.0, 0.02])
    for _ in range(2):
        right = z > c.mean()
        c = np.array([np.average(z[~right], weights=w[~right]), np.average(z[right], weights=w[right])])
    return c.mean()


def test_near_ties_that_fill_their_list_once(hip):
    """The first step that leaves limits finds more near ties than their list holds (a seventh of the rows, on the
    border of two centroids that moves on), so that the pass ends early and another one labels the rows. The rows it
    had not come to have no limit from it, and must not be held to what the memory says: here the limits of
    a fit before, with centroids so far apart that they are good for the whole fit."""
    n, d, k, tied, line = 200003, 68, 3200, 30000, 60000
    rng = np.random.default_rng(0)
    z_line, z_rest = rng.uniform(0, 1, line), rng.uniform(3, 4, n - tied - line)
    q, width = 0.4, 0.2  # the place that is the border after two steps, if the tied rows are there
    for _ in range(3):
        places = np.linspace(q - width, q + width, 201)
        off = [abs(border_after_two_steps(p, tied, z_line) - p) for p in places]
        q, width = places[int(np.argmin(off))], width / 50
    assert min(off) < 1e-5  # (rows within some 1e-4 of the border are near ties)
    X = np.full((n, d), 0.5, np.float32)
    X[:, 0] = np.concatenate([np.full(tied, q), z_line, z_rest])
    C = np.full((k, d), 0.5, np.float32)
    C[:, 0] = np.concatenate([[0.0, 0.02], 3 + np.linspace(0, 0.02, 40), 1000 + np.arange(k - 42)])
    far = C.copy()
    far[:42, 0] = 2000 + np.arange(42) * 10
    far[0, 0], far[2, 0] = 0.3, 3.5
    with hip.Handle(n, d, k, np.float32) as h:
        h.set_data(X)
        assert run(h, X, far, 6, 2)["measured"] < n
        got = run(h, X, C, 12, 2)
    want = fit(hip, X, C, 12, 0)
    assert np.array_equal(got["labels"], want["labels"])
    same(got, want)


def strips(n, d, k, dtype, seed):
    """Rows along lines of eight centroids each, the lines far apart, whose centroids go on moving a little for many
    steps; sums of such values are exact."""
    rng = np.random.default_rng(seed)
    at = rng.integers(0, k, n)
    X = np.round(rng.standard_normal((n, d)) * 64) / 1024
    C = np.zeros((k, d))
    X[:, 0] = np.round((8 * (at % 8) + rng.uniform(0, 8, n)) * 4096) / 4096
    C[:, 0] = 8.0 * (np.arange(k) % 8) + rng.uniform(3, 5, k)
    for A, c in ((X, at), (C, np.arange(k))):
        line = c // 8 - 1
        A[np.arange(len(A))[line >= 0], 1 + line[line >= 0] % (d - 1)] += 40.0 * (1 + line[line >= 0] // (d - 1))
    return X.astype(dtype), C.astype(dtype)


# each form of the long-row kernel (sums of 4, 8 and 16 centroids, one to four vectors a lane), the row-stationary
# one, tiled ones with and without the centroids' neighbours
ALONE = [("float32", 20003, d, k) for d, k in ((68, 2), (68, 3), (784, 4), (132, 5), (516, 8), (132, 8), (784, 10), (260, 16))]
ALONE += [("float32", 30001, 32, 80), ("float32", 70001, 13, 300), ("float32", 70001, 132, 130), ("float32", 70001, 101, 300),
          ("float64", 20003, 80, 130), ("float64", 40001, 101, 130)]


@pytest.mark.parametrize("dtype,n,d,k", ALONE)
def test_rows_are_left_alone_while_centroids_move(hip, dtype, n, d, k):
    X, C = strips(n, d, k, dtype, 3)
    fits = [fit(hip, X, C, s, 2) for s in range(4, 25)]
    moving = [i for i in range(20) if not np.array_equal(fits[i]["centers"], fits[i + 1]["centers"])]
    assert any(0 < fits[i]["measured"] < n / 2 for i in moving), [fits[i]["measured"] for i in moving]
    for i in (0, 3, 8, 15):
        same(fits[i], fit(hip, X, C, 4 + i, 0), dtype == "float32")


def free_bytes():
    from h2o4gpu_amd.libs import ch2o4gpu_gpu as shim
    free = np.zeros(16, np.uint64)
    status, n = shim.get_gpu_info_c(0, 0, 0, 0, 1, 0, 0, 0, 0, None, None, free, None, None, None,
                                    None, None, None, None, None, None)
    assert status == 0 and n >= 1 and free[0] > 0
    return int(free[0])


def test_a_fit_that_has_no_memory_to_spare_measures_every_row(hip, capfd):
    """Twelve bytes a row and the centroids' distances (116 MB here) are only taken from what the steps themselves
    leave: with some 60 MB more free than those need, the fit is made without limits, and has nothing to report."""
    n, d, k = 4000000, 66, 4096
    X = np.random.default_rng(1).standard_normal((n, d), dtype=np.float32)
    for _ in range(2):  # what a fit of each kind takes beside the handle (the second time, when all kernels are loaded)
        with hip.Handle(n, d, k, np.float32) as h:
            h.set_data(X)
            before = free_bytes()
            want = run(h, X, X[:k], 4, 0)
            plain = before - free_bytes()
            same(run(h, X, X[:k], 4, 2), want)
            limits = before - free_bytes() - plain
    assert limits > 100 << 20, (plain, limits)
    with hip.Handle(n, d, k, np.float32, verbose=200) as h:
        h.set_data(X)
        hogs, left = [], plain + (60 << 20)
        while free_bytes() > left + (8 << 20):  # (a handle's two models)
            kh = min(free_bytes() - left, 32 << 30) // (2 * 4 * 4096) // 256 * 256
            hogs.append(hip.Handle(kh, 4096, kh, np.float32))
        assert plain + (20 << 20) < free_bytes() < plain + limits - (20 << 20)
        capfd.readouterr()
        got = run(h, X, X[:k], 4, 2)
        err = capfd.readouterr().err
        for hog in hogs:
            hog.close()
    same(got, want)
    assert got["measured"] == -1 and err == ""


# (a centroid of equal features has a norm whose roundings all go the same way, and by how much hangs on its last bits:
# up to d / 2 eps, where random features show some 0.13 sqrt(d))
@pytest.mark.parametrize("n,d,k", [(20003, 784, 10), (20003, 1024, 3), (20003, 300, 16), (30001, 32, 80), (30001, 61, 70),
                                   (30001, 298, 130), (30001, 780, 66)])
def test_rows_of_equal_features(hip, n, d, k):
    rng = np.random.default_rng(d)
    X = np.empty((n, d), np.float32)
    X[:] = rng.uniform(1.0, 1.4, (n, 1)).astype(np.float32)
    C = X[rng.permutation(n)[:k]].copy()
    for steps in (5, 8, 12, 20, 40):
        same(fit(hip, X, C, steps, 2), fit(hip, X, C, steps, 0))


@pytest.mark.parametrize("d,k", [(68, 3), (784, 10), (260, 16), (32, 70), (13, 90)])
def test_sums_that_large_values_have_left(hip, d, k):
    """Two rows whose first features are 2^60 and -2^60 are as near to the centroid of ordinary rows as to one on an axis, to
    float32, once that one is nearer than 2^48 (2^50.5 where distances are compared at 16 ulp): they leave the ordinary rows' sum when steps measure some rows
    only, and what their size has rounded away of it must be there again."""
    rng = np.random.default_rng(d)
    m, line = 5000, 15000
    t = np.sort(rng.uniform(2, 4, line))
    c, path = np.array([4.0, 3.8]), []
    for _ in range(5):
        far = t > c.mean()
        c = np.array([t[far].mean(), t[~far].mean()])
        path.append(c[0])
    near = 2.0 ** (50.5 if d <= 64 else 48)
    unit = near / ((path[2] + path[3]) / 2)  # (a step from the fifth on is the first that sees centroids so near)
    X = np.zeros((m + line, d), np.float32)
    X[:m] = rng.uniform(0.5, 1.5, (m, d)) / 3
    X[m:, 1] = t * unit
    X[m + line // 2, 2] = 7
    big = [100, 3000]
    X[big] = 0
    X[big, 0] = 2.0 ** 60, -2.0 ** 60
    C = np.zeros((k, d), np.float32)
    C[0, 1], C[1, 0], C[2, 1] = 4.0 * unit, 1, 3.8 * unit
    C[3:, 3] = 2.0 ** 54 * np.arange(1, k - 2)
    before = fit(hip, X, C, 3, 0)
    assert (before["labels"][big] == 1).all()
    ordinary = np.setdiff1d(np.arange(m), big)
    for steps in (9, 12, 30):
        got, want = fit(hip, X, C, steps, 2), fit(hip, X, C, steps, 0)
        assert (want["labels"][big] == 0).all()
        assert np.allclose(want["centers"][1], X[ordinary].astype(np.float64).mean(0), rtol=1e-6, atol=0)
        assert np.array_equal(got["labels"], want["labels"]) and np.array_equal(got["counts"], want["counts"])
        assert np.allclose(got["centers"], want["centers"], rtol=3e-7, atol=0)


@pytest.mark.parametrize("d,k", [(68, 3), (784, 10), (32, 80), (61, 70)])
@pytest.mark.parametrize("what", ["unrounded", "scales", "sparse", "sparse integers"])
def test_sums_of_any_values(hip, d, k, what):
    """Values whose sums are not exact, features of very different sizes, features that are zero in a whole cluster:
    a mean is a float32 value, of sums whose error is some 2^-50 of it."""
    X, C = strips(20003, d, k, "float64", 7)
    rng = np.random.default_rng(d)
    if what == "scales":
        scale = 2.0 ** rng.uniform(-12, 12, d)
        X, C = X * scale, C * scale
    elif what != "unrounded":
        keep = rng.uniform(size=X.shape) < 0.02
        keep[:, :1] = True
        X = np.where(keep, np.round(16 * X) if what == "sparse integers" else X * np.pi, 0)
        C = C * (16 if what == "sparse integers" else np.pi)
    X, C = X.astype(np.float32), C.astype(np.float32)
    for steps in (6, 12, 25):
        got, want = fit(hip, X, C, steps, 2), fit(hip, X, C, steps, 0)
        assert np.array_equal(got["labels"], want["labels"]) and np.array_equal(got["counts"], want["counts"])
        assert np.allclose(got["centers"], want["centers"], rtol=3e-7, atol=0)
        assert got["measured"] >= 0


# rows without clusters: bounds that are given up for sixteen steps after three looks in vain, and begun anew
NOISE = [("float32", 20003, 32, 80), ("float32", 6001, 784, 10), ("float32", 40001, 101, 130), ("float64", 20003, 80, 130)]


def noise(dtype, n, d, k):
    rng = np.random.default_rng(n + d)
    X = (np.round(rng.standard_normal((n, d)) * 1024) / 1024).astype(dtype)
    return X, X[:k].copy()


@pytest.mark.parametrize("dtype,n,d,k", NOISE)
def test_fits_come_out_the_same_every_time(hip, dtype, n, d, k):
    """Which steps keep bounds, and how the minimum distances are made, hangs on the rows and not on how far the
    host is ahead of the device (other fits run at the same time here, every other time)."""
    import threading
    X, C = noise(dtype, n, d, k)
    Y, D = noise("float32", 400000, 64, 64)
    done = threading.Event()

    def others():
        with hip.Handle(Y.shape[0], Y.shape[1], D.shape[0], Y.dtype) as g:
            g.set_data(Y)
            while not done.is_set():
                run(g, Y, D, 3, 0)

    with hip.Handle(n, d, k, X.dtype) as h:
        h.set_data(X)
        for tol in (0.0, 1e-30):
            fits = {}
            for busy in (False, True):
                done.clear()
                thread = threading.Thread(target=others) if busy else None
                if busy:
                    thread.start()
                try:
                    for steps in range(12, 44):
                        fits.setdefault(steps, []).extend(run(h, X, C, steps, 2, tol) for _ in range(3))
                finally:
                    done.set()
                    if busy:
                        thread.join()
            for steps, f in fits.items():
                assert len({g["measured"] for g in f}) == 1, (steps, [g["measured"] for g in f])
                for g in f[1:]:
                    same(g, f[0], dtype == "float32")
                    assert dtype == "float64" or np.array_equal(g["mind"], f[0]["mind"])


@pytest.mark.parametrize("dtype,n,d,k", NOISE)
def test_bounds_given_up_and_begun_anew(hip, dtype, n, d, k):
    """Three looks in vain from the third step on, sixteen steps without limits, three more, then 32 without:
    fits that end in each stretch, and in the first steps of the next one."""
    X, C = noise(dtype, n, d, k)
    with hip.Handle(n, d, k, X.dtype) as h:
        h.set_data(X)
        for steps in (16, 24, 30, 41, 64, 80):
            want = run(h, X, C, steps, 0)
            for tol in (0.0, 1e-30):
                got = run(h, X, C, steps, 2, tol)
                assert got["it"] == steps or tol > 0
                if got["it"] != steps:  # (at rest)
                    want = run(h, X, C, steps, 0, tol)
                same(got, want, dtype == "float32")


# a little above the line from which fits keep bounds by themselves: the row-stationary step, tiled kernels of both
# precisions, long rows with a handful of centroids
DEFAULT = [("float32", 2000003, 32, 256), ("float32", 80001, 132, 500), ("float64", 60001, 101, 900), ("float32", 140001, 784, 10)]


@pytest.mark.parametrize("dtype,n,d,k", DEFAULT)
def test_fits_keep_bounds_by_themselves(hip, dtype, n, d, k):
    """Through a handle that nobody sets an option for, and through the estimator."""
    from h2o4gpu_amd import KMeans
    X, C = strips(n, d, k, dtype, 5)
    want = fit(hip, X, C, 12, 0)
    got = fit(hip, X, C, 12)
    assert want["measured"] == -1 and 0 <= got["measured"] < n / 2
    same(got, want, dtype == "float32")
    assert fit(hip, X, C, 9)["measured"] == -1
    model = KMeans(n_clusters=k, init=C, n_init=1, max_iter=12, tol=0.0).fit(X)
    assert np.array_equal(model.labels_, want["labels"])
    big = np.abs(want["centers"]).max()
    off = 0 if dtype == "float32" else 1000 * np.finfo(np.float64).eps * big
    assert np.allclose(model.cluster_centers_, want["centers"], rtol=0, atol=off)


@pytest.mark.parametrize("k", [17, 27, 100])
def test_blocks_of_one_centroid_are_not_measured(hip, k):
    """Rows ordered in space, clusters far apart: hardly a block has rows of two."""
    n = 300007
    rng = np.random.default_rng(k)
    places = np.stack(np.meshgrid(*[np.arange(5) * 16.0] * 3), -1).reshape(-1, 3)[rng.permutation(125)[:k]]
    X = (places[rng.integers(0, k, n)] + np.round(rng.standard_normal((n, 3)) * 256) / 256).astype(np.float32)
    C = (places + 1).astype(np.float32)
    got, want = fit(hip, X, C, 12, 2), fit(hip, X, C, 12, 0)
    assert want["measured"] == -1 and 0 <= got["measured"] < n / 10
    same(got, want)


def test_a_stop_signal_ends_a_fit_that_does_not_measure_every_row(hip):
    """Runs in a child process: the handler is process-wide and must not replace pytest's. The labels are those of
    the centroids the fit has come to."""
    import json
    import os
    import subprocess
    import sys
    here = os.path.dirname(os.path.abspath(__file__))
    proc = subprocess.run([sys.executable, os.path.join(here, "signal_stop_bounds_check.py")],
                          capture_output=True, text=True, timeout=100)
    assert proc.returncode == 0, proc.stdout + proc.stderr
    fits = [json.loads(line) for line in proc.stdout.strip().splitlines()]
    assert len(fits) == 4
    for f in fits:
        assert f["stopped"] and f["bounds"] and f["labels"] and f["counts"], fits
    assert proc.stderr.count("Signal caught") == 4, fits
