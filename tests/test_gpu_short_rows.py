"""Rows of three to eight float32 features against more than 16 centroids: the kernel that takes
them by itself, against the CPU oracle, where its tiles and its lane groups end."""
import numpy as np
import pytest

from parity import label_report

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float32).eps


def data(n, d, k, offset=0.0):
    rng = np.random.default_rng(n + 10 * d + k)
    X = (offset + rng.uniform(-10, 10, size=(n, d))).astype(np.float32)
    C = (offset + rng.uniform(-10, 10, size=(k, d))).astype(np.float32)
    return X, C


@pytest.mark.parametrize("d", [3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("n,k,offset", [(1, 17, 0), (1, 65, 0), (31, 32, 0), (31, 64, 0), (65, 49, 0), (4099, 27, 0), (20001, 300, 0),
                                        (3000, 900, 0), (3000, 1300, 0), (30000, 64, 100)])
def test_step_and_labels(hip, oracle, n, d, k, offset):
    X, C = data(n, d, k, offset)
    with hip.Handle(n, d, k, np.float32) as h:
        h.set_data(X)
        h.set_centroids(C)
        # (the dispatch rule; d = 5 to 8 beyond its LDS runs the row-stationary kernel's float32 instructions)
        h.set_option("fuse", 0)
        assert h.step_products() == (6 if k > (16 if d <= 4 else 48) else 0)
        h.set_option("fuse", 1)
        if k <= 300:
            assert h.step_products() == (6 if k > (16 if d <= 4 else 48) else 0)
        h.iterate(1)
        fused, counts, centres = h.labels(), h.counts(), h.centroids()
        h.set_centroids(C)
        h.assign()
        got, mind = h.labels(), h.min_distances()
    want, wmind = oracle.assign(X, C, return_mindist=True)
    label_report(oracle, X, C, got, want)
    label_report(oracle, X, C, fused, want)
    scale = (X.astype(np.float64) ** 2).sum(1).max() + (C.astype(np.float64) ** 2).sum(1).max()
    # distances are compared (and returned) at 16 ulp; each of up to 48 products and six norm parts
    # rounds at most once at the size of xx + cc
    assert np.max(np.abs(mind.astype(np.float64) - wmind)) <= (16 + 54) * EPS * scale
    wC, wcounts = oracle.update(X, fused, C)
    assert np.array_equal(counts, wcounts)
    assert np.allclose(centres, wC, rtol=4 * EPS, atol=4 * EPS * np.abs(X).max())


@pytest.mark.parametrize("d", [3, 4, 5, 8])
def test_distances_are_as_close_to_float64_as_the_float32_instructions(hip, d):
    n, k = 30000, 200
    X, C = data(n, d, k, offset=30.0)
    X64, C64 = X.astype(np.float64), C.astype(np.float64)
    truth = ((X64[:, None, :] - C64[None]) ** 2).sum(2).min(1)
    err = {}
    for variant in ("auto", "mfma_rowstat"):
        with hip.Handle(n, d, k, np.float32) as h:
            h.set_data(X)
            h.set_centroids(C)
            h.set_option("assign", variant)
            assert h.step_products() == (6 if variant == "auto" else 0)
            h.assign()
            err[variant] = np.sqrt(((h.min_distances() - truth) ** 2).mean())
    print("d=%d: rms error of the minimum distance %.3g, float32 instructions %.3g" % (d, err["auto"], err["mfma_rowstat"]))
    assert err["auto"] <= 1.01 * err["mfma_rowstat"]


@pytest.mark.parametrize("d", [3, 4, 5, 8])
def test_rows_and_centroids_no_distance_exists_for(hip, oracle, d):
    X, C = data(3000, d, 60)
    X[5, 0], X[70, d - 1], X[200, 0], X[300] = np.nan, np.inf, -np.inf, 3e38
    C[7, d - 1], C[33, 0] = np.inf, np.nan
    with hip.Handle(3000, d, 60, np.float32) as h:
        h.set_data(X)
        h.set_centroids(C)
        h.assign()
        got = h.labels()
    assert (got[[5, 70, 200, 300]] == -1).all() and not np.isin(got, [7, 33]).any()
    keep = np.ones(3000, bool)
    keep[[5, 70, 200, 300]] = False
    label_report(oracle, X[keep], np.where(np.isfinite(C).all(1)[:, None], C, np.float32(1e18)), got[keep],
                 oracle.assign(X[keep], np.where(np.isfinite(C).all(1)[:, None], C, np.float32(1e18))))
