"""Rows within rounding of a tie between two centroids: the split tiled kernel lists them and
settles them with the float32 instructions' own arithmetic (where the list, a sixteenth of the rows,
does not hold them, the pass runs again on those instructions), so the labels are those of the
float32 instructions bit for bit."""
import numpy as np
import pytest

from parity import label_report

pytestmark = pytest.mark.gpu


def labels_of(hip, X, C, split=None, steps=0):
    n, d = X.shape
    with hip.Handle(n, d, C.shape[0], np.float32) as h:
        h.set_data(X)
        h.set_centroids(C)
        if split is not None:
            h.set_option("fp32_split", split)
        products = h.step_products()
        assert products in ((3, 6) if split != 0 else (0,))
        if steps:
            h.fit(steps, 0.0)
        else:
            h.assign()
        return h.labels(), h.min_distances(), h.centroids()


@pytest.mark.parametrize("n,d,k", [(5000, 132, 129), (4097, 131, 300), (20011, 298, 257), (3000, 784, 100), (60001, 256, 1000),
                                   (129, 136, 70)])
@pytest.mark.parametrize("whole", [False, True])
def test_labels_are_the_float32_instructions(hip, n, d, k, whole):
    rng = np.random.default_rng(n + d + k)
    C = rng.uniform(0, 200, size=(k, d)).astype(np.float32)
    # a few centroids within a hair of another one: about three rows in a hundred have both nearest
    for c in range(0, k - 1, max(2, k // 2)):
        C[c + 1] = C[c] + (1e-4 * rng.standard_normal(d)).astype(np.float32)
    X = (C[rng.integers(0, k, size=n)] + 30 * rng.standard_normal((n, d))).astype(np.float32)
    if whole:  # (rows of bfloat16 values: half the products where the rows are many)
        X = np.clip(np.rint(X), 0, 255).astype(np.float32)
    got, mind, _ = labels_of(hip, X, C)
    want, wmind, _ = labels_of(hip, X, C, split=0)
    assert np.array_equal(got, want)
    if n > 1000:  # (there are ties to settle: the same products without it label some rows otherwise)
        assert not np.array_equal(labels_of(hip, X, C, split=6)[0], want)
    eps = np.finfo(np.float32).eps
    scale = (X.astype(np.float64) ** 2).sum(1).max() + (C.astype(np.float64) ** 2).sum(1).max()
    assert np.abs(mind - wmind).max() <= (4 * np.sqrt(d) + 40) * eps * scale


def test_a_fit_takes_the_same_course(hip):
    rng = np.random.default_rng(4)
    n, d, k = 60000, 200, 150
    X = (rng.uniform(0, 50, size=(40, d))[rng.integers(0, 40, size=n)] + 9 * rng.standard_normal((n, d))).astype(np.float32)
    C = X[rng.choice(n, size=k, replace=False)]
    got, want = labels_of(hip, X, C, steps=25), labels_of(hip, X, C, split=0, steps=25)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[2], want[2])


def test_more_ties_than_the_list_holds(hip, oracle):
    """Every centroid twice: every row is a tie, the pass runs again, the lower index wins."""
    rng = np.random.default_rng(8)
    n, d, k = 9000, 160, 140
    C = np.repeat(rng.standard_normal((k // 2, d)).astype(np.float32) * 10, 2, axis=0)
    X = (C[rng.integers(0, k, size=n)] + rng.standard_normal((n, d))).astype(np.float32)
    got, _, _ = labels_of(hip, X, C)
    label_report(oracle, X, C, got, oracle.assign(X, C))
    assert (got % 2 == 0).all() and np.array_equal(got, labels_of(hip, X, C, split=0)[0])


def test_rows_no_distance_exists_for(hip):
    rng = np.random.default_rng(9)
    n, d, k = 3000, 150, 90
    X, C = rng.standard_normal((n, d)).astype(np.float32), rng.standard_normal((k, d)).astype(np.float32)
    X[[3, 77, 2999], [0, 149, 20]] = np.nan, np.inf, -np.inf
    C[11, 5] = np.nan
    got, want = labels_of(hip, X, C)[0], labels_of(hip, X, C, split=0)[0]
    assert np.array_equal(got, want) and (got[[3, 77, 2999]] == -1).all()


@pytest.mark.parametrize("d", [150, 256])
def test_rows_and_centroids_that_are_not_finite_are_no_ties(hip, d):
    """A NaN centroid, or rows with infinite norms, beside rows that are near ties: only those are listed.
    (Were more listed than the list holds, the float32 instructions would run again over all rows, and
    every minimum distance would be theirs.)"""
    rng = np.random.default_rng(d)
    n, k = 8000, 120
    C = rng.uniform(0, 200, size=(k, d)).astype(np.float32)
    C[61] = C[60] + (1e-4 * rng.standard_normal(d)).astype(np.float32)
    X = (C[rng.integers(0, k, size=n)] + 30 * rng.standard_normal((n, d))).astype(np.float32)
    for case in "nan centroid", "infinite rows":
        Y, E = X.copy(), C.copy()
        if case == "nan centroid":
            E[100, 5] = np.nan
        else:
            Y[::5, 3] = np.inf
        got, mind, _ = labels_of(hip, Y, E)
        want, wmind, _ = labels_of(hip, Y, E, split=0)
        assert np.array_equal(got, want), case
        assert not np.array_equal(labels_of(hip, Y, E, split=6)[0], want), case
        assert (mind != wmind).mean() > 0.1, case


@pytest.mark.parametrize("d,k", [(20, 70), (150, 90), (130, 300)])
def test_transform_of_rows_that_are_not_finite(hip, d, k):
    """Infinite and NaN distances come out as the float32 instructions have them."""
    rng = np.random.default_rng(d)
    X, C = rng.standard_normal((300, d)).astype(np.float32), rng.standard_normal((k, d)).astype(np.float32)
    X[[3, 77, 150, 299], [0, 7, 2, 5]] = np.nan, np.inf, -np.inf, 3.4e38
    C[[11, 60], [5, 1]] = np.inf, -3.4e38
    with hip.Handle(300, d, k, np.float32) as h:
        h.set_data(X)
        h.set_centroids(C)
        assert h.step_products() == 6
        got = h.transform(X)
        h.set_option("fp32_split", 0)
        want = h.transform(X)
    finite = np.isfinite(want)
    assert np.array_equal(got[~finite], want[~finite], equal_nan=True) and np.isfinite(got[finite]).all()
    assert (~finite).sum() > 4 * k


@pytest.mark.parametrize("d,k", [(20, 70), (150, 90), (130, 300)])
def test_missing_values_cost_a_transform_no_second_pass(hip, d, k):
    """NaN rows and centroids give NaN where they stand and leave the others as the bfloat16 products have
    them; an infinite row or centroid has the whole transform run on the float32 instructions."""
    rng = np.random.default_rng(d)
    X, C = rng.standard_normal((5000, d)).astype(np.float32), rng.standard_normal((k, d)).astype(np.float32)
    with hip.Handle(5000, d, k, np.float32) as h:
        def both(X, C):
            h.set_centroids(C)
            h.set_option("fp32_split", 0)
            want = h.transform(X)
            h.set_option("fp32_split", -1)
            return h.transform(X), want
        plain, f32 = both(X, C)
        assert not np.array_equal(plain, f32)
        Y, E = X.copy(), C.copy()
        Y[[3, 4000], [0, 7]] = np.nan
        E[11, 5] = np.nan
        got, _ = both(Y, E)
        hurt = np.zeros(got.shape, bool)
        hurt[:, [3, 4000]] = hurt[11] = True
        assert np.isnan(got[hurt]).all() and np.array_equal(got[~hurt], plain[~hurt])
        for bad in (np.inf, -np.inf, 3e30):
            for where in "XC":
                Y, E = X.copy(), C.copy()
                (Y if where == "X" else E)[17, 2] = bad
                got, want = both(Y, E)
                assert np.array_equal(got, want, equal_nan=True) and not np.isfinite(want).all()
