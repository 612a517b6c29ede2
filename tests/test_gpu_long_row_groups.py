"""The long-row kernel where its steps run out: wavefronts with one group of four rows or none, odd
and even numbers of groups, workgroups of 8 and of 12 wavefronts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("d,k", [(72, 4), (264, 10), (784, 10), (1024, 3)])
@pytest.mark.parametrize("n", [1, 5, 33, 8191, 8200, 16390, 40000])
def test_long_rows_step_when_the_groups_run_out(hip, oracle, dtype, n, d, k):
    if dtype == np.float64:
        d = min(d, 512)
    rng = np.random.default_rng(n + d)
    X = rng.integers(-20, 20, size=(n, d)).astype(dtype)
    C = rng.integers(-20, 20, size=(k, d)).astype(dtype)
    with hip.Handle(n, d, k, dtype) as h:
        h.set_data(X)
        h.set_centroids(C)
        h.set_option("assign", "wave_row")
        h.iterate(1)
        L, counts, centres = h.labels(), h.counts(), h.centroids()
    D = ((X * X).sum(1)[:, None] + (C * C).sum(1)[None, :] - 2 * X @ C.T).astype(np.float64)
    assert np.array_equal(L, D.argmin(1))  # (whole numbers below 2^24: exact in any order)
    wC, wcounts = oracle.update(X, L, C)
    assert np.array_equal(counts, wcounts) and np.allclose(centres, wC, rtol=4 * np.finfo(dtype).eps)
