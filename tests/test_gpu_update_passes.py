"""The passes around the distance kernels where their work split can go wrong: row norms of many
long rows, the ordering of the rows by label, the counts per candidate of the seeding."""
import numpy as np
import pytest
import scipy.sparse
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,d", [(49151, 70), (49152, 65), (49157, 96), (50000, 97), (49409, 131), (60001, 64)])
def test_row_norms_are_the_scalar_sum(hip, dtype, n, d):
    """The squared norm of a row is its distance to a centroid at the origin: bit for bit the sum
    over j ascending with every product and every sum rounded, whichever kernel makes it."""
    rng = np.random.default_rng(n + d)
    X = rng.standard_normal((n, d)).astype(dtype)
    C = np.zeros((17, d), dtype)
    C[1:] = rng.standard_normal((16, d)).astype(dtype)
    with hip.Handle(n, d, 17, dtype) as h:
        h.set_data(X)
        h.set_centroids(C)
        h.set_option("assign", "mfma_tiled")
        out = torch.empty((17, n), dtype=torch.float32 if dtype == np.float32 else torch.float64, device="cuda")
        torch.cuda.synchronize()
        h.transform_resident(out.data_ptr())
        got = out[0].cpu().numpy()
    want = np.zeros(n, dtype)
    for j in range(d):
        want = want + X[:, j] * X[:, j]
    assert np.array_equal(got, want)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,k", [(1023, 1023), (1025, 1024), (5000, 1025), (70001, 2048), (9000, 2049), (30000, 4097)])
@pytest.mark.parametrize("how", ["random", "one", "sorted", "gaps"])
def test_rows_in_label_order(hip, dtype, n, k, how):
    """Given labels, the update's counts and means: blocks, wavefronts and rounds of 64 rows with a
    remainder, numbers of labels round a power of two, rounds of a single label, rows without one."""
    d = 1 + 160 * 1024 // min(k, 1024)  # (the sums are beyond the LDS chunks: rows are ordered by label)
    rng = np.random.default_rng(n + k)
    X = rng.integers(-50, 50, size=(n, d)).astype(dtype)  # (sums exact: any order gives the same)
    L = rng.integers(0, k, size=n).astype(np.int32)
    if how == "one":
        L[:] = k - 1
    elif how == "sorted":
        L.sort()
    elif how == "gaps":
        L[rng.random(n) < 0.3] = -1
    C = rng.standard_normal((k, d)).astype(dtype)
    with hip.Handle(n, d, k, dtype) as h:
        h.set_data(X)
        h.set_centroids(C)
        h.set_labels(L)
        h.update()
        got, counts = h.centroids(), h.counts()
    assert np.array_equal(counts, np.bincount(L[L >= 0], minlength=k))
    rows = np.flatnonzero(L >= 0)
    sums = scipy.sparse.csr_matrix((np.ones(len(rows)), (L[rows], rows)), shape=(k, n)) @ X.astype(np.float64)
    scale = (dtype(1) / np.maximum(counts, 1).astype(dtype))[:, None]
    want = np.where(counts[:, None] > 0, sums.astype(dtype) * scale, C)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("n,d,k", [(20000, 3, 2), (50001, 8, 300), (40000, 4, 9000)])
def test_candidate_weights_count_every_row_once(hip, n, d, k):
    """Rows per nearest candidate: counted in LDS up to 16384 candidates, in memory beyond."""
    rng = np.random.default_rng(k)
    X = rng.standard_normal((n, d)).astype(np.float32)
    with hip.Handle(n, d, k, np.float32) as h:
        h.set_data(X)
        h.init_parallel(5)
        info = h.parallel_seed_info()
    w, cand = np.asarray(info["weights"]), np.asarray(info["cand_rows"])
    assert len(w) == len(cand) > k and w.sum() == n
    assert k < 9000 or len(w) > 16384
    X64 = X.astype(np.float64)
    C = X64[cand]
    near = np.concatenate([((X64[i:i + 1000] ** 2).sum(1)[:, None] + (C ** 2).sum(1) - 2 * X64[i:i + 1000] @ C.T).argmin(1)
                           for i in range(0, n, 1000)])
    # (a near-tie row may count for either of its two candidates)
    assert np.abs(w - np.bincount(near, minlength=len(cand))).sum() <= 2 * max(4, n // 2000)
