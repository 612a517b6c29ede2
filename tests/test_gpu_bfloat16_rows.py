"""Rows whose every value is a bfloat16 (8-bit pixels) run half the products of the split tiled
kernel; the other half are products with zeros, so labels and distances are the same bits as
those of rows the handle does not look at (host rows of a predict or transform call). Rows that are
no longer such values when the kernel reads them are left to the float32 instructions."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d,k", [(49152, 65, 200), (50001, 100, 300), (49153, 784, 257), (60000, 132, 1024)])
@pytest.mark.parametrize("odd", [None, "first", "last", "middle"])
def test_same_bits_as_the_general_form(hip, n, d, k, odd):
    rng = np.random.default_rng(n + d + k)
    X = rng.integers(0, 256, size=(n, d)).astype(np.float32) * (rng.random((n, d)) < 0.4)
    X = np.ascontiguousarray(X, np.float32)
    if odd is not None:  # one value that is not a bfloat16, wherever the pass over the rows may end
        i, j = {"first": (0, 0), "last": (n - 1, d - 1), "middle": (n // 2 + 1, d - 3)}[odd]
        X[i, j] = 200.1234
    C = (X[rng.choice(n, size=k, replace=False)] + rng.standard_normal((k, d))).astype(np.float32)
    m = 3000
    part = np.concatenate([X[:m // 3], X[n // 2:n // 2 + m // 3], X[n - m // 3:]])
    with hip.Handle(n, d, k, np.float32) as h:
        h.set_data(X)
        h.set_centroids(C)
        assert h.step_products() == (3 if odd is None else 6)
        h.assign()
        got = h.labels()
        out = torch.empty((k, n), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        h.transform_resident(out.data_ptr())
        want, D = h.predict(part), h.transform(part)
        out = out.cpu().numpy()
    pick = np.r_[0:m // 3, n // 2:n // 2 + m // 3, n - m // 3:n]
    assert np.array_equal(got[pick], want)
    assert np.array_equal(out[:, pick], D)
    D64 = ((X[pick[::50]].astype(np.float64)[:, None, :] - C.astype(np.float64)[None, :64]) ** 2).sum(2).T
    scale = (X.astype(np.float64) ** 2).sum(1).max() + (C.astype(np.float64) ** 2).sum(1).max()
    assert np.abs(out[:64, pick[::50]] - D64).max() <= (4 * np.sqrt(d) + 40) * np.finfo(np.float32).eps * scale


@pytest.mark.parametrize("n,d,k", [(49152, 100, 300), (50001, 160, 200)])
def test_rows_rewritten_in_place(hip, n, d, k):
    """Adopted rows that stop being bfloat16 values after the handle has looked at them: assignment,
    transform and the seeding's passes see the values that are there, as the float32 instructions do."""
    rng = np.random.default_rng(n)
    X = rng.integers(0, 256, size=(n, d)).astype(np.float32)
    C = X[rng.choice(n, size=k, replace=False)]
    more = torch.from_numpy(rng.random((n, d), np.float32)).cuda()
    got, phi = [], []
    for split in (None, 0):
        rows = torch.from_numpy(X).cuda()
        out = torch.empty((k, n), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        with hip.Handle(n, d, k, np.float32) as h:
            h.set_data_device(rows.data_ptr(), keepalive=rows)
            if split is not None:
                h.set_option("fp32_split", split)
            h.set_centroids(C)
            h.assign()
            assert h.step_products() == (3 if split is None else 0)
            rows += more
            torch.cuda.synchronize()
            h.assign()
            h.transform_resident(out.data_ptr())
            labels, mind = h.labels(), h.min_distances()
            h.init_parallel(5)
            got.append((labels, mind, out.cpu().numpy()))
            phi.append(h.parallel_seed_info()["phi"])
    # (rounds of 65 to 128 candidates run six products: the sums round differently)
    assert np.allclose(phi[0], phi[1], rtol=2e-6)
    for a, b in zip(*got):
        assert np.array_equal(a, b)
