"""Random start rows drawn with the device's help: the rows the host's walk picks, whatever the
number of rows, of clusters and the seed."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(46342, 4), (40000, 3), (65537, 1), (100_000, 8), (300_001, 4096), (1_000_003, 37),
                                 (999_999, 100_000), (10_000_000, 256), (50_000_000, 1000)])
@pytest.mark.parametrize("seed", [0, 1, 12345, 2147483647])
def test_rows_equal_the_host_walk(hip, n, k, seed):
    X = torch.zeros((n, 1), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    with hip.Handle(n, 1, k, np.float32) as h:
        h.set_data_device(X.data_ptr(), keepalive=X)
        h.init_random_rows(seed)
        got = h.seed_rows()
    assert np.array_equal(got, hip.random_start_rows(seed, n, k))


def test_second_start_on_one_handle(hip):
    n, k = 200_000, 50
    X = torch.randn((n, 3), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    with hip.Handle(n, 3, k, np.float64) as h:
        h.set_data_device(X.data_ptr(), keepalive=X)
        for seed in (3, 4):
            h.init_random_rows(seed)
            rows = hip.random_start_rows(seed, n, k)
            assert np.array_equal(h.seed_rows(), rows)
            assert np.array_equal(h.centroids(), X.cpu().numpy()[rows])
            h.fit(2, 0.0)
