"""The kernels that form float32 products on the bfloat16 matrix pipe by default give the labels of the
float32 instructions bit for bit: rows within rounding of a tie are settled as those settle them, in
every kernel family and wherever a model or a tile ends."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def near_tied(n, d, k, offset=0.0, every=3):
    """Rows, and centroids one in `every` of which has a neighbour within a hair: rows near those are ties."""
    rng = np.random.default_rng(n + 7 * d + k)
    C = rng.uniform(-20, 20, size=(k, d))
    for c in range(0, k - 1, every):
        C[c + 1] = C[c] + 2e-5 * rng.standard_normal(d)
    C = (C[rng.permutation(k)] + offset).astype(np.float32)
    X = (C[rng.integers(0, k, size=n)] + 4 * rng.standard_normal((n, d))).astype(np.float32)
    return X, C


def run(hip, X, C, split=None, steps=0, fuse=1):
    with hip.Handle(X.shape[0], X.shape[1], C.shape[0], np.float32) as h:
        h.set_data(X)
        h.set_option("fuse", fuse)
        if split is not None:
            h.set_option("fp32_split", split)
        h.set_centroids(C)
        products = h.step_products()
        if steps:
            h.fit(steps, 0.0)
        else:
            h.assign()
        return h.labels(), h.centroids(), h.min_distances(), products


# row-stationary: rows of whole 16-byte vectors and not, one and several 32-centroid tiles, one chunk of
# centroids and several (d = 24 and 32 beyond some 450, d = 64 beyond 224), fewer rows than a tile
ROWSTAT = [(5000, 16, 129), (4001, 13, 300), (20001, 32, 256), (3000, 30, 70), (6000, 64, 224), (6000, 64, 700), (5003, 61, 35),
           (9000, 24, 1500), (7000, 9, 1000), (33, 40, 100), (1, 48, 65), (4000, 32, 2000)]
SHORT = [(5000, 3, 17), (4001, 4, 64), (20001, 5, 300), (3000, 6, 65), (1, 7, 50), (6000, 8, 100), (33, 3, 900)]
TILED = [(5000, 65, 300), (4097, 101, 500), (20001, 96, 257), (129, 127, 200), (3000, 112, 1000)]


@pytest.mark.parametrize("offset", [0.0, 30.0])
@pytest.mark.parametrize("n,d,k", ROWSTAT + SHORT + TILED)
def test_labels_are_the_float32_instructions(hip, n, d, k, offset):
    # (the tiled kernel lists its ties and holds a sixteenth of the rows)
    X, C = near_tied(n, d, k, offset, every=60 if d > 64 else 3)
    got, _, mind, products = run(hip, X, C, fuse=0)
    want, _, wmind, none = run(hip, X, C, split=0, fuse=0)
    assert products == 6 and none == 0
    assert np.array_equal(got, want)
    # (the data has rows that the two forms label differently unless they are settled)
    if n >= 3000:
        assert not np.array_equal(run(hip, X, C, split=6, fuse=0)[0], want)
    scale = (X.astype(np.float64) ** 2).sum(1).max() + (C.astype(np.float64) ** 2).sum(1).max()
    assert np.abs(mind - wmind).max() <= (16 + 4 * np.sqrt(d) + 40) * np.finfo(np.float32).eps * scale


@pytest.mark.parametrize("offset", [0.0, 4000.0])
@pytest.mark.parametrize("n,d,k", TILED + [(5000, 132, 200), (4097, 131, 70), (20011, 298, 300), (3000, 784, 257), (20000, 160, 256)])
def test_more_ties_than_the_list_holds(hip, n, d, k, offset):
    """A third of the centroids in pairs, or data so far from the origin that most rows are ties: the
    pass runs again on the float32 instructions, in each form the plain kernel has."""
    X, C = near_tied(n, d, k, offset)
    got, _, mind, products = run(hip, X, C)
    want, _, wmind, _ = run(hip, X, C, split=0)
    assert products == 6 and np.array_equal(got, want) and np.array_equal(mind, wmind)


def test_parts_of_a_set_are_labelled_as_the_set(hip):
    """labels of rows predicted in pieces, whatever ties each piece has, are those of the fit."""
    X, C = near_tied(30000, 150, 200, every=8)
    with hip.Handle(30000, 150, 200, np.float32) as h:
        h.set_data(X)
        h.set_centroids(C)
        h.assign()
        want = h.labels()
        assert np.array_equal(h.predict(X), want)
        for lo, hi in ((0, 40), (40, 5000), (5000, 30000)):
            assert np.array_equal(h.predict(X[lo:hi]), want[lo:hi])


# (65 features: the parts fit the fixed array in both cases, the list beside two million rows does not)
@pytest.mark.parametrize("n,d,k", [(20000, 3, 27), (5000, 8, 60), (20001, 32, 256), (9000, 24, 1500), (5000, 65, 300), (3000, 300, 200),
                                   (2000000, 65, 300), (3000, 784, 3000)])
def test_calls_without_allocation_give_the_same_labels(hip, n, d, k):
    X, C = near_tied(n, d, k, every=3 if n < 100000 else 60)
    with hip.Handle(k, d, k, np.float32) as h:
        h.set_centroids(C)
        h.set_option("fp32_split", 0)
        want = h.predict(X)
    dX, dC = torch.from_numpy(X).cuda(), torch.from_numpy(C).cuda()
    labels = torch.full((n,), -7, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    hip.predict_device_noalloc(np.float32, n, d, k, dX.data_ptr(), dC.data_ptr(), labels.data_ptr(),
                               torch.cuda.current_stream().cuda_stream)
    assert np.array_equal(labels.cpu().numpy(), want)


@pytest.mark.parametrize("n,d,k", [(60000, 32, 256), (40000, 61, 40), (50000, 13, 200), (60000, 3, 27), (40000, 7, 60), (30000, 100, 400)])
def test_a_fit_takes_the_same_course(hip, n, d, k):
    """Labels and centroids of 25 fused steps are those of the float32 instructions, whose course a
    single row labelled otherwise would leave."""
    rng = np.random.default_rng(d)
    X = (rng.uniform(0, 50, size=(k // 2, d))[rng.integers(0, k // 2, size=n)] + 9 * rng.standard_normal((n, d)))
    X = np.rint(4 * X).astype(np.float32) / 4 if d < 9 else X.astype(np.float32)
    C = X[rng.choice(n, size=k, replace=False)]
    got, want = run(hip, X, C, steps=25), run(hip, X, C, split=0, steps=25)
    assert got[3] == 6 and want[3] == 0
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("n,d,k,sets", [(30000, 30, 70, 2), (20000, 64, 40, 2), (25000, 5, 60, 3)])
def test_a_restart_is_the_fit_it_stands_for(hip, n, d, k, sets):
    """Stacked restarts against ordinary handles, both left to choose their kernels (the stacked steps
    run the float32 instructions, the others the bfloat16 products)."""
    rng = np.random.default_rng(n)
    X = (rng.uniform(-8, 8, size=(k, d))[rng.integers(0, k, size=n)] + 1.5 * rng.standard_normal((n, d))).astype(np.float32)
    if hip.stack_width(n, d, k, np.float32, sets) < sets:
        pytest.skip("shape does not hold %d sets" % sets)
    starts = [X[rng.choice(n, size=k, replace=False)] for _ in range(sets)]
    with hip.Handle(n, d, k, np.float32, sets=sets) as h:
        h.set_data(X)
        for s in range(sets):
            h.select_set(s)
            h.set_centroids(starts[s])
        assert h.step_products() == 0
        h.fit(15, 0.0)
        for s in range(sets):
            h.select_set(s)
            labels, centres, _, products = run(hip, X, starts[s], steps=15)
            assert products == 6
            assert np.array_equal(h.labels(), labels) and np.array_equal(h.centroids(), centres)


@pytest.mark.parametrize("n,d,k", [(5000, 8, 60), (20001, 32, 256), (9000, 24, 1500), (5000, 65, 300), (3000, 300, 200)])
def test_captured_calls_settle_each_replay_anew(hip, n, d, k):
    """The call without allocation recorded into a graph: replays on other rows, with few ties, with more
    than the list holds, and with few again, give what the call gives outside the graph."""
    few, C = near_tied(n, d, k, every=60)
    dX, dC = torch.from_numpy(few).cuda(), torch.from_numpy(C).cuda()
    labels = torch.empty(n, dtype=torch.int32, device="cuda")
    side = torch.cuda.Stream()

    def call(stream):
        hip.predict_device_noalloc(np.float32, n, d, k, dX.data_ptr(), dC.data_ptr(), labels.data_ptr(), stream.cuda_stream)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(side)  # (a kernel's LDS limit is raised outside the capture)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call(torch.cuda.current_stream())
    tied = torch.from_numpy(C[np.random.default_rng(3).integers(0, 2, size=n)]).cuda() * 0.5 + 0.5 * dC[torch.arange(n, device="cuda") % k]
    for rows in (torch.from_numpy(few).cuda(), tied, torch.from_numpy(few).cuda(), tied + 3000):
        dX.copy_(rows)
        torch.cuda.synchronize()
        labels.fill_(-7)
        graph.replay()
        torch.cuda.synchronize()
        got = labels.cpu().numpy()
        labels.fill_(-7)
        torch.cuda.synchronize()
        call(torch.cuda.current_stream())
        torch.cuda.synchronize()
        assert np.array_equal(got, labels.cpu().numpy()) and (got >= 0).all()
        with hip.Handle(k, d, k, np.float32) as h:
            h.set_centroids(C)
            h.set_option("fp32_split", 0)
            assert np.array_equal(got, h.predict(dX.cpu().numpy()))
