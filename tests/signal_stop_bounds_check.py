"""Child process of test_gpu_bounded_fits.py::test_a_stop_signal_ends_a_fit_that_does_not_measure_every_row: fits
that would go on for long, of rows without clusters, with limits kept and with rows ordered in space, and a SIGINT while
they run (H2O4GPU_KMEANS_SIGNALS=1: the library's handler). Not collected by pytest."""
import json
import os
import signal
import sys
import threading

import numpy as np

os.environ["H2O4GPU_KMEANS_SIGNALS"] = "1"
sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
from h2o4gpu_amd.libs import kmeans_hip  # noqa: E402

MOST = 1_000_000
for n, d, k, tol in ((100_003, 32, 80, 0.0), (100_003, 32, 80, 1e-30), (400_003, 3, 100, 0.0), (400_003, 3, 100, 1e-30)):
    X = np.random.default_rng(n + d).standard_normal((n, d), dtype=np.float32)
    with kmeans_hip.Handle(n, d, k, np.float32) as h:
        h.set_data(X)
        h.set_option("bounds", 2)
        h.set_centroids(X[:k])
        h.fit(20, 0.0)  # (kernels loaded, memory taken)
        measured = h.rows_measured()
        h.set_centroids(X[:k])
        threading.Timer(0.015, lambda: os.kill(os.getpid(), signal.SIGINT)).start()
        iterations = h.fit(MOST, tol)
        print(json.dumps({"stopped": 1 <= iterations < MOST, "bounds": measured >= 0, "iterations": iterations,
                          "labels": bool(np.array_equal(h.labels(), h.predict(X))),
                          "counts": int(h.counts().sum()) == n}), flush=True)
