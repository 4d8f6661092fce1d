"""GPU: Ozaki products, Grams and count choices of several threads, which share
the device's stream and its Ozaki workspace, give the results of the same calls
made one after the other."""
import threading

import numpy as np
import pytest

from oracle import ozaki as Z

pytestmark = pytest.mark.gpu


def test_ozaki_calls_of_several_threads(hip):
    rnd = np.random.default_rng(13)

    def product(m, n, k, count, fn):
        A, B = Z.phi_matrix(rnd, (m, k), 1.0), Z.phi_matrix(rnd, (k, n), 1.0)

        def run():
            dC = hip.DeviceArray.filled((m, n), 0xFF)
            fn(0, 0, m, n, k, 1.0, hip.DeviceArray.from_numpy(A), hip.DeviceArray.from_numpy(B), 0.0, dC, count)
            return dC.numpy()
        return run

    def choose(m, n, k):
        A, B = Z.phi_matrix(rnd, (m, k), 2.0), Z.phi_matrix(rnd, (k, n), 2.0)
        return lambda: np.array(hip.ozaki_choose(0, 0, m, n, k, hip.DeviceArray.from_numpy(A),
                                                 hip.DeviceArray.from_numpy(B)))

    # sizes that grow, so that a later call replaces the workspace
    jobs = [product(100, 80, 300, 9, hip.ozaki2_dgemm), choose(500, 400, 1500), product(300, 200, 700, 6, hip.ozaki_dgemm),
            product(700, 900, 1000, 15, hip.ozaki2_dgemm)]
    alone = [job() for job in jobs]
    wrong = []

    def work(i):
        for rep in range(20):
            if not np.array_equal(jobs[i](), alone[i]):
                wrong.append((i, rep))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
