"""GPU: factorizations and right solves of several threads, which share the
device's stream and its scratch buffer, give the bits of the same calls made
one after the other."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _spd(rnd, n):
    R = np.triu(rnd.uniform(-1, 1, (n, n)), 1) / n + np.diag(rnd.uniform(1, 2, n))
    return R, R.T @ R


def test_factor_and_solve_of_several_threads(hip):
    rnd = np.random.default_rng(11)
    jobs = []
    # sizes that grow, so that a solve's larger request replaces the buffer
    for m, n in ((0, 200), (300, 64), (0, 449), (500, 257), (0, 130), (900, 400)):
        R, S = _spd(rnd, n)
        B = rnd.standard_normal((m, n))

        def run(m=m, n=n, R=R, S=S, B=B):
            if m == 0:
                d = hip.DeviceArray.from_numpy(S)
                assert hip.potrf_upper(n, d) == 0
            else:
                d = hip.DeviceArray.from_numpy(B)
                hip.trsm_right_upper(m, n, 1.0, hip.DeviceArray.from_numpy(R), d)
            return d.numpy()

        jobs.append(run)
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
