"""GPU: CholeskyQR of several threads, which share the device's stream and the
buffers of hip_cholesky_qr, gives the bits of the same calls made one after the
other."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_cholesky_qr_of_several_threads(hip):
    rnd = np.random.default_rng(12)
    jobs = []
    # sizes that grow, so that a later call replaces the buffers
    for m, n, variant in ((500, 64, 2), (2000, 200, 0), (3000, 300, 3), (5000, 130, 2)):
        A = rnd.standard_normal((m, n))

        def run(m=m, n=n, variant=variant, A=A):
            dA, dR = hip.DeviceArray.from_numpy(A), hip.DeviceArray.filled((n, n), 0xFF)
            assert hip.cholesky_qr(m, n, dA, dR, variant=variant)[0] == 0
            return dA.numpy(), dR.numpy()

        jobs.append(run)
    alone = [job() for job in jobs]
    wrong = []

    def work(i):
        for rep in range(15):
            if not all(np.array_equal(a, b) for a, b in zip(jobs[i](), alone[i])):
                wrong.append((i, rep))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
