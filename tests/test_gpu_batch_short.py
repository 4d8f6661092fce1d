"""GPU: the simulated grid's batched rounds with segments of fewer than 16 k
(none at all among them) and ranks of a single row: the bits of one launch per
rank and round, and exact on integers."""
import numpy as np
import pytest

from tests.simutil import run_sim

pytestmark = pytest.mark.gpu

# (p, grid, m, n, k): rounds of 0 or 1, of 15 or 16, 7 or 8, 3 k and ranks of 1 or 2 rows, next to longer ones
CASES = [(4, [2, 2, 1], 300, 200, 1), (4, [2, 2, 1], 301, 203, 31), (24, [4, 2, 3], 515, 261, 47),
         (16, [4, 4, 1], 131, 1030, 13), (8, [2, 2, 2], 3, 700, 500), (24, [4, 2, 3], 4099, 2051, 95),
         (9, [3, 3, 1], 4, 100, 50), (4, [2, 2, 1], 2, 300, 19)]


@pytest.mark.parametrize("p,grid,m,n,k", CASES)
def test_short_segments(hip, monkeypatch, p, grid, m, n, k):
    rnd = np.random.default_rng(m + k)
    print(f"[short] {p} {grid} {m}x{n}x{k}", flush=True)
    A, B = rnd.standard_normal((m, k)), rnd.standard_normal((k, n))
    batch = run_sim(p, m, n, k, 0, 0, A, B, proc_grid=grid)
    monkeypatch.setenv("CA3DMM_SIM_BATCH", "0")
    assert np.array_equal(batch, run_sim(p, m, n, k, 0, 0, A, B, proc_grid=grid))
    monkeypatch.delenv("CA3DMM_SIM_BATCH")
    A, B = rnd.integers(-9, 10, (m, k)).astype(float), rnd.integers(-9, 10, (k, n)).astype(float)
    assert np.array_equal(run_sim(p, m, n, k, 0, 0, A, B, proc_grid=grid), A @ B)


@pytest.mark.parametrize("p,grid,m,n,k", CASES)
def test_short_segments_in_registers(hip, p, grid, m, n, k):
    """The grouped mode's batched form, whose rounds accumulate in registers."""
    rnd = np.random.default_rng(m + k + 1)
    A, B = rnd.standard_normal((m, k)), rnd.standard_normal((k, n))
    batched, persistent = (_grouped(p, m, n, k, A, B, grid, tile) for tile in (3, 0))
    assert np.array_equal(batched, persistent)


def _grouped(p, m, n, k, A, B, grid, tile):
    out, sim, w, args = run_sim(p, m, n, k, 0, 0, A, B, proc_grid=grid, grouped=True, keep=True)
    Ap, ldA, Bp, ldB, Cp, ldC, dC, dA, dB = args
    sim.set_tuning(8, 2, tile)
    dC.upload(np.full(out.shape, -1.0))
    sim.exec(Ap, ldA, Bp, ldB, Cp, ldC)
    got = dC.numpy()
    sim.free()
    return got
