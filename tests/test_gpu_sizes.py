"""izh_run against izh_step at the sizes where a kernel of the fused run
changes its form: tile counts around the limits of the LDS key histograms,
deposit chunks of every length, grids narrower than the deposit's window.  The bar is the fused run's own: 1e-10
relative in the diagnostics and the particles."""
import pytest

from conftest import col_err, full_row_err
from test_gpu_parity import TOL

pytestmark = pytest.mark.gpu


def run_against_step(gpu, n, grid, period, steps=5, seed=3):
    from impactz import beam as B
    from impactz.sim import Simulation
    print(f"fused against step: {n} particles, grid {grid}, period {period}", flush=True)
    pts = B.gaussian_bunch(n, seed=seed)
    a = Simulation(pts, B.Beam(), B.fodo(1), grid)
    b = Simulation(pts, B.Beam(), B.fodo(1), grid)
    b.bunch.resort_period = period
    rows = [a.diag(a.step(e)) for _, e in zip(range(steps), a.segments())]
    rec = b.run_fused(steps)
    worst = max(full_row_err(b.diag(rec[k]), rows[k]) for k in range(steps))
    pe = col_err(b.bunch.getpts(), a.bunch.getpts())
    a.close()
    b.close()
    assert worst < TOL and pe < TOL, (worst, pe)


@pytest.mark.parametrize("n,grid,period", [
    (20_003, (32, 32, 32), 2),       # 64 tiles: the pass counts its keys in LDS
    (4_001, (64, 64, 128), 3),       # 1024 tiles: the last count that does
    (4_001, (64, 128, 128), 2),      # 2048: past it, the prologue's still does
    (3_001, (256, 256, 256), 2),     # 32768: past the prologue's limit too
])
def test_key_histograms(gpu, n, grid, period):
    run_against_step(gpu, n, grid, period)


@pytest.mark.parametrize("n,grid,period", [
    (50, (4, 8, 16), 1),             # a grid inside one window
    (700, (8, 16, 4), 2),
    (262_143, (32, 32, 32), 4),      # the last bunch of 1024-slot chunks
    (262_145, (32, 16, 64), 4),      # the first of 2048
    (4_194_305, (32, 32, 32), 2),    # full-length chunks
])
def test_deposit_chunks(gpu, n, grid, period):
    run_against_step(gpu, n, grid, period, steps=3)
