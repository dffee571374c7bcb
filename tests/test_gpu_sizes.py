"""izh_run against izh_step at the sizes where a kernel of the fused run
changes its form: tile counts around the limits of the LDS key histograms,
deposit chunks of every length, grids narrower than the deposit's window.  The bar is the fused run's own: 1e-10
relative in the diagnostics and the particles."""
import numpy as np
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
    moms, rows = [], []
    for _, e in zip(range(steps), a.segments()):
        moms.append(a.step(e))
        rows.append(a.diag(moms[-1]) if n > 2 else None)
    rec = b.run_fused(steps)
    # two particles lie on a line of each plane: emittance zero, the derived
    # columns undefined; their squares, products and maxima still compare
    pick = list(range(6, 12)) + list(range(37, 44))
    worst = max(float(np.max(np.abs(rec[k][pick] / moms[k][pick] - 1))) for k in range(steps))
    if n > 2:
        worst = max([worst] + [full_row_err(b.diag(rec[k]), rows[k])
                               for k in range(steps)])
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


def open_potential(rho, h):
    """The open-boundary potential of rho[k][j][i] in numpy FP64: the doubled
    convolution with the integrated Green function."""
    nz, ny, nx = rho.shape
    ax = [np.arange(n + 2) * d - d / 2.0 for n, d in zip((nx, ny, nz), h)]
    x, y, z = ax[0][None, None, :], ax[1][None, :, None], ax[2][:, None, None]
    r = np.sqrt(x * x + y * y + z * z)
    t = (-z * z * np.arctan(x * y / (z * r)) - y * y * np.arctan(x * z / (y * r))
         - x * x * np.arctan(y * z / (x * r))) / 2.0
    t += y * z * np.log(x + r) + x * z * np.log(y + r) + x * y * np.log(z + r)
    g = np.diff(np.diff(np.diff(t, axis=0), axis=1), axis=2) / (h[0] * h[1] * h[2])

    def fold(n):
        m = np.arange(2 * n)
        return np.where(m <= n, m, 2 * n - m)
    g = g[np.ix_(fold(nz), fold(ny), fold(nx))]
    s = (2 * nz, 2 * ny, 2 * nx)
    return np.fft.irfftn(np.fft.rfftn(g) * np.fft.rfftn(rho, s=s, axes=(0, 1, 2)), s=s,
                         axes=(0, 1, 2))[:nz, :ny, :nx]


@pytest.mark.parametrize("grid", [(4, 4, 4), (8, 64, 4), (128, 8, 16), (16, 256, 8),
                                  (4, 32, 128), (64, 16, 512), (512, 4, 8)])
def test_solve_line_lengths(gpu, grid):
    """The transforms of G and of the charge at every kind of line length:
    runtime and compile-time, one block's worth and more, along each axis.
    FP64 within 1e-10 of the maximum; the mixed form's FP32 transforms
    round each of their about 3 log2(8 g) stages to 6e-8, so 1e-5 bounds
    them."""
    print(f"solve {grid}", flush=True)
    nx, ny, nz = grid
    h = (1.0e-3, 0.8e-3, 2.0e-3)
    rho = np.random.default_rng(5).random((nz, ny, nx))
    want = open_potential(rho, h)
    for prec, tol in ((gpu.FP64, TOL), (gpu.MIXED, 1e-5)):
        f = gpu.FieldQuant(*grid, precision=prec)
        d = gpu.CompDom(*grid)
        d.set([0, h[0] * (nx - 1), 0, h[1] * (ny - 1), 0, h[2] * (nz - 1)], h)
        f.upload_rho(rho)
        f.update3O(d)
        err = np.max(np.abs(f.download(gpu.PHI) - want)) / np.max(np.abs(want))
        f.close()
        assert err < tol, (prec, err)


@pytest.mark.parametrize("n,grid,period", [
    (2, (8, 8, 8), 1),               # fewer particles than a wavefront
    (257, (16, 16, 16), 2),          # two blocks, one of a single slot
    (3_000, (128, 128, 128), 2),     # a group crosses hundreds of tiles
    (131_073, (64, 64, 128), 3),     # the first bunch of two groups a block
    (524_288, (32, 32, 32), 2),      # the last pass that kicks from phi
    (524_289, (32, 32, 32), 2),      # the first that gathers E through a box
    (70_000, (4, 4, 4), 2),          # from phi, every cell at an edge
    (786_432, (64, 64, 128), 2),     # 3/2 of the nodes
    (1_048_577, (64, 64, 64), 2),    # past four times the nodes
    (1_500_001, (64, 64, 128), 2),   # the first pass of 1024 blocks
    (4_000_001, (64, 64, 128), 2),   # and of 2048
])
def test_pass_blocks(gpu, n, grid, period):
    run_against_step(gpu, n, grid, period, steps=3)


@pytest.mark.parametrize("n,grid", [
    (4_096, (32, 32, 32)),           # straight to the grid
    (4_097, (16, 16, 32)),           # the whole grid in LDS: its largest
    (4_097, (4, 8, 16)),             # and a small one
    (4_097, (32, 16, 32)),           # binned: 16 tiles
    (50_001, (128, 64, 16)),         # uneven tiles, a ragged last block
    (5_000, (128, 256, 256)),        # 16384 tiles of 8 nodes: tiles of 16
    (4_500, (4, 1024, 8)),           # a tile as wide as the grid
])
@pytest.mark.parametrize("uniform", [True, False])
def test_charge_forms(gpu, n, grid, uniform):
    """izh_charge against numpy: the contributions, rounded to the deposit's
    fixed point (2^e with sum |w| 2^e <= 2^61), sum exactly in any order, so
    what remains is the rounding of the weights and of each contribution:
    1e-13 of the largest node bounds both."""
    print(f"charge {n} {grid} uniform {uniform}", flush=True)
    from impactz import beam as B
    pts = B.gaussian_bunch(n, seed=8)
    if not uniform:
        pts[:, 7] *= np.random.default_rng(9).uniform(0.5, 2.0, n)
    b = gpu.BeamBunch.from_beam(pts, B.Beam())
    f = gpu.FieldQuant(*grid)
    d = gpu.CompDom(*grid)
    pr, _, _ = b.conv1st(0.0, 1.0, 1.0)
    d.update(pr)
    for _ in range(2):               # the second from the scratch the first made
        b.charge(d, f)
    rho = f.download(gpu.RHO)
    p = b.getpts()
    lo, h = d.range[0::2], d.msize
    want = np.zeros(grid[0] * grid[1] * grid[2])
    pos = p[:, [0, 2, 4]]
    i = ((pos - lo) * (1.0 / h) + 1.0).astype(np.int64)
    a = ((lo - pos) + i * h) * (1.0 / h)
    for c in range(8):
        o = np.array([c & 1, (c >> 1) & 1, c >> 2])
        w = np.prod(np.where(o, 1.0 - a, a), axis=1) * p[:, 7]
        k = i - 1 + o
        np.add.at(want, k[:, 0] + grid[0] * (k[:, 1] + grid[1] * k[:, 2]), w)
    err = np.max(np.abs(rho.ravel() - want)) / np.max(np.abs(want))
    b.close()
    f.close()
    assert err < 1e-13, err


@pytest.mark.parametrize("n", [1, 2_047, 2_048, 2_049, 300_007, 4_003_000])
@pytest.mark.parametrize("lossy", [False, True])
def test_download_order(gpu, n, lossy):
    """getpts returns the survivors in their original order: chunk edges of
    the packing, and more rows than it copies at a time.  The t-frame position
    is a few FP64 operations (1e-14)."""
    print(f"download {n} lossy {lossy}", flush=True)
    from impactz import beam as B
    bm = B.Beam()
    pts = B.gaussian_bunch(n, seed=4)
    b = gpu.BeamBunch.from_beam(pts, bm)
    rad = 1.5e-3 if lossy else 1.0
    b.conv1st(0.0, rad, rad)
    got = b.getpts()
    rcp = 1.0 / (bm.gamma0 - pts[:, 5])
    xt = (pts[:, 0] - pts[:, 1] * pts[:, 4] * rcp) * bm.scxl
    yt = (pts[:, 2] - pts[:, 3] * pts[:, 4] * rcp) * bm.scxl
    r = np.sqrt(xt * xt + yt * yt)
    assert np.min(np.abs(r - rad)) > 1e-12     # no particle on the edge
    keep = r < rad
    b.close()
    assert got.shape == (int(keep.sum()), 9)
    assert np.array_equal(got[:, 6:], pts[keep, 6:])
    assert np.array_equal(got[:, [1, 3, 5]], pts[keep][:, [1, 3, 5]])
    assert np.max(np.abs(got[:, 0] - xt[keep]), initial=0.0) < 1e-14


@pytest.mark.parametrize("n,grid,period", [
    (5_592_405, (64, 64, 64), 2),    # rows of the cache's 256 MB: the last ordinary ones
    (5_592_406, (64, 64, 64), 2),    # the first read past it
    (5_592_999, (64, 64, 64), 1),    # scatters only, a ragged last block
])
def test_streamed_rows(gpu, n, grid, period):
    run_against_step(gpu, n, grid, period, steps=4)
