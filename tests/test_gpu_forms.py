"""The fused run's forms with one another: rows past the caches with the FP32
boxes, with push kinds read at run time and with losses; the kick from the
potential in the mixed form at the grid's edges; the lengths of the deposit's
chunks; izh_charge's global bins; the Green function on cells of other shapes;
recycled memory, column by column."""
import numpy as np
import pytest

from conftest import col_err, full_row_err
from test_gpu_memory import records
from test_gpu_parity import TOL

pytestmark = pytest.mark.gpu

STREAMED = 5_592_501         # past the 256 MB cache, a ragged last block


def lattice(kind, radius=1.0):
    from impactz import beam as B
    if kind == "solenoid":   # coupled maps, in the first pass too
        return [B.Element(0.2, 4, 10, 3, 2.0, 0.0, radius), B.Element(0.3, 4, 10, 0, radius)]
    if kind == "kmode":      # the K-mode quadrupole's chromatic map
        return [B.Element(0.1, 4, 10, 1, 8.0, -1.0, radius), B.Element(0.3, 4, 10, 0, radius)]
    return B.fodo(1, radius=radius)


def run_against_step(gpu, n, grid, period, kind, radius=1.0, steps=6):
    from impactz import beam as B
    from impactz.sim import Simulation
    print(f"forms: {n} particles, grid {grid}, period {period}, {kind}, {radius}", flush=True)
    pts = B.gaussian_bunch(n, seed=6)
    a = Simulation(pts, B.Beam(), lattice(kind, radius), grid)
    b = Simulation(pts, B.Beam(), lattice(kind, radius), grid)
    b.bunch.resort_period = period
    moms, rows = [], []
    for _, e in zip(range(steps), a.segments()):
        moms.append(a.step(e))
        rows.append(a.diag(moms[-1]))
    rec = b.run_fused(steps)
    assert b.bunch.nptlocal == a.bunch.nptlocal
    lost = n - b.bunch.nptlocal
    worst = max(full_row_err(b.diag(rec[k]), rows[k]) for k in range(steps))
    pe = col_err(b.bunch.getpts(), a.bunch.getpts())
    a.close()
    b.close()
    assert worst < TOL and pe < TOL, (worst, pe)
    return lost


@pytest.mark.parametrize("kind,period", [("solenoid", 1), ("solenoid", 3), ("kmode", 2)])
@pytest.mark.parametrize("n", [20_003, STREAMED])
def test_run_time_kinds(gpu, n, kind, period):
    run_against_step(gpu, n, (32, 32, 32) if n < 1e6 else (64, 64, 64), period, kind)


@pytest.mark.parametrize("n,grid,period", [(20_003, (32, 32, 32), 4), (20_003, (32, 32, 32), 1),
                                           (700_001, (32, 32, 32), 3),
                                           (STREAMED, (64, 64, 64), 4),
                                           (STREAMED, (64, 64, 64), 1)])
def test_losses(gpu, n, grid, period):
    """Particles lost in scatter passes and in place, in every form."""
    lost = run_against_step(gpu, n, grid, period, "fodo", radius=2.2e-3)
    assert 0.005 * n < lost < 0.5 * n


@pytest.mark.parametrize("n,grid,period,kind", [
    (70_001, (4, 4, 4), 2, "fodo"),          # from phi, every cell at an edge
    (9_001, (4, 16, 8), 1, "fodo"),
    (3_001, (128, 128, 128), 2, "solenoid"),  # from phi, run-time kinds
    (700_001, (32, 32, 32), 3, "fodo"),       # through boxes
    (700_001, (32, 32, 32), 3, "kmode"),
    (STREAMED, (64, 64, 64), 4, "fodo"),      # past the caches, three blocks a CU in place
    (STREAMED, (64, 64, 64), 2, "solenoid"),
])
def test_mixed_forms(gpu, n, grid, period, kind):
    """The mixed form against FP64.  Its FP32 transforms and positions put an
    error of at most 1e-5 of the largest E on a kick; over the steps each
    coordinate is off by that share of what space charge has done to it, which
    the same lattice without current measures.  1e-4 of that leaves a factor
    ten for the kicks' own compensation; a particle moved to another's slot, or
    a field from a wrong node, is off by orders of magnitude more."""
    from impactz import beam as B
    from impactz.sim import Simulation
    print(f"mixed: {n} particles, grid {grid}, period {period}, {kind}", flush=True)
    pts = B.gaussian_bunch(n, seed=6)
    out = []
    for current, prec in ((0.1, gpu.FP64), (0.1, gpu.MIXED), (0.0, gpu.FP64)):
        sim = Simulation(pts, B.Beam(current=current), lattice(kind), grid, precision=prec)
        sim.bunch.resort_period = period
        sim.run_fused(6)
        out.append(sim.bunch.getpts()[:, :6])
        sim.close()
    full, mixed, free = out
    kicked = np.max(np.abs(full - free), axis=0)
    # the phase is wrapped on the way: without current it is not
    kicked[4] = np.max(np.abs(np.angle(np.exp(1j * (full[:, 4] - free[:, 4])))))
    err = np.max(np.abs(mixed - full), axis=0)
    assert np.all(kicked > 0) and np.all(err < 1e-4 * kicked), err / kicked


@pytest.mark.parametrize("n", [524_287, 524_288, 1_048_575, 1_048_576, 2_097_151, 2_097_152,
                               4_194_303, 4_194_304])
def test_chunk_lengths(gpu, n):
    """Both sides of each bunch size where the deposit's chunks double, from
    1024 slots to 16384 (chunk_len)."""
    run_against_step(gpu, n, (32, 32, 32), 3, "fodo", steps=3)


@pytest.mark.parametrize("uniform", [True, False])
def test_charge_with_global_bins(gpu, uniform):
    """More than 8192 tiles even of 16 nodes: izh_charge counts and ranks its
    particles in global memory.  The bar of the other forms: 1e-13."""
    from impactz import beam as B
    n, grid = 5_000, (512, 512, 256)
    print(f"charge {n} {grid} uniform {uniform}", flush=True)
    pts = B.gaussian_bunch(n, seed=8)
    if not uniform:
        pts[:, 7] *= np.random.default_rng(9).uniform(0.5, 2.0, n)
    b = gpu.BeamBunch.from_beam(pts, B.Beam())
    f, d = gpu.FieldQuant(*grid), gpu.CompDom(*grid)
    pr, _, _ = b.conv1st(0.0, 1.0, 1.0)
    d.update(pr)
    for _ in range(2):
        b.charge(d, f)
    rho = f.download(gpu.RHO).ravel()
    p = b.getpts()
    f.close()
    b.close()
    lo, h = d.range[0::2], d.msize
    pos = p[:, [0, 2, 4]]
    i = ((pos - lo) * (1.0 / h) + 1.0).astype(np.int64)
    a = ((lo - pos) + i * h) * (1.0 / h)
    at, val = [], []
    for c in range(8):
        o = np.array([c & 1, (c >> 1) & 1, c >> 2])
        k = i - 1 + o
        at.append(k[:, 0] + grid[0] * (k[:, 1] + grid[1] * k[:, 2]))
        val.append(np.prod(np.where(o, 1.0 - a, a), axis=1) * p[:, 7])
    at, val = np.concatenate(at), np.concatenate(val)
    nodes, inv = np.unique(at, return_inverse=True)
    want = np.bincount(inv, weights=val)
    top = np.max(np.abs(want))
    assert np.max(np.abs(rho[nodes] - want)) < 1e-13 * top
    rho[nodes] = 0.0
    assert not rho.any()


@pytest.mark.parametrize("h", [(1.0, 1.0, 0.2), (1.0, 1.0, 4.0), (1.0, 4.0, 16.0),
                               (0.3, 1.0, 30.0)])
def test_green_function_of_cells(gpu, h):
    """phi of a unit charge on the first node is the Green function itself, the
    mean of 1/r over a cell, here by Gauss's rule: near the origin from the
    corners, elsewhere from the series (525 thousand nodes).  Off by
    - the series' truncation, at most 1.5e-12 (test_green_series.py);
    - near the origin, the corners' rounding: 48 terms of up to 7 r^2 / volume,
      each rounded twice to 1.1e-16, come to 7.4e-14 r^2 / volume;
    - the transforms' rounding: three of 22 stages, 1e-14 of the largest value
      at most."""
    grid = (64, 64, 128)
    print(f"green {h}", flush=True)
    h = np.array(h) * 1e-3
    rho = np.zeros(grid[::-1])
    rho[0, 0, 0] = 1.0
    f, d = gpu.FieldQuant(*grid), gpu.CompDom(*grid)
    d.set([0, h[0] * (grid[0] - 1), 0, h[1] * (grid[1] - 1), 0, h[2] * (grid[2] - 1)], h)
    f.upload_rho(rho)
    f.update3O(d)
    phi = f.download(gpu.PHI)
    f.close()
    rng = np.random.default_rng(2)
    ijk = np.stack([rng.integers(0, n, 4000) for n in grid], axis=1)
    # whole axes and the box's surroundings; 3 half diagonals away Gauss's 16
    # points per axis are exact to rounding
    ijk = np.vstack([ijk] + [np.eye(3, dtype=int)[a] * np.arange(grid[a])[:, None]
                             for a in range(3)] + [rng.integers(0, 24, (2000, 3))])
    pos = ijk * h
    r = np.linalg.norm(pos, axis=1)
    far = r > 3 * np.linalg.norm(h) / 2
    ijk, pos = ijk[far], pos[far]
    t, w = np.polynomial.legendre.leggauss(16)
    t, w = t / 2, w / 2
    want = np.zeros(len(pos))
    for i in range(16):
        for j in range(16):
            rho2 = (pos[:, 0] + t[i] * h[0]) ** 2 + (pos[:, 1] + t[j] * h[1]) ** 2
            zz = pos[:, 2, None] + t * h[2]
            want += w[i] * w[j] * np.sum(w / np.sqrt(rho2[:, None] + zz * zz), axis=1)
    got = phi[ijk[:, 2], ijk[:, 1], ijk[:, 0]]
    reach = 12.0 * np.linalg.norm(h) / 2
    near = np.all(pos <= reach, axis=1)
    corner = np.where(near, 7.4e-14 * np.sum(pos * pos, axis=1) / np.prod(h), 0.0)
    assert np.sum(near) > 300 and np.sum(~near) > 300
    err = np.abs(got - want)
    assert np.all(err < 1.5e-12 * want + corner + 1e-14 * phi[0, 0, 0]), np.max(err / want)


def test_recycled_blocks_change_no_column(gpu):
    """Records from recycled blocks against those from fresh ones, each column
    on its own scale."""
    from impactz import beam as B
    pool = gpu.BeamBunch.from_beam(B.gaussian_bunch(60_000, seed=3), B.Beam())
    cases = [(60_000, (32, 32, 32), gpu.FP64), (20_001, (16, 64, 16), gpu.MIXED),
             (58_000, (32, 32, 32), gpu.FP64), (59_999, (64, 32, 16), gpu.MIXED)]
    first = []
    for c in cases:
        gpu.memory_trim()
        first.append(records(gpu, pool, *c))
    assert gpu.memory_info()[1] > 0
    for k in (2, 0, 3, 1, 0):
        again = records(gpu, pool, *cases[k])
        scale = np.max(np.abs(first[k]), axis=0)
        # first and odd moments are sums that cancel: on the scale of their
        # terms, the maximum of the coordinates times the particles
        amax = np.max(first[k][:, 37:43], axis=0)
        n = cases[k][0]
        for q, powers in enumerate(MOMENT_POWERS):
            scale[q] = max(scale[q], n * np.prod(amax ** np.array(powers)))
        assert np.all(np.abs(again - first[k]) <= TOL * scale), k
    pool.close()


def _powers(**kw):
    return [kw.get(c, 0) for c in ("x", "px", "y", "py", "z", "pz")]


# the powers of (x, px, y, py, z, pz) in the record's 37 sums
MOMENT_POWERS = (
    [_powers(**{c: 1}) for c in ("x", "px", "y", "py", "z", "pz")]
    + [_powers(**{c: 2}) for c in ("x", "px", "y", "py", "z", "pz")]
    + [_powers(x=1, px=1), _powers(y=1, py=1), _powers(z=1, pz=1)]
    + [_powers(**{c: k}) for c in ("x", "px", "y", "py", "z", "pz") for k in (3, 4)]
    + [_powers(**{u: a, p: b}) for u, p in (("x", "px"), ("y", "py"))
       for a, b in ((1, 2), (1, 3), (2, 1), (2, 2), (3, 1))])
