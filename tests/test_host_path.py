"""The library's host side on the CPU, over a HIP runtime that queues work and
launches nothing (fake_hip.cpp): what is still queued when a failed call
returns, what is launched and allocated, and what becomes of device memory."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

HERE = os.path.dirname(os.path.abspath(__file__))

PREAMBLE = """
import ctypes as C, sys, threading
sys.path.insert(0, {pkg!r})
fake = C.CDLL({fake!r}, mode=C.RTLD_GLOBAL)
fake.fake_pending.restype = fake.fake_launches.restype = C.c_int64
fake.fake_held.restype = fake.fake_peak.restype = C.c_size_t
fake.fake_capacity.argtypes = fake.fake_fail_alloc.argtypes = [C.c_size_t]
fake.fake_poke.argtypes = [C.c_size_t, C.c_size_t, C.c_int64]
from impactz import beam as B, hip
import numpy as np
hip.init(0)
BEAM = B.Beam()

def bunch(n, precision=hip.FP64):
    return hip.BeamBunch.from_beam(B.gaussian_bunch(n, seed=1), BEAM, precision)

def drift():
    return hip.segment(0.05, 0, 0.0, 10, 1.0, 1.0, 0.1, 0.0)

def refused(call, text=''):
    try:
        call()
    except hip.IZHError as e:
        assert text in str(e), str(e)
        return
    raise AssertionError('accepted')

def answered(steps):
    # a run's results come as one copy of the 11 words it keeps on the device
    fake.fake_poke(88, 80, steps)
"""


@pytest.fixture(scope="session")
def fake_hip(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-pthread",
                           os.path.join(HERE, "fake_hip.cpp"), "-o", lib])

    def run(script):
        head = PREAMBLE.format(pkg=os.path.join(ROOT, "impact-z_amd"), fake=lib)
        r = subprocess.run([sys.executable, "-c", head + script], capture_output=True, text=True,
                           timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr

    return run


@pytest.mark.parametrize("kernel", ["k_pass", "k_finalize", "k_deposit_tiles", "k_fft_two",
                                    "k_efield"])
def test_failed_run_leaves_nothing_queued(fake_hip, kernel):
    """After a run that fails on the way, the field's stream is its own again:
    nothing may be queued on the bunch's by then, or the field's buffers could
    pass to another owner while kernels still use them."""
    fake_hip(f"""
b = bunch(600_000)          # gathers E through a box, so every step has its E kernel
f, d = hip.FieldQuant(32, 32, 32), hip.CompDom(32, 32, 32)
fake.fake_fail_kernel({kernel.encode()!r})
refused(lambda: b.run(f, d, 0.0, [drift()] * 4, BEAM.current), 'injected')
assert fake.fake_launches({kernel.encode()!r}) == 1
assert fake.fake_pending() == 0, fake.fake_pending()
f.close()
b.close()
""")


@pytest.mark.parametrize("kernel", ["k_prologue_keys", "k_pass", "k_fft_two"])
def test_failed_job_leaves_nothing_queued(fake_hip, kernel):
    fake_hip(f"""
b = bunch(5_000)
f, d = hip.FieldQuant(16, 16, 16), hip.CompDom(16, 16, 16)
fake.fake_fail_kernel({kernel.encode()!r})
refused(lambda: hip.Job(b, f, d, 0.0, [drift()], 8, BEAM.current), 'injected')
assert fake.fake_pending() == 0, fake.fake_pending()
job = hip.Job(b, f, d, 0.0, [drift()], 8, BEAM.current, False)
job.advance(3)
fake.fake_fail_kernel(b'k_deposit_tiles')
refused(lambda: job.advance(3), 'injected')
job.close()
assert fake.fake_pending() == 0, fake.fake_pending()
f.close()
b.close()
""")


@pytest.mark.parametrize("cavity,why", [
    ("hip.segment(0.05, 103, [1e6, 324e6, 0, 1, 1], 10, 1.0, 1.0, 0.1, 0.0)", "needs its field"),
    ("hip.segment(0.05, 105, [1e6, 324e6, 0, 1, 1], 10, 1.0, 1.0, 0.1, 0.0, TABLE)", "Fourier"),
    ("hip.segment(0.05, 101, [1e6, 324e6, 0, 1, 1], 10, 1.0, 1.0, 0.1, 0.0, SERIES)", "table"),
    ("hip.segment(0.05, 102, [1e6, 0.0, 0, 1, 1], 10, 1.0, 1.0, 0.1, 0.0, TABLE)", "frequency"),
])
def test_run_refuses_a_cavity_before_it_starts(fake_hip, cavity, why):
    """A cavity in mid-lattice that has no usable field is refused with the
    bunch as it was, not after the steps before it."""
    fake_hip(f"""
TABLE = hip.RFData(np.array([[0.0, 1.0, 0.0, 0.0], [1.0, 1.0, 0.0, 0.0]]), fourier=False)
SERIES = hip.RFData(np.array([5.0, 0.0, 1.0, 1.0, 0.5, 0.2, 0.1, 0.1, 0.1]), fourier=True)
b = bunch(2_000)
f, d = hip.FieldQuant(16, 16, 16), hip.CompDom(16, 16, 16)
before = list(b.info().refpt)
fake.fake_forget_launches()
for current in (BEAM.current, 0.0):
    refused(lambda: b.run(f, d, 0.0, [drift(), drift(), {cavity}], current), {why!r})
assert fake.fake_launches(b'') == 0 and list(b.info().refpt) == before
f.close()
b.close()
""")


@pytest.mark.parametrize("n,kernel", [(100, "k_deposit_direct"), (5_000, "k_deposit_small"),
                                      (5_000, "k_fx_to_grid"), (5_000, "k_wake_field")])
def test_failed_call_on_the_field_leaves_the_bunch_free(fake_hip, n, kernel):
    """Kernels on the field's stream read the bunch's rows: after a call that
    fails, ending the bunch alone must find them done."""
    fake_hip(f"""
b = bunch({n})
f, d = hip.FieldQuant(16, 16, 16), hip.CompDom(16, 16, 16)
b.conv1st(0.05, 1.0, 1.0)
d.set([0, 1, 0, 1, 0, 1], [1 / 15] * 3)
w = hip.wake(1, 0.01, 0.02, 0.03)
fake.fake_fail_kernel({kernel.encode()!r})

def calls():
    b.wakefield(f, d, w)
    b.charge(d, f)
refused(calls, 'injected')
b.close()
assert fake.fake_pending() == 0, fake.fake_pending()
f.close()
""")


@pytest.mark.parametrize("kernel", ["k_gather_kick", "k_kick2"])
def test_failed_kick_leaves_the_field_free(fake_hip, kernel):
    """And kernels on the bunch's stream read the field's E."""
    fake_hip(f"""
b = bunch(5_000)
f, d = hip.FieldQuant(16, 16, 16), hip.CompDom(16, 16, 16)
b.conv1st(0.05, 1.0, 1.0)
d.set([0, 1, 0, 1, 0, 1], [1 / 15] * 3)
b.charge(d, f)
f.update3O(d)
b.cvbkforth1st()
fake.fake_fail_kernel({kernel.encode()!r})
if {kernel!r} == 'k_kick2':
    refused(lambda: b.kick2(0.0, 0.05, hip.element(0, 0.0, 0.1), f, d), 'injected')
else:
    refused(lambda: b.kick1(0.05, f, d), 'injected')
f.close()
assert fake.fake_pending() == 0, fake.fake_pending()
b.close()
""")


@pytest.mark.parametrize("kernel", ["k_deposit_small", "k_fx_to_grid"])
def test_charge_after_a_failed_one_starts_clean(fake_hip, kernel):
    """The accumulator is cleared by whatever reads it; a deposit that no call
    read must not add to the next one."""
    fake_hip(f"""
b = bunch(5_000)
f, d = hip.FieldQuant(16, 16, 16), hip.CompDom(16, 16, 16)
b.conv1st(0.05, 1.0, 1.0)
d.set([0, 1, 0, 1, 0, 1], [1 / 15] * 3)
b.charge(d, f)
assert fake.fake_launches(b'k_fill_u32') == 0
fake.fake_fail_kernel({kernel.encode()!r})
refused(lambda: b.charge(d, f), 'injected')
b.charge(d, f)
b.charge(d, f)
assert fake.fake_launches(b'k_fill_u32') == 1
""")


@pytest.mark.parametrize("kernel", ["k_deposit_tiles", "k_fft_two"])
def test_deposit_after_a_failed_run_starts_clean(fake_hip, kernel):
    fake_hip(f"""
b = bunch(5_000)
f, d = hip.FieldQuant(16, 16, 16), hip.CompDom(16, 16, 16)
fake.fake_fail_kernel({kernel.encode()!r})
refused(lambda: b.run(f, d, 0.0, [drift()] * 3, BEAM.current), 'injected')
assert fake.fake_launches(b'k_fill_u32') == 0
answered(3)
b.run(f, d, 0.0, [drift()] * 3, BEAM.current)
assert fake.fake_launches(b'k_fill_u32') == 1
b.run(f, d, 0.0, [drift()] * 3, BEAM.current)
assert fake.fake_launches(b'k_fill_u32') == 1
""")


def test_run_after_its_sort_state_was_lost_starts_afresh(fake_hip):
    """A run on a larger grid that finds no memory for its tile lists has
    already given up the smaller ones: the next run on the first field may not
    start from them."""
    fake_hip("""
b = bunch(5_000)
f, d = hip.FieldQuant(16, 16, 16), hip.CompDom(16, 16, 16)
g, e = hip.FieldQuant(64, 64, 64), hip.CompDom(64, 64, 64)
answered(2)
b.run(f, d, 0.0, [drift()] * 2, BEAM.current)
b.run(f, d, 0.0, [drift()] * 2, BEAM.current)
assert fake.fake_launches(b'k_prologue_keys') == 1      # the second started warm
for lost in (1, 2):
    fake.fake_fail_alloc(4 * 512)                       # the cursors of 512 tiles
    refused(lambda: b.run(g, e, 0.0, [drift()] * 2, BEAM.current))
    fake.fake_fail_alloc(0)
    b.run(f, d, 0.0, [drift()] * 2, BEAM.current)
    assert fake.fake_launches(b'k_prologue_keys') == 1 + lost
""")


def test_memory_another_thread_gives_back_is_waited_for(fake_hip):
    """Kept blocks fill the device.  The first thread that finds no memory takes
    them all and frees them; the others wait for that instead of failing."""
    fake_hip("""
b = bunch(1_000)
f = hip.FieldQuant(64, 64, 64)
before = fake.fake_held()
f.close()
assert fake.fake_held() == before                       # all of it kept
# room for the two smaller fields, but not beside what is kept
fake.fake_capacity(before + (1 << 20))
fake.fake_free_delay(20)
fields, errors, gate = [], [], threading.Barrier(2)

def make(grid):
    gate.wait()
    try:
        fields.append(hip.FieldQuant(*grid))
    except hip.IZHError as e:
        errors.append(str(e))

for _ in range(3):
    threads = [threading.Thread(target=make, args=(g,)) for g in ((32, 32, 64), (32, 64, 32))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    while fields:
        fields.pop().close()
    # every block of the 64^3 grid again
    fake.fake_free_delay(0)
    f = hip.FieldQuant(64, 64, 64)
    f.close()
    fake.fake_free_delay(20)
b.close()
""")


@pytest.mark.parametrize("call", ["b.wakefield(f, d, hip.wake(2, table=TABLE, scale=1.0))",
                                  "hip.probe_copy(3 << 20)"])
def test_kept_memory_is_no_obstacle_to_other_allocations(fake_hip, call):
    """A wake's table and the copy probe find room where kept blocks fill the
    device, and give their own memory back."""
    fake_hip(f"""
z = np.linspace(0.0, 1.0, 1000)
TABLE = hip.RFData(np.stack([z, z, z, z], axis=1), fourier=False)
b = bunch(1_000)
f, d = hip.FieldQuant(16, 16, 16), hip.CompDom(16, 16, 16)
b.conv1st(0.05, 1.0, 1.0)
d.set([0, 1, 0, 1, 0, 1], [1 / 15] * 3)
b.wakefield(f, d, hip.wake(1, 0.01, 0.02, 0.03))        # the field's own wake lines
held = fake.fake_held()
hip.FieldQuant(64, 64, 64).close()
assert fake.fake_held() > held                          # kept
fake.fake_capacity(fake.fake_held())
{call}
f.close()
b.close()
TABLE.close()
assert fake.fake_held() == 0, fake.fake_held()
""")


def test_memory_info_and_trim(fake_hip):
    fake_hip("""
assert hip.memory_info() == (0, 0)
b = bunch(1_000)
used, kept = hip.memory_info()
assert used == fake.fake_held() and kept == 0
hip.FieldQuant(32, 32, 32).close()
after, kept = hip.memory_info()
assert after == used and kept > 0 and used + kept == fake.fake_held()
hip.memory_trim()
assert hip.memory_info() == (used, 0) and fake.fake_held() == used
# another allocation of the package finds what the library keeps
hip.DeviceDoubles._rt = fake
fake.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
fake.hipFree.argtypes = [C.c_void_p]
hip.FieldQuant(32, 32, 32).close()
fake.fake_capacity(fake.fake_held() + 1000)
hip.DeviceDoubles(1000).close()
b.close()
assert hip.memory_info() == (0, 0)
""")


@pytest.mark.parametrize("n,grid,form", [(1_000_000, (64, 64, 64), "MIXED"),
                                         (20_001, (16, 32, 64), "FP64"),
                                         (300_007, (128, 64, 32), "FP64"),
                                         (5_000, (32, 32, 32), "MIXED"),
                                         (2_500_000, (32, 32, 32), "FP64")])
def test_footprint_is_what_a_job_holds(fake_hip, n, grid, form):
    """The admission footprint bounds a job's device memory."""
    fake_hip(f"""
from impactz import scan
pool = scan.Pool({n})
r = scan.Request({n}, {grid}, 40, 10.0, hip.{form})
base = hip.memory_info()[0]
lv = scan.Live(r, pool, use_graph=False)
held = hip.memory_info()[0] - base
need = scan.footprint(r.n, r.grid, r.precision, r.steps)
assert held <= need <= 1.1 * held + (1 << 20), (held, need)
lv.close()
pool.close()
""")


def test_serve_keeps_to_its_budget(fake_hip):
    """Jobs and the buffers kept of finished ones stay within the budget."""
    fake_hip("""
from impactz import scan
pool = scan.Pool(60_000)
reqs = [scan.Request(n, g, 6, 10.0, hip.FP64)
        for n, g in ((10_000, (32, 32, 32)), (60_000, (16, 16, 32)), (30_000, (16, 32, 32)),
                     (50_000, (32, 32, 32)), (20_000, (32, 16, 16)), (37_000, (32, 32, 32)))]
base = fake.fake_held()
budget = int(1.5 * max(scan.footprint(r.n, r.grid, r.precision) for r in reqs))
answered(6)
out = scan.serve(reqs, pool, budget, use_graph=False, policy="fifo")
assert out["requests"] == 6 and out["peak_bytes"] <= budget
assert fake.fake_peak() - base <= budget, (fake.fake_peak() - base, budget)
pool.close()
""")


def test_new_domain_finds_the_field_of_the_last_run(fake_hip):
    """A run that stops on the way may leave a potential without its E, which
    needs the domain both belong to: it is formed before another one is set."""
    fake_hip("""
b = bunch(5_000)            # kicks from the potential
f, d = hip.FieldQuant(16, 16, 16), hip.CompDom(16, 16, 16)
job = hip.Job(b, f, d, 0.0, [drift()], 8, BEAM.current, False)
job.advance(3)
job.close()
assert fake.fake_launches(b'k_efield') == 0
d.set([0, 1, 0, 1, 0, 1], [1 / 15] * 3)
f.upload_rho(np.ones((16, 16, 16)))
f.update3O(d)
assert fake.fake_launches(b'k_efield') == 1
f.download(hip.EX)
assert fake.fake_launches(b'k_efield') == 1
""")


def test_kept_memory_stays_within_its_bound(fake_hip):
    """A field of more than 8 GiB ends: the oldest of its blocks go back, what
    is kept stays below the bound but close to it, and the next field takes it."""
    fake_hip("""
b = bunch(1_000)
base = hip.memory_info()[0]
sizes = []
for grid in ((512, 512, 256), (512, 512, 256), (256, 512, 512)):
    f = hip.FieldQuant(*grid)
    used = hip.memory_info()[0] - base
    f.close()
    held, kept = hip.memory_info()
    assert used > 8 << 30 and held == base
    assert (7 << 30) < kept <= (8 << 30) and fake.fake_held() == base + kept, kept
b.close()
assert fake.fake_held() == 0
""")


def test_run_starts_warm_only_on_what_its_last_run_left(fake_hip):
    """The sort state of a run goes with the key grids in its field: a field made
    at the place of one that has ended, and a field whose domain another bunch
    has set, hold other ones."""
    fake_hip("""
def cold():
    before = fake.fake_launches(b'k_prologue_keys')
    b.run(f, d, 0.0, [drift()] * 2, BEAM.current)
    return fake.fake_launches(b'k_prologue_keys') - before

b, other = bunch(5_000), bunch(6_000)
f, d = hip.FieldQuant(16, 16, 16), hip.CompDom(16, 16, 16)
answered(2)
assert cold() and not cold() and not cold()
for _ in range(5):
    f.close()
    f = hip.FieldQuant(16, 16, 16)
    assert cold() and not cold()
other.run(f, d, 0.0, [drift()] * 2, BEAM.current)
assert cold() and not cold()
other.conv1st(0.05, 1.0, 1.0)
d.set([0, 1, 0, 1, 0, 1], [1 / 15] * 3)
other.charge(d, f)
assert cold() and not cold()
""")
