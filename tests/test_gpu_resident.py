"""Sweeps of small systems in one launch (a system per workgroup, in LDS):
the trajectory, counters and errors of the oracle's restatement and of the
launched kernels, over the shapes the kernel treats apart."""
import ctypes as C

import numpy as np
import pytest

from hsmc_amd import gpu
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _melted(shape, rho, seed, drop=0):
    """fcc cells `shape` at density rho with `drop` vacancies, melted by the
    oracle: configuration and box."""
    conf, box = gpu.lattice(2, shape, rho)
    conf = conf[drop:].copy()
    conf[:, 0] = np.arange(len(conf))
    cb = O.Checkerboard(conf, box, tuple(int(L / (1 + 1e-9)) // 2 * 2 for L in box), 0.3, seed)
    cb.sweeps(20)
    return cb.config(), box


# (fcc cells, density, vacancies): 8 cells a phase and 32 lanes each; a 2-cell
# axis (each neighbour cell met once); N = 1; wide cells of 16 slots; unequal edges; 64 and 80 cells a phase and 16
# lanes each, with more spheres than threads of one pass
CASES = [((3, 3, 3), 0.93, 0), ((1, 4, 4), 0.375, 0), ((1, 4, 4), 0.375, 63), ((4, 4, 4), 0.70, 1), ((5, 5, 5), 0.30, 3),
         ((3, 4, 5), 0.60, 0), ((5, 5, 5), 0.85, 0), ((4, 5, 6), 0.88, 7), ((2, 2, 6), 0.42, 2)]


@pytest.mark.parametrize("shape,rho,drop", CASES)
@pytest.mark.parametrize("sweeps", [1, 65])
def test_resident_sweeps_match_oracle(shape, rho, drop, sweeps):
    conf, box = _melted(shape, rho, 3, drop)
    ctx = gpu.Context([dict(n=len(conf), box=box, dr_max=0.2, seed=11)])
    ctx.upload(conf)
    cb = O.Checkerboard(conf, box, ctx.grid(), 0.2, 11)
    for n in (sweeps, 1, 2):
        ctx.sweeps(n)
        cb.sweeps(n)
        assert np.array_equal(ctx.download(), cb.config()), n
    c = ctx.counters()
    assert (c["attempts"], c["accepted"], c["left_cell"], c["sweeps"]) == \
        tuple(int(v) for v in cb.counters())
    ctx.close()


def test_resident_replicas_equal_launched_and_alone():
    """A batch of uneven systems: resident (the default) against launched
    phases, switching between the two in mid-run, and against each replica
    alone; counters included."""
    systems = [_melted(s, r, 5 + k, d) for k, (s, r, d) in enumerate(CASES)]
    reps = [dict(n=len(c), box=b, dr_max=0.15, seed=70 + k) for k, (c, b) in enumerate(systems)]

    def make(which):
        ctx = gpu.Context([reps[k] for k in which])
        for r, k in enumerate(which):
            ctx.upload(systems[k][0], r)
        return ctx

    everyone = range(len(reps))
    launched = make(everyone)
    launched.set_tuning(32, 4, 8)
    launched.sweeps(101)
    mixed = make(everyone)
    mixed.sweeps(33)           # resident; odd, so the launched count buffers change places
    mixed.set_tuning(32, 4, 8)
    mixed.sweeps(68)
    resident = make(everyone)
    resident.sweeps(101)
    for k in everyone:
        want = launched.download(k), launched.counters(k)
        alone = make([k])
        alone.sweeps(101)
        for ctx, r in ((mixed, k), (resident, k), (alone, 0)):
            assert np.array_equal(ctx.download(r), want[0]), k
            assert ctx.counters(r) == want[1], k
        alone.close()
    # the volume-move scan reads a cell list the resident kernel does not leave
    for sf in (1.0, 0.999, 0.99):
        assert np.array_equal(resident.any_overlap_scaled_batch(sf), launched.any_overlap_scaled_batch(sf))
    for ctx in (launched, mixed, resident):
        ctx.close()


@pytest.mark.parametrize("tuned", [False, True])
def test_sweep_counter_moved_by_an_odd_number(tuned):
    """Sweeps after the counter moves by an odd number equal those of a fresh
    context at that counter (launched sweeps fill the other count buffer)."""
    conf, box = _melted((4, 4, 4), 0.8, 9)
    outs = []
    for warm in (4, 0):
        ctx = gpu.Context([dict(n=len(conf), box=box, dr_max=0.1, seed=3)])
        if tuned:
            ctx.set_tuning(32, 2, 0)
        ctx.upload(conf)
        ctx.sweeps(warm)
        ctx.upload(conf)
        ctx.set_sweep_counter(1001)
        ctx.sweeps(7)
        outs.append(ctx.download())
        ctx.close()
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("tuned", [False, True])
def test_overfull_cells_are_reported(tuned):
    """More spheres in a cell than it holds: the same error either way, and
    other contexts go on."""
    box = (6.5, 6.5, 6.5)
    rng = np.random.default_rng(2)
    conf = np.zeros((200, 4))
    conf[:, 0] = np.arange(200)
    conf[:, 1:] = rng.random((200, 3)) * np.array(box)
    conf[:60, 1:] = 3.0 + 0.1 * rng.random((60, 3))
    ctx = gpu.Context([dict(n=200, box=box, dr_max=0.1, seed=3)])
    if tuned:
        ctx.set_tuning(32, 2, 0)
    ctx.upload(conf)
    with pytest.raises(gpu.HsmcError) as e:
        ctx.sweeps(1)
        ctx.sync()
    assert e.value.code == -1
    good, gbox = _melted((3, 3, 3), 0.45, 4)
    other = gpu.Context([dict(n=len(good), box=gbox, dr_max=0.1, seed=3)])
    other.upload(good)
    other.sweeps(3)
    other.sync()
    other.close()
    ctx.close()


@pytest.mark.parametrize("calls,fold", [((60, 60, 60), 100), ((9000,), 5000)])
def test_counters_across_a_fold_between_launches(calls, fold):
    """The 32-bit counters are folded into the totals before they could
    overflow (every 2^24 sweeps; lowered here): sweeps launched after that,
    in the same call, count too, and a reset takes them along."""
    systems = [_melted((3, 3, 3), 0.7, 6), _melted((2, 2, 6), 0.42, 7)]
    reps = [dict(n=len(c), box=b, dr_max=0.15, seed=40 + k) for k, (c, b) in enumerate(systems)]
    ctxs = [gpu.Context(reps) for _ in range(2)]
    resident, launched = ctxs
    launched.set_tuning(32, 4, 64)
    assert gpu.load().hsmc_gpu_test_fold_sweeps(resident.h, C.c_uint64(fold)) == 0
    for ctx in ctxs:
        for r, (conf, _) in enumerate(systems):
            ctx.upload(conf, r)
        for n in calls:
            ctx.sweeps(n)
    for r in (0, 1):
        assert resident.counters(r) == launched.counters(r), r
    for ctx in ctxs:
        for n in calls:
            ctx.sweeps(n)
        ctx.reset_counters()
        ctx.sweeps(3)
    for r in (0, 1):
        assert resident.counters(r) == launched.counters(r), r
    for ctx in ctxs:
        ctx.close()
