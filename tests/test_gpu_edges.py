"""Edge cases and error paths of the device layer: empty queries, arguments
out of range, and the conditions the reference turns into print-and-exit
(cell_list.c:126-129 cells narrower than a diameter, cell_list.c:229-232 a
cell over max_part).  Every error is a status code; the context stays usable
after it."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from hsmc_amd import gpu
from oracle import oracle as O

pytestmark = pytest.mark.gpu

BAD_ARG, CELL_OVERFLOW, CELL_TOO_SMALL, NOT_SUPPORTED = -5, -1, -2, -8


def _code(fn):
    with pytest.raises(gpu.HsmcError) as e:
        fn()
    return e.value.code


@pytest.fixture(scope="module")
def sys500():
    o = O.System(2, 5, rho=0.5, neigh_dr=1.0, max_part=10, seed=1)
    conf = o.config()
    L = o.box()["lx"]
    ctx = gpu.Context([dict(n=len(conf), box=(L, L, L), dr_max=0.1, seed=3)])
    ctx.upload(conf)
    yield ctx, conf, L
    ctx.close()


def test_box_limits():
    # a 2-cell sweep grid needs an edge above 2 diameters, and cells narrower
    # than 1.5 (edges in [3, 4) would give cells of 1.5 to 2)
    assert _code(lambda: gpu.Context([dict(n=4, box=(1.9, 5.0, 5.0))])) == BAD_ARG
    assert _code(lambda: gpu.Context([dict(n=8, box=(3.5, 6.0, 6.0))])) == NOT_SUPPORTED
    ctx = gpu.Context([dict(n=8, box=(2.9, 4.1, 6.2))])   # cells 1.45, 1.025, 1.033
    assert ctx.grid() == (2, 4, 6)
    ctx.close()


def test_empty_queries(sys500):
    ctx, conf, L = sys500
    assert len(ctx.overlap_batch(np.zeros(0, np.int32), np.zeros((0, 3)))) == 0
    assert len(ctx.widom_points(np.zeros((0, 3)))) == 0
    assert len(ctx.pair_dist(np.zeros(0, np.int32), np.zeros(0, np.int32))) == 0
    assert ctx.widom_uniform(1, 0, 0, 0) == 0
    ctx.sweeps(0)
    counts = ctx.npt_sweeps(0, 3.0, 0.01)
    assert counts.sum() == 0
    assert np.array_equal(ctx.download(), conf)


def test_arguments_out_of_range(sys500):
    ctx, conf, L = sys500
    bad = conf.copy()
    bad[7, 2] = L + 0.5
    assert _code(lambda: ctx.upload(bad)) == BAD_ARG
    assert _code(lambda: ctx.rdf_counts(0.01, 400, L / 2 + 0.5)) == BAD_ARG   # beyond minimum image
    assert _code(lambda: ctx.any_overlap_scaled(np.full(65, 0.99))) == BAD_ARG   # at most 64 factors
    assert _code(lambda: ctx.set_tuning(48, 2, 0)) == BAD_ARG
    assert _code(lambda: ctx.set_tuning(32, 3, 0)) == BAD_ARG   # cells per workgroup: 1, 2, 4 or 8
    assert _code(lambda: ctx.set_tuning(64, 8, 0)) == BAD_ARG   # at most 256 lanes
    assert _code(lambda: ctx.npt_sweeps(1, -1.0, 0.01)) == BAD_ARG
    assert _code(lambda: ctx.npt_sweeps(1, 3.0, 0.0)) == BAD_ARG
    assert _code(lambda: ctx.overlap_batch(np.array([len(conf)], np.int32), np.zeros((1, 3)))) == BAD_ARG
    assert _code(lambda: ctx.box(1)) == BAD_ARG   # one replica only
    net = gpu.Mlp(ctx, seed=1)
    assert _code(lambda: net.widom(0.25, 1.0, 1, 0, 1000)) == BAD_ARG   # mix must be below 1
    net.close()
    # nothing above changed the configuration
    assert np.array_equal(ctx.download(), conf)


def test_reference_exit_conditions(sys500):
    ctx, conf, L = sys500
    # cells narrower than a diameter (cell_list.c:126-129)
    assert _code(lambda: ctx.cell_list((11, 10, 10), 10)) == CELL_TOO_SMALL
    # a cell with more occupants than max_part - 1 (cell_list.c:229-232):
    # 500 spheres in 27 cells of side 3.33
    assert _code(lambda: ctx.cell_list((3, 3, 3), 10)) == CELL_OVERFLOW
    # the context is usable afterwards
    pc, nm = ctx.cell_list((10, 10, 10), 10)
    assert pc[:, 0].sum() == len(conf)
    ctx.sweeps(5)
    ctx.sync()
    assert ctx.any_overlap_scaled([1.0])[0] == 1


@pytest.mark.parametrize("n", [1, 255, 32768, 32769, 65536, 65537, 100001])
def test_rows_in_transit(n):
    """Configurations cross in chunks of 32768 rows through two buffers: every
    row arrives, up and down, as it was, beside another replica's."""
    L = max(5.0, (n / 0.3) ** (1 / 3))
    rng = np.random.default_rng(n)
    conf = np.zeros((n, 4))
    conf[:, 0] = np.arange(n)
    conf[:, 1:] = rng.random((n, 3)) * L
    other = conf[:300].copy()
    ctx = gpu.Context([dict(n=len(other), box=(L, L, L)), dict(n=n, box=(L, L, L))])
    ctx.upload(other, 0)
    ctx.upload(conf, 1)
    assert np.array_equal(ctx.download(1), conf)
    assert np.array_equal(ctx.download(0), other)
    bad = conf.copy()
    bad[n - 1, 3] = L * 1.001
    assert _code(lambda: ctx.upload(bad, 1)) == BAD_ARG
    assert np.array_equal(ctx.download(1), conf)   # a refused upload changes nothing
    ctx.close()


def test_counters_are_current_after_every_kind_of_sweep():
    """Counters read between sweeps, resets, tuning and box changes: attempts
    are N per sweep and what was counted before is kept."""
    conf, box = gpu.lattice(2, 5, 0.7)
    ctx = gpu.Context([dict(n=500, box=box, dr_max=0.1, seed=r) for r in (1, 2)])
    for r in (0, 1):
        ctx.upload(conf, r)
    total, last = 0, [0, 0]
    for step in (lambda: ctx.sweeps(3), lambda: ctx.sweeps(70), lambda: ctx.time_phase_kernel(2),
                 lambda: ctx.set_tuning(32, 2, 4), lambda: ctx.sweeps(9), lambda: ctx.time_sweeps(5),
                 lambda: ctx.npt_sweeps(3, 4.0, 0.01), lambda: ctx.scale(1.01, [1.01 * b for b in ctx.box(0)], 0),
                 lambda: ctx.autotune(8), lambda: ctx.sweeps(1)):
        before = ctx.counters(1)["sweeps"]
        step()
        for r in (0, 1):
            c = ctx.counters(r)
            assert c == ctx.counters(r)
            assert c["attempts"] == 500 * c["sweeps"] and c["sweeps"] >= before
            assert last[r] <= c["accepted"] <= c["attempts"]
            assert (c["accepted"] > last[r]) == (c["sweeps"] > before)
            last[r] = c["accepted"]
    sweeps = ctx.counters()["sweeps"]
    assert sweeps == 3 + 70 + 2 + 9 + 5 + 3 + 1
    ctx.reset_counters()
    ctx.sweeps(2)
    assert ctx.counters()["attempts"] == 1000 and ctx.counters()["sweeps"] == sweeps + 2
    ctx.close()


def _wide_steps(reps, confs, tuning):
    ctx = gpu.Context(reps)
    for r, c in enumerate(confs):
        ctx.upload(c, r)
    if tuning:
        ctx.set_tuning(*tuning)
    out = []
    for _ in range(20):
        ctx.sweeps(50)
        out += [ctx.download(r) for r in range(len(reps))]
    return ctx, out, [ctx.counters(r) for r in range(len(reps))], \
        [ctx.any_overlap_scaled_batch(sf).tolist() for sf in (0.99, 0.9)]


@pytest.mark.parametrize("replicas", [1, 3])
def test_steps_of_many_box_edges(replicas):
    """Steps of up to 5 box edges either way leave spheres far outside the box
    and left of the sweep grid: they are filed in a cell of it all the same,
    alike by every route, and the calls that follow read them in range."""
    conf, box = gpu.lattice(2, 3, 0.45)
    conf = conf[::18].copy()   # 6 spheres: no cell can hold too many
    conf[:, 0] = np.arange(6)
    reps = [dict(n=6, box=box, dr_max=10.0 * box[0], seed=3 + r) for r in range(replicas)]
    runs = [_wide_steps(reps, [conf] * replicas, t) for t in (None, (32, 2, 0), (32, 8, 16), (64, 4, 0, 1))]
    x = np.array(runs[0][1])[:, :, 1:]
    assert x.min() < -box[0] and x.max() > 2 * box[0]
    for run in runs[1:]:
        assert np.array_equal(np.array(run[1])[:, :, 1:], x)
        assert run[2:] == runs[0][2:]
    ctx = runs[0][0]
    net = gpu.Mlp(ctx, seed=1)
    f, n_free = net.proposal_scores(0.25)
    assert np.isneginf(f).sum() == len(f) - n_free
    assert net.widom(0.25, 0.9, 1, 1, 20000)["n"] == 20000
    ctx.widom_cells(1, 1, 100)
    ctx.widom_uniform(1, 1, 0, 10000)
    ctx.contact_counts(0.01, 5, 1.05)
    for run in runs:
        run[0].close()


def test_contexts_of_threads_share_kernels():
    """Two threads, each with its own contexts, launch the kernels that keep a
    system in more than 64 KB of LDS with different sizes: no launch is refused
    for the other's, and the results are those of one thread."""
    def work(n):
        conf, box = gpu.lattice(2, n, 0.6)
        out = []
        ctx = gpu.Context([dict(n=len(conf), box=box, dr_max=0.1, seed=r) for r in range(64)])
        for r in range(64):
            ctx.upload(conf, r)
        big, bbox = gpu.lattice(2, n + 3, 0.8)
        wide = gpu.Context([dict(n=len(big), box=bbox, dr_max=0.1, seed=1)])
        wide.upload(big)
        for k in range(40):
            ctx.sweeps(2)
            ctx.npt_sweeps(2, 2.0, 0.01)
            out.append(wide.widom_uniform(1, k, 0, 500000))
        out += [ctx.download(r).tobytes() for r in range(64)]
        for c in (ctx, wide):
            c.close()
        return out

    want = [work(6), work(7)]
    with ThreadPoolExecutor(2) as pool:
        got = list(pool.map(work, (6, 7)))
    assert got == want
