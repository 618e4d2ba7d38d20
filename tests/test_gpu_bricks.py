"""Brick phases (contexts of 40000 active cells and more) against the phases
cell by cell, which the oracle pins: positions and move counters are equal
bit for bit."""
import numpy as np
import pytest

from hsmc_amd import gpu

pytestmark = pytest.mark.gpu


def _sites(rng, box, fill):
    """A random part of a simple cubic lattice a little wider than a diameter."""
    m = [max(1, int(b / 1.04)) for b in box]
    g = np.stack(np.meshgrid(*[np.arange(k) for k in m], indexing="ij"), -1).reshape(-1, 3)
    xyz = g * (np.array(box) / m)
    return xyz[rng.random(len(xyz)) < fill] if fill < 1 else xyz


def _both(confs, boxes, sweeps=(5, 3), after=None):
    """Final positions and counters of every replica by each route."""
    def grid(b):  # largest even number of cells wider than a diameter
        g = int(b) // 2 * 2
        return g if b / g > 1.0 else g - 2

    assert sum(grid(b[0]) * grid(b[1]) * grid(b[2]) // 8 for b in boxes) >= 40000
    out = []
    for cells in (False, True):
        ctx = gpu.Context([dict(n=len(c), box=tuple(b), dr_max=0.2, seed=5 + r)
                           for r, (c, b) in enumerate(zip(confs, boxes))])
        for r, c in enumerate(confs):
            ctx.upload(np.column_stack([np.arange(len(c)), c]), r)
        if cells:
            ctx.set_tuning(32, 8, 4)
        ctx.sweeps(sweeps[0])
        if after:
            after(ctx)
        ctx.sweeps(sweeps[1])
        out.append([(ctx.download(r), ctx.counters(r)) for r in range(len(confs))])
        ctx.close()
    return out


def _same(a, b):
    for r, ((x, c), (y, d)) in enumerate(zip(a, b)):
        assert np.array_equal(x, y), r
        assert c == d, r
    assert sum(c["accepted"] for _, c in a) > 0


def _with_bulk(rng, boxes, fills):
    """Those replicas and enough others for the brick route."""
    boxes = [tuple(b) for b in boxes] + [(40.0, 41.0, 42.0)] * 6
    return [_sites(rng, b, f) for b, f in zip(boxes, list(fills) + [0.5] * 6)], boxes


def test_mixed_replicas():
    """Grids of 2 to 40 cells an axis (bricks with one active cell along an
    axis, uneven last bricks, neighbourhoods that meet themselves round the
    box), cells up to 1.5 wide (16 slots a cell), empty to full."""
    rng = np.random.default_rng(1)
    edges = [2.2, 2.9, 4.3, 4.7, 5.0, 6.4, 8.3, 8.9, 10.1, 13.0, 15.9, 17.2, 21.0, 26.3, 33.9, 40.5]
    boxes = [(a, edges[(3 * k + 1) % 16], edges[(7 * k + 5) % 16]) for k, a in enumerate(edges)]
    boxes += [(9.0, 9.0, 9.0), (11.0, 11.0, 11.0), (18.0, 18.0, 18.0), (2.4, 2.4, 70.0)]
    fills = [(0.02, 0.3, 0.6, 0.9, 1.0)[k % 5] for k in range(len(boxes))]
    confs, boxes = _with_bulk(rng, boxes, fills)
    confs = [c if len(c) else np.zeros((1, 3)) for c in confs]
    _same(*_both(confs, boxes))


@pytest.mark.parametrize("box", [(72.0, 73.0, 74.0), (27.0, 25.0, 620.0)])
def test_one_large_replica(box):
    _same(*_both([_sites(np.random.default_rng(2), box, 0.85)], [box]))


@pytest.mark.parametrize("wide", [False, True])
def test_uneven_density_and_overlaps(wide):
    """Bricks with more spheres than their list holds go half by half: one
    replica's spheres lie in an eighth of its box, another's overlap at random.
    With 16 slots a cell (a replica of wide cells beside them), halves that
    hold too many go cell by cell: a cluster of 3.4 spheres a cell."""
    rng = np.random.default_rng(3)
    box = (24.0, 24.0, 24.0)
    confs, boxes = _with_bulk(rng, [box, box, (4.7, 4.7, 4.7) if wide else box], [1.0, 1.0, 0.5])
    confs[0] = np.vstack([_sites(rng, (12.0, 12.0, 12.0), 1.0), 12.0 + 12.0 * rng.random((40, 3))])
    confs[1] = rng.random((6000, 3)) * np.array([24.0, 24.0, 12.0])
    if wide:
        confs[1] = np.vstack([11.0 * rng.random((3460, 3)), 12.0 + 12.0 * rng.random((40, 3))])
    _same(*_both(confs, boxes))


def test_lattice_starts():
    """Perfect lattices, whose layers fill some bricks beyond the mean."""
    confs, boxes = [], []
    for n, rho in ((6, 0.93), (9, 0.9), (10, 0.8), (11, 1.0), (12, 0.6), (13, 0.93), (30, 0.9)):
        L = (4 * n ** 3 / rho) ** (1 / 3)
        g = np.stack(np.meshgrid(*[np.arange(n)] * 3, indexing="ij"), -1).reshape(-1, 1, 3)
        basis = np.array([(0, 0, 0), (.5, .5, 0), (.5, 0, .5), (0, .5, .5)])
        confs.append(((g + basis) * (L / n)).reshape(-1, 3))
        boxes.append((L, L, L))
    _same(*_both(confs * 3, boxes * 3, sweeps=(1, 1)))


def test_positions_outside_the_box():
    """Spheres left outside by a smaller box are filed by the single wrap and
    compared by the FP64 arithmetic, as cell by cell."""
    rng = np.random.default_rng(4)
    confs, boxes = _with_bulk(rng, [(13.9, 13.9, 13.9), (5.9, 5.9, 5.9)], [0.3, 0.3])

    def shrink(ctx):
        ctx.set_box((12.1, 13.0, 13.9), 0)
        ctx.set_box((4.7, 5.9, 4.1), 1)

    _same(*_both(confs, boxes, after=shrink))


def test_boxes_scaled_between_sweeps():
    """A box change that keeps every sweep grid keeps the bricks; one that does
    not makes new ones."""
    rng = np.random.default_rng(5)
    confs, boxes = _with_bulk(rng, [(17.0, 17.0, 17.0)], [0.9])

    def grow(ctx):
        ctx.set_box((17.3, 17.3, 17.3), 0)
        ctx.sweeps(2)
        ctx.set_box((18.2, 18.2, 18.2), 0)

    _same(*_both(confs, boxes, after=grow))


def test_autotune_times_the_bricks():
    """The route stands beside the launch shapes, and tuning changes no result."""
    rng = np.random.default_rng(6)
    confs, boxes = _with_bulk(rng, [(9.0, 9.0, 9.0)], [0.8])
    _same(*_both(confs, boxes, after=lambda ctx: ctx.autotune(4)))


def test_full_stencils_on_two_cell_axes():
    """2 x 2 x 2 cells: a stencil has each cell once, and no more spheres than
    there are, though the brick's neighbourhood meets a cell up to 8 times.  16
    spheres of 20 lie in one cell and 4 in the one across the corner (they
    overlap, so that they stay): 128 + 4 meetings of 20 spheres, for a list of
    128."""
    rng = np.random.default_rng(7)
    confs, boxes = _with_bulk(rng, [(2.9, 2.9, 2.9)] * 8, [0.5] * 8)
    confs[:8] = [np.vstack([0.1 * rng.random((16, 3)), 1.45 + 0.1 * rng.random((4, 3))]) for _ in range(8)]
    _same(*_both(confs, boxes, sweeps=(10, 2)))


def test_steps_wider_than_the_box():
    """A step of up to two box edges either way leaves spheres outside the box
    (the wrap is a single one), some an edge away from where the reference's
    minimum image sees them."""
    rng = np.random.default_rng(8)
    confs, boxes = _with_bulk(rng, [(4.2, 4.2, 4.2)] * 24, [0.2] * 24)
    confs = [c if len(c) else np.zeros((1, 3)) for c in confs]

    def wide(ctx):
        for r in range(24):
            ctx.set_dr_max(16.5, r)

    a, b = _both(confs, boxes, sweeps=(2, 400), after=wide)
    assert any((x[:, 1:] > 4.2).any() for x, _ in b[:24])
    _same(a, b)


@pytest.mark.parametrize("cells,replicas", [(4, 5100), (6, 1500)])
def test_many_small_replicas(cells, replicas):
    """40800 active cells in replicas of 8 (too few for a brick each: cell by
    cell), 42000 of 27 beside a larger one (bricks): each replica as alone."""
    L = 1.07 * cells
    xyz = _sites(np.random.default_rng(9), (L, L, L), 0.7)
    systems = [(xyz, (L, L, L))] * replicas
    if cells == 6:   # beside a replica that no workgroup can keep in LDS
        systems.append((_sites(np.random.default_rng(9), (24.0, 24.0, 24.0), 0.7), (24.0, 24.0, 24.0)))

    def run(which):
        ctx = gpu.Context([dict(n=len(systems[k][0]), box=systems[k][1], dr_max=0.2, seed=3 + k) for k in which])
        for r, k in enumerate(which):
            ctx.upload(np.column_stack([np.arange(len(systems[k][0])), systems[k][0]]), r)
        ctx.sweeps(9)
        return ctx

    every = list(range(len(systems)))
    ctx = run(every)
    for k in (0, 1, replicas // 2, len(systems) - 1):
        alone = run([k])
        assert np.array_equal(ctx.download(k), alone.download()), k
        assert ctx.counters(k) == alone.counters(), k
        alone.close()
    ctx.close()
