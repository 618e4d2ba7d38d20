"""Pair histograms, scaled-overlap flags and uniform insertions at the sizes
where their kernels change: with and without a neighbour grid, tile edges of
the all-pairs kernels, the 3^3 and 5^3 stencils and their fallback on thin
boxes, bins by formula and by edges, spheres filed in LDS or in memory.
Every result is compared with FP64 numpy over all pairs, bit for bit."""
import ctypes as C
import math

import numpy as np
import pytest

from hsmc_amd import gpu

pytestmark = pytest.mark.gpu


def _context(xyz, box):
    conf = np.zeros((len(xyz), 4))
    conf[:, 0] = np.arange(len(xyz))
    conf[:, 1:] = xyz
    ctx = gpu.Context([dict(n=len(xyz), box=tuple(box))])
    ctx.upload(conf)
    return ctx


def _image(d, L):
    return np.where(d > L / 2, d - L, np.where(d < -L / 2, d + L, d))


def _near_pairs(xyz, box, reach):
    """(i, j, squared distance) of the pairs i < j closer than about reach."""
    out = []
    for a in range(0, len(xyz), 256):
        s = 0.0
        for k in range(3):
            d = _image(xyz[a:a + 256, None, k] - xyz[None, :, k], box[k])
            s = s + d * d if k else d * d
        i, j = np.nonzero(s < reach * reach * (1 + 1e-9))
        keep = j > i + a
        out.append((i[keep] + a, j[keep], s[i[keep], j[keep]]))
    return tuple(np.concatenate(v) for v in zip(*out))


def _histogram(s, dr_bin, nbins, rmax):
    dr = np.sqrt(s)
    b = ((dr[dr < rmax] - 1.0) / dr_bin).astype(np.int64)   # truncation, as in C
    ok = (b >= 0) & (b < nbins)
    return np.bincount(b[ok], minlength=nbins), int((~ok).sum())


BOXES = {
    # cubic boxes at density 0.8; N around the all-pairs tiles (64), run
    # lengths (4096) and the steps to a grid (5120, 7168)
    **{f"cube-{n}": (n, None) for n in (1, 2, 63, 64, 65, 127, 129, 1000, 4096, 4097, 5120, 5121, 7168, 7169)},
    # a grid with fewer than 3 cells along x; exactly 3 of side 2 and more;
    # exactly 5 of half a cutoff of 4.4 and more
    "thin-2": (8300, (4.5, 4.6)), "thin-3": (8400, (7.0, 8.3)), "thin-5": (8500, (11.1, 13.9)),
}


@pytest.mark.parametrize("name", list(BOXES))
def test_histograms_match_all_pairs(name):
    n, thin = BOXES[name]
    vol = max(n / 0.8, 75.0)
    box = np.array([vol ** (1 / 3)] * 3 if thin is None else [thin[0], thin[1], vol / (thin[0] * thin[1])])
    rng = np.random.default_rng(n)
    xyz = rng.random((n, 3)) * box   # overlapping points too: bins below 0 count as out of range
    xyz[0] = box                     # coordinates at the edge itself
    half = min(box) / 2
    reach = min(5.5, half)
    _, _, s = _near_pairs(xyz, box, reach)
    ctx = _context(xyz, box)
    # (bin width, bins, cutoff): contact; formula / edges (16, 17); edges in
    # LDS / not (2048, 2049); more bins than the cutoff reaches; fewer
    for dr_bin, nbins, rmax in ((0.01, 5, 1.05), (0.02, 16, 1.32), (0.02, 17, 1.34), (0.01, 400, 5.0),
                                (0.002, 2048, 5.096), (0.002, 2049, 5.098), (0.01, 300, 2.1),
                                (0.013, 40, 4.4)):
        rmax = min(rmax, half)
        if rmax <= 1.0:
            continue
        want = _histogram(s, dr_bin, nbins, rmax)
        got = ctx.rdf_counts(dr_bin, nbins, rmax)
        assert np.array_equal(got[0], want[0]), (dr_bin, nbins, rmax)
        assert got[1] == want[1], (dr_bin, nbins, rmax)
    ctx.close()


def test_histogram_bins_at_their_edges():
    """Pairs whose distance is within a few units in the last place of a bin
    edge fall in the bin the formula gives: 64 spheres far apart on a line in
    y and z, partners at 1 + b dr_bin and its neighbours along x."""
    dr_bin, nbins = 0.01, 64
    box = np.array([8.0, 24.0, 24.0])
    xyz = []
    for b in range(nbins):
        y, z = 1.5 * (b % 8) + 6.0 * (b % 2), 1.5 * (b // 8)
        d = 1.0 + b * dr_bin
        for _ in range(b % 5):
            d = np.nextafter(d, 0.0 if b % 2 else 9.0)
        xyz += [(0.0, y, z), (d, y, z)]
    xyz = np.array(xyz)
    i, j, s = _near_pairs(xyz, box, 2.0)
    ctx = _context(xyz, box)
    for n in (10, 30, nbins):
        want = _histogram(s, dr_bin, n, 1.0 + nbins * dr_bin)
        got = ctx.rdf_counts(dr_bin, n, 1.0 + nbins * dr_bin)
        assert np.array_equal(got[0], want[0]) and got[1] == want[1], n
    ctx.close()


@pytest.mark.parametrize("dr_bin", [5e-324, 1e-9, 1.0 - 1e-12, 1.0, 1.0 + 1e-12, 1e300, math.inf])
def test_histogram_of_extreme_bin_widths(dr_bin):
    """Widths at which the bins' edges fall together, onto zero or nowhere."""
    rng = np.random.default_rng(12)
    box = np.array([8.0, 8.0, 8.0])
    xyz = np.vstack([rng.random((60, 3)) * box, [[1.0, 1.0, 1.0], [1.0, 1.0, 2.0], [1.0, 1.0, 1.0]]])
    i, j, s = _near_pairs(xyz, box, 3.0)
    ctx = _context(xyz, box)
    want = _histogram(s, dr_bin, 40, 2.9)
    got = ctx.rdf_counts(dr_bin, 40, 2.9)
    assert np.array_equal(got[0], want[0]) and got[1] == want[1]
    ctx.close()


@pytest.mark.parametrize("shape,drop", [((4, 4, 4), 1), ((8, 8, 16), 0), ((16, 16, 16), 0),
                                        ((16, 16, 17), 5), ((16, 16, 20), 0), ((16, 16, 21), 3),
                                        ((4, 45, 50), 2), ((6, 38, 40), 7)])
def test_scaled_flags_match_all_pairs(shape, drop):
    """64 compressions on a jittered cubic lattice whose closest pair lies
    inside their range."""
    a = 1.012
    box = a * np.array(shape)
    rng = np.random.default_rng(sum(shape))
    sites = np.stack(np.meshgrid(*(np.arange(k) for k in shape), indexing="ij"), -1).reshape(-1, 3)
    sites = sites[np.sort(rng.permutation(len(sites))[drop:])]
    xyz = (sites * a + rng.uniform(-0.0035, 0.0035, sites.shape)) % box
    ctx = _context(xyz, box)
    i, j, s = _near_pairs(xyz, box, 1.03)
    sf = np.linspace(1.0, 0.985, 64)
    want = []
    for f in sf:
        t = 0.0
        for k in range(3):
            d = _image((xyz[i, k] - xyz[j, k]) * f, box[k] * f)
            t = t + d * d if k else d * d
        want.append(not np.any(t < 1.0))
    assert want[0] and not want[-1]
    assert np.array_equal(ctx.any_overlap_scaled(sf), np.array(want, dtype=np.uint8))
    assert ctx.any_overlap_scaled([sf[20]])[0] == want[20]
    ctx.close()


def _uniform(seed, n):
    """Points 0..n-1 of the uniform insertions' Philox4x32-10 stream."""
    mask = np.uint64(0xFFFFFFFF)
    c = [np.arange(n, dtype=np.uint64), np.zeros(n, np.uint64), np.zeros(n, np.uint64),
         np.full(n, 0x57490000, np.uint64)]
    k0, k1 = seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF
    for _ in range(10):
        a, b = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(b >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), b & mask,
             (a >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), a & mask]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return np.stack([w.astype(np.float64) / 4294967295.0 for w in c[:3]], 1)


@pytest.mark.parametrize("n,rho", [(1, 0.01), (108, 0.7), (511, 0.3), (2048, 0.45), (2049, 0.45),
                                   (1500, 0.12), (700, 0.02)])
def test_uniform_insertions_filed_in_lds_or_memory(n, rho):
    """Hits of the points themselves, decided over all spheres in numpy;
    N = 2048 / 2049 and dilute boxes (many cells) are the two sides of the
    LDS rule.  5000 points leave the last workgroup partly idle."""
    rng = np.random.default_rng(n)
    L = (n / rho) ** (1 / 3)
    xyz = rng.random((n, 3)) * L
    ctx = _context(xyz, (L, L, L))
    pts = _uniform(31 + (n << 33), 5000) * L
    near = np.full(len(pts), np.inf)
    for a in range(0, n, 64):
        s = sum(_image(pts[:, None, k] - xyz[None, a:a + 64, k], L) ** 2 for k in range(3))
        near = np.minimum(near, s.min(1))
    assert np.min(np.abs(near - 1.0)) > 1e-9   # no point for which the order of the sum matters
    for m in (1, 511, 5000):
        assert ctx.widom_uniform(31 + (n << 33), 0, 0, m) == int((near[:m] >= 1.0).sum())
    ctx.close()


@pytest.mark.parametrize("n,rho", [(2049, 0.6), (4000, 0.8), (5200, 0.9), (5400, 0.9), (3000, 0.4)])
def test_uniform_insertions_of_larger_systems(n, rho):
    """One workgroup of 1024 with up to 158 KB of LDS, or the grid in memory
    (larger, dilute, or few points on a grid that is there): the same hits, and
    the points' own over all spheres in numpy."""
    rng = np.random.default_rng(n)
    L = (n / rho) ** (1 / 3)
    xyz = rng.random((n, 3)) * L
    ctx = _context(xyz, (L, L, L))
    fresh = ctx.widom_uniform(5, 0, 0, 3000)
    ctx.widom_cells(1, 1, 1)                      # builds the grid
    assert ctx.widom_uniform(5, 0, 0, 3000) == fresh
    many = ctx.widom_uniform(5, 0, 0, 450000)
    assert many == sum(ctx.widom_uniform(5, 0, first, 150000) for first in (0, 150000, 300000))
    q = _uniform(5, 3000) * L
    free = np.ones(len(q), bool)
    for c in xyz:
        d = np.abs(q - c)
        d = np.minimum(d, L - d)
        free &= ~((d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2] < 1.0)
    assert fresh == int(free.sum())
    ctx.close()


@pytest.mark.parametrize("n", [1, 64, 257, 1025, 16384, 16385])
def test_few_queries_and_moves_by_value(n):
    """Overlap queries up to 8 at a time take no grid, more do; one call after
    another on a configuration changed by set_particles (up to 8 by value)."""
    L = max(4.2, (n / 0.6) ** (1 / 3))
    rng = np.random.default_rng(n)
    xyz = rng.random((n, 3)) * L
    ctx = _context(xyz, (L, L, L))
    for m in (1, 7, 8, 9, 40):
        idx = rng.integers(0, n, m).astype(np.int32)
        q = rng.random((m, 3)) * L
        q[0] = (0.0, L, 0.5 * L)
        want = []
        for k in range(m):
            d = _image(q[k] - xyz, L)
            s = d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]
            s[idx[k]] = 9.0
            want.append(np.any(s < 1.0))
        assert np.array_equal(ctx.overlap_batch(idx, q), np.array(want, dtype=np.uint8)), m
        # the same particle twice among few: its last place stands
        moved = np.concatenate([idx[:min(m, n)], idx[:1]]) if m < 8 else np.unique(idx)
        to = rng.random((len(moved), 3)) * L
        ctx.set_particles(moved, to)
        for i, t in zip(moved, to):
            xyz[i] = t
        assert np.array_equal(ctx.download()[:, 1:], xyz), m
    ctx.close()


@pytest.mark.parametrize("box,n,per_cell", [((4.3, 5.0, 6.7), 60, 300), ((2.5, 9.1, 4.9), 50, 129), ((2.2, 2.9, 2.6), 5, 1000),
                                            ((11.3, 12.9, 10.2), 300, 64), ((11.3, 12.9, 10.2), 300, 65),
                                            ((30.2, 31.7, 29.9), 4000, 20), ((40.0, 4.5, 30.0), 200, 128)])
def test_stratified_insertions_match_all_pairs(box, n, per_cell):
    """Grids of 2 cells an axis (the FP64 test) and of 4 and more (FP32 with a
    band), one and two points a lane with their remainders; spheres overlap at
    random, so lists of every length occur.  About 2e-4 of the points have a
    sphere whose squared distance is within the band."""
    rng = np.random.default_rng(per_cell)
    xyz = rng.random((n, 3)) * np.array(box)
    ctx = _context(xyz, box)
    hits, points, grid = ctx.widom_cells(9, 4, per_cell)
    assert grid == tuple(int(b / (1.0 + 1e-9)) for b in box)
    mask = np.uint64(0xFFFFFFFF)
    cells = int(np.prod(grid))
    w = [np.repeat(np.arange(cells, dtype=np.uint64), per_cell), np.tile(np.arange(per_cell, dtype=np.uint64), cells),
         np.full(cells * per_cell, 4, np.uint64), np.full(cells * per_cell, 0x57430000, np.uint64)]
    index = w[0].astype(np.int64)
    k0, k1 = 9, 0
    for _ in range(10):
        a, b = np.uint64(0xD2511F53) * w[0], np.uint64(0xCD9E8D57) * w[2]
        w = [(b >> np.uint64(32)) ^ w[1] ^ np.uint64(k0), b & mask, (a >> np.uint64(32)) ^ w[3] ^ np.uint64(k1), a & mask]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    at = np.stack([index // (grid[1] * grid[2]), index // grid[2] % grid[1], index % grid[2]], 1)
    q = (at + (np.stack(w[:3], 1).astype(np.float64) + 0.5) * 2.0 ** -32) * (np.array(box) / np.array(grid))
    free = np.ones(len(q), bool)
    for c in xyz:
        d = np.abs(q - c)
        d = np.minimum(d, np.array(box) - d)
        free &= ~((d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2] < 1.0)
    assert points == len(q) and hits == int(free.sum())
    ctx.close()


def _refuse_above(ctx, limit):
    assert gpu.load().hsmc_gpu_test_scratch_limit(ctx.h, C.c_uint64(limit)) == 0


def _refused(call):
    with pytest.raises(gpu.HsmcError) as e:
        call()
    assert e.value.code == -7


def test_bin_edges_after_a_refused_workspace():
    """Edges lost to a workspace that could not grow are made again (another
    context's edges lie in the freed memory meanwhile)."""
    conf, box = gpu.lattice(2, 6, 0.8)
    ctx = gpu.Context([dict(n=len(conf), box=box, dr_max=0.1)])
    ctx.upload(conf)
    ctx.sweeps(20)
    want, oor = ctx.rdf_counts(0.01, 100, 2.5)
    assert want.sum() > 0 and oor > 0
    _refuse_above(ctx, 4000)
    _refused(lambda: ctx.rdf_counts(0.01, 1000, 2.5))
    other = gpu.Context([dict(n=len(conf), box=box, dr_max=0.1)])
    other.upload(conf)
    other.rdf_counts(0.02, 100, 2.5)
    other.close()
    _refuse_above(ctx, 2 ** 63)
    got, out = ctx.rdf_counts(0.01, 100, 2.5)
    assert np.array_equal(got, want) and out == oor
    ctx.close()


def test_grids_after_a_refused_workspace():
    """A grid that a larger replica's refused one has displaced is built again:
    search grid, its cleared counts, and the descriptors' grid."""
    small, sbox = gpu.lattice(2, 3, 0.7)
    large, lbox = gpu.lattice(2, 12, 0.7)
    ctx = gpu.Context([dict(n=len(small), box=sbox), dict(n=len(large), box=lbox)])
    ctx.upload(small, 0)
    ctx.upload(large, 1)
    q = np.random.default_rng(3).random((500, 3)) * np.array(sbox)
    free, desc = ctx.widom_points(q, 0), gpu.point_descriptors(ctx, q, 0)
    part_cell, _ = ctx.cell_list((4, 4, 4), 12, 0)
    ctx.widom_points(q, 0)
    # each limit lets some of the larger grid's buffers through
    for limit in (3000, 9000, 20000, 40000, 50000):
        _refuse_above(ctx, limit)
        _refused(lambda: ctx.widom_points(q, 1))
        _refused(lambda: gpu.point_descriptors(ctx, q, 1))
        _refused(lambda: ctx.cell_list((20, 20, 20), 12, 1))
        _refuse_above(ctx, 2 ** 63)
        assert np.array_equal(ctx.widom_points(q, 0), free)
        assert np.array_equal(gpu.point_descriptors(ctx, q, 0), desc)
        assert np.array_equal(ctx.cell_list((4, 4, 4), 12, 0)[0], part_cell)
        assert np.array_equal(ctx.widom_points(q, 0), free)
    assert ctx.any_overlap_scaled([0.999], 1)[0] == 1
    ctx.close()


def test_out_of_range_pairs_beyond_32_bits_in_one_workgroup():
    """N = 128^3 on a lattice, cutoff 0.4 of the edge: each of the 125 cells'
    workgroups meets 4.7 * 10^9 pairs within the cutoff, nearly all beyond the
    bins.  Every site sees the same distances, so the pairs of one make the
    count."""
    n, a = 128, 1.05
    L = n * a
    cells = np.stack(np.meshgrid(*[np.arange(n)] * 3, indexing="ij"), -1).reshape(-1, 3)
    ctx = _context(cells * a, (L, L, L))
    rmax, nbins, dr_bin = 0.39991 * L, 20, 0.02   # bins to 1.4: the first neighbours, at 1.05
    counts, oor = ctx.rdf_counts(dr_bin, nbins, rmax)
    m = np.minimum(np.arange(n), n - np.arange(n)).astype(float) * a
    r = np.sqrt(m[:, None, None] ** 2 + m[None, :, None] ** 2 + m[None, None, :] ** 2).ravel()
    assert np.abs(r - rmax).min() > 1e-6
    within = int((r < rmax).sum()) - 1
    assert counts[2] == 3 * n ** 3 and counts.sum() == 3 * n ** 3
    total = n ** 3 * within // 2
    assert total // 125 > 2 ** 32
    assert oor == total - 3 * n ** 3
    ctx.close()


def test_rows_of_counts_are_bounded_on_thin_boxes():
    """N = 528000 on a box of 2 search cells across (a thread per sphere): the
    workgroups' rows of 8192 bins stay within 2048, and every sphere is
    reached."""
    n, a = 33000, 1.05
    cells = np.stack(np.meshgrid(np.arange(4), np.arange(4), np.arange(n), indexing="ij"), -1).reshape(-1, 3)
    ctx = _context(cells * a, (4 * a, 4 * a, n * a))
    _refuse_above(ctx, 2048 * 8194 * 4)
    counts, oor = ctx.rdf_counts(0.0001, 8192, 1.3)
    assert counts[500] + counts[499] == 3 * len(cells) == counts.sum() and oor == 0
    assert ctx.any_overlap_scaled([1.0, 0.96, 0.95]).tolist() == [1, 1, 0]
    ctx.close()
