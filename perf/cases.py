"""Performance cases of the framework: the calls a simulation program makes,
from one trial move of 256 spheres to a million spheres in one batch.

Eight kinds of call, each through hsmc_amd.gpu:

  serial    the reference's serial chain, one move at a time: overlap_batch
            of one trial position, set_particles when it is free
  nvt       a run segment: sweeps of one system or of a batch of replicas,
            then every replica's configuration and move counters
  npt       an isobaric run segment of a batch: NpT sweeps, then boxes,
            volume-move counters and configurations
  sample    one production sample: sweeps between samples, then the
            observables of each replica (contact histogram, uniform Widom
            insertions and, where asked, g(r) and the scaled-overlap flags of
            the thermodynamic pressure)
  rdf       one g(r) sample
  widom     one chemical-potential sample with cell-stratified insertions
  learned   one with the learned proposal (scores, cumulative mass and
            insertions of a configuration not seen before)
  train     the proposal network's training on one stored configuration

Observables follow at least one sweep, so each sample meets a configuration
the context has built no grid for, as in a production run.  Every fluid
starts from an fcc lattice (with vacancies where N is not of the form
4 nx ny nz) and is melted by the framework's own sweeps, seeded by the case's
seed; "train" uses a hot fcc crystal made here, so that exact() can restate
it in 64 bits.  The launch shape is the library's default.
"""
import math

import numpy as np
import torch

from hsmc_amd import gpu

# input sizes of the network (include/hsmc_gpu.h)
NIN, NH = gpu.MLP_IN, gpu.MLP_HIDDEN


def listed():
    return [
        # the drop-in serial mode (keyword gpu_sweep serial) at the size of
        # the reference's published tables: latency of the smallest calls
        dict(name="serial 256", kind="serial", nx=4, ny=4, nz=4, drop=0, rho=0.70, moves=32),
        # the same size with the parallel sweep: a launch-bound segment
        dict(name="nvt 256", kind="nvt", replicas=1, nx=4, ny=4, nz=4, spread=0, drop=0, rho=0.70,
             rho_to=0.70, sweeps=100, melt=1000),
        # the headline system
        dict(name="nvt 32000", kind="nvt", replicas=1, nx=20, ny=20, nz=20, spread=0, drop=0,
             rho=0.85, rho_to=0.85, sweeps=100, melt=1000),
        # the batched workload: N = 108 to 13500, rho 0.30 to 0.93
        dict(name="nvt batch of 256", kind="nvt", replicas=256, nx=3, ny=3, nz=3, spread=13, drop=0,
             rho=0.30, rho_to=0.93, sweeps=100, melt=100),
        # the published NpT table: four pressures, N = 256, 25 sweeps a sample
        dict(name="npt 32 x 256", kind="npt", replicas=32, nx=4, ny=4, nz=4, drop=0, press=1.472,
             press_to=5.274, dv=0.02, dr=0.15, sweeps=25, melt=500),
        # the large NpT system: N = 256000 at beta P = 8 and 11
        dict(name="npt 4 x 256000", kind="npt", replicas=4, nx=40, ny=40, nz=40, drop=0, press=8.0,
             press_to=11.0, dv=0.001, dr=0.1, sweeps=4, melt=60),
        # the published NVT and Widom tables: 8 replicas, 10 sweeps a sample
        dict(name="sample 8 x 256", kind="sample", replicas=8, nx=4, ny=4, nz=4, drop=0, rho=0.70,
             gap=10, insertions=100000, bins=0, factors=0, melt=1000),
        # every observable of an NVT run at a mid size
        dict(name="sample 4000", kind="sample", replicas=1, nx=10, ny=10, nz=10, drop=0, rho=0.80,
             gap=10, insertions=1000000, bins=400, factors=20, melt=1000),
        # g(r) to 5 diameters in 400 bins on the headline system
        dict(name="rdf 32000", kind="rdf", nx=20, ny=20, nz=20, drop=0, rho=0.85, bins=400,
             dr_bin=0.01, melt=1000),
        # 10^7 insertions on the large dense system
        dict(name="widom 108000", kind="widom", nx=30, ny=30, nz=30, drop=0, rho=0.90,
             insertions=10000000, melt=600),
        # the learned proposal on the same system at its usual count
        dict(name="learned 108000", kind="learned", nx=30, ny=30, nz=30, drop=0, rho=0.90,
             insertions=250000, voxel=0.25, melt=600),
        # training on uniform insertions, batches of 4096
        dict(name="train 4000", kind="train", nx=10, ny=10, nz=10, drop=0, rho=0.80, points=131072,
             epochs=2, batch=4096, voxel=0.25),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_cells(rng, lo, hi):
    """fcc cells per axis, near a cube, and a few vacancies (odd N)."""
    n = _log_int(rng, lo, hi)
    jitter = [min(hi, max(lo, n + rng.choice((0, 0, -1, 1)))) for _ in range(3)]
    return dict(nx=jitter[0], ny=jitter[1], nz=jitter[2], drop=rng.choice((0, 1, 3, 7)))


def draw(rng):
    kind = rng.choice(("serial", "nvt", "nvt", "npt", "sample", "rdf", "widom", "learned", "train"))
    rho = round(rng.uniform(0.45, 0.93), 3)
    if kind == "serial":
        return dict(kind=kind, **_draw_cells(rng, 3, 10), rho=rho, moves=rng.randint(8, 48))
    if kind == "nvt":
        replicas = rng.choice((1, 1, _log_int(rng, 2, 64)))
        spread = rng.randint(0, 4) if replicas > 1 else 0
        top = 30 if replicas == 1 else max(3, int((250000 / replicas / 4) ** (1 / 3)) - spread)
        return dict(kind=kind, replicas=replicas, **_draw_cells(rng, 3, top), spread=spread,
                    rho=rho, rho_to=round(rng.uniform(0.30, 0.93), 3) if replicas > 1 else rho,
                    sweeps=_log_int(rng, 10, 200), melt=200)
    if kind == "npt":
        replicas = _log_int(rng, 1, 48)
        top = max(3, int((1000000 / replicas / 4) ** (1 / 3)))
        cells = _draw_cells(rng, 3, min(top, 40))
        n = 4 * cells["nx"] * cells["ny"] * cells["nz"]
        press = round(rng.uniform(1.4, 11.0), 3)
        return dict(kind=kind, replicas=replicas, **cells, press=press,
                    press_to=round(rng.uniform(1.4, 11.0), 3) if replicas > 1 else press,
                    dv=round(max(0.001, 0.32 / math.sqrt(n)), 5), dr=0.1,
                    sweeps=rng.randint(1, 20 if n * replicas < 200000 else 4), melt=60)
    if kind == "sample":
        replicas = rng.choice((1, 1, rng.randint(2, 12)))
        return dict(kind=kind, replicas=replicas, **_draw_cells(rng, 3, 20 if replicas == 1 else 6),
                    rho=rho, gap=rng.randint(1, 20),
                    insertions=_log_int(rng, 10000, 2000000 // replicas),
                    bins=rng.choice((0, 100, 400)), factors=rng.choice((0, 1, 20, 64)), melt=300)
    if kind == "rdf":
        return dict(kind=kind, **_draw_cells(rng, 4, 25), rho=rho, bins=rng.choice((77, 200, 400, 800)),
                    dr_bin=rng.choice((0.005, 0.01, 0.02)), melt=300)
    if kind == "widom":
        return dict(kind=kind, **_draw_cells(rng, 4, 30), rho=rho,
                    insertions=_log_int(rng, 100000, 20000000), melt=200)
    if kind == "learned":
        return dict(kind=kind, **_draw_cells(rng, 6, 30), rho=round(rng.uniform(0.70, 0.93), 3),
                    insertions=_log_int(rng, 20000, 1000000), voxel=rng.choice((0.2, 0.25, 0.3)),
                    melt=200)
    return dict(kind=kind, **_draw_cells(rng, 4, 14), rho=round(rng.uniform(0.70, 0.93), 3),
                points=_log_int(rng, 10000, 131072), epochs=rng.randint(1, 2),
                batch=rng.choice((1024, 4096, 5000)), voxel=0.25)


# ---- configurations -----------------------------------------------------------

def _fcc(nx, ny, nz, drop, rho, rng):
    """N x {id, x, y, z} of an fcc lattice with `drop` random vacancies, at
    the density rho of the spheres that are left, and its box."""
    base = np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]])
    cells = np.stack(np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz), indexing="ij"), -1)
    sites = (cells.reshape(-1, 1, 3) + base).reshape(-1, 3)
    if drop:
        sites = sites[np.sort(rng.permutation(len(sites))[drop:])]
    a = (len(sites) / (rho * nx * ny * nz)) ** (1.0 / 3.0)
    conf = np.zeros((len(sites), 4))
    conf[:, 0] = np.arange(len(sites))
    conf[:, 1:] = sites * a
    return conf, (nx * a, ny * a, nz * a)


def _context(systems, seed, dr, melt):
    """A context of the given (configuration, box) systems, melted."""
    ctx = gpu.Context([dict(n=len(c), box=box, dr_max=dr, seed=1000 * (seed + 1) + r)
                       for r, (c, box) in enumerate(systems)])
    for r, (c, _) in enumerate(systems):
        ctx.upload(c, r)
    if melt:
        ctx.sweeps(melt)
        ctx.sync()
    return ctx


def _one(case, seed, dr=0.1, melt=None):
    """The melted context of a one-replica case."""
    rng = np.random.default_rng(seed)
    system = _fcc(case["nx"], case["ny"], case["nz"], case["drop"], case["rho"], rng)
    return _context([system], seed, dr, case["melt"] if melt is None else melt)


def _nvt_systems(case, rng):
    """(configuration, box) of each replica: cells per axis grow through
    `spread` steps, densities run from rho to rho_to."""
    R, steps = case["replicas"], max(1, case["spread"])
    out = []
    for r in range(R):
        s = r % steps
        rho = case["rho"] + (case["rho_to"] - case["rho"]) * (r / (R - 1) if R > 1 else 0.0)
        out.append(_fcc(case["nx"] + s, case["ny"] + s, case["nz"] + s, case["drop"], rho, rng))
    return out


def _cs_density(press):
    """Carnahan-Starling density at beta P sigma^3 = press."""
    lo, hi = 0.01, 1.2
    for _ in range(80):
        mid = 0.5 * (lo + hi)
        e = math.pi / 6.0 * mid
        z = (1 + e + e * e - e ** 3) / (1 - e) ** 3
        lo, hi = (mid, hi) if mid * z < press else (lo, mid)
    return 0.5 * (lo + hi)


def _pressures(case):
    R = case["replicas"]
    return [case["press"] + (case["press_to"] - case["press"]) * ((r % 4) / 3 if R > 3 else r / max(1, R - 1))
            for r in range(R)]


def _crystal(case, seed):
    """A hot fcc crystal: every sphere displaced at random by less than half
    the gap to its neighbours, so none overlap."""
    rng = np.random.default_rng(seed)
    conf, box = _fcc(case["nx"], case["ny"], case["nz"], case["drop"], case["rho"], rng)
    a = box[0] / case["nx"]
    reach = 0.499 * (a / math.sqrt(2.0) - 1.0)
    step = rng.normal(size=(len(conf), 3))
    step *= reach * rng.random((len(conf), 1)) ** (1 / 3) / np.linalg.norm(step, axis=1, keepdims=True)
    conf[:, 1:] = (conf[:, 1:] + step) % np.array(box)
    return conf, box


def _he_uniform(seed):
    """Starting weights of a network to be trained, packed."""
    rng = np.random.default_rng(seed + 77)
    w1 = rng.uniform(-1, 1, (NIN, NH)) * math.sqrt(6.0 / NIN)
    w2 = rng.uniform(-1, 1, (NH, NH)) * math.sqrt(6.0 / NH)
    w3 = rng.uniform(-1, 1, NH) * math.sqrt(6.0 / NH)
    z = np.zeros(NH)
    return np.concatenate([w1.ravel(), z, w2.ravel(), z, w3, [0.0]]).astype(np.float32)


def _trained_like(seed, beta=20.0):
    """A network close to what training converges to, -beta max(0, 1 - d) of
    the nearest sphere, with small random weights beside it."""
    rng = np.random.default_rng(seed + 99)
    w1 = rng.normal(size=(NIN, NH)) * 0.05
    w2 = rng.normal(size=(NH, NH)) * 0.05
    w3 = rng.normal(size=NH) * 0.05
    w1[0, 0], w2[0, 0], w3[0] = -1.0, 1.0, -beta
    z = np.zeros(NH)
    return np.concatenate([w1.ravel(), z, w2.ravel(), z, w3, [0.0]]).astype(np.float32)


# ---- prepare ------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case, kind=kind, seed=seed, sample=0)
    rng = np.random.default_rng(seed)
    if kind == "serial":
        st["ctx"] = _one(case, seed, melt=1000)
        st["conf"] = st["ctx"].download()
        st["box"] = np.array(st["ctx"].box())
        st["pick"] = rng.integers(0, len(st["conf"]), case["moves"])
        st["step"] = (rng.random((case["moves"], 3)) - 0.5) * 0.1
    elif kind == "nvt":
        st["ctx"] = _context(_nvt_systems(case, rng), seed, 0.1, case["melt"])
    elif kind == "npt":
        st["press"] = _pressures(case)
        systems = [_fcc(case["nx"], case["ny"], case["nz"], case["drop"], _cs_density(p), rng)
                   for p in st["press"]]
        st["ctx"] = _context(systems, seed, case["dr"], case["melt"])
    elif kind == "sample":
        systems = [_fcc(case["nx"], case["ny"], case["nz"], case["drop"], case["rho"], rng)
                   for _ in range(case["replicas"])]
        st["ctx"] = _context(systems, seed, 0.1, case["melt"])
        # sf of compressions by xi = 1e-4, 2e-4, ... (compute_press.c:253-255)
        st["sf"] = [(1.0 - 1e-4 * k) ** (1.0 / 3.0) for k in range(1, case["factors"] + 1)]
    elif kind in ("rdf", "widom"):
        st["ctx"] = _one(case, seed)
        if kind == "widom":
            _, cells, _ = st["ctx"].widom_cells(0, 0, 1)
            st["per_cell"] = max(1, round(case["insertions"] / cells))
    elif kind == "learned":
        st["ctx"] = _one(case, seed)
        st["net"] = gpu.Mlp(st["ctx"], seed=5)
        st["net"].set(_trained_like(seed))
    elif kind == "train":
        conf, box = _crystal(case, seed)
        st["ctx"] = _context([(conf, box)], seed, 0.1, 0)
        st["net"] = gpu.Mlp(st["ctx"], seed=5)
        st["weights"] = _he_uniform(seed)
    return st


# ---- run ----------------------------------------------------------------------

def _configurations(ctx):
    """Every replica's configuration, one array."""
    if ctx.R == 1:
        return ctx.download()
    return np.concatenate([ctx.download(r) for r in range(ctx.R)])


def _cut(ctx, r, bins, dr_bin):
    """g(r) cutoff: the bins' reach, at most half the shortest edge."""
    return min(1.0 + bins * dr_bin, 0.499 * min(ctx.box(r)))


def run(state):
    case, kind, ctx = state["case"], state["kind"], state["ctx"]
    state["sample"] += 1
    if kind == "serial":
        conf, L = state["conf"], state["box"]
        accepted = []
        for i, step in zip(state["pick"], state["step"]):
            q = conf[i, 1:] + step
            q = np.where(q > L, q - L, np.where(q < 0.0, q + L, q))
            free = not ctx.overlap_batch([i], [q])[0]
            if free:
                ctx.set_particles([i], [q])
                conf[i, 1:] = q
            accepted.append(free)
        return np.array(accepted), ctx.download()
    if kind == "nvt":
        ctx.sweeps(case["sweeps"])
        moves = [list(ctx.counters(r).values()) for r in range(ctx.R)]
        return _configurations(ctx), np.array(moves, dtype=np.int64)
    if kind == "npt":
        moves = ctx.npt_sweeps(case["sweeps"], state["press"], case["dv"])
        boxes = np.array([ctx.box(r) for r in range(ctx.R)])
        return moves.astype(np.int64), boxes, _configurations(ctx)
    if kind == "sample":
        ctx.sweeps(case["gap"])
        contact, out_of_range, hits, rdf, flags = [], [], [], [], []
        for r in range(ctx.R):
            c, o = ctx.contact_counts(0.01, 5, 1.05, r)
            contact.append(c)
            out_of_range.append(o)
            hits.append(ctx.widom_uniform(state["seed"], state["sample"], 0, case["insertions"], r))
            if case["bins"]:
                rdf.append(ctx.rdf_counts(0.01, case["bins"], _cut(ctx, r, case["bins"], 0.01), r)[0])
            if state["sf"]:
                flags.append(ctx.any_overlap_scaled(state["sf"], r))
        return [np.array(v) for v in (contact, out_of_range, hits, rdf, flags) if v]
    if kind == "rdf":
        ctx.sweeps(1)
        return ctx.rdf_counts(case["dr_bin"], case["bins"], _cut(ctx, 0, case["bins"], case["dr_bin"]))
    if kind == "widom":
        ctx.sweeps(1)
        hits, points, _ = ctx.widom_cells(state["seed"], state["sample"], state["per_cell"])
        return hits, points
    if kind == "learned":
        ctx.sweeps(1)
        return state["net"].widom(case["voxel"], 0.9, state["seed"], state["sample"], case["insertions"])
    net = state["net"]
    net.set(state["weights"])
    loss = net.train(case["voxel"], state["seed"], 0, case["points"], epochs=case["epochs"],
                     batch=case["batch"], lr=2e-3, beta=20.0)
    return loss, net.get()


# ---- work ---------------------------------------------------------------------

def _spheres(case):
    n = 4 * case["nx"] * case["ny"] * case["nz"] - case["drop"]
    if case["kind"] == "nvt":
        steps = max(1, case["spread"])
        return sum(4 * (case["nx"] + r % steps) * (case["ny"] + r % steps) * (case["nz"] + r % steps)
                   - case["drop"] for r in range(case["replicas"]))
    return n * case.get("replicas", 1)


def work(case):
    """Compulsory bytes and flops of one pass.  A pair test is 8 flops (three
    differences, three squares, two sums); a sweep's attempt tests the
    spheres of a 3 x 3 x 3 block of unit cells and moves 64 bytes (position
    in and out, slot id and cell count); a call's spheres are read once."""
    kind, n, rho = case["kind"], _spheres(case), case.get("rho", 0.85)
    near = 27.0 * rho
    sweep = dict(bytes=64.0 * n, flops=8.0 * near * n)
    if kind == "serial":
        m = case["moves"]
        return dict(bytes=m * 24.0 * (near + 1) + 32.0 * n, flops=m * near * 8.0)
    if kind in ("nvt", "npt"):
        return dict(bytes=sweep["bytes"] * case["sweeps"] + 32.0 * n, flops=sweep["flops"] * case["sweeps"])
    if kind == "sample":
        b, f = sweep["bytes"] * case["gap"], sweep["flops"] * case["gap"]
        ins = case["insertions"] * case["replicas"]
        b += 24.0 * n * (2 + (case["bins"] > 0) + (case["factors"] > 0))
        # contact pairs, insertions that meet a sphere after a few tests, g(r) pairs
        f += 8.0 * (0.5 * near * n + 4.0 * ins + (case["factors"] > 0) * 0.5 * near * n)
        if case["bins"]:
            f += 8.0 * 0.5 * n * rho * 4.19 * (1 + 0.01 * case["bins"]) ** 3
        return dict(bytes=b, flops=f)
    if kind == "rdf":
        r = 1 + case["bins"] * case["dr_bin"]
        edge = (n / rho) ** (1 / 3)
        return dict(bytes=sweep["bytes"] + 24.0 * n + 8.0 * case["bins"],
                    flops=sweep["flops"] + 8.0 * 0.5 * n * rho * 4.19 * min(r, 0.5 * edge) ** 3)
    if kind == "widom":
        return dict(bytes=sweep["bytes"] + 24.0 * n, flops=sweep["flops"] + 8.0 * 4.0 * case["insertions"])
    if kind == "learned":
        # a byte a voxel says which can hold a point; a score is 9856 flops on about 1% of them
        voxels = n / rho / case["voxel"] ** 3
        return dict(bytes=sweep["bytes"] + 24.0 * n + voxels,
                    flops=sweep["flops"] + 0.01 * voxels * 9856.0 + 8.0 * 4.0 * case["insertions"])
    rows = case["points"]
    # descriptor and target rows written once, read in each epoch; forward and
    # backward are three times the forward's products
    return dict(bytes=rows * 52.0 * (1 + case["epochs"]), flops=rows * (case["epochs"] * 3 * 9856.0 + 2 * 8.0 * 60))


# ---- exact --------------------------------------------------------------------

def exact(case, seed):
    """Training restated in 64 bits.  The other kinds return whole numbers
    and Markov-chain configurations, which have no such value."""
    if case["kind"] != "train":
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    f64 = dict(dtype=torch.float64, device=dev)
    conf, box = _crystal(case, seed)
    x = torch.tensor(conf[:, 1:], **f64)
    L = torch.tensor(box, **f64)
    u = torch.tensor(_philox_uniform(seed, case["points"]), **f64) * L
    m = torch.tensor([math.ceil(b / case["voxel"]) for b in box], **f64)
    edge = L / m
    centre = (torch.minimum(torch.floor(u / edge), m - 1) + 0.5) * edge
    # distances beyond the narrowest side of the descriptor grid (cells at
    # least 1.5 wide) count as that side
    far = min(b / max(1, math.floor(b / 1.5)) for b in box)

    def nearest(q, k):
        out = []
        for part in q.split(4096):
            d = part[:, None, :] - x[None, :, :]
            d = d - L * torch.round(d / L)
            out.append((d * d).sum(-1).topk(k, largest=False, sorted=True).values)
        return torch.cat(out).clamp(max=far * far).sqrt()

    X = nearest(centre, NIN) - 1.0
    T = -20.0 * torch.clamp(1.0 - nearest(u, 1)[:, 0], min=0.0)
    p = torch.tensor(_he_uniform(seed).astype(np.float64), **f64)
    m1, m2 = torch.zeros_like(p), torch.zeros_like(p)
    step, loss = 0, 0.0
    for _ in range(case["epochs"]):
        total = 0.0
        for b0 in range(0, case["points"], case["batch"]):
            xb, tb = X[b0:b0 + case["batch"]], T[b0:b0 + case["batch"]]
            q = p.clone().requires_grad_(True)
            w1, b1, w2, b2, w3, b3 = torch.split(q, [NIN * NH, NH, NH * NH, NH, NH, 1])
            h = torch.relu(xb @ w1.view(NIN, NH) + b1)
            y = torch.relu(h @ w2.view(NH, NH) + b2) @ w3 + b3
            sq = ((y - tb) ** 2).sum()
            g, = torch.autograd.grad(sq / len(xb), q)
            total += float(sq.detach())
            step += 1
            m1 = 0.9 * m1 + 0.1 * g
            m2 = 0.999 * m2 + 0.001 * g * g
            p = p - 2e-3 * (m1 / (1 - 0.9 ** step)) / ((m2 / (1 - 0.999 ** step)).sqrt() + 1e-8)
        loss = total / case["points"]
    return loss, p.cpu().numpy()


def _philox_uniform(seed, n):
    """n x 3 uniforms in [0, 1] of Philox4x32-10 stream (seed, sample 0), as
    the uniform insertions draw them: counter {i, 0, 0, "WI" << 16}."""
    mask = np.uint64(0xFFFFFFFF)
    c = [np.arange(n, dtype=np.uint64), np.zeros(n, np.uint64), np.zeros(n, np.uint64),
         np.full(n, 0x57490000, np.uint64)]
    k0, k1 = seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF
    for _ in range(10):
        a = np.uint64(0xD2511F53) * c[0]
        b = np.uint64(0xCD9E8D57) * c[2]
        c = [(b >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), b & mask,
             (a >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), a & mask]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return np.stack([w.astype(np.float64) / 4294967295.0 for w in c[:3]], 1)
