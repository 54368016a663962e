"""The work that users of this framework have it do, as measurable cases.

Six kinds of call, each through the public Python entry points:

* ``pass``   -- the whole FoF-seeded SOD pass of a resident catalogue
  (``Context.run_pass``): what a survey or zoom run does once per snapshot.
* ``replay`` -- the same pass replayed as one HIP graph
  (``Context.run_pass_graph``): repeated passes over one set of buffers,
  where launches and host round trips are what is left.
* ``sod``    -- ``Context.sod_fof`` on a catalogue that is already sorted and
  seeded: another set of thresholds or profile bins over the same halos.
* ``chain``  -- cell sort, CIC deposit, CIC^-1, seeds, member counts and the
  density order, stage by stage (the reference's cic, cicm1, tri_cic on
  device arrays), with grids of nx or 2 nx nodes per side.
* ``host``   -- the drop-ins ``cic``, ``cicm1`` and ``tri_cic`` on host arrays
  in FP64, as the Fortran modules call them.
* ``greedy`` -- the drop-in ``spherover`` on host arrays.

Catalogues are the library's seeded NFW clumps on a uniform background, the
clump-size law and the fractions of the benchmark's workloads.
"""
import math

import numpy as np
import torch

import psod_amd as P

DEV = "cuda:0"
TABLE = 8192  # rows of a program's table of greedy halos
MULTI = "200,500,740.74,359.3"  # several thresholds at once, as the profiles use


def listed():
    return [
        # smallest use: the 32^3 catalogue of the smoke run
        dict(name="pass_32", kind="pass", nx=32, npart=32 ** 3, nclump=40,
             nhi=3000, ncentral=0, deltas="200", nbins=32, rmin=0.01, rmax=2.0,
             velocity=True, keep_grid=True, up=1),
        # a small box passed over and over: launches and gaps count
        dict(name="replay_128", kind="replay", nx=128, npart=128 ** 3,
             nclump=2000, nhi=20000, ncentral=0, deltas="200", nbins=32,
             rmin=0.01, rmax=2.0, velocity=False, keep_grid=False, up=1),
        # a mid-size box with fewer particles than cells and a 2 nx grid
        dict(name="pass_256_up2", kind="pass", nx=256, npart=11_999_987,
             nclump=9000, nhi=60000, ncentral=0, deltas="200,500", nbins=60,
             rmin=0.01, rmax=1.0, velocity=False, keep_grid=True, up=2),
        # the multi-threshold profile run with velocities at 512^3
        dict(name="pass_512_multi", kind="pass", nx=512, npart=512 ** 3,
             nclump=60000, nhi=200000, ncentral=0, deltas=MULTI, nbins=64,
             rmin=0.005, rmax=3.0, velocity=True, keep_grid=True, up=1),
        # a zoom: one central halo holds 5% of the particles
        dict(name="pass_512_zoom", kind="pass", nx=512, npart=512 ** 3,
             nclump=25000, nhi=100000, ncentral=6_250_000, deltas="200",
             nbins=32, rmin=0.01, rmax=2.0, velocity=False, keep_grid=False,
             up=1),
        # the benchmark's workload: 1024^3 particles, 500,000 halos
        dict(name="pass_1024", kind="pass", nx=1024, npart=1024 ** 3,
             nclump=500000, nhi=2000000, ncentral=0, deltas="200", nbins=32,
             rmin=0.01, rmax=2.0, velocity=False, keep_grid=False, up=1),
        # new thresholds and bins over halos already seeded
        dict(name="sod_256", kind="sod", nx=256, npart=256 ** 3, nclump=8000,
             nhi=100000, ncentral=0, deltas="97,200,500", nbins=60, rmin=0.01,
             rmax=1.0, velocity=True, up=1),
        # the reference's grid (2 nx nodes per side), stage by stage
        dict(name="chain_256_up2", kind="chain", nx=256, npart=256 ** 3,
             nclump=8000, nhi=60000, ncentral=0, up=2, shift=0),
        # a ragged particle count with a shifted grid
        dict(name="chain_512_ragged", kind="chain", nx=512,
             npart=99_999_989, nclump=45000, nhi=200000, ncentral=0, up=1,
             shift=3),
        # the reference's 128^3 zone on host arrays
        dict(name="host_128", kind="host", nx=128, npart=128 ** 3,
             nclump=2000, nhi=20000, ncentral=0, up=2),
        dict(name="greedy_128", kind="greedy", nx=128, npart=128 ** 3,
             nclump=2000, nhi=20000, ncentral=0, up=2, ncut=4, delta=200.0,
             delta2=800.0),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["pass", "pass", "replay", "sod", "chain", "chain",
                       "host", "greedy"])
    if kind in ("host", "greedy"):
        nx = 128 if rng.random() < 0.5 else 64
        n = int(nx ** 3 * rng.uniform(0.7, 1.0))
        return dict(kind=kind, nx=nx, npart=n, nclump=int(n * _log(rng, 4e-4, 1e-3)),
                    nhi=int(_log(rng, 3000, 20000)), ncentral=0, up=2,
                    **(dict(ncut=4, delta=rng.choice([200.0, 500.0]),
                            delta2=800.0) if kind == "greedy" else {}))
    top = {"pass": 9, "replay": 8, "sod": 9, "chain": 9}[kind]
    nx = 1 << rng.randint(5, top)
    n = int(nx ** 3 * rng.uniform(0.6, 1.2)) | 1
    nhi = int(_log(rng, max(500.0, 1.5e-3 * n), max(3000.0, 6e-3 * n)))
    c = dict(kind=kind, nx=nx, npart=n,
             nclump=max(8, int(n * _log(rng, 2e-4, 8e-4))), nhi=nhi,
             ncentral=int(n * rng.uniform(0.02, 0.05)) if rng.random() < 0.25
             else 0,
             up=2 if nx <= 256 and rng.random() < 0.3 else 1)
    if kind == "chain":
        c["shift"] = rng.randint(0, 7)
        return c
    c.update(deltas=rng.choice(["200", "200,500", MULTI]),
             nbins=rng.randint(20, 64), rmin=rng.choice([0.005, 0.01]),
             rmax=rng.choice([1.0, 2.0]), velocity=rng.random() < 0.5)
    if kind != "sod":
        c["keep_grid"] = rng.random() < 0.3
    return c


def _params(case):
    return P.sod_params(case["nx"], case["npart"],
                        deltas=tuple(float(v) for v in case["deltas"].split(",")),
                        delta2=800.0, nbins=case["nbins"],
                        rmin_frac=case["rmin"], rmax_frac=case["rmax"],
                        velocity=case["velocity"])


def _catalogue(ctx, case, seed, with_vel):
    g = P.gen_params(case["npart"], case["nclump"], nlo=20, nhi=case["nhi"],
                     seed=seed + 1, ncentral=case["ncentral"])
    pos, vel, lab, ids, tab = ctx.generate(g, with_vel=with_vel)
    return pos, vel, lab, ids, len(tab["size"])


def prepare(case, seed):
    kind = case["kind"]
    # a captured graph belongs to one set of buffers, so a program that
    # replays keeps a context for them; the other calls share one
    ctx = P.Context(0) if kind == "replay" else P.default_context()
    vel_on = case.get("velocity", False)
    pos, vel, lab, ids, nh = _catalogue(ctx, case, seed, vel_on)
    s = dict(case=case, ctx=ctx, nh=nh)
    if kind in ("host", "greedy"):
        s["pos"], s["ids"] = pos.cpu().numpy(), ids.cpu().numpy()
        if kind == "greedy":
            nx, ng = case["nx"], case["up"] * case["nx"]
            grid = P.cic(s["pos"], ng, xxmin=-0.5)
            rho = P.cicm1(s["pos"], grid, xxmin=-0.5)
            s["isort"], s["nnew"] = P.tri_cic(rho)
            s["table"] = {}
        return s
    s.update(pos=pos, vel=vel, lab=lab, ids=ids)
    ng = case["up"] * case["nx"]
    if kind == "chain":
        return s
    s["p"] = _params(case)
    s["out"] = ctx.alloc_halo_out(nh, case["nbins"])
    s["grid"] = (torch.empty((ng, ng, ng), dtype=torch.float32, device=DEV)
                 if case.get("keep_grid") else None)
    if kind == "sod":
        s["cat"] = ctx.cell_sort(pos, case["nx"], labels=lab)
        grid = ctx.cic_deposit(s["cat"], ng)
        s["seeds"] = ctx.seeds(s["cat"], grid, nh)
        s["nmem"] = ctx.label_counts(lab, nh)
    return s


def run(s):
    case, ctx, kind = s["case"], s["ctx"], s["case"]["kind"]
    nx, ng = case["nx"], case["up"] * case["nx"]
    if kind == "host":
        grid = P.cic(s["pos"], ng, xxmin=-0.5)
        rho = P.cicm1(s["pos"], grid, xxmin=-0.5)
        isort, nnew = P.tri_cic(rho)
        return dict(grid=grid, rho=rho, isort=isort, nnew=nnew)
    if kind == "greedy":
        r = P.spherover(s["pos"], s["ids"], s["isort"], s["nnew"], nx,
                        ncut=case["ncut"], seuil=case["delta"],
                        seuil2=case["delta2"])
        # the records go to the program's halo table, of a fixed length
        o = dict(status=r["status"], alive=r["alive"],
                 structure=r["structure"])
        for k, v in dict(r["halos"], rad_bins=r["rad_bins"],
                         mass_bins=r["mass_bins"]).items():
            t = s["table"].setdefault(
                k, np.zeros((TABLE,) + v.shape[1:], v.dtype))
            m = min(TABLE, len(v))
            t[:m] = v[:m]
            t[m:] = 0
            o[k] = t
        return dict(o, nrec=len(r["rad_bins"]))
    if kind == "chain":
        cat = ctx.cell_sort(s["pos"], nx, labels=s["lab"])
        grid = ctx.cic_deposit(cat, ng, shift=case["shift"])
        rho, _ = ctx.cic_interp(cat, grid, shift=case["shift"])
        seeds = ctx.seeds(cat, grid, s["nh"], shift=case["shift"])
        nmem = ctx.label_counts(cat["lab_sorted"], s["nh"])
        isort, nnew = ctx.density_order(rho)
        # the order of the records inside a cell is left open, so records,
        # their permutation and labels are not compared; what is computed
        # from them is
        return dict(cell_start=cat["cell_start"], grid=grid, rho=rho,
                    seeds=seeds, nmem=nmem, isort=isort, nnew=nnew)
    if kind == "sod":
        return ctx.sod_fof(s["p"], s["cat"], s["pos"], s["seeds"], s["nmem"],
                           vel=s["vel"], ids=s["ids"], out=s["out"])
    kw = dict(ng=ng, vel=s["vel"], ids=s["ids"], grid=s["grid"], out=s["out"])
    if kind == "replay":
        o, _ = ctx.run_pass_graph(s["p"], s["pos"], s["lab"], s["nh"], **kw)
    else:
        o = ctx.run_pass(s["p"], s["pos"], s["lab"], s["nh"], **kw)
    return o if s["grid"] is None else dict(o, grid=s["grid"])


def work(case):
    """Bytes: positions, labels, velocities and ids read once where they are
    used, every output written once.  Flops: the two CIC weightings (8
    corners of about 6 operations) where they are part of the call."""
    n, nx, nh = case["npart"], case["nx"], case["nclump"]
    g3 = (case["up"] * nx) ** 3
    kind = case["kind"]
    row = 4 * (7 + 4) + 8 * (4 * 4 + 2 + 6) + 4 * case.get("nbins", 0)
    if kind == "host":
        return dict(bytes=12 * n + 8 * g3 + 8 * n + 4 * n, flops=96 * n)
    if kind == "greedy":
        return dict(bytes=12 * n + 8 * n + 4 * n + 9 * n, flops=12 * n)
    if kind == "chain":
        return dict(bytes=16 * n + 4 * nx ** 3 + 4 * g3 + 4 * n + 4 * n +
                    8 * nh, flops=96 * n)
    b = 16 * n + nh * row + (4 * g3 if case.get("keep_grid") else 0)
    if kind == "sod":
        return dict(bytes=16 * n + nh * row, flops=12 * n)
    return dict(bytes=b, flops=96 * n)


# ---- the same results in 64 bits, plain torch -------------------------------
def _cells(x, ng, shift):
    """Lower node and offset per axis of scaled coordinates (double)."""
    i = torch.floor(x)
    return (i.long() + shift) % ng, x - i


def _cic(pos, ng, shift=0, weight=None, chunk=1 << 24):
    g = torch.zeros(ng ** 3, dtype=torch.float64, device=DEV)
    n = pos.shape[0]
    w0 = 1.0 / n if weight is None else weight
    for a in range(0, n, chunk):
        i, f = _cells(pos[a:a + chunk].double() * ng, ng, shift)
        for c in range(8):
            b = [c & 1, (c >> 1) & 1, c >> 2]
            w = torch.full((i.shape[0],), w0, dtype=torch.float64, device=DEV)
            k = torch.zeros_like(i[:, 0])
            for d in (2, 1, 0):
                w = w * (f[:, d] if b[d] else 1.0 - f[:, d])
                k = k * ng + (i[:, d] + b[d]) % ng
            g.index_add_(0, k, w)
    return g.mul_(float(ng) ** 3).view(ng, ng, ng)


def _cicm1(pos, grid, shift=0, chunk=1 << 24):
    ng = grid.shape[0]
    rho = torch.zeros(pos.shape[0], dtype=torch.float64, device=DEV)
    flat = grid.view(-1)
    for a in range(0, pos.shape[0], chunk):
        i, f = _cells(pos[a:a + chunk].double() * ng, ng, shift)
        r = rho[a:a + chunk]
        for c in range(8):
            b = [c & 1, (c >> 1) & 1, c >> 2]
            k = torch.zeros_like(i[:, 0])
            w = torch.ones_like(f[:, 0])
            for d in (2, 1, 0):
                w = w * (f[:, d] if b[d] else 1.0 - f[:, d])
                k = k * ng + (i[:, d] + b[d]) % ng
            r += flat[k] * w
    return rho


def _halos(case, pos, vel, lab, nh):
    """The floating outputs of the SOD of every label, brute force."""
    nx, n = case["nx"], case["npart"]
    x = pos.double() * nx
    x = torch.where(x >= nx, x - nx, x)
    rho = _cicm1(pos, _cic(pos, case["up"] * nx))
    cell = torch.floor(x)
    mpart = float(nx) ** 3 / n
    deltas = [float(v) for v in case["deltas"].split(",")]
    z = dict(radius=np.zeros((nh, P.MAXDELTA)), overdens=np.zeros((nh, P.MAXDELTA)),
             rint=np.zeros((nh, P.MAXDELTA)), mint=np.zeros((nh, P.MAXDELTA)),
             overdens2=np.zeros(nh), com_pos=np.zeros((nh, 3)),
             com_vel=np.zeros((nh, 3)))

    def gap(a, b):
        d = a - b
        return d - nx * torch.round(d / nx)

    def od(k, r):
        return k * mpart / (4.0 / 3.0 * math.pi * r ** 3)

    for h in range(nh):
        mem = torch.nonzero(lab == h).squeeze(1)
        seed = mem[torch.argmax(rho[mem])]
        far = gap(cell, cell[seed]).abs().amax(dim=1)
        cand = torch.nonzero(far <= 1).squeeze(1)
        near = x[far <= 2]
        s = torch.empty(len(cand), dtype=torch.float64, device=DEV)
        for a in range(0, len(cand), 1024):
            d2 = gap(x[cand[a:a + 1024], None], near[None]).square().sum(-1)
            t = torch.where(d2 <= 1.0, (d2 + 1.0 / 4096.0).rsqrt(), 0.0)
            s[a:a + 1024] = t.sum(1)
        c = cand[torch.argmax(s)]
        rel = gap(x, x[c])
        r, order = torch.sort(rel.square().sum(1).sqrt())
        k = torch.arange(1, n + 1, dtype=torch.float64, device=DEV)
        o = od(k, r)
        for i, dl in enumerate(deltas):
            ks = int(torch.nonzero((o <= dl) & (k >= 10))[0]) + 1
            r1, r2 = float(r[ks - 2]), float(r[ks - 1])
            o1, o2 = od(ks - 1, r1), od(ks, r2)
            lr = math.log(r2) if not o1 > o2 else math.log(r1) + (
                math.log(dl) - math.log(o1)) * (math.log(r2) - math.log(r1)) / (
                math.log(o2) - math.log(o1))
            z["radius"][h, i], z["overdens"][h, i] = r1, o1
            z["rint"][h, i] = math.exp(lr)
            z["mint"][h, i] = dl * 4.0 / 3.0 * math.pi * math.exp(3 * lr)
            if i == 0:
                up = torch.nonzero(o[1:ks] > 800.0)
                if len(up):
                    z["overdens2"][h] = float(o[int(up[-1]) + 1])
                inside = order[:ks - 1]
                com = (x[c] + rel[inside].mean(0)) / nx
                z["com_pos"][h] = (com - torch.floor(com)).cpu().numpy()
                if vel is not None:
                    z["com_vel"][h] = vel[inside].double().mean(0).cpu().numpy()
    return z


def exact(case, seed):
    kind = case["kind"]
    if kind == "greedy":
        return None
    ctx = P.default_context()
    pos, vel, lab, _, nh = _catalogue(ctx, case, seed,
                                      case.get("velocity", False))
    ng = case["up"] * case["nx"]
    if kind == "host":
        # xxmin = -0.5: nodes shifted by half the box; mpf = 1/N in real(4)
        w = float(np.float32(1.0 / case["npart"]))
        g = _cic(pos, ng, shift=ng // 2, weight=w)
        return dict(grid=g, rho=_cicm1(pos, g, shift=ng // 2), isort=None,
                    nnew=None)
    if kind == "chain":
        g = _cic(pos, ng, shift=case["shift"])
        return dict(cell_start=None, grid=g,
                    rho=_cicm1(pos, g, shift=case["shift"]), seeds=None,
                    nmem=None, isort=None, nnew=None)
    small = case["nx"] <= 64 and nh <= 300
    if not small and not case.get("keep_grid"):
        return None  # the search of every halo takes too long
    z = _halos(case, pos, vel, lab, nh) if small else {}
    if case.get("keep_grid"):
        z["grid"] = _cic(pos, ng)
    return z
