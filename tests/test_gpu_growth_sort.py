"""Sorted bands and cubes of the large halos' growth: keys ranked in LDS bins,
bands cut into pieces that fit there, and the cases left to the bitonic
network (many coincident distances).  The routes (cube sorted whole, radial
bins in one workgroup, staged launches) and the oracle have to agree."""
import numpy as np
import pytest

from parity import check_sod

pytestmark = pytest.mark.gpu

NX = 64


def halos(kind, sizes, seed):
    """Clumps of the given sizes over a thin background, labelled."""
    rng = np.random.default_rng(seed)
    n = NX ** 3
    pos, lab = [], []
    for i, m in enumerate(sizes):
        c = (np.array([12 + 20 * (i % 3), 12 + 20 * (i // 3 % 3),
                       12 + 20 * (i // 9)]) + 0.3) / NX
        u = rng.normal(size=(m, 3))
        u /= np.linalg.norm(u, axis=1)[:, None]
        if kind == "ball":  # overdensity 200 throughout: crossings anywhere
            r = (m / (200 * 4.18879)) ** (1 / 3) * rng.random(m) ** (1 / 3)
        else:
            r = 6.0 * rng.random(m) ** 2
        x = r[:, None] * u
        if kind == "lattice":  # many particles at each distance
            x = np.round(x * 4) / 4
        pos.append(c + x / NX)
        lab.append(np.full(m, i))
    k = n - sum(sizes)
    pos.append(rng.random((k, 3)))
    lab.append(np.full(k, -1))
    pos = (np.concatenate(pos) % 1.0).astype(np.float32)
    return pos, np.concatenate(lab).astype(np.int32)


@pytest.mark.parametrize("kind", ["cusp", "ball", "lattice"])
@pytest.mark.parametrize("sizes", [(130, 700, 1025, 4095, 4097),
                                   (6000, 8100, 12000),
                                   (30000, 60000, 90000)])
def test_growth_routes_agree(orc, kind, sizes, monkeypatch):
    import torch
    import psod_amd as P
    pos, lab = halos(kind, sizes, len(sizes))
    n, nh = len(pos), len(sizes)
    ctx = P.Context(0)
    dpos = torch.from_numpy(pos).cuda()
    dlab = torch.from_numpy(lab).cuda()
    ids = torch.arange(n, dtype=torch.int64, device="cuda")
    vel = torch.from_numpy(np.random.default_rng(1).normal(
        size=(n, 3)).astype(np.float32)).cuda()
    cat = ctx.cell_sort(dpos, NX, labels=dlab)
    seeds = ctx.seeds(cat, ctx.cic_deposit(cat, NX), nh)
    nmem = ctx.label_counts(dlab, nh)
    deltas = (200.0, 450.0)
    p = P.sod_params(NX, n, deltas=deltas, delta2=800.0, nbins=32,
                     rmin_frac=0.01, rmax_frac=1.5, mmin=100.0, small_max=1,
                     velocity=True)

    def run():
        o = ctx.sod_fof(p, cat, dpos, seeds, nmem, vel=vel, ids=ids)
        torch.cuda.synchronize()
        return {k: v.cpu().numpy() for k, v in o.items()}

    out = {"whole": run()}
    monkeypatch.setenv("PSOD_LIGHT_CAP", "0")
    out["bins"] = run()
    ctx.set_tunables(giant_min=1)
    out["staged"] = run()
    monkeypatch.delenv("PSOD_LIGHT_CAP")
    a = out["whole"]
    exact = ("centre", "count", "radius", "count2", "profile", "status",
             "nboundary")
    for r in ("bins", "staged"):
        for k in exact:
            np.testing.assert_array_equal(a[k], out[r][k], err_msg=f"{r} {k}")
    ctx.close()
    if kind == "lattice":
        return  # ties everywhere: decided by float32 distances
    cs, perm = orc.cell_sort(pos, NX, 8)
    fp = orc.fof_params(NX, n, deltas=deltas, delta2=800.0, nbins=32,
                        rmin_frac=0.01, rmax_frac=1.5, mmin=100.0)
    r = orc.sod_fof(pos, cs, perm, 8, seeds.cpu().numpy().astype(np.int64),
                    nmem.cpu().numpy().astype(np.int64), fp,
                    vel=vel.cpu().numpy(), ids=ids.cpu().numpy())
    check_sod(a, r, len(deltas))
