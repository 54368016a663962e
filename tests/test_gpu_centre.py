"""Centre search: the bounded search (windows of 8 records, boxes of 16
candidates, pilots, items) against the exhaustive one, where every candidate
is summed, on catalogues whose cells span the sizes at which the windows
start (64 records) up to thousands."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nclump,nhi,ncentral,seed", [
    (16, 3, 800, 1500, 1),     # few cells, seeds near the periodic edge
    (32, 40, 6000, 0, 2),
    (64, 200, 20000, 40000, 3),
    (64, 900, 1500, 0, 4),     # many halos just above the bound
])
def test_bounded_search_matches_exhaustive(nx, nclump, nhi, ncentral, seed):
    import torch
    import psod_amd as P
    n = nx ** 3
    ctx = P.Context(0)
    pos, _, lab, ids, tab = ctx.generate(
        P.gen_params(n, nclump, nlo=20, nhi=nhi, seed=seed,
                     ncentral=ncentral), with_vel=False)
    nh = len(tab["size"])
    cat = ctx.cell_sort(pos, nx, labels=lab)
    grid = ctx.cic_deposit(cat, nx)
    seeds = ctx.seeds(cat, grid, nh)
    nmem = ctx.label_counts(lab, nh)
    # small_max = 1: every halo takes the large path
    p = P.sod_params(nx, n, small_max=1)
    out = {}
    for name, bound_min in (("bounded", 1), ("exhaustive", 1 << 30)):
        ctx.set_tunables(bound_min=bound_min)
        out[name] = ctx.sod_fof(p, cat, pos, seeds, nmem, ids=ids)
    torch.cuda.synchronize()
    for k in ("centre", "count", "radius", "status"):
        np.testing.assert_array_equal(out["bounded"][k].cpu().numpy(),
                                      out["exhaustive"][k].cpu().numpy(),
                                      err_msg=k)
    assert (out["bounded"]["centre"] >= 0).all()
    ctx.close()
