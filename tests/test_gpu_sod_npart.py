"""The batched SOD indexes records by cell_start alone: a catalogue whose
npart says less (the plain method and the growth never read it) gives the same
halos, its centre search included."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("npart", [1, 1000])
def test_sod_fof_does_not_depend_on_npart(npart):
    import torch
    import psod_amd as P
    nx = 64
    n = nx ** 3
    ctx = P.Context(0)
    pos, _, lab, ids, tab = ctx.generate(
        P.gen_params(n, 60, nlo=20, nhi=20000, seed=8), with_vel=False)
    nh = len(tab["size"])
    cat = ctx.cell_sort(pos, nx, labels=lab)
    grid = ctx.cic_deposit(cat, nx)
    seeds = ctx.seeds(cat, grid, nh)
    nmem = ctx.label_counts(lab, nh)
    p = P.sod_params(nx, n, small_max=64)
    ctx.set_tunables(bound_min=1)
    # the smaller npart first: its scratch is not the other call's
    a = ctx.sod_fof(p, dict(cat, npart=npart), pos, seeds, nmem, ids=ids)
    assert ctx.sod_stats()["centre_skipped"] > 0  # windows were in use
    b = ctx.sod_fof(p, cat, pos, seeds, nmem, ids=ids)
    torch.cuda.synchronize()
    for k in ("centre", "count", "radius", "status", "profile", "ngather"):
        np.testing.assert_array_equal(a[k].cpu().numpy(), b[k].cpu().numpy(),
                                      err_msg=k)
    ctx.close()
