"""Deposit and interpolation of a catalogue whose cell_start counts more
records than the npart of the call (which only scales the deposit): the lists
of pieces are sized by npart, and what does not fit them is done whole."""
import ctypes as C

import numpy as np
import pytest


def dense(nx, n, seed):
    """n particles, all but 1000 of them in one 8^3 block."""
    rng = np.random.default_rng(seed)
    pos = rng.random((n, 3), dtype=np.float32)
    pos[1000:] = (pos[1000:] * np.float32(6.0) + np.float32(9.0)) / np.float32(nx)
    return pos


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ng", [(32, 32), (32, 64)])
@pytest.mark.parametrize("npart", [1 << 17, 300001, 1 << 20])
def test_deposit_with_fewer_particles_than_records(nx, ng, npart):
    import torch
    import psod_amd as P
    from psod_amd import _lib
    L = _lib.load()
    ctx = P.Context(0)
    n = 1200007
    pos = torch.from_numpy(dense(nx, n, npart)).cuda()
    cat = ctx.cell_sort(pos, nx)
    got = ctx.cic_deposit(dict(cat, npart=npart), ng)
    # without lists of pieces: the same sums and the same scale
    want = torch.empty_like(got)
    torch.cuda.synchronize()
    _lib.check(L.psod_cic_deposit_noalloc(
        ctx.h, npart, nx, C.c_void_p(cat["cell_start"].data_ptr()),
        C.c_void_p(cat["rec"].data_ptr()), ng, 0,
        C.c_void_p(want.data_ptr())))
    ctx.synchronize()
    torch.testing.assert_close(got, want, rtol=0, atol=0)
    full = ctx.cic_deposit(cat, ng).double() * (n / npart)
    torch.testing.assert_close(got.double(), full, rtol=3e-7, atol=0)
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("npart", [1 << 21, (1 << 21) + 4097])
def test_seeds_with_fewer_particles_than_records(npart):
    import torch
    import psod_amd as P
    ctx = P.Context(0)
    nx, n, nh = 32, 5000003, 50
    pos = torch.from_numpy(dense(nx, n, 3)).cuda()
    lab = torch.randint(-1, nh, (n,), dtype=torch.int32, device="cuda")
    cat = ctx.cell_sort(pos, nx, labels=lab)
    grid = ctx.cic_deposit(cat, nx)
    want = ctx.seeds(cat, grid, nh)
    got = ctx.seeds(dict(cat, npart=npart), grid, nh)
    assert (want >= 0).all()
    torch.testing.assert_close(got, want, rtol=0, atol=0)
    ctx.close()
