"""Interpolation of blocks shared by several workgroups: blocks of exactly,
one fewer and one more than a multiple of the records of a piece (4096), and
totals on both sides of the count from which blocks are shared."""
import ctypes as C

import numpy as np
import pytest

EDGES = [0, 1, 4095, 4096, 4097, 8191, 8192, 8193, 12289]


def catalogue(nx, total, seed):
    """EDGES records in the first blocks of a row, the rest even over the
    other blocks (fewer than 4096 each), labels at random."""
    rng = np.random.default_rng(seed)
    nblk = (nx // 8) ** 3
    cnt = np.zeros(nblk, np.int64)
    cnt[:len(EDGES)] = EDGES
    rest = total - sum(EDGES)
    q, r = divmod(rest, nblk - len(EDGES))
    cnt[len(EDGES):] = q
    cnt[len(EDGES):len(EDGES) + r] += 1
    assert q + 1 < 4096
    blk = np.repeat(np.arange(nblk), cnt)
    nb = nx // 8
    org = np.stack([blk % nb, blk // nb % nb, blk // nb ** 2], 1) * 8
    # offsets of at most 8 - 2^-10 cells: the sum stays in the block
    pos = ((org + rng.integers(0, 8192, (total, 3)) / 1024.0) / nx).astype(
        np.float32)
    p = rng.permutation(total)
    return pos[p], rng.integers(-1, 5, total).astype(np.int32), blk[p], cnt


@pytest.mark.gpu
@pytest.mark.parametrize("nx,total", [
    (64, 1 << 20), (128, (1 << 21) - 1), (128, 1 << 21),
    (128, (1 << 21) + 4097)])
@pytest.mark.parametrize("up,shift", [(1, 0), (2, 3)])
def test_blocks_at_the_edges_of_pieces(nx, total, up, shift):
    import torch
    import psod_amd as P
    from psod_amd import _lib
    L = _lib.load()
    ng, nh = up * nx, 5
    pos, lab, blk, cnt = catalogue(nx, total, total)
    ctx = P.Context(0)
    cat = ctx.cell_sort(torch.from_numpy(pos).cuda(), nx,
                        labels=torch.from_numpy(lab).cuda())
    cs = cat["cell_start"].cpu().numpy()
    np.testing.assert_array_equal(np.diff(cs[::512]), cnt)
    grid = torch.rand((ng, ng, ng), dtype=torch.float32, device="cuda") + 0.5
    rs = torch.full((total,), float("nan"), device="cuda")
    ro = torch.full((total,), float("nan"), device="cuda")
    key = torch.full((nh,), -1, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    ptr = lambda t: C.c_void_p(t.data_ptr())
    _lib.check(L.psod_cic_interp(ctx.h, total, nx, ptr(cat["cell_start"]),
                                 ptr(cat["rec"]), ng, shift, ptr(grid),
                                 ptr(rs), ptr(ro), ptr(cat["lab_sorted"]), nh,
                                 ptr(key)))
    rec = cat["rec"].cpu().numpy()
    idx = rec[:, 3].view(np.int32)
    # the sum of 8 products in double, as torch gives it
    x = torch.from_numpy(pos).cuda().double() * ng
    i0 = torch.floor(x).long()
    f = x - i0
    want = torch.zeros(total, dtype=torch.float64, device="cuda")
    g = grid.double().ravel()
    for c in range(8):
        o = torch.tensor([c & 1, (c >> 1) & 1, c >> 2], device="cuda")
        i = (i0 + o + shift) % ng
        w = torch.where(o == 1, f, 1 - f)
        want += g[(i[:, 2] * ng + i[:, 1]) * ng + i[:, 0]] * w.prod(1)
    want, ro, rs = want.cpu().numpy(), ro.cpu().numpy(), rs.cpu().numpy()
    # one rounding to float of a sum of 8 positive terms in double
    np.testing.assert_allclose(ro, want, rtol=2.0 ** -23)
    np.testing.assert_array_equal(rs, ro[idx])
    k = (ro.view(np.uint32).astype(np.uint64) << np.uint64(32)) | \
        (np.uint64(0xFFFFFFFF) - np.arange(total, dtype=np.uint64))
    wk = np.array([k[lab == h].max() for h in range(nh)], np.uint64)
    np.testing.assert_array_equal(key.cpu().numpy().view(np.uint64), wk)
    ctx.close()
