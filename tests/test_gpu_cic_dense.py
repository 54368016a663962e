"""CIC deposit and interpolation where one tile or block holds very many
records: tiles deposited in pieces, blocks interpolated by several workgroups,
at the sizes where the splitting begins and with remainders."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def catalogue(nx, nback, ndense, seed):
    """nback uniform particles and ndense in two cells of one block, one of
    them at the block's upper corner (its nodes belong to other tiles too)."""
    rng = np.random.default_rng(seed)
    pos = rng.random((nback + ndense, 3), dtype=np.float32)
    cell = np.where(rng.random((ndense, 1)) < 0.5, 15, 11)
    pos[nback:] = ((cell + rng.random((ndense, 3))) / nx).astype(np.float32)
    lab = rng.integers(-1, 7, nback + ndense).astype(np.int32)
    return pos, lab


def nodes(cat, ng):
    """Lower node and float32 offsets of every record, in record order."""
    nx, R = cat["nx"], ng // cat["nx"]
    nb = nx // 8
    cs = cat["cell_start"].cpu().numpy()
    blk = np.repeat(np.arange(nb ** 3), np.diff(cs[::512]))
    rec = cat["rec"].cpu().numpy()
    q = rec[:, :3] * np.float32(R)
    lo = np.floor(q)
    b = np.stack([blk % nb, blk // nb % nb, blk // nb ** 2], 1)
    return b * 8 * R + lo.astype(np.int64), (q - lo).astype(np.float32)


def corners(i0, f, ng, shift, dtype):
    w = [1 - f.astype(dtype), f.astype(dtype)]
    for c in range(8):
        o = np.array([c & 1, (c >> 1) & 1, c >> 2])
        i = (i0 + o + shift) % ng
        yield ((i[:, 2] * ng + i[:, 1]) * ng + i[:, 0],
               w[o[0]][:, 0], w[o[1]][:, 1], w[o[2]][:, 2])


@pytest.mark.parametrize("ndense", [(1 << 17) - 3000, 1 << 17,
                                    (1 << 17) + 32769, 900001])
@pytest.mark.parametrize("nx,ng,shift", [(32, 32, 0), (32, 64, 5), (8, 8, 3)])
def test_dense_tiles(nx, ng, shift, ndense):
    import torch
    import psod_amd as P
    if nx == 8:
        ndense //= 2
    pos, _ = catalogue(max(nx, 16), 40000, ndense, ndense)
    ctx = P.default_context()
    cat = ctx.cell_sort(torch.from_numpy(pos).cuda(), nx)
    grid = ctx.cic_deposit(cat, ng, shift=shift).cpu().numpy().ravel()
    i0, f = nodes(cat, ng)
    hi = np.zeros(ng ** 3)
    lo = np.zeros(ng ** 3)
    for i, wx, wy, wz in corners(i0, f, ng, shift, np.float32):
        w = np.rint(wx * wy * wz * np.float32(2.0 ** 36)).astype(np.int64)
        hi += np.bincount(i, weights=w >> 20, minlength=ng ** 3)
        lo += np.bincount(i, weights=w & 0xFFFFF, minlength=ng ** 3)
    s = (hi.astype(np.int64) << 20) + lo.astype(np.int64)
    norm = float(ng) ** 3 / len(pos)
    want = (s.astype(np.float64) * 2.0 ** -36 * norm).astype(np.float32)
    np.testing.assert_array_equal(grid, want)


@pytest.mark.parametrize("ndense", [16380, 16384, 32768 + 257, 500003])
@pytest.mark.parametrize("ng,shift", [(32, 0), (64, 3)])
def test_dense_blocks(ng, shift, ndense):
    import torch
    import psod_amd as P
    nx, nhalo = 32, 7
    # the background keeps the count above that where blocks are shared
    pos, lab = catalogue(nx, (1 << 21) + 11, ndense, ndense)
    ctx = P.default_context()
    cat = ctx.cell_sort(torch.from_numpy(pos).cuda(), nx,
                        labels=torch.from_numpy(lab).cuda())
    grid = ctx.cic_deposit(cat, ng, shift=shift)
    key = torch.full((nhalo,), -1, dtype=torch.int64, device="cuda")
    rho, rs = ctx.cic_interp(cat, grid, shift=shift, sorted_out=True,
                             nhalo=nhalo, seed_key=key)
    i0, f = nodes(cat, ng)
    g = grid.cpu().numpy().ravel().astype(np.float64)
    want = np.zeros(len(pos))
    for i, wx, wy, wz in corners(i0, f, ng, shift, np.float64):
        want += g[i] * wx * wy * wz
    rs = rs.cpu().numpy()
    # one rounding to float of a sum of 8 positive terms in double
    np.testing.assert_allclose(rs, want, rtol=2.0 ** -23)
    idx = cat["rec"].cpu().numpy()[:, 3].view(np.int32)
    got = np.empty(len(pos), np.float32)
    got[idx] = rs
    np.testing.assert_array_equal(rho.cpu().numpy(), got)
    k = (got.view(np.uint32).astype(np.uint64) << np.uint64(32)) | \
        (np.uint64(0xFFFFFFFF) - np.arange(len(pos), dtype=np.uint64))
    wk = np.array([k[lab == h].max() for h in range(nhalo)], np.uint64)
    np.testing.assert_array_equal(key.cpu().numpy().view(np.uint64), wk)


def test_non_finite_positions_add_nothing():
    """A record whose offsets are not finite has weight 0 at every node."""
    import torch
    import psod_amd as P
    pos, _ = catalogue(32, 5000, 0, 1)
    ctx = P.default_context()
    cat = ctx.cell_sort(torch.from_numpy(pos).cuda(), 32)
    want = ctx.cic_deposit(cat, 32).cpu().numpy()
    rec = cat["rec"]
    i0, f = nodes(cat, 32)
    keep = np.ones(5000, bool)
    keep[::50] = False
    rec[torch.from_numpy(np.flatnonzero(~keep)).cuda(), 1] = float("nan")
    got = ctx.cic_deposit(cat, 32).cpu().numpy().ravel()
    s = np.zeros(32 ** 3, np.int64)
    for i, wx, wy, wz in corners(i0[keep], f[keep], 32, 0, np.float32):
        w = np.rint(wx * wy * wz * np.float32(2.0 ** 36)).astype(np.int64)
        np.add.at(s, i, w)
    ref = (s.astype(np.float64) * 2.0 ** -36 * (32.0 ** 3 / 5000)).astype(
        np.float32)
    np.testing.assert_array_equal(got, ref)
    assert want.sum() > got.sum()
