"""Centre search beside a record whose position is not finite: the windows of
8 records must not lose the finite ones that share a window with it."""
import numpy as np
import pytest

NX = 64


def cell_key(c):
    nb = NX // 8
    b = ((c[:, 2] >> 3) * nb + (c[:, 1] >> 3)) * nb + (c[:, 0] >> 3)
    return (b << 9) | ((c[:, 2] & 7) << 6) | ((c[:, 1] & 7) << 3) | (c[:, 0] & 7)


def catalogue():
    """Four cells in a row along x, all else within 3 cells of them empty:
    62 holds 8 particles close together at its upper x face (the best S, 616,
    with the help of 7 particles of cell 63); 63 holds those 7 in its sub-cell
    (0, 4, 4) and 56 far from the face; 61 holds 9 close together (S 576, more
    than the 8 have without the 7); 60 holds 60 out of everyone's reach, which
    make 61 the more promising cell.  The last particle of the catalogue lies
    in 63 and in the 7's sub-cell; the count of records before cell 63 is a
    multiple of 8, so that they and it are one window."""
    rng = np.random.default_rng(3)
    back = rng.random((NX ** 3, 3), dtype=np.float32)
    d = np.abs(back * NX - np.array([62.5, 20.5, 20.5]))
    d = np.minimum(d, NX - d)
    back = back[(d > 3.6).any(1)]
    mid = 20.5625
    a = 2 * np.pi * np.arange(7) / 7
    ring = np.stack([np.full(7, 63.03), mid + 0.05 * np.cos(a),
                     mid + 0.05 * np.sin(a)], 1)
    tight = lambda x, m: np.array([x, mid, mid]) + \
        1e-4 * rng.standard_normal((m, 3))
    far = np.stack([rng.uniform(63.96, 63.99, 56), rng.uniform(20.52, 20.98, 56),
                    rng.uniform(20.52, 20.98, 56)], 1)
    more = np.stack([rng.uniform(60.005, 60.035, 60), rng.uniform(20.02, 20.98, 60),
                     rng.uniform(20.02, 20.98, 60)], 1)
    near = np.concatenate([tight(62.99, 8), tight(61.05, 9), ring, far,
                           more]) / NX
    pos = np.concatenate([back, near.astype(np.float32)])
    cells = np.floor(pos * np.float32(NX)).astype(np.int64)
    key = cell_key(cells)
    k63 = cell_key(np.array([[63, 20, 20]]))[0]
    pad = -int((key < k63).sum()) % 8
    fill = np.full((pad, 3), 0.3 / NX, np.float32) + \
        rng.random((pad, 3), dtype=np.float32) * np.float32(0.1 / NX)
    pos = np.concatenate([fill, pos])
    first = len(fill) + len(back)
    last = np.array([[63.06, mid, mid]], np.float32) / NX
    return np.concatenate([pos, last]).astype(np.float32), first


def infinite_x(pos):
    """The last particle with x = +inf and a y whose cell sort lands in cell
    63 all the same: the integer cell of +inf is 2^31 - 1 - NX after the wrap,
    so its block offset along x is -9 modulo the blocks, two rows of blocks
    back and the last block along x."""
    out = pos.copy()
    out[-1] = (np.inf, (pos[-1, 1] * NX + 16) / NX, pos[-1, 2])
    return out


@pytest.mark.gpu
def test_window_with_an_infinite_record():
    import torch
    import psod_amd as P
    base, first = catalogue()
    n = len(base)
    # the finite particle moved out of every cell around the halo
    without = base.copy()
    without[-1] = (0.3 / NX, 0.3 / NX, 0.3 / NX)
    ctx = P.Context(0)
    p = P.sod_params(NX, n, deltas=(200.0,), small_max=1)
    seeds = torch.tensor([first], dtype=torch.int32, device="cuda")
    nmem = torch.tensor([18], dtype=torch.int32, device="cuda")
    ctx.set_tunables(bound_min=1)
    got = {}
    for name, x in (("without", without), ("inf", infinite_x(base))):
        pos = torch.from_numpy(x).cuda()
        cat = ctx.cell_sort(pos, NX)
        if name == "inf":  # as planned: 8 records from a multiple of 8
            cs = cat["cell_start"].cpu().numpy()
            k63 = cell_key(np.array([[63, 20, 20]]))[0]
            rec = cat["rec"].cpu().numpy()[cs[k63]:cs[k63 + 1]]
            assert cs[k63] % 8 == 0 and len(rec) == 64
            assert np.isinf(rec[:8, 0]).sum() == 1
            assert (rec[:8, 3].view(np.int32) >= first + 17).all()
        o = ctx.sod_fof(p, cat, pos, seeds, nmem)
        torch.cuda.synchronize()
        got[name] = (int(o["centre"][0]), int(o["count"][0, 0]))
    ctx.close()
    assert first <= got["without"][0] < first + 8
    assert got["inf"] == got["without"]
