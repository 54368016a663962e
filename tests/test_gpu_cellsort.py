"""Cell sort on the device at the edges of its passes: one and two radix
passes, the chunk sizes, block groups of 1, 2 and 4 (by density), groups
larger than a workgroup holds, ragged counts, with and without labels and
permutation."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def cell_keys(pos, nx):
    """Cell key of every particle, float32 arithmetic as documented."""
    xs = pos * np.float32(nx)
    xs = np.where(xs >= nx, xs - np.float32(nx), xs)
    c = np.floor(xs).astype(np.int64)
    b, l = c >> 3, c & 7
    nb = nx >> 3
    blk = (b[:, 2] * nb + b[:, 1]) * nb + b[:, 0]
    key = (blk << 9) | (l[:, 2] << 6) | (l[:, 1] << 3) | l[:, 0]
    return key, xs - (8 * b).astype(np.float32)


@pytest.mark.parametrize("nx,n,clump,labels,perm", [
    (8, 1, 0.0, True, True),            # one block, one particle
    (8, 60001, 0.0, True, False),       # dense single block, large group
    (16, 3071, 0.0, False, True),       # groups of 4 blocks in one workgroup
    (32, 32768, 0.5, True, True),       # one pass, half in one cell
    (32, 300007, 0.0, True, True),      # density 9: single-block groups
    (64, 1048577, 0.2, True, False),    # first count with chunks of 8192
    (128, 2500000, 0.1, True, True),    # 10 digit bits in one pass
    (256, 3000001, 0.3, False, True),   # two passes, sparse, one huge group
    (512, 5000011, 0.0, True, False),   # two passes of 8 bits, very sparse
    (1024, 4194303, 0.1, True, False),  # 9 and 10 bits
])
def test_cell_sort_matches_keys(nx, n, clump, labels, perm):
    import torch
    import psod_amd as P
    rng = np.random.default_rng(nx + n)
    pos = rng.random((n, 3), dtype=np.float32)
    k = int(clump * n)
    if k:  # a clump inside a few cells
        pos[:k] = (0.3 + rng.random((k, 3)) * 1.5 / nx).astype(np.float32)
    pos[0] = 1.0  # the periodic edge is cell 0
    if n > 2:
        pos[1] = 0.0
        pos[2] = np.nextafter(np.float32(1.0), np.float32(0.0))
    lab = rng.integers(-1, 1000, n).astype(np.int32)
    ctx = P.default_context()
    cat = ctx.cell_sort(torch.from_numpy(pos).cuda(), nx,
                        labels=torch.from_numpy(lab).cuda() if labels else None,
                        want_perm=perm)
    torch.cuda.synchronize()
    key, u = cell_keys(pos, nx)
    cs = cat["cell_start"].cpu().numpy()
    ref = np.zeros(nx ** 3 + 1, np.int64)
    np.cumsum(np.bincount(key, minlength=nx ** 3), out=ref[1:])
    np.testing.assert_array_equal(cs, ref)
    rec = cat["rec"].cpu().numpy()
    idx = np.ascontiguousarray(rec[:, 3]).view(np.int32)
    np.testing.assert_array_equal(np.sort(idx), np.arange(n))
    assert np.all(np.diff(key[idx]) >= 0)  # cell order
    np.testing.assert_array_equal(rec[:, :3], u[idx])  # exact offsets
    if perm:
        np.testing.assert_array_equal(cat["perm"].cpu().numpy(), idx)
    if labels:
        np.testing.assert_array_equal(cat["lab_sorted"].cpu().numpy(), lab[idx])
