"""Greedy spherover on the device at the edges of its launches: seeds whose
gathered particles are sorted whole in LDS, whose crossing lies in the first
radial bins, whose crossing needs more keys than LDS holds, cubes of more
cells than a gather workgroup has threads, both marking-block sizes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ncentral,nclump,nhi,ncut,rmax,mmin,seuil", [
    (8, 300, 0, 100, 3, 1.0, 20.0, 200.0),       # smallest grid, tiny sorts
    (32, 20000, 20, 500, 5, 1.0, 100.0, 200.0),  # > 8192 keys inside R
    (64, 5000, 60, 2000, 10, 1.5, 100.0, 200.0),  # > 8192 gathered, fewer in R
    (32, 0, 60, 3000, 2, 1.0, 20.0, 500.0),      # small cubes
    (32, 9000, 20, 2000, 9, 2.0, 50.0, 300.0),   # 8^3 marking blocks
])
def test_greedy_sizes_match_oracle(orc, nx, ncentral, nclump, nhi, ncut, rmax,
                                   mmin, seuil):
    import psod_amd as P
    pos, _, _, ids, _ = orc.generate(
        orc.gen_params(nx ** 3, nclump, nlo=20, nhi=nhi, seed=5,
                       ncentral=ncentral), with_vel=False)
    rho = orc.cicm1(pos, orc.cic(pos, 2 * nx, xxmin=-0.5), xxmin=-0.5)
    _, isort, nnew = orc.tri_cic(rho)
    kw = dict(ncut=ncut, seuil=seuil, mmin=mmin, nbins=40, rmax_frac=rmax)
    r = orc.sod_greedy(pos, ids, isort, nnew,
                       orc.greedy_params(nx, ref_order=0, **kw))
    g = P.spherover(pos, ids, isort, nnew, nx, **kw)
    assert g["status"] == r["status"]
    hr, hg = r["halos"], g["halos"]
    assert len(hg["ipart"]) == len(hr["ipart"]) > 0
    # whole numbers equal; distances come from the same FP64 expressions
    for k in ("ipart", "seed", "centre", "iamas", "masse", "masse2", "rayon",
              "amass", "xc", "yc", "zc", "overdens", "accepted"):
        np.testing.assert_array_equal(hg[k], hr[k], err_msg=k)
    np.testing.assert_array_equal(g["mass_bins"], r["mass_bins"])
    np.testing.assert_allclose(g["rad_bins"], r["rad_bins"], rtol=1e-15)
    if r["status"] == P.OK:  # an aborted zone leaves later seeds' flags open
        np.testing.assert_array_equal(g["alive"], r["alive"])
        np.testing.assert_array_equal(g["structure"], r["structure"])
