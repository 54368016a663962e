"""Greedy spherover where a seed fails: the zone ends at the first failing
seed in seed order, whatever order the seeds ran in.  Records, captured
particles, structure ids and the seed named by the error are those of the
sequential loop (the oracle)."""
import re

import numpy as np
import pytest

NX, NCUT = 64, 2
BIG = 9000  # not closed within 2 cells: (BIG / 200 / (4 pi / 3))^(1/3) = 2.2


def catalogue(chain, others):
    """A unit-density background and compact clumps.  `chain` clumps lie 3
    cells apart in seed order, so that each waits for the one before it;
    `others` are far from them and from each other.  Entries are clump sizes;
    the seeds are the clumps' first particles in that order."""
    rng = np.random.default_rng(7)
    back = rng.random((NX ** 3, 3))
    at = [(4.5 + 3 * i, 8.5, 8.5) for i in range(len(chain))] + \
         [(8.5 + 12 * (i % 4), 40.5, 20.5 + 12 * (i // 4))
          for i in range(len(others))]
    parts, seeds, n = [back], [], len(back)
    for c, m in zip(at, list(chain) + list(others)):
        parts.append((np.array(c) + rng.uniform(-0.25, 0.25, (m, 3))) / NX)
        seeds.append(n)
        n += m
    pos = np.concatenate(parts).astype(np.float32)
    return pos, np.array(seeds, np.int32)


CASES = {
    # the last seed fails at once; the chain needs a round per seed
    "isolated_last": ([300] * 12, [BIG], list(range(13))),
    # it fails at once, then a chain seed, which comes first; seeds after it
    # have captured their particles by then
    "chain_too": ([300] * 5 + [BIG] + [300] * 4, [BIG, 250, 260],
                  list(range(13))),
    # the first seed of all fails beside seeds that run in the same round
    "first": ([BIG, 300, 300], [250, 260], list(range(5))),
    # a seed early in the order fails, isolated, after seeds of a later place
    "between": ([300] * 9, [BIG, 250], [0, 1, 2, 3, 9, 4, 5, 6, 7, 8, 10]),
}


@pytest.mark.gpu
@pytest.mark.parametrize("nsel", [4_000_000, 5000])
@pytest.mark.parametrize("name", list(CASES))
def test_zone_ends_at_the_first_failing_seed(orc, name, nsel):
    import torch  # noqa: F401  (its HIP runtime is loaded first)
    import psod_amd as P
    chain, others, order = CASES[name]
    pos, seeds = catalogue(chain, others)
    isort = np.zeros(len(pos), np.int32)
    isort[:len(order)] = seeds[order] + 1
    ids = np.arange(len(pos), dtype=np.int64) * 3 + 5
    nnew = len(order)
    kw = dict(ncut=NCUT, mmin=50.0, nbins=8)
    r = orc.sod_greedy(pos, ids, isort, nnew, orc.greedy_params(
        NX, ref_order=0, nsel=min(nsel, len(pos)), **kw))
    fail = [k for k, o in enumerate(order) if (chain + others)[o] == BIG][0]
    want = P.E_CAPACITY if nsel < BIG else P.E_UNCLOSED
    assert r["status"] == want and len(r["halos"]["ipart"]) == fail
    g = P.spherover(pos, ids, isort, nnew, NX, nsel=nsel, **kw)
    assert g["status"] == want
    from psod_amd import _lib
    msg = _lib.load().psod_last_error().decode()
    assert re.search(rf"\bseed {fail + 1}\b", msg), msg
    for k in ("ipart", "seed", "centre", "iamas", "masse", "masse2", "rayon",
              "overdens", "accepted"):
        np.testing.assert_array_equal(g["halos"][k], r["halos"][k], err_msg=k)
    np.testing.assert_array_equal(g["mass_bins"], r["mass_bins"])
    np.testing.assert_array_equal(g["alive"], r["alive"])
    np.testing.assert_array_equal(g["structure"], r["structure"])
