"""Counts near 2^31: records are indexed with 32 bits and kernels step past
the end of their lists before they compare, so the entry points that sort
particles into cells refuse counts within 2^16 of it, before they touch the
device (no GPU is needed to see it)."""
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIMIT = (1 << 31) - (1 << 16)


def call(L, name, n):
    """The entry point with n particles and a null context: its message."""
    from psod_amd import _lib
    args = {
        "psod_cell_sort": (None, n, None, None, 64, None, None, None, None),
        "psod_pass": (None, None, n, 64, 64, None, None, None, None, 1, None,
                      None),
        "psod_pass_graph": (None, None, n, 64, 64, None, None, None, None, 1,
                            None, None, None),
        "psod_autotune": (None, None, n, 64, None, None, None, None, 1, 1,
                          None, None, None),
        "psod_host_spherover": (None, n, None, None, None, 0, None, 1, None,
                                None, None, None, None, None, None),
    }[name]
    assert getattr(L, name)(*args) == _lib.E_ARG
    return L.psod_last_error().decode()


@pytest.mark.parametrize("name", ["psod_cell_sort", "psod_pass",
                                  "psod_pass_graph", "psod_autotune",
                                  "psod_host_spherover"])
def test_counts_near_2_31_are_refused_first(name):
    from psod_amd import _lib
    L = _lib.load()
    for n in (LIMIT + 1, (1 << 31) - 1, 1 << 31, 1 << 40):
        assert re.search(rf"{n} particles, at most {LIMIT}", call(L, name, n))
    for n in (1, LIMIT):
        assert "null context" in call(L, name, n)


def test_header_states_the_limit():
    src = open(os.path.join(ROOT, "include", "psod.h")).read()
    assert int(re.search(r"PSOD_NPART_MAX (\d+)LL", src).group(1)) == LIMIT
