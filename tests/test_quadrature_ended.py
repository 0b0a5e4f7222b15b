"""Samples whose recurrence ends early (small sectors: all later couplings are zero)
take no longer together than one by one."""
import time

import numpy as np
import pytest

from qsi_subspace_ed_amd import ftlm


def _best(f):
    f()
    out = []
    for _ in range(5):
        t0 = time.perf_counter()
        f()
        out.append(time.perf_counter() - t0)
    return min(out)


@pytest.mark.parametrize("n", [1, 5])
def test_time_and_values(n):
    R, M = 64, 2000
    a = np.zeros((R, M))
    b = np.zeros((R, M))
    rng = np.random.default_rng(1)
    a[:, :n] = rng.standard_normal((R, n))
    b[:, :n - 1] = 0.5 + rng.random((R, n - 1))
    got = ftlm.quadrature(a, b)
    for r in range(R):
        e, w = ftlm.tridiag_eig(a[r, :n], b[r, :n])
        assert np.array_equal(got[r][0], e) and np.array_equal(got[r][1], w)
    one = _best(lambda: [ftlm.tridiag_eig(a[r, :int(np.flatnonzero(b[r] == 0.0)[0]) + 1],
                                          b[r, :n]) for r in range(R)])
    assert _best(lambda: ftlm.quadrature(a, b)) <= 2 * one
