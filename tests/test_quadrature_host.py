"""ftlm.quadrature, all samples of a sector in one native call, against
tridiag_eig sample by sample: bit for bit for one sample and for more than there
are threads, one step and many, samples that end early, (R, M - 1) couplings and
strided arrays; and its refusals."""
import numpy as np
import pytest

from qsi_subspace_ed_amd import ftlm


@pytest.mark.parametrize("R,M", [(0, 4), (1, 1), (1, 2), (3, 5), (17, 1), (64, 100), (130, 33)])
def test_samples(R, M):
    rng = np.random.default_rng(R + M)
    a = rng.standard_normal((R, 2 * M))[:, ::2]
    b = 0.5 + rng.random((M, R)).T
    if M > 4:
        b[::3, 3] = 0.0
        b[1::3, 0] = 0.0
    got = ftlm.quadrature(a, b)
    assert len(got) == R
    for r, (e, w) in enumerate(got):
        z = np.flatnonzero(b[r] == 0.0)
        m = int(z[0]) + 1 if z.size else M
        we, ww = ftlm.tridiag_eig(a[r][:m], b[r][:m])
        assert np.array_equal(e, we) and np.array_equal(w, ww)
    for (e, w), (e1, w1) in zip(got, ftlm.quadrature(a, b[:, :M - 1])):
        assert np.array_equal(e, e1) and np.array_equal(w, w1)


def test_refusals():
    a, b = np.ones((3, 6)), np.ones((3, 6))
    b[1, 2] = np.nan
    with pytest.raises(RuntimeError, match="convergence"):
        ftlm.quadrature(a, b)
    with pytest.raises(IndexError):
        ftlm.quadrature(a, np.ones((2, 6)))
    with pytest.raises(RuntimeError):
        ftlm.quadrature(np.ones((2, 0)), np.ones((2, 0)))


def test_ragged():
    """Samples of different lengths, and couplings given only as far as their
    sample goes, are taken one by one."""
    rng = np.random.default_rng(0)
    a = np.empty(3, dtype=object)
    b = []
    for r, m in enumerate((4, 7, 1)):
        a[r] = rng.standard_normal(m)
        b.append(np.append(0.5 + rng.random(m - 1), 0.0))
    for (e, w), x, y in zip(ftlm.quadrature(a, b), a, b):
        we, ww = ftlm.tridiag_eig(x, y)
        assert np.array_equal(e, we) and np.array_equal(w, ww)
    a2 = rng.standard_normal((2, 6))
    b2 = np.array([[0.5, 0.7, 0.0], [0.4, 0.0, 0.0]])
    assert [e.size for e, _ in ftlm.quadrature(a2, b2)] == [3, 2]
