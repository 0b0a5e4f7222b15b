"""Observables of few operators: no more time than a few applies and dot products
take, and on a large basis of two-word states the same values as among more
operators, which go through another kernel."""
import time

import numpy as np
import pytest

import qsi_subspace_ed_amd as q
from qsi_subspace_ed_amd import latgen
from qsi_subspace_ed_amd import observables as obs

pytestmark = pytest.mark.gpu


def _best(f, n=7):
    f()
    out = []
    for _ in range(n):
        t0 = time.perf_counter()
        f()
        out.append(time.perf_counter() - t0)
    return min(out) * 1e6


@pytest.mark.parametrize("repeats", [(2, 2, 3), (2, 2, 4), (2, 3, 3)])
@pytest.mark.parametrize("long", [False, True])
def test_time(cuda, repeats, long):
    """One operator on one vector against the same by torch: an apply into a vector
    that is allocated for it and freed, as the call does, and a dot product; 1.5
    times as long and 30 us allowed."""
    jd = latgen.Supercell(repeats).to_dict()
    basis = q.enumerate_basis_device(jd, 0)
    if long:
        op = q.GpuOp(basis, q.build_hamiltonian_g(jd, [-0.9, -0.5, -0.3, -0.7]))
    else:
        op = obs.ring_operators(basis, jd)[0]
    psi = cuda.randn(basis.dim(), 1, dtype=cuda.float64, device="cuda")

    def ref():
        v = psi.t().contiguous()[0]
        y = cuda.empty_like(v)
        op.evaluate(v, y)
        cuda.dot(v, y).item()
        del y
        cuda.cuda.empty_cache()

    got = _best(lambda: obs.expectations([op], psi))
    want = _best(ref)
    assert got <= 1.5 * want + 30.0, (got, want)


def test_two_word_states(cuda):
    jd = latgen.Supercell((2, 3, 3)).to_dict()
    basis = q.enumerate_basis_device(jd, 0)
    ops = obs.ring_operators(basis, jd)[:17]
    psi = cuda.randn(basis.dim(), 1, dtype=cuda.float64, device="cuda",
                     generator=cuda.Generator(device="cuda").manual_seed(1))
    psi /= cuda.linalg.norm(psi)
    # sums of D products of unit vectors
    tol = 2 * basis.dim() * 2.0 ** -53
    more = obs.expectations(ops, psi)
    for n in (1, 2, 3, 16):
        assert np.abs(obs.expectations(ops[:n], psi) - more[:n]).max() <= tol
    more = obs.cross_correlations(ops, psi)
    for n in (2, 8, 9):
        assert np.abs(obs.cross_correlations(ops[:n], psi) - more[:n, :n]).max() <= tol
