"""Expectations and correlations of many small operators in one pass, against
the oracle: column counts at the edges of the 16-column products and of the
128 columns formed in LDS (129 goes through stored columns), bases below and
above 64 rows, operators of several terms, with Z strings and with diagonal
parts, operators too long for the pass, and NaN in a vector.

Every result is a sum of at most D products of two columns whose entries are
sums of at most 20 products, so it differs from the oracle's by at most about
(D + 20) eps sum |products|; the tolerance is that bound at D = 5940."""
import numpy as np
import pytest

import qsi_subspace_ed_amd as q
from oracle import pyoracle as orc
from qsi_subspace_ed_amd import latgen
from qsi_subspace_ed_amd import observables as obs
from qsi_subspace_ed_amd.operators import SymbolicOpSum, SymbolicPMROperator

pytestmark = pytest.mark.gpu
TOL = (5940 + 20) * 2.3e-16


def _sums(jd, n_ops, kind, seed):
    """n_ops operators: single rings; or 1-5 rings, some with a Z on another
    spin, some with a diagonal term, one empty; or 17 ring terms."""
    rings, rings_h, _ = q.get_ring_ops(jd)
    every = rings + rings_h
    rng = np.random.default_rng(seed)
    out = []
    for l in range(n_ops):
        H = SymbolicOpSum()
        if kind == "ring":
            H.add_term(1.0, every[l % len(every)])
        elif kind == "long":
            for k in range(17):
                H.add_term(float(rng.standard_normal()), every[(l + k) % len(every)])
        elif l != 1:
            for _ in range(int(rng.integers(1, 6))):
                o = every[int(rng.integers(len(every)))]
                if rng.random() < 0.3:
                    o = o * SymbolicPMROperator.from_ops("z", [int(rng.integers(8))])
                H.add_term(float(rng.standard_normal()), o)
            if rng.random() < 0.5:
                H.add_term(float(rng.standard_normal()),
                           SymbolicPMROperator.from_ops("zz", [0, int(rng.integers(1, 8))]))
        out.append(H)
    return out


def _check(got, want, scale):
    assert got.shape == want.shape
    assert np.all(np.abs(got - want) <= TOL * scale)


@pytest.mark.parametrize("repeats,sector", [((1, 1, 2), 0), ((2, 2, 2), 0), ((2, 2, 2), 1)])
@pytest.mark.parametrize("n_ops,n_vec,kind", [
    (1, 1, "ring"), (15, 1, "mixed"), (16, 1, "ring"), (17, 1, "mixed"), (4, 17, "mixed"),
    (25, 5, "mixed"), (64, 2, "ring"), (128, 1, "mixed"), (129, 1, "ring"), (43, 3, "mixed"),
    (3, 2, "long")])
def test_against_oracle(cuda, repeats, sector, n_ops, n_vec, kind):
    jd = latgen.Supercell(repeats).to_dict()
    states = q.enumerate_basis(jd, sector)
    sums = _sums(jd, n_ops, kind, 7)
    basis = q.GpuBasis(states, len(jd["atoms"]))
    ops = [q.GpuOp(basis, H) for H in sums]
    ob = orc.Basis(states)
    rng = np.random.default_rng(n_ops + n_vec)
    psi = rng.standard_normal((states.shape[0], n_vec))
    psi /= np.linalg.norm(psi, axis=0)
    d = cuda.from_numpy(psi).cuda()
    # |O_l psi_i| |O_m psi_j| bounds the sums of |products|
    norm = np.array([[np.linalg.norm(orc.evaluate_add(ob, H, psi[:, i].copy(),
                                                      np.zeros(len(states))))
                      for i in range(n_vec)] for H in sums])
    _check(obs.expectations(ops, d), orc.expectations(ob, sums, psi),
           norm[:, :, None] * np.ones(n_vec) + 1e-300)
    _check(obs.cross_correlations(ops, d), orc.cross_correlations(ob, sums, psi),
           norm[:, None, :, None] * norm[None, :, None, :] + 1e-300)


def test_nan_stays_in_its_vector(cuda):
    jd = latgen.Supercell((2, 2, 2)).to_dict()
    basis = q.GpuBasis(q.enumerate_basis(jd), 32)
    ops = [q.GpuOp(basis, H) for H in _sums(jd, 5, "mixed", 3)]
    psi = np.random.default_rng(1).standard_normal((basis.dim(), 2))
    clean = obs.cross_correlations(ops, cuda.from_numpy(psi).cuda())
    psi[17, 1] = np.nan
    got = obs.cross_correlations(ops, cuda.from_numpy(psi).cuda())
    assert np.array_equal(got[:, :, 0, 0], clean[:, :, 0, 0])
