"""The thick-restart solvers' Rayleigh-Ritz: what the solve engine returns where a
request's projected matrix is not finite, on both sides of the order up to which
the device diagonalises it; vectors that keep their norm over restarts; and
operators that are not symmetric."""
import numpy as np
import pytest

import qsi_subspace_ed_amd as q
from qsi_subspace_ed_amd import latgen, serve
from qsi_subspace_ed_amd.operators import SymbolicOpSum, SymbolicPMROperator

pytestmark = pytest.mark.gpu


def _point():
    return serve.point_coeffs([-0.9, -0.5, -0.3, -0.7], q.get_loc_z() @ [0.05, -0.02, 0.07])


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("slot", [0, 5])
@pytest.mark.parametrize("ncv", [8, 15, 48, 49])
def test_engine_not_finite(cuda, value, slot, ncv):
    """A request with a coefficient that is not finite, beside good requests and
    in the column of an earlier one: its values are all NaN, theirs unchanged."""
    jd = latgen.Supercell((2, 2, 2)).to_dict()
    op = q.GpuOp(q.enumerate_basis_device(jd, 0), serve.slotted_hamiltonian(jd))
    good = _point()
    bad = good.copy()
    bad[slot] = value
    eng = serve.Engine(op, max_cols=3, nev=3, ncv=ncv, tol=1e-10, max_restarts=4, autotune=False)

    def run(reqs):
        ids = [eng.submit(c, s) for c, s in reqs]
        got = {f.id: f for f in eng.run_all()}
        return [got[i] for i in ids]

    want = [f.evals for f in run([(good, 3), (good, 4), (good, 5)])]
    assert np.isfinite(want).all()
    got = run([(good, 3), (bad, 6), (good, 5), (good, 4), (bad, 7)])
    for k, w in ((0, 0), (2, 2), (3, 1)):
        assert np.array_equal(got[k].evals, want[w])
    for k in (1, 4):
        assert np.isnan(got[k].evals).all() and got[k].nconv == 0


@pytest.mark.parametrize("nev,ncv", [(8, 32), (10, 40), (12, 47), (12, 48)])
def test_vectors_keep_their_norm(cuda, nev, ncv):
    """A thick restart keeps Ritz vectors without normalising them again, so the
    rotations that form their coefficients must not grow or shrink vectors on
    average: an error of one sign in c^2 + s^2 adds up.  A vector sees about ten
    sweeps of ncv rotations in each of four cycles, each rounding its square norm
    by 2^-53 (root mean square) either way: a random walk of sqrt(40 ncv) 2^-53,
    and 1 / sqrt(nev) of that for the mean of nev vectors.  Six of these are
    allowed."""
    from test_gpu_restart import _basis, _terms
    states, spins, W = _basis(1, 10, 513, 513)
    H = _terms(spins, 24, 10, z=False, open_spins=False)
    for k, p in enumerate(spins):
        H.add_term(0.37 * 1.61 ** (k % 7) + 0.011 * k, SymbolicPMROperator.from_ops("z", [p]))
    op = q.GpuOp(q.GpuBasis(states, W), H)
    _, vecs, _, _ = op.eigsh(nev=nev, ncv=ncv, tol=1e-30, max_restarts=3, seed=3, n_evecs=nev,
                             raise_on_noconv=False)
    off = ((vecs * vecs).sum(0) - 1.0).cpu().numpy()
    assert abs(off.mean()) <= 6 * np.sqrt(40 * ncv / nev) * 2.0 ** -53, off


# Operators that are not symmetric: thick-restart Lanczos does not converge on
# them, and what is returned at the restart limit follows from the rounding of
# every step.  The values are what the solvers with one kernel per sum and
# Rayleigh-Ritz on the host return; they are kept to the bit.
def _hamiltonian(jd):
    H = q.build_hamiltonian_g(jd, [-0.9, -0.5, -0.3, -0.7])
    q.add_local_field(H, jd, [0.05, -0.02, 0.07])
    return H


def _operator(kind, slots):
    """An operator that is not symmetric: rings of a cluster one cell wide pass
    through a spin twice and lack their reverses ("unpaired"); or flips whose
    reverses have another coefficient, slot, sign or Z string."""
    if kind == "unpaired":
        jd = latgen.Supercell((1, 2, 2)).to_dict()
        H = serve.slotted_hamiltonian(jd) if slots else _hamiltonian(jd)
        return q.GpuOp(q.enumerate_basis_device(jd, 0), H)
    rng = np.random.default_rng(5)
    states = np.zeros((513, 2), dtype=np.uint64)
    states[:, 0] = np.sort(rng.choice(1 << 10, 513, replace=False))
    H = SymbolicOpSum()
    for k in range(16):
        at = [int(v) for v in rng.choice(10, 3, replace=False)]
        a = str(rng.choice(["+", "-"]))
        b = "-" if a == "+" else "+"
        slot = k % 4
        c = float(rng.standard_normal())
        O = SymbolicPMROperator.from_ops([a, b, "z"], at)
        R = SymbolicPMROperator.from_ops([b, a, "z"], at)
        if kind == "coefficient":
            H.add_term(c, O)
            H.add_term(c if k else 0.7 * c, R)
        elif kind == "slot":
            H.add_term(1.0, O, slot=slot)
            H.add_term(1.0, R, slot=slot if k else 1)
        elif kind == "sign":
            R.sign = R.sign if k else -R.sign
            H.add_term(1.0, O, slot=slot)
            H.add_term(1.0, R, slot=slot)
        else:
            H.add_term(c, O)
            H.add_term(c, R if k else SymbolicPMROperator.from_ops([b, a], at[:2]) *
                       SymbolicPMROperator.from_ops("z", [(at[2] + 1) % 10]))
    for p in range(10):
        H.add_term(0.3 + 0.11 * p, SymbolicPMROperator.from_ops("z", [p]))
    return q.GpuOp(q.GpuBasis(states, 10), H)


ENGINE = {
    ("unpaired", 1, 8): ["-0x1.9fe0d4c2c7c0cp+1", "-0x1.7072c5b6d0d7cp+1"],
    ("unpaired", 3, 15): ["-0x1.9bf524818ecb4p+1", "-0x1.6fa7a1920b2adp+1"],
    ("unpaired", 4, 40): ["-0x1.e14f6f44a4fd6p+1", "-0x1.6ff32dbf933dap+1"],
    ("coefficient", 3, 15): ["-0x1.16f86942d6129p+3", "-0x1.17086c65509b9p+3"],
    ("coefficient", 4, 40): ["-0x1.16f88457e3d0ap+3", "-0x1.17086e0fb5686p+3"],
    ("slot", 3, 15): ["-0x1.1877479e14638p+3", "-0x1.0bc5c954f6703p+3"],
    ("slot", 4, 40): ["-0x1.187747d8455e1p+3", "-0x1.0bc682daf1cdap+3"],
    ("sign", 3, 15): ["-0x1.15c12481f49a8p+3", "-0x1.0b422f2ee88dbp+3"],
    ("sign", 4, 40): ["-0x1.15c104ff95c17p+3", "-0x1.0b43c0a9874dap+3"],
    ("z", 3, 15): ["-0x1.16f0dd958dff8p+3", "-0x1.170022242d1f7p+3"],
    ("z", 4, 40): ["-0x1.16f0d32ec16c0p+3", "-0x1.17001f54ce088p+3"],
}


@pytest.mark.parametrize("kind,nev,ncv", list(ENGINE))
def test_engine_not_symmetric(cuda, kind, nev, ncv):
    """The first and the last of five requests on three columns."""
    op = _operator(kind, True)
    eng = serve.Engine(op, max_cols=3, nev=nev, ncv=ncv, tol=1e-10, max_restarts=4,
                       autotune=False, cache_connectivity=False)
    c = np.random.default_rng(2).uniform(-1.0, -0.2, size=(5, op.n_slots))
    ids = [eng.submit(c[k], 11 + k) for k in range(5)]
    got = {f.id: f.evals[0] for f in eng.run_all()}
    assert [float(got[ids[k]]).hex() for k in (0, 4)] == ENGINE[kind, nev, ncv]


EIGSH = {
    ("unpaired", 1, 8): ["-0x1.85801080438b4p+1"],
    ("unpaired", 3, 15): [
        "-0x1.880140e659e0dp+1", "-0x1.5db61958a620cp+1", "-0x1.2ec5de7bffba5p+1"],
    ("unpaired", 4, 40): [
        "-0x1.7d7baec051c76p+1", "-0x1.737b84701f64fp+1", "-0x1.5cb90754572f2p+1",
        "-0x1.04f10d5fb1ff0p+1"],
    ("coefficient", 3, 15): [
        "-0x1.16f77984bc2c1p+3", "-0x1.032bf7a933870p+3", "-0x1.01d9850bfff13p+3"],
    ("coefficient", 4, 40): [
        "-0x1.16f77963bde57p+3", "-0x1.03281b4ccf654p+3", "-0x1.01d90e88b3bc8p+3",
        "-0x1.fde173ff380d4p+2"],
    ("slot", 3, 15): ["-0x1.4dd4ce9d6be9ep+3", "-0x1.1e06b85639decp+3", "-0x1.0bb6c10d340aap+3"],
    ("slot", 4, 40): [
        "-0x1.4dd4ce9d6bea4p+3", "-0x1.1e06b85639dd3p+3", "-0x1.0bb6c10d8a04fp+3",
        "-0x1.0381eccf9cf2ep+3"],
    ("sign", 3, 15): ["-0x1.49cfdf30570c4p+3", "-0x1.1830bca798542p+3", "-0x1.0b9e600ddbccap+3"],
    ("sign", 4, 40): [
        "-0x1.49cf772b4be51p+3", "-0x1.1858fbe961848p+3", "-0x1.064ca6a064eb2p+3",
        "-0x1.ee510a93e7c47p+2"],
    ("z", 3, 15): ["-0x1.16e5d80e0ad31p+3", "-0x1.03a0d26f18c47p+3", "-0x1.01a406039092dp+3"],
    ("z", 4, 40): [
        "-0x1.16e5e0820c03ap+3", "-0x1.039f3c19c5468p+3", "-0x1.01ace8cf41a5cp+3",
        "-0x1.fdbfc88094235p+2"],
}


@pytest.mark.parametrize("kind,nev,ncv", list(EIGSH))
def test_eigsh_not_symmetric(cuda, kind, nev, ncv):
    evals = _operator(kind, False).eigsh(nev=nev, ncv=ncv, tol=1e-10, max_restarts=4, seed=3,
                                         raise_on_noconv=False)[0]
    assert [float(v).hex() for v in evals] == EIGSH[kind, nev, ncv]
