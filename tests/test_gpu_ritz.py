"""What the solve engine returns where a request's projected matrix is not finite,
on both sides of the order up to which the device diagonalises it."""
import numpy as np
import pytest

import qsi_subspace_ed_amd as q
from qsi_subspace_ed_amd import latgen, serve

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
    from qsi_subspace_ed_amd.operators import SymbolicPMROperator
    states, spins, W = _basis(1, 10, 513, 513)
    H = _terms(spins, 24, 10, z=False, open_spins=False)
    for k, p in enumerate(spins):
        H.add_term(0.37 * 1.61 ** (k % 7) + 0.011 * k, SymbolicPMROperator.from_ops("z", [p]))
    op = q.GpuOp(q.GpuBasis(states, W), H)
    _, vecs, _, _ = op.eigsh(nev=nev, ncv=ncv, tol=1e-30, max_restarts=3, seed=3, n_evecs=nev,
                             raise_on_noconv=False)
    off = ((vecs * vecs).sum(0) - 1.0).cpu().numpy()
    assert abs(off.mean()) <= 6 * np.sqrt(40 * ncv / nev) * 2.0 ** -53, off
