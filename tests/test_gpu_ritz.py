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
