"""The thick-restart solver's device passes at their edges, against a dense
diagonalisation: search spaces on both sides of the projection kernels' 16 and
32 columns and of the device Rayleigh-Ritz's 48, odd and even orders, the
smallest ones, bases below one workgroup's rows and beyond, and subspaces that end
early.  The solver stops at a relative residual of 1e-10: eigenvalues lie within
that of the exact ones (times the norm of H), and vectors with a gap to the rest
of the spectrum within 1e-10 * |H| / gap, checked as residuals below 1e-9 |H|."""
import numpy as np
import pytest

import qsi_subspace_ed_amd as q
from test_gpu_window import _basis, _terms

pytestmark = pytest.mark.gpu


def _dense(op):
    r, c, v, d = op.connectivity()
    A = np.diag(d).astype(np.float64)
    np.add.at(A, (r, c), v)
    return A


@pytest.mark.parametrize("bits,keep", [(6, 40), (9, 500), (9, 512), (10, 513), (11, 1500)])
@pytest.mark.parametrize("nev,ncv", [(1, 2), (1, 3), (2, 9), (3, 15), (5, 16), (5, 17), (6, 24),
                                     (4, 32), (4, 33), (8, 47), (8, 48), (8, 49), (10, 63)])
def test_lowest(cuda, bits, keep, nev, ncv):
    if ncv < 9 and keep > 64:
        keep, bits = 64, 6  # a search in two or three vectors takes hundreds of restarts
    states, spins, W = _basis(1, bits, keep, keep)
    H = _terms(spins, 24, bits, z=False, open_spins=False)
    # a diagonal without repeated values: no degenerate levels
    from qsi_subspace_ed_amd.operators import SymbolicPMROperator
    for k, p in enumerate(spins):
        H.add_term(0.37 * 1.61 ** (k % 7) + 0.011 * k, SymbolicPMROperator.from_ops("z", [p]))
    op = q.GpuOp(q.GpuBasis(states, W), H)
    A = _dense(op)
    assert np.array_equal(A, A.T)  # every term is followed by its conjugate
    want = np.linalg.eigvalsh(A)
    norm = np.abs(want).max()
    n = min(nev, keep - 1)
    evals, vecs, _, _ = op.eigsh(nev=nev, ncv=ncv, tol=1e-10, max_restarts=20000, seed=3, n_evecs=n)
    assert np.abs(evals[:n] - want[:n]).max() <= 1e-9 * norm
    V = vecs.cpu().numpy()
    for i in range(n):
        v = V[:, i]
        assert abs(np.linalg.norm(v) - 1.0) <= 1e-9
        assert np.linalg.norm(A @ v - evals[i] * v) <= 1e-9 * norm


@pytest.mark.parametrize("bits,keep", [(6, 40), (10, 513)])
@pytest.mark.parametrize("nev,ncv", [(1, 6), (3, 15), (3, 16), (3, 17), (4, 24), (4, 32), (4, 33),
                                     (5, 48), (5, 49), (5, 63)])
def test_engine(cuda, bits, keep, nev, ncv):
    """Seven points on three columns of the solve engine, on both sides of its
    kernels' column limits and of the device Rayleigh-Ritz's: columns that
    restart in different steps, are refilled, and (small basis, large search
    space) exhaust their space."""
    from qsi_subspace_ed_amd import serve
    from qsi_subspace_ed_amd.operators import SymbolicOpSum, SymbolicPMROperator
    states, spins, W = _basis(1, bits, keep, keep)
    H = SymbolicOpSum()
    # conjugate pairs share a slot; a field without repeated values
    for k, (_, o, _) in enumerate(_terms(spins, 24, bits, z=False, open_spins=False).off_diag_terms):
        H.add_term(1.0, o, slot=k // 2 % 4)
    for k, p in enumerate(spins):
        H.add_term(0.37 * 1.61 ** (k % 7) + 0.011 * k, SymbolicPMROperator.from_ops("z", [p]))
    op = q.GpuOp(q.GpuBasis(states, W), H)
    pts = np.random.default_rng(ncv).uniform(-1.0, -0.2, size=(op.n_slots, 7))
    eng = serve.Engine(op, max_cols=3, nev=nev, ncv=ncv, tol=1e-10, max_restarts=20000)
    ids = [eng.submit(pts[:, k], 11 + k) for k in range(7)]
    got = {f.id: f.evals for f in eng.run_all()}
    for k, i in enumerate(ids):
        A = np.empty((keep, keep))
        for c0 in range(0, keep, 64):
            R = min(64, keep - c0)
            c = cuda.from_numpy(np.repeat(pts[:, k:k + 1], R, axis=1)).cuda()
            y = cuda.empty((keep, R), dtype=cuda.float64, device="cuda")
            op.apply_block(cuda.eye(keep, dtype=cuda.float64, device="cuda")[:, c0:c0 + R]
                           .contiguous(), y, coeffs=c)
            A[:, c0:c0 + R] = y.cpu().numpy()
        assert np.array_equal(A, A.T)
        want = np.linalg.eigvalsh(A)
        n = min(nev, keep - 1)
        assert np.abs(got[i][:n] - want[:n]).max() <= 1e-9 * np.abs(want).max()


@pytest.mark.parametrize("nev,ncv", [(1, 8), (3, 15), (3, 20), (4, 40)])
def test_engine_not_symmetric(cuda, nev, ncv):
    """A cluster one cell wide: its rings pass through a spin twice, H is not
    symmetric and requests end at their restart limit.  The engine's unfused
    steps give a request the same bits alone and among others."""
    from qsi_subspace_ed_amd import latgen, serve
    jd = latgen.Supercell((1, 2, 2)).to_dict()
    basis = q.enumerate_basis_device(jd, 0)
    pts = np.random.default_rng(ncv).uniform(-1.0, -0.2, size=(serve.N_SLOTS, 5))
    pts[4:] *= 0.1

    def run(ks):
        op = q.GpuOp(basis, serve.slotted_hamiltonian(jd))
        eng = serve.Engine(op, max_cols=5, nev=nev, ncv=ncv, tol=1e-10, max_restarts=7,
                           autotune=False)
        ids = [eng.submit(pts[:, k], 11 + k) for k in ks]
        got = {f.id: f.evals for f in eng.run_all()}
        return [got[i] for i in ids]

    together = run(range(5))
    for k in range(5):
        assert np.array_equal(run([k])[0], together[k])
