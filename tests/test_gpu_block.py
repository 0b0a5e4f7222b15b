"""The searching block apply where its split can go wrong: column counts on both
sides of every lane-group size (one column, an odd last column beside a pair, 64
columns), rows that are no multiple of a tile or of a workgroup's four tiles,
fewer rows than a wavefront, more terms than one round's 256 or than the rows'
entries hold, one- and two-word states, Z strings, operators with and without
coefficient classes, strided blocks at odd offsets, and accumulation.  Every
column is the column computed alone, bit for bit (and the cached connectivity's,
where the operator has classes), and agrees with the single-vector apply."""
import numpy as np
import pytest

import qsi_subspace_ed_amd as q
from test_gpu_window import _basis, _terms

pytestmark = pytest.mark.gpu


def _classed(H, n_cls):
    """The same terms with coefficients out of n_cls values."""
    vals = [0.75 - 0.5 * k for k in range(n_cls)]
    H.off_diag_terms = [(vals[i % n_cls],) + t[1:] for i, t in enumerate(H.off_diag_terms)]
    return H


@pytest.mark.parametrize("words,bits,keep", [(1, 6, 17), (1, 6, 64), (2, 7, 65), (1, 9, 257),
                                             (2, 12, 1500), (1, 13, 8191)])
@pytest.mark.parametrize("n", [0, 1, 64, 130, 256, 300, 700])
@pytest.mark.parametrize("n_cls", [0, 3])
def test_columns(cuda, words, bits, keep, n, n_cls):
    states, spins, W = _basis(words, bits, keep, keep)
    H = _terms(spins, n, n + bits, z=n % 2 == 0, open_spins=n == 64)
    if n_cls:
        H = _classed(H, n_cls)
    basis = q.GpuBasis(states, W)
    op = q.GpuOp(basis, H)
    D = basis.dim()
    rng = np.random.default_rng(n + D)
    x = rng.standard_normal((D, 64))
    x[::7, ::3] = 1e-16  # below the apply tolerance
    x = cuda.from_numpy(x).cuda()
    y0 = cuda.from_numpy(rng.standard_normal((D, 64))).cuda()
    alone, single = cuda.empty_like(x), cuda.empty_like(x)
    for c in range(64):
        op.apply_block(x[:, c:c + 1], alone[:, c:c + 1])
        ys = cuda.empty(D, dtype=cuda.float64, device="cuda")
        op.evaluate(x[:, c].contiguous(), ys)
        single[:, c] = ys
    # two orders of the same n + 1 products, each within (n + 2) ulp/2 of
    # sum |c| |x| <= (n + 1) max|c| max|x|
    cmax = max([abs(t[0]) for t in H.off_diag_terms] + [0.3])
    tol = 2 * (n + 2) * 2.0 ** -53 * (n + 1) * cmax * float(x.abs().max())
    assert float((alone - single).abs().max()) <= tol
    for R in (2, 3, 7, 8, 16, 33, 63, 64):
        for c0 in (0, 1) if R < 64 else (0,):
            y = y0.clone()
            op.apply_block(x[:, c0:c0 + R], y[:, c0:c0 + R])
            assert cuda.equal(y[:, c0:c0 + R], alone[:, c0:c0 + R]), (R, c0)
            assert cuda.equal(y[:, :c0], y0[:, :c0]) and cuda.equal(y[:, c0 + R:], y0[:, c0 + R:])
    # accumulation starts from Y, so it is compared column by column
    for R in (2, 7, 64):
        y, ya = y0.clone(), y0.clone()
        op.apply_block(x[:, :R], y[:, :R], accumulate=True)
        for c in range(R):
            op.apply_block(x[:, c:c + 1], ya[:, c:c + 1], accumulate=True)
        assert cuda.equal(y, ya), R
    if n_cls and n:
        assert op.cache_connectivity(True) > 0
        y = cuda.empty_like(x)
        op.apply_block(x, y)
        assert cuda.equal(y, alone)


@pytest.mark.parametrize("words,bits,keep", [(1, 6, 17), (2, 7, 65), (1, 12, 1500), (1, 13, 8191)])
@pytest.mark.parametrize("cfg", [0, 1, 2, 4, 8, 9, 10, 13])
def test_cached_columns(cuda, words, bits, keep, cfg):
    """Every configuration over cached connectivity gives the searching apply's
    columns bit for bit, at every width, odd and strided blocks included."""
    states, spins, W = _basis(words, bits, keep, keep)
    H = _classed(_terms(spins, 130, bits, z=True, open_spins=False), 3)
    basis = q.GpuBasis(states, W)
    op, cached = q.GpuOp(basis, H), q.GpuOp(basis, H)
    assert cached.cache_connectivity(True) > 0
    cached.set_block_cfg(cfg)
    D = basis.dim()
    rng = np.random.default_rng(D)
    x = cuda.from_numpy(rng.standard_normal((D, 64))).cuda()
    y0 = cuda.from_numpy(rng.standard_normal((D, 64))).cuda()
    for R in (1, 2, 3, 5, 7, 8, 16, 21, 33, 63, 64):
        c0 = 1 if R < 64 else 0
        for add in (False, True):
            y, yc = y0.clone(), y0.clone()
            op.apply_block(x[:, c0:c0 + R], y[:, c0:c0 + R], accumulate=add)
            cached.apply_block(x[:, c0:c0 + R], yc[:, c0:c0 + R], accumulate=add)
            assert cuda.equal(y, yc), (R, add)


@pytest.mark.parametrize("R", [1, 3, 8, 21, 64])
@pytest.mark.parametrize("cached", [False, True])
def test_recurrence(cuda, R, cached):
    """Block Lanczos over sectors of 1500, 17 and 4096 states (tiles cut short,
    empty tiles, workgroups without a tile of some sector): each column's
    coefficients are those of the three-term recurrence in float64 on the CPU.
    Six steps; rounding grows with the condition of the steps before, so 1e-11
    relative to the largest coefficient, as for the sectors run alone."""
    from qsi_subspace_ed_amd import ftlm
    ops, V, want = [], [], []
    for bits, keep in ((12, 1500), (6, 17), (12, 4096)):
        states, spins, W = _basis(1, bits, keep, keep)
        H = _classed(_terms(spins, 40, 5, z=False, open_spins=False), 3)
        ops.append(q.GpuOp(q.GpuBasis(states, W), H))
        V.append(np.random.default_rng(keep).standard_normal((keep, R)))
        if cached:
            ops[-1].cache_connectivity(True)
        r, c, v, d = ops[-1].connectivity()
        A = np.diag(d)
        np.add.at(A, (r, c), v)
        b = V[-1] / np.linalg.norm(V[-1], axis=0)
        a, be, al_s, be_s = np.zeros_like(b), np.zeros(R), [], []
        for _ in range(6):
            w = A @ b
            al = np.sum(b * w, axis=0)
            w -= al * b + be * a
            be = np.linalg.norm(w, axis=0)
            a, b = b, w / be
            al_s.append(al)
            be_s.append(be)
        want.append((np.array(al_s).T, np.array(be_s).T))
    al, be, _ = ftlm.lanczos_block(ops, [cuda.from_numpy(v).cuda() for v in V], 6)
    for s, (wa, wb) in enumerate(want):
        scale = max(np.abs(wa).max(), np.abs(wb).max())
        assert np.abs(al[s] - wa).max() <= 1e-11 * scale, s
        assert np.abs(be[s] - wb).max() <= 1e-11 * scale, s


@pytest.mark.parametrize("R", [31, 32, 63, 64])
@pytest.mark.parametrize("cfg", [8, 9, 10])
def test_cached_wide(cuda, R, cfg):
    """Blocks large enough for four columns per lane (the last lane repeats up to
    three), beside the same columns sixteen at a time, which are not."""
    from qsi_subspace_ed_amd import latgen
    jd = latgen.Supercell((1, 3, 4)).to_dict()
    H = q.build_hamiltonian_g(jd, [-0.9, -0.5, -0.3, -0.7])
    q.add_local_field(H, jd, [0.05, -0.02, 0.07])
    op = q.GpuOp(q.enumerate_basis_device(jd, 0), H)
    assert op.cache_connectivity(True) > 0
    op.set_block_cfg(cfg)
    D = op.rows()
    assert D * R >= 1 << 22 > D * 16
    x = cuda.randn(D, R + 1, dtype=cuda.float64, device="cuda",
                   generator=cuda.Generator(device="cuda").manual_seed(R))
    y = cuda.full_like(x, 7.0)
    op.apply_block(x[:, 1:], y[:, 1:])
    assert bool((y[:, 0] == 7.0).all())
    for c0 in range(1, R + 1, 16):
        w = min(16, R + 1 - c0)
        z = cuda.empty((D, w), dtype=cuda.float64, device="cuda")
        op.apply_block(x[:, c0:c0 + w].contiguous(), z)
        assert cuda.equal(y[:, c0:c0 + w], z), c0
