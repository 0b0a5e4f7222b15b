"""The window apply kernel against the lane kernel, bit for bit, where its
matching can go wrong: bases of 127 to 129 and 255 to 257 states (tiles of 128
rows, windows of 128 ranks, and the lane kernel below that), term lists at the
edges of its chunks of 64, sectors that the terms close and do not close,
one- and two-word states whose varying bits straddle the words, ranges beyond the
windows of a term, Z strings and projectors; the dot-product instances through the
Lanczos coefficients; and the automatic choice on both sides of its size."""
import numpy as np
import pytest

import qsi_subspace_ed_amd as q
from qsi_subspace_ed_amd import latgen
from qsi_subspace_ed_amd.operators import SymbolicOpSum, SymbolicPMROperator

pytestmark = pytest.mark.gpu

# spins that vary in the synthetic bases, lowest first
SPINS = {1: [0, 1, 2, 3, 5, 8, 13, 21, 30, 31, 32, 40, 55],
         2: [0, 1, 2, 5, 31, 32, 62, 63, 64, 65, 66, 80, 95]}


def _basis(words, bits, keep, seed):
    """keep of the 2^bits states over the varying spins, as (D, 2) [lo, hi]."""
    spins = SPINS[words][:bits] if words == 1 else SPINS[words][-bits:]
    idx = np.arange(1 << bits, dtype=np.uint64)
    if keep < idx.size:
        idx = np.sort(np.random.default_rng(seed).choice(idx, keep, replace=False))
    out = np.zeros((idx.size, 2), dtype=np.uint64)
    for b, p in enumerate(spins):
        out[:, p // 64] |= ((idx >> np.uint64(b)) & np.uint64(1)) << np.uint64(p % 64)
    return out, spins, (56 if words == 1 else 96)


def _terms(spins, n, seed, z, open_spins):
    """n flips of one to three spins, each followed by its conjugate where the
    list has room; with open_spins some flip a spin that no projector fixes
    (their targets do not keep the rows' order)."""
    rng = np.random.default_rng(seed)
    H = SymbolicOpSum()
    conj = {"+": "-", "-": "+"}
    while len(H.off_diag_terms) < n:
        k = int(rng.integers(1, 4))
        at = [int(v) for v in rng.choice(spins, k, replace=False)]
        ops = [str(v) for v in rng.choice(["+", "-", "x"] if open_spins else ["+", "-"], k)]
        rest = [p for p in spins if p not in at]
        extra = [int(rng.choice(rest))] if rng.random() < 0.5 else []
        tail = [str(rng.choice(["p", "z"] if z else ["p"]))] if extra else []
        c = float(rng.standard_normal())
        H.add_term(c, SymbolicPMROperator.from_ops(ops + tail, at + extra))
        if len(H.off_diag_terms) < n:
            H.add_term(c, SymbolicPMROperator.from_ops([conj.get(o, o) for o in ops] + tail,
                                                       at + extra))
    H.add_term(0.3, SymbolicPMROperator.from_ops("z", [spins[0]]))
    return H


def _same(cuda, states, n_spins, H):
    basis = q.GpuBasis(states, n_spins)
    basis.build_lowkeys()
    D = states.shape[0]
    x = np.random.default_rng(D).standard_normal(D)
    x[::7] = 1e-16  # below the apply tolerance
    x = cuda.from_numpy(x).cuda()
    y0 = cuda.from_numpy(np.random.default_rng(1).standard_normal(D)).cuda()
    for verified in (False, True):
        got = {}
        for v in ("lane", "window"):
            op = q.GpuOp(basis, H)
            if verified:
                op.verify_lowkeys()
            op.set_variant(v)
            y, ya = cuda.empty_like(x), y0.clone()
            op.evaluate(x, y)
            op.evaluate_add(x, ya)
            a, b = op.lanczos_coeffs(4, v0=y0)
            got[v] = (y.cpu().numpy(), ya.cpu().numpy(), a, b)
        for u, w in zip(got["lane"], got["window"]):
            assert np.array_equal(u, w, equal_nan=True), verified


@pytest.mark.parametrize("words", [1, 2])
@pytest.mark.parametrize("bits,keep", [(7, 127), (7, 128), (8, 129), (8, 255), (8, 256), (9, 257),
                                       (12, 4096), (12, 1500), (13, 8191)])
@pytest.mark.parametrize("z", [False, True])
@pytest.mark.parametrize("open_spins", [False, True])
def test_synthetic(cuda, words, bits, keep, z, open_spins):
    states, spins, W = _basis(words, bits, keep, keep)
    _same(cuda, states, W, _terms(spins, 24, bits, z, open_spins))


@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 128, 129, 200])
def test_term_counts(cuda, n):
    states, spins, W = _basis(1, 11, 2048, 0)
    _same(cuda, states, W, _terms(spins, n, n, False, False))


@pytest.mark.parametrize("repeats,sector", [((2, 2, 2), 1), ((1, 3, 3), 0), ((2, 2, 3), 0),
                                            ((1, 3, 5), 0), ((2, 3, 3), 0)])
def test_ice(cuda, repeats, sector):
    jd = latgen.Supercell(repeats).to_dict()
    H = q.build_hamiltonian_g(jd, [-0.9, -0.5, -0.3, -0.7])
    q.add_local_field(H, jd, [0.05, -0.02, 0.07])
    basis = q.enumerate_basis_device(jd, sector)
    x = cuda.randn(basis.dim(), dtype=cuda.float64, device="cuda",
                   generator=cuda.Generator(device="cuda").manual_seed(3))
    ys = []
    for v in ("lane4", "window", "auto"):
        op = q.GpuOp(basis, H)
        op.set_variant(v)
        y = cuda.empty_like(x)
        op.evaluate(x, y)
        ys.append((y, op.lanczos_coeffs(3, v0=x)))
    basis.build_lowkeys()
    for v in ("window", "auto"):
        op = q.GpuOp(basis, H)
        op.verify_lowkeys()  # 2 in the ice sectors, 1 in the one-pair sector
        op.set_variant(v)
        y = cuda.empty_like(x)
        op.evaluate(x, y)
        ys.append((y, op.lanczos_coeffs(3, v0=x)))
    for y, (a, b) in ys[1:]:
        assert cuda.equal(y, ys[0][0])
        assert np.array_equal(a, ys[0][1][0]) and np.array_equal(b, ys[0][1][1])
