"""Choices of kernels against the kernels they choose from: the automatic one is
not left behind by the fixed ones where it was measured to lose, and the default
block configuration not by the other."""
import numpy as np
import pytest

import qsi_subspace_ed_amd as q
from qsi_subspace_ed_amd import latgen

pytestmark = pytest.mark.gpu


def _times(cuda, ops, n=20, rounds=5):
    """Shortest time (us) of n applies of each of ops, taken in turn."""
    x = cuda.randn(ops[0].rows(), dtype=cuda.float64, device="cuda")
    y = cuda.empty_like(x)
    best = [np.inf] * len(ops)
    for _ in range(rounds + 1):
        for k, op in enumerate(ops):
            a, b = (cuda.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(n):
                op.evaluate(x, y)
            b.record()
            b.synchronize()
            best[k] = min(best[k], a.elapsed_time(b) / n * 1e3)
    return best


def _graph_times(cuda, ops, n=50, rounds=5):
    """The same for the applies of a graph of n."""
    x = cuda.randn(ops[0].rows(), dtype=cuda.float64, device="cuda")
    y = cuda.empty_like(x)
    best, graphs = [], []
    for op in ops:
        op.evaluate(x, y)
        cuda.cuda.synchronize()
        g = cuda.cuda.CUDAGraph()
        with cuda.cuda.graph(g):
            for _ in range(n):
                op.evaluate(x, y)
        graphs.append(g)
        best.append(np.inf)
    for _ in range(rounds + 1):
        for k, g in enumerate(graphs):
            a, b = (cuda.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            g.replay()
            b.record()
            b.synchronize()
            best[k] = min(best[k], a.elapsed_time(b) / n * 1e3)
    return best


def _ops(basis, H, variants):
    out = []
    for v in variants:
        op = q.GpuOp(basis, H)
        op.set_variant(v)
        out.append(op)
    return out


@pytest.mark.parametrize("missing", [0.0, 0.01, 0.03, 0.1])
def test_scattered_misses(cuda, missing):
    """64 spins with states left out at random: where terms lead out of the basis
    all over, the window kernel takes up to twice the lane kernel's time."""
    jd = latgen.Supercell((2, 2, 4)).to_dict()
    H = q.build_hamiltonian_g(jd, [-0.9, -0.5, -0.3, -0.7])
    states = q.enumerate_basis_device(jd, 0).states()
    keep = np.random.default_rng(1).random(states.shape[0]) >= missing
    basis = q.GpuBasis(np.ascontiguousarray(states[keep]), 64)
    auto, lane = _times(cuda, _ops(basis, H, ("auto", "lane4")))
    assert auto <= 1.2 * lane, (auto, lane)
    if missing == 0.0:
        assert auto <= 0.9 * lane, (auto, lane)


def test_one_pair_sector(cuda):
    """A sector that few terms lead out of, together, stays on the window kernel."""
    jd = latgen.Supercell((1, 3, 5)).to_dict()
    H = q.build_hamiltonian_g(jd, [-0.9, -0.5, -0.3, -0.7])
    basis = q.enumerate_basis_device(jd, 1)
    auto, lane = _times(cuda, _ops(basis, H, ("auto", "lane4")))
    assert auto <= 0.9 * lane, (auto, lane)


@pytest.mark.parametrize("repeats", [(2, 2, 2), (1, 3, 3)])
def test_autotuned_small(cuda, repeats):
    """Tuning an operator on a small basis, where the automatic choice has a kernel
    of its own, does not leave it slower than before."""
    jd = latgen.Supercell(repeats).to_dict()
    H = q.build_hamiltonian_g(jd, [-0.9, -0.5, -0.3, -0.7])
    basis = q.enumerate_basis_device(jd, 0)
    tuned, auto = _ops(basis, H, ("auto", "auto"))
    assert tuned.autotune(0, reps=3)[0] in q._lib.VARIANTS
    a, b = _times(cuda, (tuned, auto), n=100)
    assert a <= 1.2 * b, (a, b)


def _first_terms(H, n):
    out = q.SymbolicOpSum()
    for c, o, _ in H.off_diag_terms[:n]:
        out.add_term(c, o)
    return out


@pytest.mark.parametrize("repeats", [(1, 3, 3), (2, 2, 4)])
@pytest.mark.parametrize("n", [1, 4, 8])
def test_few_terms(cuda, repeats, n):
    """Operators of few terms: a row does them in a round or two.  Applies of a
    captured graph: on their own those of the smaller basis take the host's time."""
    jd = latgen.Supercell(repeats).to_dict()
    H = _first_terms(q.build_hamiltonian_g(jd, [-0.9, -0.5, -0.3, -0.7]), n)
    basis = q.enumerate_basis_device(jd, 0)
    auto, lane = _graph_times(cuda, _ops(basis, H, ("auto", "lane4")))
    assert auto <= 1.15 * lane, (auto, lane)


def test_default_block(cuda):
    """Eight cached columns, one per lane (the default configuration): at most 1.28
    times as long as in pairs, of whose gathers it makes twice as many."""
    jd = latgen.Supercell((2, 2, 4)).to_dict()
    op = q.GpuOp(q.enumerate_basis_device(jd, 0),
                 q.build_hamiltonian_g(jd, [-0.9, -0.5, -0.3, -0.7]))
    op.cache_connectivity()
    X = cuda.randn(op.rows(), 8, dtype=cuda.float64, device="cuda")
    Y = cuda.empty_like(X)
    best = {}
    for _ in range(5):
        for cfg in (1, 9):
            op.set_block_cfg(cfg)
            a, b = (cuda.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(10):
                op.apply_block(X, Y)
            b.record()
            b.synchronize()
            best[cfg] = min(best.get(cfg, np.inf), a.elapsed_time(b))
    assert best[1] <= 1.28 * best[9], best
