"""The wavefront-per-row apply that the automatic choice takes on small bases,
against the lane kernel, bit for bit: rows that do not fill a workgroup's four
wavefronts, term lists at the edges of its chunks of 64, one- and two-word states,
Z strings, targets outside the basis, and both sides of the size where it ends."""
import numpy as np
import pytest

import qsi_subspace_ed_amd as q
from test_gpu_window import _basis, _terms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("words,bits,keep", [(1, 6, 1), (1, 6, 5), (2, 7, 127), (1, 12, 1500),
                                             (2, 12, 4096), (1, 13, 8191)])
@pytest.mark.parametrize("n", [0, 1, 63, 64, 65, 200])
@pytest.mark.parametrize("z", [False, True])
def test_rows(cuda, words, bits, keep, n, z):
    states, spins, W = _basis(words, bits, keep, keep)
    H = _terms(spins, n, n + bits, z, open_spins=n == 65)
    basis = q.GpuBasis(states, W)
    x = np.random.default_rng(keep).standard_normal(keep)
    x[::7] = 1e-16  # below the apply tolerance
    x[3::50] = np.inf
    x = cuda.from_numpy(x).cuda()
    y0 = cuda.from_numpy(np.random.default_rng(1).standard_normal(keep)).cuda()
    got = []
    for v in ("lane", "auto"):
        op = q.GpuOp(basis, H)
        op.set_variant(v)
        y, ya = cuda.empty_like(x), y0.clone()
        op.evaluate(x, y)
        op.evaluate_add(x, ya)
        got.append((y.cpu().numpy(), ya.cpu().numpy()))
    for u, w in zip(*got):
        assert np.array_equal(u, w, equal_nan=True)


@pytest.mark.parametrize("keep", [16383, 16384, 16385])
def test_limit(cuda, keep):
    idx = np.arange(keep, dtype=np.uint64) * np.uint64(3)
    states = np.stack([idx, np.zeros_like(idx)], axis=1)
    H = _terms(list(range(12)), 70, 1, False, False)
    basis = q.GpuBasis(states, 20)
    x = cuda.from_numpy(np.random.default_rng(keep).standard_normal(keep)).cuda()
    ys = []
    for v in ("lane", "auto"):
        op = q.GpuOp(basis, H)
        op.set_variant(v)
        y = cuda.empty_like(x)
        op.evaluate(x, y)
        ys.append(y)
    assert cuda.equal(*ys)
