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
