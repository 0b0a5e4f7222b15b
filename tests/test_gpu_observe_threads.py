"""Observables from several host threads at once: calls with few and with many
columns, whose kernels ask for different amounts of LDS, do not disturb each
other (the limit is a process-wide attribute of the kernel)."""
import threading

import numpy as np
import pytest

import qsi_subspace_ed_amd as q
from qsi_subspace_ed_amd import latgen
from qsi_subspace_ed_amd import observables as obs

pytestmark = pytest.mark.gpu


def test_threads(cuda):
    jd = latgen.Supercell((2, 2, 2)).to_dict()
    basis = q.enumerate_basis_device(jd, 0)
    ops = obs.ring_operators(basis, jd)
    counts = [4, 32, 9, 31]
    psi = cuda.randn(basis.dim(), 4, dtype=cuda.float64, device="cuda",
                     generator=cuda.Generator(device="cuda").manual_seed(1))
    want = [obs.cross_correlations(ops[:n], psi) for n in counts]
    cuda.cuda.synchronize()
    wrong = []

    def work(k):
        try:
            for _ in range(50):
                if not np.array_equal(obs.cross_correlations(ops[:counts[k]], psi), want[k]):
                    wrong.append(counts[k])
        except Exception as e:  # noqa: BLE001
            wrong.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(counts))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
