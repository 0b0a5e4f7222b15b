"""The kernel name under which the benchmark looks up measured traffic is the one of
the kernel that the library launches."""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402
import qsi_subspace_ed_amd as q  # noqa: E402
from qsi_subspace_ed_amd import latgen  # noqa: E402
from qsi_subspace_ed_amd.operators import SymbolicOpSum, SymbolicPMROperator  # noqa: E402


def _name(H, mode):
    return bench.variant_kernel("window", 1, low_mode=mode, H=H)


def test_window():
    rings = q.build_hamiltonian_g(latgen.Supercell((2, 2, 2)).to_dict(), [-1.0] * 4)
    assert _name(rings, 2) == "k_apply_win<1, false, false, false>"
    assert _name(rings, 1) == "k_apply_win<1, false, false, true>"
    # rings of a cluster one cell wide lack their reverses
    narrow = q.build_hamiltonian_g(latgen.Supercell((1, 2, 2)).to_dict(), [-1.0] * 4)
    assert _name(narrow, 2) == "k_apply_win<1, false, false, true>"
    one = SymbolicOpSum()
    one.add_term(1.0, SymbolicPMROperator.from_ops("+-", [0, 1]))
    assert _name(one, 2) == "k_apply_win<1, false, false, true>"
    # a spin flipped outside the projector
    open_spin = SymbolicOpSum()
    open_spin.add_term(1.0, SymbolicPMROperator.from_ops("x", [3]))
    assert _name(open_spin, 2) == "k_apply_win<1, false, false, true>"
