"""bench.py's byte model of the spectral passes against counts of the arrays that a
step's launches read and write (in half spectra; a spectral table is half of one)."""

import pytest

import bench
import cases


@pytest.mark.parametrize("absorbing", [True, False])
def test_spectral_pass_bytes(absorbing):
    f = cases.case_3d(N=(40, 36, 30), Nt=2, absorbing=absorbing)
    spec = (40 // 2 + 1) * 36 * 30 * 8
    # (inputs, outputs, tables): the gradient leaves kappa F and the z output, the
    # divergence and the absorption terms as many outputs as inputs
    last = [(1, 2, 1), (3, 3, 1)] + ([(2, 2, 2)] if absorbing else [])
    # (read, written): the gradient's second launch makes three outputs from two fields
    y = [(1, 1), (2, 3), (3, 3), (3, 3)] + ([(2, 2), (2, 2)] if absorbing else [])
    # one plane pass makes all three gradient outputs
    plane = [(1, 3, 1)] + last[1:]
    mean = lambda v: sum(v) / len(v)  # noqa: E731
    assert bench.kernel_bytes(f, "last_axis") == pytest.approx(mean([spec * (i + o + t / 2) for i, o, t in last]))
    assert bench.kernel_bytes(f, "y_pass") == pytest.approx(mean([spec * (r + w) for r, w in y]))
    assert bench.kernel_bytes(f, "yz_plane") == pytest.approx(mean([spec * (i + o + t / 2) for i, o, t in plane]))
