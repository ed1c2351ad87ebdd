"""A launch configuration cached by the autotuner for one handle must not reach a
handle of the same shape whose environment switches other kernels on or off."""

import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


def test_generic_last_axis_stays_generic_after_a_tuned_handle(kw, monkeypatch):
    """The axisymmetric handle's tuning has no pencils to time, so its cached
    entry holds the 2-D default, narrow last-axis tiles; KW_LAST_NT=0 asks for the
    generic kernel, whose results differ from the tiles' in the last bits."""
    f = cases.case_2d_p0_lossless(N=96, Nt=40, pml=8, het=True)
    a = cases.case_axisym(Nx=96, Ny=96, Nt=8, source="p0")
    monkeypatch.setenv("KW_ROW_NT", "0")  # nothing to tune in the rows: only the last axis can differ
    print("[gpu tune overrides] 96x96: axisymmetric handle tuned first, then KW_LAST_NT=0", flush=True)
    with kw.Simulation(a, record=("p",)) as sim:
        sim.autotune(trial_steps=2)
    monkeypatch.setenv("KW_LAST_NT", "0")
    ref = kw.run(f, record=("p",))["p"]
    with kw.Simulation(f, record=("p",)) as sim:
        sim.autotune(trial_steps=2)
        sim.run()
        got = sim.fetch("p")
    np.testing.assert_array_equal(got, ref)


def test_padded_rows_keep_specialised_pencils_after_a_generic_handle(kw, monkeypatch):
    """Generic pencils read spectrum rows of Nx/2+1 values, so a handle with padded
    rows cannot take the configuration of one that ran them."""
    f = cases.case_3d(N=(64, 48, 32), Nt=20, pml=4, source="p")
    monkeypatch.setenv("KW_PAD_SPECTRA", "1")
    ref = kw.run(f, record=("p",))["p"]
    print("[gpu tune overrides] 64x48x32: generic pencils tuned first, then padded rows", flush=True)
    with monkeypatch.context() as m:
        m.setenv("KW_PENCIL_NT", "0")
        m.setenv("KW_LAST_NT", "0")
        with kw.Simulation(f, record=("p",)) as sim:
            sim.autotune(trial_steps=2)
    with kw.Simulation(f, record=("p",)) as sim:
        sim.autotune(trial_steps=2)
        sim.run()
        got = sim.fetch("p")
    assert cases.rel_l2(got, ref) <= 1e-5  # tuned launch shapes: the same formulas to FP32 rounding
