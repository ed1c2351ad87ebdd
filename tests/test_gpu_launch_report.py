"""kw_sim_launch_config names the workgroup sizes and radix plans that run, and the
autotuner times each launch shape once."""

import pytest

import cases

pytestmark = pytest.mark.gpu


def config(kw, f):
    with kw.Simulation(f, record=("p",)) as sim:
        return sim.launch_config()


def test_narrow_last_axis_reports_its_plan(kw):
    """A 512-point last axis of a 2-D grid: 4-column tiles of 192 threads, plan 0."""
    c = config(kw, cases.case_2d_absorbing_psource(N=(48, 512), Nt=4))
    print(f"[gpu launch report] 48x512: {c}", flush=True)
    assert (c["last_nt"], c["last_plan"]) == (192, 0)


def test_64_thread_pencils_report_128(kw, monkeypatch):
    monkeypatch.setenv("KW_PENCIL_NT", "64")
    c = config(kw, cases.case_3d(N=(32, 160, 192), Nt=4, pml=4, source="p"))
    print(f"[gpu launch report] KW_PENCIL_NT=64: {c}", flush=True)
    assert c["ypass_nt"] == 128 and c["last_nt"] == 128


@pytest.mark.parametrize("shape, row, y, last, plans", [
    ((54, 45, 50), 256, 256, 256, (4, 4)), ((42, 252, 392), 256, 256, 512, (4, 4)),
    ((36, 525, 35), 256, 512, 256, (4, 4)), ((36, 640, 32), 256, 1024, 256, (4, 0)),
    ((64, 36, 525), 128, 256, 1024, (4, 4)), ((60, 250), 256, 0, 128, (0, 4)), ((25, 27, 30), 0, 0, 0, (0, 0))])
def test_compiled_lengths_report_their_kernels(kw, shape, row, y, last, plans):
    """Lengths with one instantiation each (plan 4), beside tuned and generic ones."""
    f = cases.case_3d(N=shape, Nt=4, pml=3, source="p") if len(shape) == 3 else \
        cases.case_2d_absorbing_psource(N=shape, Nt=4)
    c = config(kw, f)
    print(f"[gpu launch report] {shape}: {c}", flush=True)
    assert (c["row_nt"], c["ypass_nt"], c["last_nt"]) == (row, y, last)
    assert (c["ypass_plan"], c["last_plan"]) == plans


def test_generic_kernels_report_zero(kw, monkeypatch):
    for k in ("KW_ROW_NT", "KW_PENCIL_NT", "KW_LAST_NT"):
        monkeypatch.setenv(k, "0")
    c = config(kw, cases.case_3d(N=(54, 45, 48), Nt=4, pml=4, source="p"))
    assert (c["row_nt"], c["ypass_nt"], c["last_nt"], c["ypass_plan"], c["last_plan"]) == (0, 0, 0, 0, 0)


def test_autotuner_times_each_shape_once(kw):
    """A tuned y axis beside a last axis with one instantiation: the base, three row
    workgroup sizes, three row targets, and three y-pass sizes.  The first step of a
    trial and the timed ones launch one density kernel each."""
    f = cases.case_3d(N=(64, 48, 35), Nt=12, pml=4, source="p")
    with kw.Simulation(f, record=("p",)) as sim:
        sim.set_profiling(True)
        sim.autotune(trial_steps=3)
        launches = sim.profile()["x_density"][1]
    print(f"[gpu launch report] 64x48x35: {launches} density launches", flush=True)
    assert launches == (1 + 3 + 3 + 3) * 4
