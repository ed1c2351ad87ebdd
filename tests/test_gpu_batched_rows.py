"""Batched equals alone across the row kernels' two forms: a small grid run alone
transforms the components of density and pressure side by side (the wide form), a
batch of it always one after the other.  The update's statements are the same code
in both, and multiply-adds fuse within one source expression only, so results are
equal bit for bit."""

import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [160, 192, 256, 384, 512, 768])
@pytest.mark.parametrize("medium", ["power", "stokes", "lossless"])
def test_batched_rows_equal_alone(kw, nx, medium):
    items = []
    for seed in (3, 4):
        f = cases.case_3d(N=(nx, 32, 48), Nt=12, pml=4, source="p", absorbing=medium != "lossless", nonlinear=True,
                          alpha_power=2.0 if medium == "stokes" else 1.5, seed=seed)
        if medium == "stokes":
            f["absorbing_flag"] = np.full_like(f["absorbing_flag"], 2)
        items.append(f)
    print(f"[gpu batched rows] {nx}x32x48 {medium}", flush=True)
    rec = ("p", "p_max", "p_final", "u_final")
    with kw.Server(batching=True, max_active=4, steps_per_quantum=5) as srv:
        ids = [srv.submit(f, record=rec) for f in items]
        for i in ids:
            assert srv.wait(i, timeout=100.0) and srv.state(i) == "done", srv.error(i)
        outs = [srv.outputs(i) for i in ids]
    for f, got in zip(items, outs):
        ref = kw.run(f, record=rec)
        for k in ref:
            np.testing.assert_array_equal(got[k], ref[k], err_msg=k)
