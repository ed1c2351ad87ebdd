"""Row kernels with full workgroups at lengths outside the tuned ones: the form
that transforms the components one after the other, which a volume of ordinary
size runs and a small grid does not (a workgroup of few row pairs takes the wide
form).  KW_ROW_WGS=64 asks for so few workgroups that these small grids fill theirs:
P row pairs each, P > RowCfg::PWIDE.  Against the FP64 oracle and the runtime-radix
kernels as in test_gpu_lengths.py (relative L2 1e-4 and 1e-5), and bit for bit
against the default workgroups: the pairs per workgroup and the form of the kernel
leave every row's transform and update as they are."""

import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu

# (shape, P): P pairs for rows that do not divide by 2 P, an odd number of rows (a last
# row alone), and a last stage that leaves threads idle; two, three and four stages
VOLUMES = [
    ((216, 32, 32), 7, dict(source="p", nonlinear=True)),
    ((105, 45, 49), 14, dict(source="p", mode="dirichlet", many=True)),
    ((135, 35, 45), 11, dict(source="p", absorbing=False, nonlinear=True)),
    ((98, 45, 45), 15, dict(source="uxyz", mode="additive-no-correction")),
    ((343, 27, 25), 5, dict(source="p", many=True)),
    ((640, 20, 20), 3, dict(source="uxyz", mode="dirichlet", absorbing=False)),
    ((1000, 18, 16), 2, dict(source="ux", nonlinear=True)),
    ((81, 50, 49), 16, dict(source=None, p0=True)),
    ((49, 63, 45), 16, dict(source="p", het=False, nonlinear=True)),
]
PLANES = [((216, 1000), 7, dict(stokes=True, nonlinear=True)), ((375, 525), 4, dict(mode="dirichlet")),
          ((270, 625), 4, dict(stokes=True, many=True)), ((150, 1024), 8, dict(stokes=True))]
REC = ("p", "p_max", "p_rms", "p_max_all", "p_final", "u_final")


def check(kw, oracle, monkeypatch, f, pairs, name):
    print(f"[gpu full rows] {name}: {pairs} pairs per workgroup", flush=True)
    few = kw.run(f, record=REC)
    monkeypatch.setenv("KW_ROW_WGS", "64")
    got = kw.run(f, record=REC)
    ref = oracle.run(f, record=REC)
    for k in ("KW_ROW_NT", "KW_PENCIL_NT", "KW_LAST_NT", "KW_PLANE"):
        monkeypatch.setenv(k, "0")
    gen = kw.run(f, record=REC)
    for k in ref:
        assert cases.rel_l2(got[k], ref[k]) <= 1e-4, (k, cases.rel_l2(got[k], ref[k]))
        assert cases.rel_l2(got[k], gen[k]) <= 1e-5, (k, cases.rel_l2(got[k], gen[k]))
        np.testing.assert_array_equal(got[k], few[k], err_msg=k)


@pytest.mark.parametrize("shape, pairs, kind", VOLUMES)
def test_volume_rows(kw, oracle, monkeypatch, shape, pairs, kind):
    check(kw, oracle, monkeypatch, cases.case_3d(N=shape, Nt=12, pml=4, **kind), pairs, f"volume {shape}")


@pytest.mark.parametrize("shape, pairs, kind", PLANES)
def test_plane_rows(kw, oracle, monkeypatch, shape, pairs, kind):
    check(kw, oracle, monkeypatch, cases.case_2d_absorbing_psource(N=shape, Nt=16, **kind), pairs, f"plane {shape}")
