"""The step's boundary planes, norm and friction velocity on grids that do not fill their
blocks, against the oracle (the bars of test_gpu_step)."""

import numpy as np
import pytest

import lsbflow_amd as L
from lsbflow_amd.core import setup_case
from tests.conftest import rel_l2
from tests.test_gpu_step import check_fields, run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "nx,ny,nz",
    [
        (36, 10, 8),   # 180 modes (11 blocks of 16 and a part), 9 planes for 16 groups
        (40, 12, 16),  # 240 modes (whole blocks), 17 planes: one group takes two
        (32, 2, 24),   # the smallest ny (no Nyquist row)
    ],
)
@pytest.mark.parametrize("model,top_bc,bctype", [(0, 0, 3), (2, 2, 0)])
def test_partial_blocks(nx, ny, nz, model, top_bc, bctype):
    case = L.cases.CASES["c1_dns"].with_(name="small", nx=nx, ny=ny, nz=nz, sgsflag=1, sgsmodel=model, top_bc=top_bc,
                                         bctype=bctype, dt=2e-4, pert_rms=1e-2)
    st, g = run_both(case, 3)
    check_fields(st, g)


@pytest.mark.parametrize(
    "nx,ny",
    [(32, 2), (64, 16), (512, 256), (50, 24), (54, 30), (90, 48), (96, 50), (150, 10), (192, 96), (400, 36), (450, 60), (480, 240)],
)
@pytest.mark.parametrize("precision", [0, 1])
def test_ceiling_blend_x_lines(nx, ny, precision, monkeypatch):
    """The blended ceiling by x lines (no y transforms) against the 2-D transforms
    (LSB_NO_XBLEND=1): even and odd line counts per block, both kinds of lengths.  The two
    differ by the rounding of one plane's transforms, log2(nx ny) levels of 1e-16 each:
    1e-12 on the velocities of three steps, 1e-9 on the pressure (a divergence over
    k^2 dt); the mixed form's FP32 chain can round those differences up to its own
    3e-7 per field value, 1e-6 and 1e-4."""
    case = L.cases.CASES["c1_dns"].with_(name="blend", nx=nx, ny=ny, nz=16, sgsflag=1, sgsmodel=0, top_bc=2, samp=0.3,
                                         dt=1e-4, pert_rms=1e-2)
    u, v, w = L.cases.initial_condition(case)
    out = {}
    for sep in ("0", "1"):
        monkeypatch.setenv("LSB_NO_XBLEND", sep)
        c = setup_case(case, precision=precision)
        try:
            c.state_set(u, v, w)
            c.timestep(3)
            out[sep] = c.state_get()
        finally:
            c.close()
    for k in ("uf", "vf", "wf", "pf"):
        assert np.all(np.isfinite(out["0"][k])), k
        err = rel_l2(out["0"][k], out["1"][k])
        bar = ((1e-12, 1e-9), (1e-6, 1e-4))[precision][k == "pf"]
        print(nx, ny, precision, k, f"{err:.2e}", flush=True)
        assert err < bar, (k, err)
