"""The dynamic model in its two passes over u' and g' against the stages and the filter as
passes of their own (LSB_NO_DYNFUSE=1): the same bits, for both stored types."""

import numpy as np
import pytest

import lsbflow_amd as L
from lsbflow_amd._lib import LsbError
from lsbflow_amd.core import setup_case
from tests.test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu

# tiles are 62 columns at most (evened out over the row) by 6 rows, sliding over z
GRIDS = [
    (32, 8, 16),     # one tile in x, ny = 6 + 2
    (60, 30, 32),    # one tile of 60 columns
    (64, 36, 48),    # two of 32, whole row tiles
    (192, 50, 64),   # four of 48, a last tile of two rows
    (1152, 16, 16),  # FP64 only: the mixed model refuses rows above 1024 points
]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nx,ny,nz", GRIDS)
@pytest.mark.parametrize("b,dyn_avg,forcing", [(2.0, 0, 1), (1.0, 1, 0), (1.0, 0, 0)])
def test_two_passes_bit_identical(nx, ny, nz, b, dyn_avg, forcing, precision, monkeypatch):
    """(a, b) = (1, 2), whose sum 4 goes into the weights, and (1, 1), which divides by 3."""
    case = L.cases.CASES["c2_dyn_les"].with_(name=f"dynf{nx}x{ny}", nx=nx, ny=ny, nz=nz, dyn_avg=dyn_avg, b=b,
                                             dt=1e-4, pert_rms=1e-2)
    u, v, w = L.cases.initial_condition(case)
    out = {}
    for sep in ("0", "1"):
        monkeypatch.setenv("LSB_NO_DYNFUSE", sep)
        c = setup_case(case, precision=precision, forcing=forcing)
        try:
            if forcing:
                c.set_sponge(0.3, 0.25, 0.70)
            c.state_set(u, v, w)
            if precision and nx > 1024:
                with pytest.raises(LsbError):
                    c.timestep(2)
                return
            c.timestep(3)
            out[sep] = c.state_get()
        finally:
            c.close()
    for k in ("uf", "vf", "wf", "pf", "nlnif", "nlnmif"):
        assert np.all(np.isfinite(out["0"][k])), k
        assert np.array_equal(out["0"][k], out["1"][k]), k


@pytest.mark.parametrize("precision", [0, 1])
def test_state_holds_what_the_two_passes_use(precision):
    """The dynamic model's state takes three fields more than the sigma model's (M:L, M:M and
    the plane means' partial sums); allocations are rounded, one field at most."""
    hip, taken = Hip(), []
    for model in (2, 1):
        case = L.cases.CASES["c2_dyn_les"].with_(name="mem", nx=128, ny=64, nz=64, sgsmodel=model)
        with setup_case(case, precision=precision) as c:
            before = hip.free_bytes()
            c.state_set(*L.cases.initial_condition(case))
            c.timestep(2)
            c.synchronize()
            taken.append(before - hip.free_bytes())
    field = 130 * 64 * 65 * 8
    print(f"precision {precision}: {(taken[1] - taken[0]) / field:.1f} fields", flush=True)
    assert taken[1] - taken[0] <= 4 * field
