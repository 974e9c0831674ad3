"""The wall-normal kernels at the sizes where their launch shape changes.

Row blocks: n up to 128 / 129 (4 blocks of 16) against above; pencils: few, between, and
enough to fill the chip; columns that leave a partial last tile.  dfdz and the homogeneous
solve against the same products in numpy (FP64 sums in another order, bar 1e-12 relative
L2); the pressure step and the velocity solves against their unfused or FP64 forms (FP64:
another order of the same sums, 1e-10 in the velocities and 1e-7 in the pressure; mixed: the
FP32 rounding of the velocity solve's correction, 1e-6).
"""

import numpy as np
import pytest

import lsbflow_amd as L
from lsbflow_amd.core import Config, Context, setup_case
from tests.conftest import rel_l2
from tests.test_gpu_helmholtz_c3 import Hip, c3_rhs, solve_dev

pytestmark = pytest.mark.gpu

NZ = [16, 63, 64, 127, 128, 129, 130, 144]
HORIZ = [(20, 12), (160, 108), (324, 216)]  # 240 pencils, 17,280, 69,984: few, between, wide


@pytest.mark.parametrize("nx,ny", HORIZ)
@pytest.mark.parametrize("nz", NZ)
def test_derivative_and_solve(nx, ny, nz):
    rng = np.random.default_rng(nz * 7 + nx)
    with Context(Config(nx=nx, ny=ny, nz=nz)) as ctx:
        m, g = ctx.mats(), ctx.grid()
        u = rng.standard_normal((nz + 1, ny, nx))
        ref = (m["mdz"] @ u.reshape(nz + 1, -1)).reshape(u.shape)
        ed = rel_l2(ctx.dfdz(u), ref)
        sigma = 250.0
        k2 = (g["wavx"] ** 2)[None, :] + (g["wavy"] ** 2)[:, None] + sigma
        q = m["simat"] @ u[1:-1].reshape(nz - 1, -1)
        q /= m["diag"][:, None] - k2.reshape(1, -1)
        ref = np.zeros_like(u)
        ref[1:-1] = (m["smat"] @ q).reshape(nz - 1, ny, nx)
        es = rel_l2(ctx.solve_helmholtz(u, sigma), ref)
    print(f"{nx}x{nz + 1}x{ny}: dfdz {ed:.1e} solve {es:.1e}", flush=True)
    assert ed < 1e-12 and es < 1e-12


def run(case, precision):
    with setup_case(case, precision=precision) as ctx:
        ctx.state_set(*L.cases.initial_condition(case))
        ctx.timestep(3)
        return ctx.state_get()


@pytest.mark.parametrize("nx,ny", [(32, 12), (160, 108), (216, 162)])  # 384, 17,280, 34,992 pencils
@pytest.mark.parametrize("nz", [63, 128, 129])
def test_step_against_unfused(nx, ny, nz, monkeypatch):
    case = L.cases.CASES["c2_dyn_les"].with_(nx=nx, ny=ny, nz=nz, sgsmodel=2, dt=5e-5, samp=0.1)
    got = run(case, 0)
    monkeypatch.setenv("LSB_NO_ZPRESS", "1")
    monkeypatch.setenv("LSB_NO_ZHELM", "1")
    ref = run(case, 0)
    errs = {k: rel_l2(got[k], ref[k]) for k in ("uf", "vf", "wf", "pf")}
    monkeypatch.delenv("LSB_NO_ZPRESS")
    monkeypatch.delenv("LSB_NO_ZHELM")
    got = run(case, 1)
    monkeypatch.setenv("LSB_NO_ZHELM32", "1")
    ref = run(case, 1)
    mixed = {k: rel_l2(got[k], ref[k]) for k in ("uf", "vf", "wf")}
    print(f"{nx}x{nz + 1}x{ny}: {errs} mixed {mixed}", flush=True)
    assert max(errs[k] for k in ("uf", "vf", "wf")) < 1e-10 and errs["pf"] < 1e-7
    assert max(mixed.values()) < 1e-6


@pytest.mark.parametrize("nx,ny", HORIZ[:2] + [(162, 108)])
@pytest.mark.parametrize("nz", [16, 64, 127, 129, 170, 172, 192])
@pytest.mark.parametrize("sigma", [0.0, 2.0e5])
def test_fp32_and_refined_solve(nx, ny, nz, sigma, monkeypatch):
    """The one-kernel solves against the FP64 solution: FP32's rounding times the solve's
    conditioning (1.7e-7 at most here; the separate kernels' error up to the order of its
    sums), and after the refinement that error times itself, at least four digits below.
    The two routes sum in different orders, so equal bits would mean that one of them ran
    twice."""
    hip = Hip()
    with setup_case(L.cases.CASES["c2_dyn_les"].with_(nx=nx, ny=ny, nz=nz)) as ctx:
        rhs = c3_rhs(nz + 1, nx * ny, 2).reshape(2, nz + 1, ny, nx)
        u64 = solve_dev(ctx, hip, rhs, sigma, 0)
        u32, ur = (solve_dev(ctx, hip, rhs, sigma, m) for m in (1, 2))
        monkeypatch.setenv("LSB_NO_ZREFINE", "1")
        s32, sr = (solve_dev(ctx, hip, rhs, sigma, m) for m in (1, 2))
    e = [rel_l2(x, u64) for x in (u32, ur, s32, sr)]
    print(f"{nx}x{nz + 1}x{ny} sigma {sigma}: FP32 {e[0]:.1e} refined {e[1]:.1e}; separate {e[2]:.1e} {e[3]:.1e}",
          flush=True)
    assert np.all(ur[:, 0] == 0.0) and np.all(ur[:, nz] == 0.0) and np.all(u32[:, nz] == 0.0)
    assert not np.array_equal(u32, s32) and not np.array_equal(ur, sr)
    assert e[0] < 1e-6 and e[1] < 1e-4 * e[0]
    assert e[0] < 4.0 * e[2] and e[1] < 4.0 * max(e[3], 1e-15)
