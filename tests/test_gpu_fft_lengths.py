"""The horizontal transforms at the lengths with a factor 3 or 5.

Every x length (nx/2) and y length (ny) of the register-resident passes that is not a
power of two, one plane count that leaves a partial last block of rows, kx columns that
leave a partial last tile.  FP64 transforms against numpy's (pocketfft): both round each
of the log2(N) butterfly levels, relative L2 a few eps, bar 4e-15; the fused gradient
transform and the products against the oracle's nonlinear term (bar 1e-10, the operator
bar); the mixed form's fused forward pass and right-hand side against the FP64 step, which
FP32 rounding of the nonlinear chain leaves within 1e-5.
"""

import ctypes as C

import numpy as np
import pytest

import lsbflow_amd as L
from lsbflow_amd import _lib
from lsbflow_amd.core import Config, Context, setup_case
from oracle import Oracle, OracleConfig
from tests.conftest import rel_l2
from tests.test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu

XLEN = [24, 25, 27, 30, 36, 40, 45, 48, 50, 54, 60, 72, 75, 80, 81, 90, 96, 100, 108, 120, 135, 144, 150, 160, 162, 180,
        192, 200, 216, 225, 240]
YLEN = [n for n in XLEN if n % 2 == 0]
PAIRS = [(2 * m, YLEN[(5 * i) % len(YLEN)]) for i, m in enumerate(XLEN)]
NZP = 5


def test_pairs_cover_every_length():
    assert {ny for _, ny in PAIRS} == set(YLEN)


@pytest.mark.parametrize("nx,ny", PAIRS + [(128, 60), (120, 64), (250, 60), (60, 24)])
def test_transform_pair(nx, ny):
    rng = np.random.default_rng(nx * 1000 + ny)
    with Context(Config(nx=nx, ny=ny, nz=NZP - 1)) as ctx:
        x = np.zeros((2, NZP, ny, nx + 2))
        x[..., :nx] = rng.standard_normal((2, NZP, ny, nx))
        ref = np.fft.fft(np.fft.rfft(x[..., :nx])[..., : nx // 2], axis=-2) / (nx * ny)
        spec = ctx.fwd(x)
        ef = rel_l2(spec.reshape(ref.shape + (2,)), np.stack([ref.real, ref.imag], axis=-1))
        s = rng.standard_normal((2, NZP, ny, nx))
        full = np.zeros((2, NZP, ny, nx // 2 + 1), dtype=complex)
        full[..., : nx // 2] = np.fft.ifft(np.ascontiguousarray(s).view(complex), axis=-2, norm="forward")
        back = ctx.inv(s)
        ei = rel_l2(back[..., :nx], np.fft.irfft(full, n=nx, norm="forward"))
        assert np.all(back[..., nx:] == 0.0)
    print(f"{nx}x{ny}: forward {ef:.1e} inverse {ei:.1e}", flush=True)
    assert ef < 4e-15 and ei < 4e-15


def case_of(nx, ny):
    return L.cases.CASES["c2_dyn_les"].with_(nx=nx, ny=ny, nz=12, sgsmodel=2, xnu=2e-5, dt=2.5e-4, samp=0.1)


@pytest.mark.parametrize("nx,ny", PAIRS[::2] + [(50, 60)])
def test_nonlinear_term(nx, ny):
    case = case_of(nx, ny).with_(sgsflag=0)
    keys = OracleConfig.__dataclass_fields__
    o = Oracle(OracleConfig(**{k: v for k, v in case.as_dict().items() if k in keys}))
    o.ubar, o.ubarp, o.ubarpp = L.cases.base_flow(case)
    uif = np.stack(L.cases.initial_condition(case.with_(pert_rms=0.05)))
    ref, _ = o.nlterm_skewsym(uif, np.zeros_like(uif[0]), 0)
    with setup_case(case) as ctx:
        got = ctx.nlterm_skewsym(uif)
    e = rel_l2(got, ref)
    print(f"{nx}x{ny}: nonlinear term {e:.1e}", flush=True)
    assert e < 1e-10


@pytest.mark.parametrize("nx,ny", PAIRS)
def test_mixed_step_against_fp64(nx, ny):
    case = case_of(nx, ny)
    out = []
    for precision in (0, 1):
        with setup_case(case, precision=precision) as ctx:
            ctx.state_set(*L.cases.initial_condition(case))
            ctx.timestep(4)
            out.append(ctx.state_get())
    errs = {k: rel_l2(out[1][k], out[0][k]) for k in ("uf", "vf", "wf", "nlnif")}
    print(f"{nx}x{ny}: mixed vs FP64 {errs}", flush=True)
    assert max(errs.values()) < 1e-5


def test_noalloc_beyond_its_scratch_stays_accepted():
    """One field of 480 x 240 x 301 exceeds the 2^25-double scratch, which the lengths with a
    factor 3 or 5 do not use: accepted, the bits of lsb_horfft_dev."""
    nx, ny, nz = 480, 240, 300
    hip, lib = Hip(), _lib.lib()
    with Context(Config(nx=nx, ny=ny, nz=nz)) as ctx:
        s = np.random.default_rng(3).standard_normal((nz + 1, ny, nx))
        spec = hip.alloc(s.nbytes)
        hip.put(spec, s)
        got = []
        for fn in (lib.lsb_horfft_dev, lib.lsb_horfft_dev_noalloc):
            out = hip.alloc((nz + 1) * ny * (nx + 2) * 8)
            _lib.check(fn(ctx.h, out, spec, 1, 1, None), "horfft")
            ctx.synchronize()
            got.append(hip.get(out, (nz + 1, ny, nx + 2)))
            assert hip.lib.hipFree(out) == 0
        assert hip.lib.hipFree(spec) == 0
    assert np.array_equal(*got)


def device_fields(hip, nf, nx, ny, nzp, seed):
    """(nf spectral fields on the device, room for their physical ones, its shape)"""
    s = np.random.default_rng(seed).standard_normal((nf, nzp, ny, nx))
    shape = (nf, nzp, ny, nx + 2)
    spec, out = hip.alloc(s.nbytes), hip.alloc(8 * int(np.prod(shape)))
    hip.put(spec, s)
    hip.put(out, np.zeros(shape))
    return spec, out, shape


def capture(hip, stream, enqueue):
    graph, ex = C.c_void_p(), C.c_void_p()
    assert hip.lib.hipStreamBeginCapture(stream, 1) == 0
    enqueue()
    assert hip.lib.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert hip.lib.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)) == 0
    assert hip.lib.hipGraphDestroy(graph) == 0
    return ex


@pytest.mark.parametrize("nz,nf", [(100, 3), (250, 2)])
def test_inverse_takes_no_memory(nz, nf):
    """Three fields of 93 MB (a piece of one field and one of two) and two of 232 MB (two pieces
    of the planes of each) leave the device's free memory as it was, and have the bits of
    fifty planes at a time."""
    nx, ny, np50 = 480, 240, 50
    hip, lib = Hip(), _lib.lib()
    with Context(Config(nx=nx, ny=ny, nz=nz)) as ctx, Context(Config(nx=nx, ny=ny, nz=np50 - 1)) as few:
        spec, out, shape = device_fields(hip, nf, nx, ny, nz + 1, 3)
        for f in range(nf):
            for k in range(0, nz, np50):
                o, i = (C.c_void_p(p.value + 8 * (f * (nz + 1) + k) * ny * n) for p, n in ((out, nx + 2), (spec, nx)))
                _lib.check(lib.lsb_horfft_dev(few.h, o, i, 1, 1, None), "horfft")
        few.synchronize()
        want = hip.get(out, shape)[:, :nz]
        hip.put(out, np.zeros(shape))
        free = hip.free_bytes()
        _lib.check(lib.lsb_horfft_dev(ctx.h, out, spec, 1, nf, None), "horfft")
        ctx.synchronize()
        assert hip.free_bytes() == free
        assert np.array_equal(hip.get(out, shape)[:, :nz], want)
        for p in (spec, out):
            assert hip.lib.hipFree(p) == 0


def test_first_inverse_under_capture():
    """A first inverse transform inside a stream capture, one field of 337 MB (two pieces of
    its planes): the graph replays to the eager bits."""
    nx, ny, nz = 480, 240, 365
    hip, lib = Hip(), _lib.lib()
    with Context(Config(nx=nx, ny=ny, nz=nz)) as ctx, Context(Config(nx=nx, ny=ny, nz=nz)) as ref:
        spec, out, shape = device_fields(hip, 1, nx, ny, nz + 1, 5)
        want = hip.alloc(8 * int(np.prod(shape)))
        _lib.check(lib.lsb_horfft_dev(ref.h, want, spec, 1, 1, None), "horfft")
        ref.synchronize()
        stream = C.c_void_p(ctx.stream())
        ex = capture(hip, stream, lambda: _lib.check(lib.lsb_horfft_dev(ctx.h, out, spec, 1, 1, stream), "horfft"))
        for _ in range(3):
            hip.put(out, np.zeros(shape))
            assert hip.lib.hipGraphLaunch(ex, stream) == 0
            ctx.synchronize()
            assert np.array_equal(hip.get(out, shape), hip.get(want, shape))
        hip.lib.hipGraphExecDestroy(ex)
        for p in (spec, out, want):
            assert hip.lib.hipFree(p) == 0


def test_captured_inverse_outlives_larger_calls():
    """A graph of the inverse captured after an eager one of the same size (280 MB) replays to
    the eager bits also after eager calls with more fields, and beside a transform of the same
    context on another stream: it holds no buffer of the context."""
    nx, ny, nz = 480, 240, 100
    hip, lib = Hip(), _lib.lib()

    def inverse(ctx, f, nf, stream):
        _lib.check(lib.lsb_horfft_dev(ctx.h, f[1], f[0], 1, nf, stream), "horfft")

    with Context(Config(nx=nx, ny=ny, nz=nz)) as ctx, Context(Config(nx=nx, ny=ny, nz=nz)) as other:
        a, b = (device_fields(hip, nf, nx, ny, nz + 1, 10 + nf) for nf in (3, 4))
        s1, s2 = C.c_void_p(ctx.stream()), C.c_void_p(other.stream())
        inverse(ctx, a, 3, s1)
        inverse(ctx, b, 4, s1)
        ctx.synchronize()
        want = [hip.get(x[1], x[2]) for x in (a, b)]
        ex = capture(hip, s1, lambda: inverse(ctx, a, 3, s1))
        for _ in range(3):
            for x in (a, b):
                hip.put(x[1], np.zeros(x[2]))
            assert hip.lib.hipGraphLaunch(ex, s1) == 0
            inverse(ctx, b, 4, s2)
            ctx.synchronize()
            other.synchronize()
            for x, w in zip((a, b), want):
                assert np.array_equal(hip.get(x[1], x[2]), w)
        hip.lib.hipGraphExecDestroy(ex)
        for x in (a, b):
            for p in x[:2]:
                assert hip.lib.hipFree(p) == 0


@pytest.mark.parametrize("nx,ny,nz", [(32, 16, 16), (128, 64, 32), (512, 256, 16), (48, 24, 16), (180, 150, 16), (480, 240, 16)])
def test_fp64_forward_y_with_rhs(nx, ny, nz, monkeypatch):
    """The forward y pass with the right-hand side in its epilogue against the two passes
    (LSB_NO_YRHS=1): the smallest, middle and largest lengths of both kinds, with partial
    tiles of 16 kx columns, over three steps (each order of the schemes).  They differ by
    roundings of the three pieces of N (a few 1e-16 of the largest, which the sum can leave
    1e3 below): 1e-12 for N and the velocities; the pressure, a divergence divided by
    k^2 dt, 1e-9."""
    case = L.cases.CASES["c1_dns"].with_(name="yrhs", nx=nx, ny=ny, nz=nz, dt=1e-4, pert_rms=1e-2)
    u, v, w = L.cases.initial_condition(case)
    out = {}
    for sep in ("0", "1"):
        monkeypatch.setenv("LSB_NO_YRHS", sep)
        c = setup_case(case)
        try:
            c.state_set(u, v, w)
            c.timestep(3)
            out[sep] = c.state_get()
        finally:
            c.close()
    for k in ("uf", "vf", "wf", "pf", "nlnif", "nlnmif"):
        assert np.all(np.isfinite(out["0"][k])), k
        assert rel_l2(out["0"][k], out["1"][k]) < (1e-9 if k == "pf" else 1e-12), k
