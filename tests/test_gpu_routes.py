"""Each kernel that the size rules choose between, held to the oracle or to the
kernels it replaces on sizes that reach it."""
import numpy as np
import pytest

from tests.helpers import host_case, oracle_sim

pytestmark = pytest.mark.gpu


def _sim(n, precision="f64", seed=21, swirl=True):
    """A simulation of n cells, for operators with winds of both signs everywhere
    (swirl; no state to step), and its fields."""
    import json

    from tests.test_gpu_parity import _gpu_sim, _swirl
    nl, Gr, RS, Th, fields = host_case(*n, seed=seed)
    nl = json.loads(json.dumps(nl))
    nl["mi355x"]["precision"] = precision
    if swirl:
        fields = _swirl(Gr, fields)
    return _gpu_sim(nl, Gr, RS, Th, fields), Gr, RS, Th, fields


@pytest.mark.parametrize("n", [(24, 20, 16), (96, 13, 33), (64, 64, 75), (128, 64, 64)])
@pytest.mark.parametrize("zero", [False, True])
def test_rk3_call_keeps_x_and_y_tendencies(gpu, n, zero):
    """After the advection with its RK3 stage (FP64) the tendency arrays hold the
    x and y contributions, the same bits as after the x and y passes alone,
    also where the y and z passes run as one kernel (the first three grids by
    default, the last on request): every stage, added to what the arrays
    held and written over it."""
    import torch
    from pycles_amd import _capi
    from pycles_amd.Advection import advect_fused, advect_rk3
    sim = _sim(n)[0]
    PV = sim.PV
    g = torch.Generator(device="cuda").manual_seed(3)
    held = 1e-3 * torch.randn(PV.tendencies.shape, generator=g, device="cuda", dtype=torch.float64)
    PV.tendencies.copy_(held)
    for p in (_capi.ADV_PASS_X, _capi.ADV_PASS_Y):
        advect_fused(sim.SA, sim.MA, sim.Gr, sim.Ref, PV, tend_zero=zero, passes=p)
    want = PV.tendencies.clone()
    cp = PV.values * (1.0 + 1e-3)
    sim.TS.dt = 0.5
    for rk in range(3):
        for flags in (0, _capi.ADV_FUSE_YZ):
            sim.TS.rk_step = rk
            PV.tendencies.copy_(held)
            out = torch.zeros_like(PV.values)
            advect_rk3(sim.SA, sim.MA, sim.TS, sim.Gr, sim.Ref, PV, tend_zero=zero, passes=flags,
                       arrays=(out, None if rk == 0 else cp))
            torch.cuda.synchronize()
            assert torch.equal(PV.tendencies, want), (rk, flags)


def _projection(n, code, shift, gw=3):
    """One projection of seeded fields whose arrays start `shift` elements off a
    16-byte boundary: u, v, w, p and div as numpy arrays, and the inputs."""
    import torch
    from pycles_amd import _capi
    from pycles_amd import _device as D
    nx, ny, nz = n
    nzg, N = nz + 2 * gw, nx * ny * (nz + 2 * gw)
    dx = (50.0, 60.0, 20.0)
    dt = D.torch_dtype(code)
    rng = np.random.default_rng(nx + nz)
    alpha = 0.8 + 0.5 * np.arange(nzg) / nzg
    prof = {"rho0": 1.0 / alpha, "rho0_half": 1.0 / (alpha - 0.004), "alpha0": alpha, "alpha0_half": alpha - 0.004,
            "p0": 1e5 - np.arange(nzg), "p0_half": 1e5 - np.arange(nzg)}
    dp = {k: torch.from_numpy(v).cuda() for k, v in prof.items()}
    ref = _capi.Ref(*[dp[k].data_ptr() for k in ("rho0", "rho0_half", "alpha0", "alpha0_half", "p0", "p0_half")])
    f = rng.standard_normal((3, nzg, ny, nx)).astype(np.float64 if code == D.F64 else np.float32)
    for a in f[:2]:
        a[:gw], a[nzg - gw:] = a[gw:2 * gw][::-1], a[nzg - 2 * gw:nzg - gw][::-1]
    f[2, gw - 1] = f[2, nzg - gw] = f[2, nzg - gw - 1] = 0.0
    buf = torch.zeros(5 * N + 4, dtype=dt, device="cuda")
    buf[shift:shift + 3 * N] = torch.from_numpy(f).cuda().reshape(-1)
    esz = buf.element_size()
    ptr = [buf.data_ptr() + esz * (shift + q * N) for q in range(5)]
    plan = _capi.PressurePlan(_capi.Dims(n, gw, dx), prof["rho0"].ctypes.data, prof["rho0_half"].ctypes.data, code)
    plan.update(ref, *ptr, 0.75, None, D.stream())
    torch.cuda.synchronize()
    return buf[shift:shift + 5 * N].cpu().numpy().reshape(5, nzg, ny, nx), f, prof, dx


def _projection_oracle(n, f, prof, dx, gw=3):
    """The oracle's projection of the same fields: u, v, w, p, div."""
    from oracle import oracle as O
    nx, ny, nz = n
    oref = O.Ref(*[prof[k] for k in ("p0", "p0_half", "alpha0", "alpha0_half", "rho0", "rho0_half")])
    sim = O.OracleSimulation(O.make_dims(nx, ny, nz, gw, *dx), oref, False, None)
    for k, a in zip("uvw", f):
        sim.pv(k)[...] = np.pad(a.astype(np.float64).transpose(2, 1, 0), ((gw, gw), (gw, gw), (0, 0)), mode="wrap")
    sim.pressure_update()
    inner = lambda a: np.asarray(a)[gw:-gw, gw:-gw].transpose(2, 1, 0)  # noqa: E731
    return [inner(sim.pv(k)) for k in "uvw"] + [inner(sim.dv[k]) for k in ("dynamic_pressure", "divergence")]


# (size, precision, form): 0 general, levels beyond whole segments (8 FP64, 16
# FP32); 1 stored pivots for few columns, below and above 64 KB of LDS and at
# its last level count; 2 and 3 planes
FORMS = [((16, 32, 317), "f64", 0), ((256, 128, 83), "f64", 0), ((16, 32, 501), "f32", 0), ((128, 256, 131), "f32", 0),
         ((64, 128, 41), "f64", 1), ((64, 64, 100), "f64", 1), ((32, 32, 250), "f64", 1), ((16, 32, 315), "f64", 1),
         ((64, 128, 41), "f32", 1), ((64, 64, 100), "f32", 1), ((32, 32, 250), "f32", 1), ((16, 32, 499), "f32", 1),
         ((256, 128, 70), "f64", 2), ((256, 128, 70), "f32", 2), ((64, 64, 75), "f64", 3), ((64, 64, 75), "f32", 3)]


@pytest.mark.parametrize("n,precision,form", FORMS)
def test_projection_form_against_the_oracle(gpu, n, precision, form):
    """Each form of the projection, by 16-byte accesses and with the fields off
    a 16-byte boundary: the two give the same bits (the same operations on the
    same values), and the first agrees with the oracle, in FP64 to the
    bound of test_pressure_parity (1e-12 of each field's maximum, in proportion
    to the transforms' length above 2^12 points), in FP32 to that of
    test_pressure_f32 (2e-5; these domains are at most 512 cells wide), and its
    divergence, about ten FP32 roundings of terms that are at most twice the
    maximum, to 2e-6."""
    from pycles_amd import _capi
    from pycles_amd import _device as D
    code = D.precision_code(precision)
    assert _capi.pressure_form(_capi.Dims(n, 3, (50.0, 60.0, 20.0)), code) == form
    print(n, precision, "aligned", flush=True)
    got, f, prof, dx = _projection(n, code, 0)
    print("shifted", flush=True)
    off = _projection(n, code, 1)[0]
    assert np.array_equal(got, off)
    want = _projection_oracle(n, f, prof, dx)
    sl = slice(3, -3)
    r = 1e-12 * max(1.0, np.log2(n[0] * n[1]) / 12)
    tol = {"f64": (r,) * 4 + (1e-12,), "f32": (2e-5,) * 4 + (2e-6,)}[precision]
    for q, name in enumerate(("u", "v", "w", "p", "div")):
        a, b = (got[q], want[q]) if name != "div" else (got[q][sl], want[q][sl])
        err = np.abs(a.astype(np.float64) - b).max() / np.abs(b).max()
        print(name, err, flush=True)
        assert err <= tol[q], (name, err)


def test_separate_passes_against_the_oracle(gpu):
    """The x, y and z passes of moist WENO5 launched one by one (FP64, partial
    tiles in every direction): the oracle's bits."""
    import torch
    from pycles_amd import _capi
    from pycles_amd.Advection import advect_fused
    sim, Gr, RS, Th, fields = _sim((24, 20, 16), seed=7)
    for p in (_capi.ADV_PASS_X, _capi.ADV_PASS_Y, _capi.ADV_PASS_Z):
        advect_fused(sim.SA, sim.MA, sim.Gr, sim.Ref, sim.PV, passes=p)
    torch.cuda.synchronize()
    osim = oracle_sim(Gr, RS, Th, fields, True)
    osim.scalar_advection_update()
    osim.momentum_advection_update()
    gw = Gr.dims.gw
    for n in ("u", "v", "w", "s", "qt"):
        g = sim.PV.get_tendency_array(n, Gr)[gw:-gw, gw:-gw, gw:-gw]
        assert np.array_equal(g, osim.pt(n)[gw:-gw, gw:-gw, gw:-gw]), n


@pytest.mark.parametrize("n,fused", [((64, 64, 64), True), ((64, 64, 76), False)])
def test_yz_switch(gpu, n, fused):
    """On both sides of the FP64 switch (256 and 304 blocks) the default call
    gives the bits of the passes launched one by one, and a timed step brackets
    the passes that the untimed one runs, with its bits."""
    import torch
    from pycles_amd import _capi
    from pycles_amd.Advection import advect_fused, yz_fused
    sim = _sim(n)[0]
    PV = sim.PV
    assert yz_fused(sim.SA, sim.MA, PV) == fused
    out = []
    for seq in ((0,), (_capi.ADV_PASS_X, _capi.ADV_PASS_Y, _capi.ADV_PASS_Z)):
        PV.zero_tendencies()
        for p in seq:
            advect_fused(sim.SA, sim.MA, sim.Gr, sim.Ref, PV, passes=p)
        out.append(PV.tendencies.clone())
    assert torch.equal(out[0], out[1])
    steps = []
    for timed in (False, True):
        s = _sim(n, swirl=False)[0]
        s.begin_run()
        s.timers = [] if timed else None
        s.step()
        torch.cuda.synchronize()
        steps.append((s.PV.values.clone(), s.PV.tendencies.clone()))
    names = {a for a, _ in s.timers}
    assert ("adv_yz_rk3" in names, "adv_z_rk3" in names) == (fused, not fused)
    assert torch.equal(steps[0][0], steps[1][0]) and torch.equal(steps[0][1], steps[1][1])
