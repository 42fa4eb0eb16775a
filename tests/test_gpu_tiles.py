"""Kernels that tile or split their domain, at the sizes where a tile, a
remainder or a vector path can go wrong, against numpy or the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dims(n, gw, dx=(50.0, 60.0, 20.0)):
    from pycles_amd import _capi
    return _capi.Dims(tuple(n), gw, dx)


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("n,gw", [((1, 1, 2), 2), ((3, 2, 5), 5), ((64, 3, 26), 3), ((65, 9, 27), 3), ((130, 5, 75), 4),
                                  ((63, 4, 64), 8)])
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_layout_tiles(n, gw, precision):
    """Ingress and egress move values, so they are exact (the FP32 form up to
    the one rounding of its store), over partial tiles in i and k, one-cell
    extents and ghost rims wider than the domain."""
    import torch
    from pycles_amd import _capi
    from pycles_amd import _device as D
    nx, ny, nz = n
    nzg = nz + 2 * gw
    rng = np.random.default_rng(5)
    field = rng.standard_normal((nzg, ny, nx))
    base = 300.0 + rng.standard_normal(nzg)
    i = (np.arange(nx + 2 * gw) - gw) % nx
    j = (np.arange(ny + 2 * gw) - gw) % ny
    ref = np.ascontiguousarray((field + base[:, None, None])[:, j][:, :, i].transpose(2, 1, 0))
    code = D.precision_code(precision)
    np_t = np.float64 if precision == "f64" else np.float32
    src, b = _dev(ref), _dev(base)
    dev = torch.full((nzg, ny, nx), -7.0, dtype=D.torch_dtype(code), device="cuda")
    _capi.layout_ingress(_dims(n, gw), src.data_ptr(), dev.data_ptr(), b.data_ptr(), code, D.stream())
    want = ((field + base[:, None, None]) - base[:, None, None]).astype(np_t)
    assert np.array_equal(dev.cpu().numpy(), want)
    back = torch.full(ref.shape, -9.0, dtype=torch.float64, device="cuda")
    _capi.layout_egress(_dims(n, gw), dev.data_ptr(), back.data_ptr(), b.data_ptr(), code, D.stream())
    full = want.astype(np.float64) + base[:, None, None]
    assert np.array_equal(back.cpu().numpy(), full[:, j][:, :, i].transpose(2, 1, 0))
    # without a base: the values themselves
    _capi.layout_egress(_dims(n, gw), dev.data_ptr(), back.data_ptr(), None, code, D.stream())
    assert np.array_equal(back.cpu().numpy(), want.astype(np.float64)[:, j][:, :, i].transpose(2, 1, 0))


@pytest.mark.parametrize("n,gw", [((70, 9, 13), 3), ((6, 6, 5), 3), ((65, 8, 40), 2)])
def test_sgs_and_diffusion_tiles_bitwise(n, gw):
    """The SGS and diffusion marches over partial column tiles and uneven z
    chunks, FP64, bitwise against the oracle (each operator's calls apart as
    well as in one pass)."""
    import torch
    from oracle import oracle as O
    from pycles_amd import _capi
    from pycles_amd import _device as D
    nx, ny, nz = n
    nzg = nz + 2 * gw
    rng = np.random.default_rng(nx)
    dx = (50.0, 60.0, 20.0)
    dims, odims = _dims(n, gw, dx), O.make_dims(nx, ny, nz, gw, *dx)
    alpha = 0.8 + 0.01 * np.arange(nzg)
    half = alpha - 0.004
    prof = {"rho0": 1.0 / alpha, "rho0_half": 1.0 / half, "alpha0": alpha, "alpha0_half": half,
            "p0": 1e5 - 200.0 * np.arange(nzg), "p0_half": 1e5 - 200.0 * np.arange(nzg) + 90.0}
    oref = O.Ref(prof["p0"], prof["p0_half"], alpha, half, prof["rho0"], prof["rho0_half"])
    dp = {k: _dev(v) for k, v in prof.items()}
    ref = _capi.Ref(*[dp[k].data_ptr() for k in ("rho0", "rho0_half", "alpha0", "alpha0_half", "p0", "p0_half")])
    f = {k: rng.standard_normal((nzg, ny, nx)) for k in ("u", "v", "w", "s", "qt", "n2", "tu", "tv", "tw", "ts", "tq")}
    f["T"] = 290.0 + rng.standard_normal((nzg, ny, nx))
    f["n2"] *= 1e-3

    def ghosted(a):
        return np.ascontiguousarray(np.pad(a.transpose(2, 1, 0), ((gw, gw), (gw, gw), (0, 0)), mode="wrap"))

    sim = O.OracleSimulation(odims, oref, True, O.Lookup(np.linspace(100.0, 380.0, 16), np.linspace(1.0, 2.0, 16)),
                             sgs={"cs": 0.17, "prt": 1.0 / 3.0})
    for k in ("u", "v", "w", "s", "qt"):
        sim.pv(k)[...] = ghosted(f[k])
        sim.pt(k)[...] = ghosted(f["t" + k[0]])
    sim.dv["buoyancy_frequency"][...] = ghosted(f["n2"])
    sim.dv["temperature"][...] = ghosted(f["T"])
    sim.kinematics_update()
    sim.sgs_update()
    t = {k: _dev(v) for k, v in f.items()}
    smag, nu, dif = (torch.full((nzg, ny, nx), -1.0, dtype=torch.float64, device="cuda") for _ in range(3))
    vel = [t[k].data_ptr() for k in ("u", "v", "w")]
    st = D.stream()
    _capi.sgs_smagorinsky(dims, vel, t["n2"].data_ptr(), 0.17, 1.0 / 3.0, smag.data_ptr(), nu.data_ptr(), dif.data_ptr(),
                          D.F64, st)
    lv = slice(1, nzg - 1)

    def inner(a):
        return np.asarray(a)[gw:-gw, gw:-gw].transpose(2, 1, 0)

    assert np.array_equal(smag.cpu().numpy()[lv], inner(sim.smag)[lv])
    assert np.array_equal(nu.cpu().numpy()[lv], inner(sim.dv["viscosity"])[lv])
    assert np.array_equal(dif.cpu().numpy()[lv], inner(sim.dv["diffusivity"])[lv])
    # the ghost levels' outer ends, which the reference leaves at zero
    for a in (smag, nu, dif):
        assert not a[0].any() and not a[-1].any()
    # their periodic images (the oracle's own stop at ghost column 1, where
    # the reference reads before its array)
    sim.smag[...] = ghosted(smag.cpu().numpy())
    sim.dv["viscosity"][...] = ghosted(nu.cpu().numpy())
    sim.dv["diffusivity"][...] = ghosted(dif.cpu().numpy())
    sim.scalar_diffusion_update()
    sim.momentum_diffusion_update()
    S, M, E = _capi.DIFF_SCALARS, _capi.DIFF_MOMENTUM, _capi.DIFF_ENTROPY_SOURCE
    for flags in ([S | M | E], [S, M | E], [S, M, E]):
        tend = {k: _dev(f["t" + k]) for k in "uvwsq"}
        for fl in flags:
            _capi.diffusion(dims, ref, vel, [tend[k].data_ptr() for k in "uvw"] if fl & M else None,
                            [t["s"].data_ptr(), t["qt"].data_ptr()], [tend["s"].data_ptr(), tend["q"].data_ptr()], None,
                            nu.data_ptr(), dif.data_ptr(), smag.data_ptr(), t["T"].data_ptr(), fl, D.F64, st)
        for k, n_ in (("u", "u"), ("v", "v"), ("w", "w"), ("s", "s"), ("q", "qt")):
            assert np.array_equal(tend[k].cpu().numpy()[gw:-gw], inner(sim.pt(n_))[gw:-gw]), (flags, n_)


@pytest.mark.parametrize("n,gw", [((8, 6, 3), 3), ((9, 7, 5), 5), ((64, 33, 20), 3), ((13, 1, 11), 2), ((1, 3, 4), 4)])
@pytest.mark.parametrize("precision,shift", [("f64", 0), ("f32", 0), ("f32", 1), ("f64", 1)])
def test_rk3_stage_tiles(n, gw, precision, shift):
    """The RK3 stage over planes that do and do not divide into 16-byte
    accesses, fields off a 16-byte boundary (shift), columns no deeper than
    their ghost rim, and every boundary type, bitwise against numpy in the
    field's precision (the update uses uncontracted + and *)."""
    import torch
    from pycles_amd import _capi
    from pycles_amd import _device as D
    nx, ny, nz = n
    nzg, N = nz + 2 * gw, nx * ny * (nz + 2 * gw)
    np_t = np.float64 if precision == "f64" else np.float32
    code = D.precision_code(precision)
    bcs = [1.0, -1.0, 2.0, -0.5]
    rng = np.random.default_rng(7)
    val, ten, cpy = (rng.standard_normal((4, nzg, ny, nx)).astype(np_t) for _ in range(3))
    sl = slice(gw, gw + nz)
    dt = 0.7

    def up(a):
        buf = torch.zeros(4 * N + 4, dtype=D.torch_dtype(code), device="cuda")
        buf[shift:shift + 4 * N] = _dev(a).reshape(-1)
        return buf, [buf.data_ptr() + (shift + q * N) * buf.element_size() for q in range(4)]

    def down(b):
        return b[shift:shift + 4 * N].cpu().numpy().reshape(4, nzg, ny, nx)

    for rk in range(3):
        for zero in (0, 1):
            bv, pv = up(val)
            bt, pt = up(ten)
            bc_, pc = up(cpy)
            _capi.rk3_stage(_dims(n, gw), pv, pt, pc, bcs, rk, dt, code, D.stream(), zero)
            d = np_t(dt)
            x = val + ten * d
            want_c = cpy.copy()
            if rk == 0:
                want_c[:, sl] = val[:, sl]
            elif rk == 1:
                x = np_t(0.75) * cpy + np_t(0.25) * x
            else:
                x = np_t(1.0 / 3.0) * cpy + np_t(2.0 / 3.0) * x
            want = val.copy()
            want[:, sl] = x[:, sl]
            for q, bc in enumerate(bcs):
                f = want[q]
                for m in range(gw):
                    if bc == 1.0:
                        f[gw - 1 - m], f[nzg - gw + m] = f[gw + m], f[nzg - gw - 1 - m]
                    elif bc == 2.0:
                        f[gw - 1 - m], f[nzg - gw + m] = f[gw], f[nzg - gw - 1]
                    elif m == 0:
                        f[gw - 1] = f[nzg - gw] = 0.0
                    else:
                        f[gw - 1 - m], f[nzg - gw + m] = np_t(bc) * f[gw - 1 + m], np_t(bc) * f[nzg - gw - m]
            assert np.array_equal(down(bv), want), (rk, zero)
            assert np.array_equal(down(bc_), want_c), (rk, zero)
            assert np.array_equal(down(bt), np.zeros_like(ten) if zero else ten), (rk, zero)


@pytest.mark.parametrize("n,gw", [((8, 8, 6), 3), ((9, 7, 5), 5), ((68, 61, 4), 2), ((1, 1, 2), 2), ((256, 130, 13), 3)])
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_statistics_tiles(n, gw, precision):
    """Level statistics over planes that do and do not divide into 16-byte
    accesses and shares, with and without a second factor and a mask, and the
    cloud statistics over partial column groups and depths that do not divide
    by the wavefronts, against numpy.  Sums of N terms in two orders differ by
    at most N eps times the sum of their magnitudes; extremes and counts are
    exact."""
    import torch
    from pycles_amd import _capi
    from pycles_amd import _device as D
    nx, ny, nz = n
    nzg, N = nz + 2 * gw, nx * ny
    code = D.precision_code(precision)
    np_t = np.float64 if precision == "f64" else np.float32
    rng = np.random.default_rng(11)
    a, b = (rng.standard_normal((nzg, ny, nx)).astype(np_t) for _ in range(2))
    mask = (rng.random((nzg, ny, nx)) < 0.3).astype(np_t)
    mask[0] = 0.0
    ba, bb = 5.0 + rng.random(nzg), -2.0 + rng.random(nzg)
    dims = _dims(n, gw)
    ws = torch.empty(_capi.horizontal_stats_workspace_bytes(dims), dtype=torch.uint8, device="cuda")
    ta, tb, tm, tba, tbb = (_dev(x) for x in (a, b, mask, ba, bb))
    eps = np.finfo(np.float64).eps
    for second in (False, True):
        for masked in (False, True):
            out = torch.empty((6, nzg), dtype=torch.float64, device="cuda")
            _capi.horizontal_stats(dims, ta.data_ptr(), tba.data_ptr(), tb.data_ptr() if second else None,
                                   tbb.data_ptr() if second else None, tm.data_ptr() if masked else None, code,
                                   out.data_ptr(), ws.data_ptr(), D.stream())
            got = out.cpu().numpy()
            v = a.astype(np.float64) + ba[:, None, None]
            if second:
                v = v * (b.astype(np.float64) + bb[:, None, None])
            m = mask.astype(np.float64) if masked else np.ones_like(v)
            cnt = m.sum(axis=(1, 2))
            div = np.maximum(cnt, 1.0) if masked else float(N)
            for q in range(3):
                want = (v ** (q + 1) * m).sum(axis=(1, 2)) / div
                mag = (np.abs(v) ** (q + 1) * m).sum(axis=(1, 2)) / div
                assert np.all(np.abs(got[q] - want) <= (N + 8) * eps * mag), (second, masked, q)
            w = np.where(m != 0.0, v, np.nan)
            for k in range(nzg):
                hi, lo = (-9e12, 9e12) if not m[k].any() else (np.nanmax(w[k]), np.nanmin(w[k]))
                assert got[3, k] == hi and got[4, k] == lo
            assert np.array_equal(got[5], cnt)
    ql = np.where(rng.random((nzg, ny, nx)) < 0.2, rng.random((nzg, ny, nx)), 0.0).astype(np_t)
    ql[gw] = 0.0
    rho = 1.2 - 0.01 * np.arange(nzg)
    tq, tr = _dev(ql), _dev(rho)
    ws = torch.empty(_capi.cloud_stats_workspace_bytes(dims), dtype=torch.uint8, device="cuda")
    out = torch.empty(nz + 4, dtype=torch.float64, device="cuda")
    _capi.cloud_stats(dims, tr.data_ptr(), tq.data_ptr(), code, out.data_ptr(), ws.data_ptr(), D.stream())
    got = out.cpu().numpy()
    q = ql[gw:gw + nz].astype(np.float64)
    assert np.array_equal(got[:nz], (q > 0).sum(axis=(1, 2)) * (1.0 / N))
    assert got[nz] == (q > 0).any(axis=0).sum() / float(N)
    k = np.flatnonzero((q > 0).any(axis=(1, 2)))
    assert got[nz + 1] == ((k[0] + 0.5) * 20.0 if k.size else 99999.9)
    assert got[nz + 2] == ((k[-1] + 0.5) * 20.0 if k.size else -99999.9)
    lwp = (rho[:nz, None, None] * q * 20.0).sum() / N
    assert abs(got[nz + 3] - lwp) <= (N * nz + 8) * eps * lwp


@pytest.mark.parametrize("n,gw", [((70, 9, 13), 3), ((6, 5, 5), 5), ((8, 8, 600), 3), ((64, 128, 5), 2), ((512, 260, 300), 3)])
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_dry_thermo_tiles(n, gw, precision):
    """The dry thermodynamics over partial column tiles, uneven and longest
    chunks (large planes, deep columns), added to and overwriting the w
    tendency, against its closed form in numpy.  FP64: exp, log and pow within
    an ulp or two of numpy's and five more roundings, 1e-14 relative; the
    buoyancy and N^2 are differences of nearly equal terms, 1e-14 of those
    terms.  FP32 stores round once more (6e-8)."""
    import torch
    from pycles_amd import _capi
    from pycles_amd import _device as D
    nx, ny, nz = n
    nzg = nz + 2 * gw
    code = D.precision_code(precision)
    np_t = np.float64 if precision == "f64" else np.float32
    rng = np.random.default_rng(3)
    p0 = 1e5 * np.exp(-0.5 * np.arange(nzg) / nzg)
    a0 = 287.1 * 300.0 * (p0 / 1e5) ** 0.28 / p0
    base = 6864.8 + 2.0 + 0.01 * np.arange(nzg)
    dev = rng.standard_normal((nzg, ny, nx)).astype(np.float32)
    s = (base[:, None, None] + dev.astype(np.float64)) if precision == "f64" else dev
    full = base[:, None, None] + dev.astype(np.float64)
    wt0 = rng.standard_normal((nzg, ny, nx)).astype(np_t)
    dp = {k: _dev(v) for k, v in (("p0", p0), ("a0", a0), ("base", base))}
    ref = _capi.Ref(*[dp["a0"].data_ptr()] * 4, dp["p0"].data_ptr(), dp["p0"].data_ptr())
    bs = _capi.ScalarBase(dp["base"].data_ptr(), None) if precision == "f32" else None
    p3, a3 = p0[:, None, None], a0[:, None, None]
    T = 298.15 * np.exp((full - 6864.8 + 287.1 * np.log(p3 / 1e5)) / 1004.0)
    al = 287.1 * T / p3
    b = 9.80665 * (al - a3) / a3
    b[-1] = 0.0
    th = T / (p3 / 1e5) ** (287.1 / 1004.0)
    n2 = np.zeros_like(T)
    thz = th.copy()
    thz[0] = 0.0
    n2[2:-1] = 9.80665 / th[2:-1] * 0.5 * (thz[3:] - thz[1:-2]) / 20.0
    dw = np.zeros_like(T)
    dw[:nzg - 2] = 0.5 * (b[:nzg - 2] + b[1:nzg - 1])
    r = 1e-14 if precision == "f64" else 1e-14 + 6e-8
    ts = _dev(s)
    for over in (0, 1):
        out = [torch.full((nzg, ny, nx), -5.0, dtype=D.torch_dtype(code), device="cuda") for _ in range(5)]
        wt = _dev(wt0)
        _capi.thermo_dry(_dims(n, gw), ref, ts.data_ptr(), wt.data_ptr(), *[o.data_ptr() for o in out], bs, code, D.stream(),
                         over)
        gT, gal, gb, gth, gn2 = (o.cpu().numpy().astype(np.float64) for o in out)
        assert np.all(np.abs(gT - T) <= r * T)
        assert np.all(np.abs(gal - al) <= r * al)
        k = nzg - 1
        assert np.all(np.abs(gb[:k] - b[:k]) <= 3e-14 * 9.80665 + (r - 1e-14) * np.abs(b[:k])) and np.all(gb[k] == -5.0)
        assert np.all(np.abs(gth[1:] - th[1:]) <= r * th[1:]) and np.all(gth[0] == -5.0)
        assert np.all(np.abs(gn2[2:-1] - n2[2:-1]) <= 3e-14 * 9.80665 / 20.0 + (r - 1e-14) * np.abs(n2[2:-1]))
        want = dw + (0.0 if over else wt0.astype(np.float64))
        want[nzg - 2:] = wt0[nzg - 2:]
        assert np.all(np.abs(wt.cpu().numpy().astype(np.float64) - want) <= 6e-14 * 9.80665 + (r - 1e-14) * np.abs(want))


@pytest.mark.parametrize("n,gw,shift", [((8, 8, 5), 5, 0), ((16, 8, 9), 3, 1), ((8, 64, 2), 2, 0), ((64, 64, 64), 3, 0),
                                        ((32, 16, 104), 3, 1), ((16, 8, 315), 3, 0), ((16, 8, 316), 3, 0),
                                        ((256, 128, 12), 3, 0), ((512, 256, 3), 3, 1), ((64, 128, 40), 3, 0), ((64, 128, 41), 3, 0),
                                        ((256, 64, 75), 3, 0), ((256, 64, 160), 3, 0), ((8, 1024, 5), 3, 0)])
def test_projection_forms(n, gw, shift):
    """The projection in the forms its size rules choose (kx planes in one
    kernel, with and without staged pivots; few columns with stored pivots in
    LDS, up to 315 FP64 levels; the general solve; blocks of less than half a
    wavefront; few and many sequences per block) and off a 16-byte boundary (shift), FP64 against the
    oracle: 1e-12 of each field's maximum, as test_pressure_parity.  The CFL
    maximum is exact for the velocities that come back."""
    import torch
    from oracle import oracle as O
    from pycles_amd import _capi
    from pycles_amd import _device as D
    nx, ny, nz = n
    nzg, N = nz + 2 * gw, nx * ny * (nz + 2 * gw)
    dx = (50.0, 60.0, 20.0)
    rng = np.random.default_rng(nx + nz)
    alpha = 0.8 + 0.5 * np.arange(nzg) / nzg
    half = alpha - 0.004
    prof = {"rho0": 1.0 / alpha, "rho0_half": 1.0 / half, "alpha0": alpha, "alpha0_half": half,
            "p0": 1e5 - np.arange(nzg), "p0_half": 1e5 - np.arange(nzg)}
    oref = O.Ref(prof["p0"], prof["p0_half"], alpha, half, prof["rho0"], prof["rho0_half"])
    dp = {k: _dev(v) for k, v in prof.items()}
    ref = _capi.Ref(*[dp[k].data_ptr() for k in ("rho0", "rho0_half", "alpha0", "alpha0_half", "p0", "p0_half")])
    f = {k: rng.standard_normal((nzg, ny, nx)) for k in "uvw"}
    for a, sgn in ((f["u"], 1), (f["v"], 1), (f["w"], -1)):
        if sgn > 0:
            a[:gw], a[nzg - gw:] = a[gw:2 * gw][::-1], a[nzg - 2 * gw:nzg - gw][::-1]
        else:
            a[gw - 1] = a[nzg - gw] = a[nzg - gw - 1] = 0.0
    sim = O.OracleSimulation(O.make_dims(nx, ny, nz, gw, *dx), oref, False, None)
    for k in "uvw":
        sim.pv(k)[...] = np.pad(f[k].transpose(2, 1, 0), ((gw, gw), (gw, gw), (0, 0)), mode="wrap")
    sim.pressure_update()
    buf = torch.zeros(3 * N + 4, dtype=torch.float64, device="cuda")
    for q, k in enumerate("uvw"):
        buf[shift + q * N:shift + (q + 1) * N] = _dev(f[k]).reshape(-1)
    ptr = [buf.data_ptr() + 8 * (shift + q * N) for q in range(3)]
    p, div = (torch.zeros((nzg, ny, nx), dtype=torch.float64, device="cuda") for _ in range(2))
    cfl = torch.full((1,), 1e30, dtype=torch.float64, device="cuda")
    dims = _dims(n, gw, dx)
    plan = _capi.PressurePlan(dims, prof["rho0"].ctypes.data, prof["rho0_half"].ctypes.data, D.F64)
    plan.update(ref, *ptr, p.data_ptr(), div.data_ptr(), 0.75, cfl.data_ptr(), D.stream())
    got = buf[shift:shift + 3 * N].cpu().numpy().reshape(3, nzg, ny, nx)

    def err(a, name, dv=False):
        b = np.asarray((sim.dv[name] if dv else sim.pv(name)))[gw:-gw, gw:-gw].transpose(2, 1, 0)
        return np.abs(a - b).max() / np.abs(b).max()

    for q, k in enumerate("uvw"):
        assert err(got[q], k) <= 1e-12, k
    assert err(p.cpu().numpy(), "dynamic_pressure", True) <= 1e-12
    sl = slice(gw, gw + nz)
    odiv = np.asarray(sim.dv["divergence"])[gw:-gw, gw:-gw, gw:-gw].transpose(2, 1, 0)
    assert np.abs(div.cpu().numpy()[sl] - odiv).max() <= 1e-12 * np.abs(odiv).max()
    c = 0.75 * ((np.abs(got[0, sl]) * (1.0 / dx[0]) + np.abs(got[1, sl]) * (1.0 / dx[1])) + np.abs(got[2, sl]) * (1.0 / dx[2]))
    assert float(cfl[0]) == c.max() + 1e-11


@pytest.mark.parametrize("n", [(3, 5, 4), (64, 64, 6), (45, 47, 5), (160, 130, 2)])
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_level_means_tiles(n, precision):
    """Level means of several fields in one call: bitwise the one-field calls',
    and numpy's to N eps of the mean magnitude; planes below, at and beyond
    whole batches of a block's loads."""
    import torch
    from pycles_amd import _capi
    from pycles_amd import _device as D
    code = D.precision_code(precision)
    nzg, N = n[2] + 4, n[0] * n[1]
    rng = np.random.default_rng(2)
    f = rng.standard_normal((3, nzg, n[1], n[0])).astype(np.float64 if precision == "f64" else np.float32)
    t = _dev(f)
    many, one = (torch.full((3, nzg), 9.0, dtype=torch.float64, device="cuda") for _ in range(2))
    _capi.level_means(_dims(n, 2), [t[q].data_ptr() for q in range(3)], many.data_ptr(), code, D.stream())
    for q in range(3):
        _capi.level_mean(_dims(n, 2), t[q].data_ptr(), one[q].data_ptr(), code, D.stream())
    assert torch.equal(many, one)
    d = f.astype(np.float64)
    assert np.all(np.abs(many.cpu().numpy() - d.mean(axis=(2, 3))) <= (N + 8) * np.finfo(np.float64).eps * np.abs(d).mean(axis=(2, 3)))


@pytest.mark.parametrize("n,orders", [((12, 12, 6), (5, 5)), ((20, 11, 7), (9, 5)), ((24, 10, 6), (9, 9)), ((68, 13, 6), (7, 7)),
                                      ((64, 37, 5), (5, 5)), ((1024, 10, 5), (5, 5)), ((1032, 10, 5), (9, 9)),
                                      ((2048, 10, 5), (9, 9)),
                                      ((22, 10, 5), (9, 9)), ((21, 10, 5), (5, 5))])
@pytest.mark.parametrize("moist,shift", [(True, 0), (False, 0), (True, 1)])
def test_advection_x_forms_bitwise(n, orders, moist, shift):
    """FP64 tendencies, bitwise against the oracle, over the x pass's forms:
    rows of whole vectors (one block of several rows, rows that do and do not
    divide ny, one row per block, rows beyond its limit), odd rows and fields
    off a 16-byte boundary (shift); tendencies zero on entry and accumulated."""
    import torch
    from oracle import oracle as O
    from pycles_amd import _capi
    from pycles_amd import _device as D
    nx, ny, nz = n
    gw = (max(orders) + 1) // 2
    nzg, N = nz + 2 * gw, nx * ny * (nz + 2 * gw)
    dx = (50.0, 60.0, 20.0)
    rng = np.random.default_rng(nx * ny)
    alpha = 0.8 + 0.3 * np.arange(nzg) / nzg
    half = alpha - 0.004
    prof = {"rho0": 1.0 / alpha, "rho0_half": 1.0 / half, "alpha0": alpha, "alpha0_half": half, "p0": alpha, "p0_half": alpha}
    oref = O.Ref(prof["p0"], prof["p0_half"], alpha, half, prof["rho0"], prof["rho0_half"])
    dp = {k: _dev(v) for k, v in prof.items()}
    ref = _capi.Ref(*[dp[k].data_ptr() for k in ("rho0", "rho0_half", "alpha0", "alpha0_half", "p0", "p0_half")])
    names = ["u", "v", "w", "s"] + (["qt"] if moist else [])
    f = {k: rng.standard_normal((nzg, ny, nx)) for k in names}
    t0 = {k: rng.standard_normal((nzg, ny, nx)) for k in names}
    lt = O.Lookup(np.linspace(100.0, 380.0, 16), np.linspace(1.0, 2.0, 16)) if moist else None
    buf = torch.zeros(2 * len(names) * N + 4, dtype=torch.float64, device="cuda")

    def slot(q):
        return buf[shift + q * N:shift + (q + 1) * N]

    for zero in (0, 1):
        sim = O.OracleSimulation(O.make_dims(nx, ny, nz, gw, *dx), oref, moist, lt, scalar_order=orders[0],
                                 momentum_order=orders[1])
        for q, k in enumerate(names):
            start = t0[k] if k == "w" or not zero else np.zeros_like(t0[k])
            sim.pv(k)[...] = np.pad(f[k].transpose(2, 1, 0), ((gw, gw), (gw, gw), (0, 0)), mode="wrap")
            sim.pt(k)[...] = np.pad(start.transpose(2, 1, 0), ((gw, gw), (gw, gw), (0, 0)), mode="wrap")
            slot(q).copy_(_dev(f[k]).reshape(-1))
            slot(len(names) + q).copy_(_dev(t0[k]).reshape(-1))  # stale where zero: to be replaced
        sim.scalar_advection_update()
        sim.momentum_advection_update()
        ptr = [slot(q).data_ptr() for q in range(2 * len(names))]
        v, t = ptr[:len(names)], ptr[len(names):]
        if nx == 2048:
            # rows whose staged form exceeds the LDS are refused whatever the form
            with pytest.raises(_capi.PyclesError, match="does not fit in LDS"):
                _capi.advection(_dims(n, gw, dx), ref, v[:3], t[:3], v[3:], t[3:], None, *orders, D.F64, D.stream(), 0)
            return
        _capi.advection(_dims(n, gw, dx), ref, v[:3], t[:3], v[3:], t[3:], None, *orders, D.F64, D.stream(),
                        _capi.ADV_TEND_ZERO if zero else 0)
        for q, k in enumerate(names):
            got = slot(len(names) + q).cpu().numpy().reshape(nzg, ny, nx)[gw:-gw]
            want = np.asarray(sim.pt(k))[gw:-gw, gw:-gw, gw:-gw].transpose(2, 1, 0)
            assert np.array_equal(got, want), (k, zero, np.abs(got - want).max())


@pytest.mark.parametrize("n,orders", [((70, 9, 13), (5, 5)), ((64, 12, 70), (5, 5)), ((33, 11, 9), (7, 7)), ((65, 10, 150), (9, 5)),
                                      ((24, 13, 21), (9, 9))])
@pytest.mark.parametrize("moist", [True, False])
def test_fp32_advection_forms(n, orders, moist):
    """FP32 tendencies against the FP64 oracle on the same values, at every
    order, over partial tiles and several z chunks, with level profiles that
    change by more than the deviations from one level to the next (moist) and
    without profiles (dry).  Bound: with D the largest offset in a window, a
    face's reconstruction is within 400 eps D (weights and candidates: about
    30 operations each on terms of up to 6 D, and the rounded profile
    differences), twice per direction; the parts of a tendency round to eps
    of their size at each of the passes' additions."""
    import torch
    from oracle import oracle as O
    from pycles_amd import _capi
    from pycles_amd import _device as D
    nx, ny, nz = n
    gw = (max(orders) + 1) // 2
    nzg = nz + 2 * gw
    dx = (50.0, 60.0, 20.0)
    rng = np.random.default_rng(nx + ny + nz)
    alpha = 0.8 + 0.3 * np.arange(nzg) / nzg
    half = alpha - 0.004
    prof = {"rho0": 1.0 / alpha, "rho0_half": 1.0 / half, "alpha0": alpha, "alpha0_half": half, "p0": alpha, "p0_half": alpha}
    oref = O.Ref(prof["p0"], prof["p0_half"], alpha, half, prof["rho0"], prof["rho0_half"])
    dp = {k: _dev(v) for k, v in prof.items()}
    ref = _capi.Ref(*[dp[k].data_ptr() for k in ("rho0", "rho0_half", "alpha0", "alpha0_half", "p0", "p0_half")])
    names = ["u", "v", "w", "s"] + (["qt"] if moist else [])
    f = {k: rng.standard_normal((nzg, ny, nx)).astype(np.float32) for k in names}
    base = {k: np.cumsum(rng.uniform(-3.0, 5.0, nzg)) for k in names[3:]} if moist else {}
    lt = O.Lookup(np.linspace(100.0, 380.0, 16), np.linspace(1.0, 2.0, 16)) if moist else None
    sim = O.OracleSimulation(O.make_dims(nx, ny, nz, gw, *dx), oref, moist, lt, scalar_order=orders[0],
                             momentum_order=orders[1])
    dev, tend = {}, {}
    for k in names:
        full = f[k].astype(np.float64) + (base[k][:, None, None] if k in base else 0.0)
        sim.pv(k)[...] = np.pad(full.transpose(2, 1, 0), ((gw, gw), (gw, gw), (0, 0)), mode="wrap")
        sim.pt(k)[...] = 0.0
        dev[k], tend[k] = _dev(f[k]), torch.zeros((nzg, ny, nx), dtype=torch.float32, device="cuda")
    sim.scalar_advection_update()
    sim.momentum_advection_update()
    bd = {k: _dev(v) for k, v in base.items()}
    sb = _capi.ScalarBase(*[bd[k].data_ptr() for k in names[3:]]) if moist else None
    _capi.advection(_dims(n, gw, dx), ref, [dev[k].data_ptr() for k in names[:3]], [tend[k].data_ptr() for k in names[:3]],
                    [dev[k].data_ptr() for k in names[3:]], [tend[k].data_ptr() for k in names[3:]], sb, *orders, D.F32,
                    D.stream(), 0)
    eps = np.finfo(np.float32).eps
    umax = 1.5 * max(np.abs(f[k]).max() for k in names[:3])  # a centred value is at most (4/3) max
    for k in names:
        amp = np.abs(f[k]).max()
        b = base.get(k, np.zeros(nzg))
        jump = max(np.abs(b[m:] - b[:-m]).max() for m in range(1, 6))
        scale = 2.0 * umax * 1.4 * sum(1.0 / d for d in dx)  # two faces of each direction, alpha rho
        tol = scale * (400 * eps * (2 * amp + jump) + 8 * eps * (amp + np.abs(b).max()))
        got = tend[k].cpu().numpy()[gw:-gw].astype(np.float64)
        want = np.asarray(sim.pt(k))[gw:-gw, gw:-gw, gw:-gw].transpose(2, 1, 0)
        err = np.abs(got - want).max()
        print(k, "error / bound", err / tol, flush=True)
        assert err <= tol, (k, err, tol)


@pytest.mark.parametrize("n", [(8, 8, 5), (16, 64, 7), (64, 32, 9), (512, 64, 6), (2048, 16, 3), (256, 128, 70)])
def test_fp32_projection_alignment(n):
    """The FP32 projection by 16-byte accesses and, with the fields off a
    16-byte boundary, by single ones: the same operations on the same values,
    so the same bits."""
    import torch
    from pycles_amd import _capi
    from pycles_amd import _device as D
    nx, ny, nz = n
    gw = 3
    nzg, N = nz + 2 * gw, nx * ny * (nz + 2 * gw)
    alpha = 0.8 + 0.5 * np.arange(nzg) / nzg
    prof = {"rho0": 1.0 / alpha, "rho0_half": 1.0 / (alpha - 0.004), "alpha0": alpha, "alpha0_half": alpha - 0.004, "p0": alpha,
            "p0_half": alpha}
    dp = {k: _dev(v) for k, v in prof.items()}
    ref = _capi.Ref(*[dp[k].data_ptr() for k in ("rho0", "rho0_half", "alpha0", "alpha0_half", "p0", "p0_half")])
    f = _dev(np.random.default_rng(nx).standard_normal(3 * N).astype(np.float32))
    plan = _capi.PressurePlan(_dims(n, gw, (50.0, 60.0, 20.0)), prof["rho0"].ctypes.data, prof["rho0_half"].ctypes.data, D.F32)
    out = []
    for shift in (0, 1):
        buf = torch.zeros(5 * N + 4, dtype=torch.float32, device="cuda")
        buf[shift:shift + 3 * N] = f
        ptr = [buf.data_ptr() + 4 * (shift + q * N) for q in range(5)]
        plan.update(ref, *ptr, 0.75, None, D.stream())
        out.append(buf[shift:shift + 5 * N].cpu().numpy())
    assert np.isfinite(out[0]).all() and np.abs(out[0][3 * N:]).max() > 0
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("n", [(17, 13, 9), (70, 9, 13), (24, 31, 40), (10, 25, 20)])
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_saturation_adjustment_columns(n, precision):
    """Columns do not depend on the plane that holds them: the columns of a plane
    that does not fill the kernels' blocks of 256, below and above one block,
    give the bits that they give within a plane of whole blocks."""
    import torch
    from pycles_amd.Simulation3d import Simulation3d
    from tests.helpers import host_case
    from tests.test_gpu_parity import _saturating
    nx, ny, nz = n
    N = (128, 32)
    state, out = None, []
    for px, py in (N, (nx, ny)):
        nl, Gr, RS, Th, fields = host_case(px, py, nz, seed=4)
        nl["mi355x"]["precision"] = precision
        fields = _saturating(Gr, fields)
        sim = Simulation3d().initialize(nl, Gr=Gr, Ref=RS, Th=Th, fields=fields)
        if state is None:
            state = {k: (sim.PV.field(k).clone(), sim.PV.base.get(k)) for k in sim.PV.index_name}
        else:
            for k, (f, base) in state.items():
                sim.PV.field(k).copy_(f[:, :ny, :nx])
                if base is not None:
                    sim.PV.base[k] = base
        sim.Th.update(sim.Gr, sim.Ref, sim.PV, sim.DV, wt_overwrite=True)
        out.append({k: sim.DV.field(k).clone() for k in ("temperature", "qv", "ql", "alpha", "buoyancy", "buoyancy_frequency")}
                   | {"w": sim.PV.tend("w").clone(), "qt": sim.PV.field("qt").clone()})
    torch.cuda.synchronize()
    assert float((out[1]["ql"] > 0).double().mean()) > 0.05
    for k, a in out[1].items():
        assert torch.equal(a, out[0][k][:, :ny, :nx].contiguous()), k
