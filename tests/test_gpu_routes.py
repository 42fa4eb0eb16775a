"""Each kernel that the size rules choose between, held to the oracle or to the
kernels it replaces on sizes that reach it."""
import numpy as np
import pytest

from tests.helpers import host_case, oracle_sim

pytestmark = pytest.mark.gpu


def _sim(n, precision="f64", seed=21):
    """A simulation of n cells with a divergence-free swirl and its fields."""
    import json

    from tests.test_gpu_parity import _gpu_sim, _swirl
    nl, Gr, RS, Th, fields = host_case(*n, seed=seed)
    nl = json.loads(json.dumps(nl))
    nl["mi355x"]["precision"] = precision
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
