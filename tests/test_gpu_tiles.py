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
