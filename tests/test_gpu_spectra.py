"""The transforms' dense sides (caller meshes read and written by the first
and last pass) and the power spectrum's runs of modes: every run length, auto
and cross spectra."""
import numpy as np
import pytest
import torch

from oracle import spec as ospec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('shape', [(16, 32, 64), (12, 18, 30), (9, 10, 15), (64, 128, 256), (6, 5, 2)])
def test_dense_sides_at_any_alignment(dev, shape):
    """A mesh 4 bytes off the passes' float2 alignment goes through the padded
    layout: the same bits as an aligned one."""
    from pmwd_amd import _lib
    n = int(np.prod(shape))
    h = _lib.context_any_cell(shape, torch.device('cuda', torch.cuda.current_device())).bind()
    nc = 2 * shape[0] * shape[1] * (shape[2] // 2 + 1)
    x = torch.randn(n, device=dev, generator=torch.Generator(dev).manual_seed(3))
    got = []
    for off in (0, 1):
        a = torch.empty(n + 2, device=dev)[off:off + n].copy_(x)
        spec = torch.empty(nc + 2, device=dev)[off:off + nc]
        back = torch.empty(n + 2, device=dev)[off:off + n]
        _lib.check(_lib.lib().pmx_rfftn(h, _lib.ptr(a), _lib.ptr(spec)))
        _lib.check(_lib.lib().pmx_irfftn(h, _lib.ptr(spec), _lib.ptr(back)))
        assert torch.equal(a, x)
        got.append((spec.clone(), back.clone()))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    # float32 rounding of the two transforms, as the tests of each length
    assert float((got[0][1] - x).norm() / x.norm()) < 2e-6


# runs of 1, 2, 4 and 8 groups, the last one of an axis shorter; flat meshes
@pytest.mark.parametrize('shape', [(130, 126, 66), (192, 200, 180), (16, 512, 1022), (256, 250, 255),
                                   (1, 64, 64), (31, 1, 30)])
@pytest.mark.parametrize('kw', [dict(), dict(bins=1.0), dict(deconv=2), dict(cross=True)])
def test_runs_match_oracle(dev, shape, kw):
    import pmwd_amd as pa
    kw = dict(kw)
    rng = np.random.default_rng(sum(shape))
    f = rng.standard_normal(shape).astype(np.float32)
    g = rng.standard_normal(shape).astype(np.float32) if kw.pop('cross', False) else None
    out = pa.powspec(torch.as_tensor(f, device=dev), 1.7,
                     g=torch.as_tensor(g, device=dev) if g is not None else None, **kw)
    with np.errstate(invalid='ignore'):
        want = ospec.powspec(f, 1.7, g=g, **kw)
    k, P, N, bins = (t.cpu().numpy() for t in out)
    np.testing.assert_array_equal(N, want[2])
    np.testing.assert_allclose(k, want[0], rtol=1e-12)
    # each mode's float32 |F|^2 (and the deconvolution's powers) is a few
    # roundings off; the tolerances of the smaller meshes
    scale = np.nanmax(np.abs(want[1]))
    tol = 1e-5 if kw.get('deconv') else 2e-6
    np.testing.assert_allclose(P, want[1], rtol=tol, atol=tol * scale)
