"""Which value scatters go by tiles: enough particles, enough tiles, and enough
particles a tile; the others take float atomics.  Either way the numbers are
the float64 scatter's."""
import numpy as np
import pytest
import torch

from oracle import pm as opm

pytestmark = pytest.mark.gpu

MIN = 131072


@pytest.mark.parametrize('mesh,n,nc,tiled', [
    ((64, 64, 64), MIN, 1, True),        # 64 tiles
    ((64, 64, 64), MIN - 1, 1, False),
    ((64, 64, 64), 2 * MIN, 1, True),
    ((64, 64, 64), 2 * MIN - 1, 2, True),
    ((64, 64, 48), MIN, 1, False),       # 48 tiles: enough for several channels only
    ((64, 64, 48), MIN, 2, True),
    ((48, 48, 48), MIN, 3, True),        # 27 tiles
    ((32, 48, 64), MIN, 3, False),       # 24 tiles
    ((16, 16, 16), 2 * MIN, 3, False),   # one tile
    ((128, 256, 256), MIN, 3, True),     # 2048 tiles, 64 particles each
    ((128, 256, 272), MIN, 3, False),    # 2176 tiles
    ((128, 128, 352), 135168, 1, True),  # 1408 tiles, 96 particles each
    ((128, 128, 352), 135167, 1, False),
])
@pytest.mark.parametrize('kind', ['scatter', 'readout_grad'])
def test_tile_rule(dev, monkeypatch, kind, mesh, n, nc, tiled):
    import pmwd_amd as pa
    from pmwd_amd import _lib
    monkeypatch.delenv('PMX_VALUES_MIN', raising=False)
    monkeypatch.setattr(_lib, '_ctx_cache', {})
    conf = pa.Configuration(1.7, mesh, mesh_shape=1)
    rng = np.random.default_rng(n + nc)
    pmid = rng.integers(0, mesh, (n, 3)).astype(np.int16)
    disp = (2 * conf.cell_size * rng.standard_normal((n, 3))).astype(np.float32)
    val = rng.standard_normal((n, nc)).astype(np.float32)
    t = lambda a: torch.as_tensor(a, device=dev)
    ptcl = pa.Particles(conf, t(pmid), t(disp))
    ctx = _lib.context(conf.mesh_shape, conf.cell_size, dev)
    _lib.check(_lib.lib().pmx_timing_enable(ctx.h, 1))
    if kind == 'scatter':
        got = pa.scatter(ptcl, conf, val=t(val))
    else:
        m = torch.zeros(mesh + (nc,), device=dev, requires_grad=True)
        out = pa.gather(ptcl, conf, m, val=torch.zeros((n, nc), device=dev))
        (got,) = torch.autograd.grad(out, m, t(val))
        tiled = tiled and (nc > 2 or n >= 2 * MIN)   # else with the positions' in one launch
    assert (_lib.timing_read(ctx)['deposit'][1] > 0) == tiled
    _lib.check(_lib.lib().pmx_timing_enable(ctx.h, 0))
    want = opm.scatter(pmid, disp, conf.cell_size, conf.mesh_shape, val=val.astype(np.float64),
                       mesh=np.zeros(mesh + (nc,)), dtype=np.float64)
    # the weights carry the float32 rounding of disp / cell, as in the density's test
    assert np.linalg.norm(got.cpu().numpy() - want) < 1e-6 * np.linalg.norm(want)


def test_empty_tiles_add_nothing(dev, monkeypatch):
    """Tiles without particles leave a caller's mesh alone, bit for bit."""
    import pmwd_amd as pa
    from pmwd_amd import _lib
    monkeypatch.setenv('PMX_VALUES_MIN', '0')
    monkeypatch.setattr(_lib, '_ctx_cache', {})
    mesh = (64, 33, 40)
    conf = pa.Configuration(1.7, mesh, mesh_shape=1)
    gen = torch.Generator(device=dev).manual_seed(5)
    base = torch.randn(mesh + (3,), device=dev, generator=gen)
    base[40:, :, :] = -0.0
    n = 1000   # all in the cells [2, 12) of each axis: one tile
    pmid = torch.randint(2, 12, (n, 3), device=dev, generator=gen).to(torch.int16)
    disp = torch.rand((n, 3), device=dev, generator=gen) * conf.cell_size
    ptcl = pa.Particles(conf, pmid, disp)
    val = torch.randn((n, 3), device=dev, generator=gen)
    got = pa.scatter(ptcl, conf, mesh=base, val=val)
    rest = torch.ones(mesh, dtype=torch.bool, device=dev)
    rest[:16, :16, :16] = False
    assert torch.equal(got[rest].view(torch.int32), base[rest].view(torch.int32))
    np.testing.assert_allclose((got - base).double().sum((0, 1, 2)).cpu(), val.double().sum(0).cpu(),
                               rtol=1e-4, atol=1e-3)
