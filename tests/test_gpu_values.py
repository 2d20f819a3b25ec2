"""The default-geometry CIC of value channels (scatter, gather and their
adjoints) against the any-geometry kernels and the float64 oracle, at meshes
with full, clipped and single tiles."""
import numpy as np
import pytest
import torch

from oracle import pm as opm

pytestmark = pytest.mark.gpu

# full 16^3 tiles; tiles clipped on every axis; one tile per axis smaller than
# 16; a one-cell axis; more particles than a workgroup in one tile
CASES = [((16, 16, 32), 2), ((20, 12, 35), 1), ((5, 7, 9), 1), ((1, 17, 33), 1), ((24, 24, 24), 1.5)]


@pytest.fixture(autouse=True)
def in_tiles(monkeypatch):
    """Contexts that scatter values in tiles at any particle count."""
    from pmwd_amd import _lib
    monkeypatch.setenv('PMX_VALUES_MIN', '0')
    monkeypatch.setattr(_lib, '_ctx_cache', {})


def _setup(dev, shape, ratio, std=2.0, seed=0):
    import pmwd_amd as pa
    conf = pa.Configuration(1.7, shape, mesh_shape=ratio)
    pmid, disp = opm.gen_grid(shape, conf.mesh_shape, conf.cell_size)
    rng = np.random.default_rng(seed)
    disp = (disp + std * conf.cell_size * rng.standard_normal(disp.shape)).astype(np.float32)
    ptcl = pa.Particles(conf, torch.as_tensor(pmid, device=dev), torch.as_tensor(disp, device=dev))
    return conf, ptcl, pmid, disp, rng


def _pad(a):
    """Zero channels up to four, which the any-geometry kernels take."""
    return np.concatenate([a, np.zeros(a.shape[:-1] + (4 - a.shape[-1],), np.float32)], axis=-1)


@pytest.mark.parametrize('nc', [1, 2, 3])
@pytest.mark.parametrize('shape,ratio', CASES)
def test_readout_and_adjoints_equal_the_any_geometry_kernels(dev, shape, ratio, nc):
    import pmwd_amd as pa
    conf, ptcl, pmid, disp, rng = _setup(dev, shape, ratio)
    mesh = rng.standard_normal(conf.mesh_shape + (nc,)).astype(np.float32)
    val = rng.standard_normal((len(pmid), nc)).astype(np.float32)
    t = lambda a: torch.as_tensor(a, device=dev).requires_grad_(True)

    def run(m, v):
        d, m, v = t(disp), t(m), t(v)
        p = ptcl.replace(disp=d)
        out = pa.gather(p, conf, m, val=v)
        (gd,) = torch.autograd.grad(out, d, v.detach())
        sc = pa.scatter(p, conf, val=v)
        sd, sv = torch.autograd.grad(sc, (d, v), m.detach())
        return [x.detach().cpu().numpy() for x in (out, gd, sd, sv)]

    got, want = run(mesh, val), run(_pad(mesh), _pad(val))
    for a, b in ((0, False), (1, True), (2, True), (3, False)):
        np.testing.assert_array_equal(got[a], want[a] if b else want[a][:, :nc])


@pytest.mark.parametrize('nc', [1, 2, 3])
@pytest.mark.parametrize('shape,ratio', CASES)
def test_value_scatter_matches_float64(dev, shape, ratio, nc):
    """Onto a mesh of the caller's, with values over ten decades.  Tolerance:
    the weights carry the float32 rounding of disp / cell (std 2 cells), the
    1e-6 of the density scatter."""
    import pmwd_amd as pa
    conf, ptcl, pmid, disp, rng = _setup(dev, shape, ratio, seed=1)
    base = rng.standard_normal(conf.mesh_shape + (nc,)).astype(np.float32)
    val = (rng.standard_normal((len(pmid), nc)) * 10.0 ** rng.uniform(-8, 2, (len(pmid), 1)))
    val = val.astype(np.float32)
    got = pa.scatter(ptcl, conf, mesh=torch.as_tensor(base, device=dev),
                     val=torch.as_tensor(val, device=dev)).cpu().numpy()
    want = opm.scatter(pmid, disp, conf.cell_size, conf.mesh_shape, mesh=base.astype(np.float64),
                       val=val.astype(np.float64), dtype=np.float64)
    assert np.linalg.norm(got - want) < 1e-6 * np.linalg.norm(want)
    # the mesh cotangent of a readout is the same scatter, onto zeros
    m = torch.as_tensor(base, device=dev).requires_grad_(True)
    out = pa.gather(ptcl, conf, m, val=torch.zeros((len(pmid), nc), device=dev))
    (gm,) = torch.autograd.grad(out, m, torch.as_tensor(val, device=dev))
    want = want - base
    assert np.linalg.norm(gm.cpu().numpy() - want) < 1e-6 * np.linalg.norm(want)


def test_infinite_and_nan_values_reach_the_same_cells(dev):
    import pmwd_amd as pa
    conf, ptcl, pmid, disp, rng = _setup(dev, (20, 12, 35), 1, seed=2)
    val = rng.standard_normal((len(pmid), 1)).astype(np.float32)
    val[7], val[100], val[101], val[5000] = np.inf, np.nan, -np.inf, np.inf
    one = pa.scatter(ptcl, conf, val=torch.as_tensor(val, device=dev)).cpu().numpy()[..., 0]
    four = pa.scatter(ptcl, conf, val=torch.as_tensor(_pad(val), device=dev)).cpu().numpy()[..., 0]
    np.testing.assert_array_equal(np.isnan(one), np.isnan(four))
    np.testing.assert_array_equal(np.isposinf(one), np.isposinf(four))
    np.testing.assert_array_equal(np.isneginf(one), np.isneginf(four))
    fine = np.isfinite(one)
    np.testing.assert_allclose(one[fine], four[fine], rtol=1e-5, atol=1e-5)


def test_value_scatter_under_capture_without_scratch(dev):
    """A context that holds no particle scratch yet still scatters values
    under graph capture (nothing may be allocated there)."""
    import pmwd_amd as pa
    from pmwd_amd import _lib
    conf, ptcl, pmid, disp, rng = _setup(dev, (20, 12, 35), 1, seed=3)
    val = torch.as_tensor(rng.standard_normal((len(pmid), 2)).astype(np.float32), device=dev)
    want = pa.scatter(ptcl, conf, val=val)
    side = torch.cuda.Stream(device=dev)
    with torch.cuda.stream(side):
        fresh = _lib.Context(conf.mesh_shape, conf.cell_size, dev)
        with _lib.context_scope(lambda key, make: fresh):
            side.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                got = pa.scatter(ptcl, conf, val=val)
    for _ in range(3):
        got.fill_(float('nan'))
        graph.replay()
        again = pa.scatter(ptcl, conf, val=val)
        torch.cuda.synchronize()
        np.testing.assert_allclose(got.cpu().numpy(), want.cpu().numpy(), rtol=1e-5, atol=1e-5)
        np.testing.assert_allclose(again.cpu().numpy(), want.cpu().numpy(), rtol=1e-5, atol=1e-5)
    del graph
    fresh.close()


@pytest.mark.parametrize('n', [131071, 131072])
def test_value_scatter_either_side_of_the_tile_rule(dev, n, monkeypatch):
    """Few particles are scattered with atomics, more in tiles: the same
    numbers to the scatter's tolerance."""
    import pmwd_amd as pa
    monkeypatch.delenv('PMX_VALUES_MIN')
    conf, ptcl, pmid, disp, rng = _setup(dev, (64, 32, 65), 1, seed=3)
    val = rng.standard_normal((n, 3)).astype(np.float32)
    got = pa.scatter(ptcl[:n], conf, val=torch.as_tensor(val, device=dev)).cpu().numpy()
    want = opm.scatter(pmid[:n], disp[:n], conf.cell_size, conf.mesh_shape, val=val.astype(np.float64),
                       mesh=np.zeros(conf.mesh_shape + (3,)), dtype=np.float64)
    assert np.linalg.norm(got - want) < 1e-6 * np.linalg.norm(want)
