"""Tile layouts of meshes with more tiles than one workgroup scans (8192), and
with exactly as many: states that alternate, so that the capacity layout
fails, then counts first, then holds again; and forward and reverse runs whose
tiles outgrow their capacities, which redoes the move exactly.  Thin meshes
have the tiles without the cells."""
import numpy as np
import pytest
import torch

from oracle import pm as opm
from test_gpu_pipeline import assert_same, run, run_adj

pytestmark = pytest.mark.gpu

FLAT = [((1, 1024, 2048), 8192), ((1, 544, 3856), 8194), ((1, 2048, 2048), 16384)]
# extents that the tile-ordered copies of the pipelines can pack
THIN = [((32, 1024, 1024), 8192), ((33, 1024, 1024), 12288)]


def _tiles(mesh):
    return int(np.prod([-(-s // 16) for s in mesh]))


@pytest.mark.parametrize('mesh,tiles', FLAT)
def test_alternating_states(dev, mesh, tiles):
    import pmwd_amd as pa
    from pmwd_amd import _lib
    assert _tiles(mesh) == tiles
    conf = pa.Configuration(1.7, mesh, mesh_shape=1)
    rng = np.random.default_rng(1)
    n = 300000
    pmid = [rng.integers(0, mesh, (n, 3)).astype(np.int16) for _ in range(2)]
    pmid.append((pmid[1] % 200).astype(np.int16))   # every particle in 2% of the tiles
    disp = (2 * conf.cell_size * rng.standard_normal((n, 3))).astype(np.float32)
    t = lambda a: torch.as_tensor(a, device=dev)
    states = [pa.Particles(conf, t(p), t(disp)) for p in pmid]
    want = []
    for s, p in zip(states, pmid):
        with _lib.context_scope(lambda key, make: make()):
            want.append(pa.scatter(s, conf, val=1.0))
        ref = opm.scatter(p, disp, conf.cell_size, mesh, mesh=np.zeros(mesh), val=1.0, dtype=np.float64)
        assert np.linalg.norm(want[-1].cpu().numpy() - ref) < 1e-6 * np.linalg.norm(ref)
    perm = torch.randperm(n, generator=torch.Generator().manual_seed(3)).to(dev)
    for i in (0, 0, 2, 1, 2, 2, 2, 0, 1, 0):
        assert torch.equal(pa.scatter(states[i], conf, val=1.0), want[i])
        assert torch.equal(pa.scatter(states[i][perm], conf, val=1.0), want[i])


def _collapse(mesh, n, steps, d, rate):
    """Particles streaming to the box centre, and whether some tile outgrows
    the capacity sized from the step before (its count + an eighth + 32)."""
    rng = np.random.default_rng(4)
    centre = 0.5 * np.array(mesh)
    q = centre + (rng.random((n, 3)) - 0.5) * np.minimum(np.array(mesh), 400)
    pmid = np.floor(q).astype(np.int16) % np.array(mesh, np.int16)
    disp = (q - np.floor(q)).astype(np.float32)
    vel = (rate * (centre - q)).astype(np.float32)
    grew, last = 0, None
    x = pmid + disp.astype(np.float64)
    for _ in range(steps):
        x = x + d * vel
        cell = np.floor(x).astype(np.int64) % np.array(mesh)
        key = np.ravel_multi_index((cell // 16).T, [-(-s // 16) for s in mesh])
        count = np.bincount(key, minlength=_tiles(mesh))
        if last is not None:
            grew += int(np.any(count > last + (last >> 3) + 32))
        last = count
    return pmid, disp, vel, grew


@pytest.mark.parametrize('mesh,tiles', THIN)
def test_forward_collapse(dev, mesh, tiles):
    import pmwd_amd as pa
    assert _tiles(mesh) == tiles
    conf = pa.Configuration(1.0, mesh, mesh_shape=1)
    pmid, disp, vel, grew = _collapse(mesh, 100000, 5, 0.5, 0.3)
    assert grew >= 2
    k, d = np.zeros(5, np.float32), np.full(5, 0.5, np.float32)
    assert_same(run(conf, dev, pmid, disp, vel, k, d, k, True),
                run(conf, dev, pmid, disp, vel, k, d, k, False))


@pytest.mark.parametrize('mesh,tiles', THIN)
def test_reverse_collapse(dev, mesh, tiles):
    import pmwd_amd as pa
    conf = pa.Configuration(1.0, mesh, mesh_shape=1)
    pmid, disp, vel, grew = _collapse(mesh, 100000, 5, 0.5, 0.3)
    assert grew >= 2
    rng = np.random.default_rng(24)
    arrs = [disp, vel] + [rng.standard_normal(disp.shape).astype(np.float32) for _ in range(2)]
    k, d = np.zeros(5, np.float32), np.full(5, 0.5, np.float32)
    got, gd = run_adj(conf, dev, pmid, arrs, 0.0, k, d, k, True)
    want, wd = run_adj(conf, dev, pmid, arrs, 0.0, k, d, k, False)
    assert_same(got, want)
    np.testing.assert_allclose(gd, wd, rtol=1e-12, atol=1e-300)
