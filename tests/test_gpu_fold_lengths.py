"""The deposit's fold in the row pass of 3 2^k axes, as of powers of two: same
bits as the separate fold pass, small and large row blocks, forward and
reverse (three meshes a launch)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('shape', [(32, 32, 192), (64, 16, 384), (16, 32, 768), (48, 16, 1536),
                                   (192, 192, 192), (32, 32, 128)])
def test_fold_in_the_row_pass(dev, shape, monkeypatch):
    from pmwd_amd import _lib
    import pmwd_amd as pa
    n = 20000
    gen = torch.Generator(dev).manual_seed(sum(shape))
    mesh = torch.tensor(shape, device=dev)
    pmid = (torch.rand((n, 3), generator=gen, device=dev) * mesh).to(torch.int16)
    disp = torch.randn((n, 3), generator=gen, device=dev)
    vel = torch.randn((n, 3), generator=gen, device=dev)
    conf = pa.Configuration(1.0, tuple(s // 2 for s in shape), mesh_shape=2, a_start=1 / 4,
                            a_nbody_maxstep=1 / 4)
    cosmo = pa.boltzmann(pa.SimpleLCDM(conf), conf)
    cot = torch.randn((n, 3), generator=gen, device=dev)
    got = []
    for on in ('1', '0'):
        monkeypatch.setenv('PMX_FOLD_ON_LOAD', on)
        monkeypatch.setattr(_lib, '_ctx_cache', {})
        d = disp.clone().requires_grad_(True)
        v = vel.clone().requires_grad_(True)
        p, _ = pa.nbody(pa.Particles(conf, pmid, d, vel=v), None, cosmo, conf)
        got.append([p.disp.detach(), p.vel.detach(), *torch.autograd.grad(p.disp, [d, v], cot)])
    for a, b in zip(*got):
        assert torch.equal(a, b)
