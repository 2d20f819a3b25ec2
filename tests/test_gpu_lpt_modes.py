"""The modes belong to the caller: writing to them between lpt() and the
backward pass neither fails nor changes the gradient."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('kind', ['leaf', 'result', 'conj'])
@pytest.mark.parametrize('order', [1, 2])
def test_modes_written_before_the_backward(dev, order, kind):
    import pmwd_amd as pa
    shape = (16, 12, 20)
    conf = pa.Configuration(3.0, shape, mesh_shape=1, a_start=1 / 16, lpt_order=order)
    cosmo = pa.boltzmann(pa.SimpleLCDM(conf), conf)
    gen = torch.Generator(dev).manual_seed(1)
    modes = pa.linear_modes(torch.randn(shape, generator=gen, device=dev), cosmo, conf)
    cots = [torch.randn((conf.ptcl_num, 3), generator=gen, device=dev) for _ in range(2)]
    got = []
    for write in (False, True):
        leaf = modes.clone().requires_grad_(True)
        m = leaf if kind == 'leaf' else (leaf * 2 if kind == 'result' else (leaf * 2).conj())
        p, _ = pa.lpt(m, cosmo, conf)
        if write and kind == 'leaf':
            with torch.no_grad():
                m.mul_(3).add_(1)
        elif write:
            m.mul_(3).add_(1)
        got.append(torch.autograd.grad([p.disp, p.vel], [leaf], cots)[0])
    assert torch.equal(got[0], got[1])
