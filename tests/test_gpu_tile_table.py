"""The binning passes' per-workgroup tile table: particles in lattice order
fill it with few tiles, in random order with more than it holds, below and
above the count where the large workgroups start; states that alternate make
the capacity layout fail, then count first, then hold again.  The deposit sums
integers, so every order and every layout gives the same bits."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _state(conf, dev, seed, std):
    import pmwd_amd as pa
    g = torch.Generator(device=dev).manual_seed(seed)
    ptcl = pa.Particles.gen_grid(conf, device=dev)
    disp = ptcl.disp + std * conf.cell_size * torch.randn(ptcl.disp.shape, generator=g, device=dev)
    return ptcl.replace(disp=disp.contiguous(), vel=torch.zeros_like(disp))


@pytest.mark.parametrize('shape', [(40, 40, 40), (64, 128, 129)])
def test_orders_and_alternating_states_give_the_same_density(dev, shape):
    import pmwd_amd as pa
    from pmwd_amd import _lib
    conf = pa.Configuration(1.7, shape, mesh_shape=1)
    states = [_state(conf, dev, 1, 0.5), _state(conf, dev, 2, 8.0)]
    # the second all in one corner of the box: every tile but a few overflows
    lo = states[1].replace(pmid=states[1].pmid % 16)
    perm = torch.randperm(len(lo), generator=torch.Generator().manual_seed(3)).to(dev)
    want = []
    for s in states + [lo]:
        with _lib.context_scope(lambda key, make: make()):
            want.append(pa.scatter(s, conf))
    assert abs(float(want[0].double().sum()) / np.prod(shape) - 1) < 1e-6
    for i in (0, 0, 2, 1, 2, 2, 2, 0, 1, 0):
        s = (states + [lo])[i]
        assert torch.equal(pa.scatter(s, conf), want[i])
        assert torch.equal(pa.scatter(s[perm], conf), want[i])


@pytest.mark.parametrize('shape', [(16, 24, 40), (64, 128, 129)])
def test_steps_of_shuffled_particles(dev, shape):
    import pmwd_amd as pa
    conf = pa.Configuration(1.7, shape, mesh_shape=1, a_start=1 / 4, a_stop=1 / 2,
                            a_nbody_maxstep=1 / 8)
    cosmo = pa.growth_integ(pa.SimpleLCDM(conf), conf)
    s = _state(conf, dev, 4, 1.0)
    perm = torch.randperm(len(s), generator=torch.Generator().manual_seed(5)).to(dev)
    a, _ = pa.nbody(s, None, cosmo, conf)
    b, _ = pa.nbody(s[perm], None, cosmo, conf)
    for name in ('disp', 'vel', 'acc'):
        assert torch.equal(getattr(a, name)[perm], getattr(b, name)), name
    # reverse run: the same arrays in another order
    cot = a.replace(disp=torch.ones_like(a.disp), vel=a.vel.clone())
    p, pc, _ = pa.nbody_adj(a, cot, cosmo, conf)
    q, qc, _ = pa.nbody_adj(a[perm], cot[perm], cosmo, conf)
    for x, y in ((p.disp, q.disp), (p.vel, q.vel), (pc.disp, qc.disp), (pc.vel, qc.vel)):
        assert torch.equal(x[perm], y)
