"""Gradients of lpt() and linear_modes() with respect to their modes: the
library's adjoints against autograd through the same steps as tensor ops, over
half-length rows of every kind, odd rows and both orders; and the grid that
the library writes."""
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu

# fixed and run-time lengths on each axis, small and large row blocks, odd
# rows, an axis of one
SHAPES = [(16, 16, 16), (64, 128, 256), (12, 10, 8), (9, 8, 10), (8, 9, 15), (20, 33, 66),
          (64, 64, 128), (1, 24, 6), (130, 128, 128), (96, 96, 192)]


def rel(a, b):
    return float(torch.linalg.vector_norm(a - b) / torch.linalg.vector_norm(b))


def setup(dev, shape, order):
    import pmwd_amd as pa
    ratio = 1.5 if all(s % 2 == 0 for s in shape) else 1   # displaced grids where they fit
    conf = pa.Configuration(3.0, shape, mesh_shape=ratio, a_start=1 / 16, lpt_order=order)
    return pa, conf, pa.boltzmann(pa.SimpleLCDM(conf), conf)


@pytest.mark.parametrize('shape', SHAPES)
@pytest.mark.parametrize('order', [1, 2])
def test_lpt_gradient(dev, shape, order, monkeypatch):
    pa, conf, cosmo = setup(dev, shape, order)
    gen = torch.Generator(dev).manual_seed(4)
    white = torch.randn(shape, generator=gen, device=dev)
    modes = pa.linear_modes(white, cosmo, conf)
    cots = [torch.randn((conf.ptcl_num, 3), generator=gen, device=dev) for _ in range(2)]
    out = []
    for fused in (True, False):
        if not fused:
            monkeypatch.setattr(sys.modules['pmwd_amd.lpt'], '_fused_graph', lambda *a: False)
        m = modes.clone().requires_grad_(True)
        p, _ = pa.lpt(m, cosmo, conf)
        out.append([p.pmid, p.disp.detach(), p.vel.detach(),
                    *torch.autograd.grad([p.disp, p.vel], [m], cots)])
    assert torch.equal(out[0][0], out[1][0])
    # up to five float32 transforms in a row, a few 1e-7 each
    for a, b in zip(out[0][1:], out[1][1:]):
        assert rel(a, b) < 5e-6
    # and the forward without a graph has the same bits
    with torch.no_grad():
        p, _ = pa.lpt(modes, cosmo, conf)
    assert torch.equal(p.disp, out[0][1]) and torch.equal(p.vel, out[0][2])


@pytest.mark.parametrize('shape', SHAPES)
@pytest.mark.parametrize('complex_', [False, True])
def test_linear_modes_gradient(dev, shape, complex_, monkeypatch):
    pa, conf, cosmo = setup(dev, shape, 2)
    gen = torch.Generator(dev).manual_seed(6)
    half = shape[:2] + (shape[2] // 2 + 1,)
    cx = lambda: torch.complex(*(torch.randn(half, generator=gen, device=dev) for _ in range(2)))
    white = cx() if complex_ else torch.randn(shape, generator=gen, device=dev)
    cot = cx()
    out = []
    for fused in (True, False):
        if not fused:
            monkeypatch.setattr(sys.modules['pmwd_amd.modes'], '_fused_graph', lambda *a: False)
        w = white.clone().requires_grad_(True)
        # a lazily conjugated cotangent, as autograd hands down
        m = pa.linear_modes(w, cosmo, conf, a=0.5)
        out.append([m.detach(), *torch.autograd.grad([m], [w], [cot.conj()])])
    for a, b in zip(*out):
        assert rel(a, b) < 2e-6


@pytest.mark.parametrize('shape,ratio', [((5, 6, 7), 1), ((16, 12, 20), 1.5), ((3, 1, 2), 2)])
def test_grid(dev, shape, ratio):
    """The grid on the device equals the one of tensor ops on the host."""
    import pmwd_amd as pa
    mesh = tuple(int(s * ratio) for s in shape)
    conf = pa.Configuration(2.0, shape, mesh_shape=mesh)
    a = pa.Particles.gen_grid(conf, vel=True, acc=True, device=dev)
    b = pa.Particles.gen_grid(conf, vel=True, acc=True, device='cpu')
    for x in ('pmid', 'disp', 'vel', 'acc'):
        assert torch.equal(getattr(a, x).cpu(), getattr(b, x)), x
        assert getattr(a, x).dtype == getattr(b, x).dtype
