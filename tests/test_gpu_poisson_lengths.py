"""The Poisson solve and its adjoint on x and y axes of compile-time length:
every chain of stages, powers of two and 3 2^k, forward and adjoint, against a
float64 solve and by the inner product."""
import numpy as np
import pytest
import torch

from oracle import pm as opm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('shape', [(96, 192, 48), (192, 96, 64), (384, 6, 64), (768, 384, 18),
                                   (6, 768, 32), (64, 128, 40), (256, 64, 16), (128, 512, 6),
                                   (512, 256, 4), (6, 1024, 34), (1024, 8, 66)])
def test_solve_and_adjoint(dev, shape):
    from pmwd_amd import _lib
    rng = np.random.default_rng(6)
    dens = (1 + 0.3 * rng.standard_normal(shape)).astype(np.float32)
    cot = rng.standard_normal((3,) + shape).astype(np.float32)
    coef = float(np.float32(1.5) * np.float32(0.3))
    c = _lib.context(shape, 1.5, dev)
    to = lambda a: torch.as_tensor(a, device=dev)
    grad, back = to(np.empty_like(cot)), to(np.empty_like(dens))
    d, g = to(dens), to(cot)
    _lib.check(_lib.lib().pmx_poisson_grad(c.bind(), _lib.ptr(d), coef, _lib.ptr(grad)))
    _lib.check(_lib.lib().pmx_poisson_grad_adj(c.bind(), _lib.ptr(g), coef, _lib.ptr(back)))
    want = opm.gravity_mesh(dens, 0.3, 1.5, shape, dtype=np.float64)
    # six float32 transforms in a row, each a few 1e-7, as of the other lengths
    for a in range(3):
        err = np.linalg.norm(grad[a].cpu().numpy() - np.asarray(want[a], np.float64))
        assert err < 5e-6 * np.linalg.norm(want[a])
    # <cot, G (dens - 1)> = <G^T cot, dens - 1>; each side a sum over the mesh
    # of terms rounded at 1e-6
    lhs = float((g.double() * grad.double()).sum())
    rhs = float((back.double() * (d.double() - 1)).sum())
    assert abs(lhs - rhs) < 5e-6 * float((g.double() * grad.double()).abs().sum())
    # the adjoint alone, against float64 solves of other fields
    for k in range(3):
        f = 1 + rng.standard_normal(shape)
        w = opm.gravity_mesh(f.astype(np.float32), 0.3, 1.5, shape, dtype=np.float64)
        lhs = sum(float((cot[a].astype(np.float64) * np.asarray(w[a], np.float64)).sum()) for a in range(3))
        rhs = float((back.cpu().numpy().astype(np.float64) * (f.astype(np.float32).astype(np.float64) - 1)).sum())
        scale = sum(float(np.abs(cot[a].astype(np.float64) * np.asarray(w[a], np.float64)).sum()) for a in range(3))
        assert abs(lhs - rhs) < 5e-6 * scale
