"""Lagrangian perturbation theory initial conditions (pmwd/lpt.py:13-212).

2LPT on the particle grid with the HIP real FFTs: first-order potential,
the second-order source from six strain fields, then ``-ik`` gradients for
the displacements and canonical velocities.  The whole of it is one library
call, and so is its adjoint with respect to the modes; gradients with respect
to the cosmology run the k-space multiplies and real-space combinations as
device tensor ops around the FFT kernels.
"""
import ctypes

import numpy as np
import torch
from torch.autograd.function import once_differentiable

from .boltzmann import growth
from .cosmo_param import check_theta, host_value, lpt_growth_derivs
from .cosmology import E2
from .gravity import laplace, neg_grad, nyquist_mask
from .particles import Particles, _gen_grid_dev, _grid_axes, _grid_on_device, _grid_tables
from .pm_util import fftfreq, fftfwd, fftinv


def _strain(kvec, i, j, pot, conf):
    """Strain component (lpt.py:13-37); Nyquist zeroed only when i != j."""
    k_i, k_j = kvec[i], kvec[j]
    if i != j:
        k_i = torch.where(nyquist_mask(k_i, conf.ptcl_spacing), torch.zeros_like(k_i), k_i)
        k_j = torch.where(nyquist_mask(k_j, conf.ptcl_spacing), torch.zeros_like(k_j), k_j)
    s = (-k_i * k_j) * pot
    return fftinv(s, shape=conf.ptcl_grid_shape).to(conf.float_dtype)


def _L(kvec, pot, conf):
    """Second-order source (lpt.py:40-76) with pot_n = pot_m."""
    L = torch.zeros(conf.ptcl_grid_shape, dtype=conf.float_dtype, device=pot.device)
    dim = conf.dim
    diag = [_strain(kvec, i, i, pot, conf) for i in range(dim)]
    for i in range(dim):
        for j in range(dim - 1, i, -1):
            L = L + diag[i] * diag[j]
    for i in range(dim - 1):
        for j in range(i + 1, dim):
            s = _strain(kvec, i, j, pot, conf)
            L = L - s * s
    return L


def _growth_f32(a, cosmo, conf, order):
    """float32 D_n(a) and a^2 H(a) D_n'(a) (lpt.py:196-201)."""
    D = float(np.float32(growth(a, cosmo, conf, order=order)))
    dD = growth(a, cosmo, conf, order=order, deriv=1)
    return D, float(np.float32(a**2 * np.sqrt(E2(a, cosmo)) * dD))


def _needs_graph(modes, theta):
    if not torch.is_grad_enabled():
        return False
    if modes.requires_grad:
        return True
    return theta is not None and any(t.requires_grad for t in theta.values())


def _growth_table(cosmo, conf):
    fac = np.zeros(4, dtype=np.float32)
    for order in range(1, 1 + conf.lpt_order):
        fac[2 * order - 2:2 * order] = _growth_f32(conf.a_start, cosmo, conf, order)
    return fac


def _plain(t):
    """Contiguous values without lazy conjugation or negation."""
    return t.resolve_conj().resolve_neg().contiguous()


def _lpt_call(m, conf, fac, dtab):
    """disp and vel from complex64 modes in one library call."""
    from . import _lib
    c = _lib.context(conf.ptcl_grid_shape, conf.ptcl_spacing, m.device)
    disp = torch.empty((int(conf.ptcl_num), 3), dtype=torch.float32, device=m.device)
    vel = torch.empty_like(disp)
    _lib.check(_lib.lib().pmx_lpt_grid(c.bind(), _lib.ptr(m), float(conf.ptcl_cell_vol),
                                       int(conf.lpt_order), fac.ctypes.data_as(ctypes.c_void_p),
                                       _lib.ptr(dtab), _lib.ptr(disp), _lib.ptr(vel)))
    return disp, vel, c


class _LptFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, modes, conf, fac, dtab):
        m = _plain(modes.detach())
        disp, vel, ctx.pmx = _lpt_call(m, conf, fac, dtab)
        # the second order's strains come from the modes again; the caller may
        # write to its own between the passes
        if conf.lpt_order > 1:
            ctx.save_for_backward(m.clone() if m.data_ptr() == modes.data_ptr() else m)
        ctx.conf, ctx.fac = conf, fac
        return disp, vel

    @staticmethod
    @once_differentiable
    def backward(ctx, disp_cot, vel_cot):
        from . import _lib
        conf = ctx.conf
        m = ctx.saved_tensors[0] if conf.lpt_order > 1 else None
        gd, gv = _plain(disp_cot), _plain(vel_cot)
        n0, n1, n2 = conf.ptcl_grid_shape
        out = torch.empty((n0, n1, n2 // 2 + 1), dtype=torch.complex64, device=gd.device)
        # the forward's context: autograd may run this on another thread
        _lib.check(_lib.lib().pmx_lpt_vjp(
            ctx.pmx.bind(), _lib.ptr(m), float(conf.ptcl_cell_vol), int(conf.lpt_order),
            ctx.fac.ctypes.data_as(ctypes.c_void_p), _lib.ptr(gd), _lib.ptr(gv), _lib.ptr(out)))
        return out, None, None, None


def _lpt_fused(modes, cosmo, conf):
    """The whole of lpt() in the library: pmid from pmx_grid, the
    displacements and velocities from pmx_lpt_grid."""
    dev = modes.device
    if conf.lpt_order == 0 or not _grid_on_device(conf, dev):
        # gen_grid's arrays are fresh: the library adds to them in place
        ptcl = Particles.gen_grid(conf, vel=True, device=dev)
        if conf.lpt_order:
            from . import _lib
            fac = _growth_table(cosmo, conf)
            m = _plain(modes.detach().to(torch.complex64))
            c = _lib.context(conf.ptcl_grid_shape, conf.ptcl_spacing, dev)
            _lib.check(_lib.lib().pmx_lpt(c.bind(), _lib.ptr(m), float(conf.ptcl_cell_vol),
                                          int(conf.lpt_order), fac.ctypes.data_as(ctypes.c_void_p),
                                          _lib.ptr(ptcl.disp), _lib.ptr(ptcl.vel)))
        return ptcl, None
    tables = _grid_tables(_grid_axes(conf), dev)
    pmid, _ = _gen_grid_dev(conf, tables, False)
    fac = _growth_table(cosmo, conf)
    if _needs_graph(modes, None):
        disp, vel = _LptFn.apply(modes, conf, fac, tables[1])
    else:
        disp, vel, _ = _lpt_call(_plain(modes.detach().to(torch.complex64)), conf, fac, tables[1])
    return Particles(conf, pmid, disp, vel=vel), None


def _fused_graph(modes, theta, conf):
    """Whether gradients go through pmx_lpt_vjp: those of complex64 modes of
    the particle grid.  Growth factors with gradients keep the tensor path."""
    n0, n1, n2 = conf.ptcl_grid_shape
    return (conf.lpt_order > 0 and modes.dtype == torch.complex64
            and tuple(modes.shape) == (n0, n1, n2 // 2 + 1)
            and _grid_on_device(conf, modes.device)
            and (theta is None or not any(t.requires_grad for t in theta.values())))


def lpt(modes, cosmo, conf, theta=None):
    """LPT at ``conf.lpt_order`` (lpt.py:136-212); returns (ptcl, obsvbl).

    This is one library call (``pmx_lpt_grid``), and its gradient with respect
    to the modes another (``pmx_lpt_vjp``).  Other
    gradients run the same steps as device tensor ops around the library FFTs,
    which autograd differentiates.  ``theta`` ({'Omega_m': t}) makes the growth
    factors differentiable with respect to Omega_m; see ``cosmo_param``.
    """
    if conf.dim != 3:
        raise ValueError(f'dim={conf.dim} not supported')
    if conf.lpt_order not in (0, 1, 2, 3):
        raise ValueError(f'lpt_order={conf.lpt_order} not supported')
    if conf.lpt_order > 2:
        raise NotImplementedError('lpt_order=3 is not implemented (as in pmwd)')
    theta = check_theta(theta, cosmo)
    if not _needs_graph(modes, theta) or _fused_graph(modes, theta, conf):
        return _lpt_fused(modes, cosmo, conf)
    dev = modes.device
    modes = modes / conf.ptcl_cell_vol
    kvec = fftfreq(conf.ptcl_grid_shape, conf.ptcl_spacing, dtype=conf.float_dtype, device=dev)
    pots = []
    if conf.lpt_order > 0:
        pots.append(laplace(kvec, modes))
    if conf.lpt_order > 1:
        pots.append(laplace(kvec, fftfwd(_L(kvec, pots[0], conf))))
    ptcl = Particles.gen_grid(conf, vel=True, device=dev)
    disp, vel = ptcl.disp.clone(), ptcl.vel.clone()
    a = conf.a_start
    for order in range(1, 1 + conf.lpt_order):
        D, a2HDp = _growth_f32(a, cosmo, conf, order)
        if theta is not None and 'Omega_m' in theta:
            _, D_om, _, v_om = lpt_growth_derivs(a, cosmo, conf, order)
            f32 = lambda x: torch.tensor(x, dtype=conf.float_dtype, device=dev)
            D = host_value(f32(D), theta, torch.tensor(D_om, dtype=torch.float64))
            a2HDp = host_value(f32(a2HDp), theta, torch.tensor(v_om, dtype=torch.float64))
        for i, k in enumerate(kvec):
            g = neg_grad(k, pots[order - 1], conf.ptcl_spacing)
            g = fftinv(g, shape=conf.ptcl_grid_shape).to(conf.float_dtype).reshape(-1)
            disp[:, i] = disp[:, i] + D * g
            vel[:, i] = vel[:, i] + a2HDp * g
    return ptcl.replace(disp=disp.contiguous(), vel=vel.contiguous()), None
