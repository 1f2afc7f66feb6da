"""Gaussian laser pulse initialiser (chimeraCL/laser.py:3-37), on the GPU."""
from __future__ import annotations

import numpy as np

from . import _lib
from .methods.generic_methods_hip import ptr


def add_gausian_pulse(solver, laser):
    """Ez_m0 pulse, forward transform, G = -i w sign(kx) E, vacuum
    propagation over x0 - x_foc, then B = rot(G)/w^2 and the backward
    transforms of B and E (laser.py:3-37).  The pulse and the spectral
    set-up run in FP64; in the mixed form the FP64 result is rounded once
    into the FP32 planes."""
    k0 = 2 * np.pi * laser["k0"]
    a0, Lx, R, x0, x_foc = (laser[k] for k in ("a0", "Lx", "R", "x0", "x_foc"))
    a, D = solver.Args, solver.DataDev
    stream = solver.comm.stream()
    if not solver.comm.mixed:
        Ez, Ez_fb, Gz_fb, sp = D["Ez_m0"], D["Ez_fb_m0"], D["Gz_fb_m0"], solver._sp
        _lib.call("chm_laser_pulse_f64", ptr(Ez), a["Nx"], a["Nr"], a["Xmin"], a["dx"], a["Rmin"],
                  a["dr"], k0, a0, x0, Lx, R, stream)
        solver.fb_transform(scals=["Ez"], dir=0)
        _lib.call("chm_laser_spectral_f64", sp, ptr(D["w_m0"]), ptr(Ez_fb), ptr(Gz_fb), x0 - x_foc, stream)
    else:
        _mixed_pulse(solver, k0, a0, x0, Lx, R, x_foc)
    solver.restore_B_fb()
    solver.fb_transform(vects=["B", "E"], dir=1)


def _mixed_pulse(solver, k0, a0, x0, Lx, R, x_foc):
    """Builds the spectral pulse (mode 0) in FP64 from the solver's own FP64
    tables and rounds E_fb, G_fb into its FP32 planes.  (An FP64 twin Solver
    built for this took as long as the solver itself, with all of its planes
    and tables, in every call.)"""
    import torch
    a, D, dev, stream = solver.Args, solver.DataDev, solver.comm.device, solver.comm.stream()
    Nx, Nr, Nk = a["Nx"], a["Nr"], a["Nr"] - 1
    sp = _lib.Spectral(Nx=Nx, Nr=Nr, M=0, dt_inv=a["dt_inv"])
    sp.kx, sp.twiddle = ptr(D["kx"]), ptr(D["fft_twiddle"])
    sp.phase_minus, sp.phase_plus = ptr(D["phase_minus"]), ptr(D["phase_plus"])
    dht = torch.empty(_lib.lib.chm_dht_table_elems(Nk, Nk), dtype=torch.float64, device=dev)
    _lib.call("chm_pad_table", ptr(D["DHT_m0"]), Nk, Nk, ptr(dht), None, None, None, stream)
    sp.DHT[0] = ptr(dht)
    Ez = torch.empty((Nr, Nx), dtype=torch.float64, device=dev)
    E_fb, G_fb = (torch.empty((Nk, Nx), dtype=torch.complex128, device=dev) for _ in range(2))
    ws = torch.empty(_lib.lib.chm_transform_workspace_bytes(Nx, Nr, 0, 1, 8), dtype=torch.uint8,
                     device=dev)
    real, fb = _lib.Planes(m0=ptr(Ez)), _lib.Fb()
    fb.m[0] = ptr(E_fb)
    _lib.call("chm_laser_pulse_f64", ptr(Ez), Nx, Nr, a["Xmin"], a["dx"], a["Rmin"], a["dr"], k0, a0,
              x0, Lx, R, stream)
    _lib.call("chm_transform_f64", sp, real, fb, 1, 0, 0, 0, ptr(ws), ws.numel(), stream)
    _lib.call("chm_laser_spectral_f64", sp, ptr(D["w_m0"]), ptr(E_fb), ptr(G_fb), x0 - x_foc, stream)
    D["Ez_fb_m0"].copy_(E_fb)
    D["Gz_fb_m0"].copy_(G_fb)
