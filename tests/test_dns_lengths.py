"""The fluid solver at the larger lengths that have a plan of their own, up to
the largest: one exchange buffer from 320 on, more than one wavefront a row
above 128, workgroups of 1024 threads and 72 KB of LDS at 512.

The steps are restated with torch's FP64 transforms (numpy's would take
minutes at 512^3), which the CPU test pins to the oracle.  Tolerances as for
the smaller lengths: 1e-11 of the largest magnitude on the GPU (a transform
rounds by 1e-16 log2(n^3), a step has seven), 1e-13 on the CPU at n = 20."""
import math

import numpy as np
import pytest
import torch

from oracle import dns_ref as D

L2PI = 2.0 * math.pi


def modes(n, dev):
    k = torch.arange(n, device=dev, dtype=torch.float64)
    k = torch.where(k <= n // 2, k, k - n)
    kx = torch.arange(n // 2 + 1, device=dev, dtype=torch.float64)
    return kx[None, None, :], k[None, :, None], k[:, None, None]


def back(a, n):
    return torch.stack([torch.fft.irfftn(c, s=(n, n, n), norm="forward") for c in a])


def ahead(a):
    return torch.stack([torch.fft.rfftn(c, norm="forward") for c in a])


def curl(U, k):
    kx, ky, kz = k
    return torch.stack([1j * (ky * U[2] - kz * U[1]), 1j * (kz * U[0] - kx * U[2]),
                        1j * (kx * U[1] - ky * U[0])])


def project(U, k):
    kx, ky, kz = k
    k2 = kx * kx + ky * ky + kz * kz
    k2[0, 0, 0] = 1.0
    d = (kx * U[0] + ky * U[1] + kz * U[2]) / k2
    return torch.stack([U[0] - kx * d, U[1] - ky * d, U[2] - kz * d])


def steps(u, nu, dt, ns):
    """velocity, vorticity and EPS_FLU after ns steps in a box of 2 pi"""
    n = u.shape[-1]
    k = modes(n, u.device)
    k2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
    r = k2.sqrt() / (n / 2)
    f = torch.where(r <= D.RTRUNC, torch.ones_like(r), torch.where(
        r <= 1.0, torch.cos((math.pi / 2) * (r - D.RTRUNC) / (1.0 - D.RTRUNC)) ** 4,
        torch.zeros_like(r)))
    e = torch.exp(-nu * k2 * dt)
    eps = 0.0

    def rhs(v, V, first):
        nonlocal eps
        z = back(curl(V, k), n)
        if first:
            eps = nu * float((z * z).sum())
        T = project(ahead(torch.cross(v, z, dim=0)), k)
        T[:, 0, 0, 0] = 0.0   # the mean's |k|^2 is "infinity"
        return T

    U = ahead(u)
    for _ in range(ns):
        U = ahead(u)
        R = rhs(u, U, True)
        Un, U = (U + 0.5 * dt * R) * e, (U + dt * R) * e
        U = project(Un + 0.5 * dt * rhs(back(U, n), U, False), k) * f
        u = back(U, n)
    return u, back(curl(U, k), n), eps


def velocity(n, k0, seed, dev):
    """divergence-free, unit rms, energy around k0"""
    g = torch.Generator(device=dev).manual_seed(seed)
    k = modes(n, dev)
    k2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
    amp = k2.sqrt() * torch.exp(-k2 / (k0 * k0))
    for c in k:
        amp = amp * (c.abs() < n // 2)
    w = torch.stack([torch.complex(*(torch.randn(k2.shape, generator=g, device=dev,
                                                 dtype=torch.float64) for _ in range(2)))
                     for _ in range(3)])
    u = back(project(w * amp, k), n)
    return u / (u * u).mean().sqrt()


def test_restatement_is_the_oracle():
    n, nu, dt = 20, 0.01, 0.01
    u0 = velocity(n, 4.0, 3, "cpu")
    s = D.DnsRef(n, L2PI, nu, dt)
    s.set_velocity(u0.numpy())
    for _ in range(3):
        s.step()
    u, w, eps = steps(u0, nu, dt, 3)
    wr = D.btran(s.vorticity(), n)
    assert np.abs(u.numpy() - s.u).max() <= 1e-13 * np.abs(s.u).max()
    assert np.abs(w.numpy() - wr).max() <= 1e-13 * np.abs(wr).max()
    assert abs(eps - s.eps) <= 1e-13 * s.eps


@pytest.mark.gpu
@pytest.mark.parametrize("n,reuse", [(160, False), (192, True), (256, False), (320, False),
                                     (384, True), (512, False)])
def test_gpu_larger_lengths(n, reuse):
    from gazpart_amd.dns import Dns
    u0 = velocity(n, n / 10.0, n, "cuda")
    nu, dt, ns = 0.01, 0.1 / n, 2
    d = Dns(n, L2PI, nu, dt, reuse_spectral=reuse)
    d.set_velocity(u0.cpu().numpy())
    k = modes(n, "cuda")
    w0 = back(curl(ahead(u0), k), n)
    assert (torch.from_numpy(d.vorticity()).cuda() - w0).abs().max() <= 1e-11 * w0.abs().max()
    del w0
    d.step(ns)
    u, w, eps = steps(u0, nu, dt, ns)
    assert (torch.from_numpy(d.velocity()).cuda() - u).abs().max() <= 1e-11 * u.abs().max()
    assert (torch.from_numpy(d.vorticity()).cuda() - w).abs().max() <= 1e-11 * w.abs().max()
    assert abs(d.info()["eps"] - eps) <= 1e-11 * eps
    assert (u - u0).abs().max() > 1e-3 * u0.abs().max()
