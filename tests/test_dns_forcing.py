"""The forcing of a wide band: steps in turns of a few megabytes of amplitudes.

Tolerance as for the narrow band: 1e-11 of the largest velocity."""
import math

import numpy as np
import pytest

from oracle import dns_ref as D

L2PI = 2.0 * math.pi


@pytest.mark.gpu
def test_wide_band_matches_the_oracle():
    """17,000 modes: five steps of amplitudes a turn, seven steps in one call"""
    import torch
    from gazpart_amd.dns import Dns
    from test_dns_lengths import velocity
    n, nu, dt = 32, 0.02, 0.002
    fp = dict(kmin=0.5, kmax=40.0, sigma=0.5, tforce=0.1, seed=-11)
    u0 = velocity(n, 2.0, 23, torch.device("cpu")).numpy()
    d = Dns(n, L2PI, nu, dt, forcing=fp)
    d.set_velocity(u0)
    f = D.OuForcing(n, L2PI, fp["kmin"], fp["kmax"], fp["sigma"], fp["tforce"], fp["seed"])
    s = D.DnsRef(n, L2PI, nu, dt, forcing=f)
    s.set_velocity(u0)
    assert d.info()["nforce"] == len(f.modes) > 16_000
    d.step(7)
    for _ in range(7):
        s.step()
    assert np.abs(d.velocity() - s.u).max() <= 1e-11 * np.abs(s.u).max()


@pytest.mark.gpu
def test_wide_band_takes_one_step_of_amplitudes():
    """A million modes at 128^3 are 50 MB of amplitudes a step; the device keeps
    one step's of them (a factor of two is let pass)."""
    import torch
    from gazpart_amd.dns import Dns
    n, keep, held = 128, [], []
    for fp in (None, dict(kmin=0.5, kmax=1e3, sigma=0.5, tforce=0.1, seed=-11)):
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        keep.append(Dns(n, L2PI, 0.01, 1e-3, forcing=fp))
        held.append(free - torch.cuda.mem_get_info()[0])
    modes = n * n * (n // 2 + 1)   # all but the mean are in the band
    assert held[1] - held[0] <= 2 * 48 * modes + 4 * modes
