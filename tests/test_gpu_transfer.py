"""Transfers between the caller's memory and the device: the state comes back
as it was given whatever the number of particles (one chunk, several, a last
chunk of one particle; fewer or more particles than before in the same
context).

No tolerance: FP64 values are copied, the mixed form keeps the velocities and
spins as float32 (round to nearest)."""
import numpy as np
import pytest

@pytest.fixture(scope="module")
def G():
    import gazpart_amd
    return gazpart_amd


def _state(np_, L, seed):
    g = np.random.default_rng(seed)
    st = g.uniform(0.1, L - 0.1, (13, np_))
    st[3:6] = g.standard_normal((3, np_)) * 3.0
    q = g.standard_normal((4, np_))
    st[6:10] = q / np.sqrt((q * q).sum(axis=0))
    st[10:13] = g.standard_normal((3, np_)) * 40.0
    st[3:6, :1] = [[1e-33], [-0.0], [1e-41]]     # the reference's ZERO, a signed zero, a denormal
    return st


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [0, 1])
def test_state_round_trip(G, prec):
    from gazpart_amd import workload as W
    L = 2.0 * np.pi
    ctx = G.Context(16, L, 0.01, 1.0, 1e-3, precision=prec, dpmax=0.2)
    ctx.set_species(np.stack([W.species_spheroid(0.02, 1.0 + 0.1 * k, 1000.0) for k in range(3)]))
    for np_ in (1, 2, 255, 256, 257, 9_830, 39_322, 39_322, 300_001, 5):
        st = _state(np_, L, np_)
        sid = (np.arange(np_) % 3).astype(np.int32)
        ctx.set_particles(st, sid)
        want = st.copy()
        if prec:
            for rows in (slice(3, 6), slice(10, 13)):
                want[rows] = st[rows].astype(np.float32)
        got = ctx.get_particles()
        np.testing.assert_array_equal(got, want, err_msg=str(np_))
        assert (np.signbit(got) == np.signbit(want)).all()
    with pytest.raises(G.GpError):
        ctx.set_particles(st, np.full(5, 3, dtype=np.int32))
    np.testing.assert_array_equal(ctx.get_particles(), want)
