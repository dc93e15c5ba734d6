"""Transfers between the caller's memory and the device, and the advance's
workgroup order: the state comes back as it was given whatever the number of
particles (one chunk, several, a last chunk of one particle; fewer or more
particles than before in the same context), and no order of the workgroups
changes a result.

No tolerance: FP64 values are copied, the mixed form keeps the velocities and
spins as float32 (round to nearest), and the order of independent particles
leaves every bit."""
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


@pytest.mark.gpu
@pytest.mark.parametrize("n,scheme", [(24, 3), (33, 4)])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("np_,nz", [(163_840, 20), (170_003, 20), (20_011, 16)])
def test_workgroup_order_changes_no_result(G, n, scheme, prec, np_, nz):
    """nz layers of collision cells: the layer order of the advance's
    workgroups (four workgroups or more a layer and y block; the last case has
    fewer and keeps the plain order), against one range per XCD"""
    from gazpart_amd import workload as W
    wl = W.build_workload("order", n, np_, scheme=scheme, apr=2.0, emaj_dx=0.02, st=1.0, seed=np_)
    out = []
    for xcd in (0, 1):
        ctx = G.Context(wl.n, wl.L, wl.visc, wl.rhof, wl.dtime, scheme=scheme, precision=prec,
                        dpmax=wl.L / (2.0 * nz + 0.5), xcd_remap=xcd, graph=2)
        ctx.bind_field(wl.field)
        ctx.set_species(wl.species)
        ctx.set_particles(wl.state, wl.species_id)
        ctx.step(4)
        out.append(ctx.get_particles())
    np.testing.assert_array_equal(out[0], out[1])
    assert not np.array_equal(out[0], wl.state)


def test_layer_order_takes_every_workgroup_once():
    """the order itself, restated: every workgroup exactly once"""
    for nb in (32, 33, 100, 157, 274, 3907):
        for layers in (1, 2, 3, 7, nb // 32):
            if layers < 1 or nb < 32 * layers:
                continue
            per = (nb + 8 * layers - 1) // (8 * layers)
            seen = []
            for b in range(8 * layers * per):
                y, t = b & 7, b >> 3
                j, z = t % per, t // per
                k, n = 8 * z + y, 8 * layers
                lo, hi = k * nb // n, (k + 1) * nb // n
                if lo + j < hi:
                    seen.append(lo + j)
            assert sorted(seen) == list(range(nb)), (nb, layers)


@pytest.mark.gpu
@pytest.mark.parametrize("np_,cells", [(300, 14), (3_000, 14), (3_000, 9), (20_000, 12)])
def test_collision_pass_matches_the_candidate_list(G, np_, cells):
    """The filters, the solve list and the one-collision pass against the
    materialised candidate list solved pair by pair: cells of less and of
    more than a particle on average, contacts from none (their rounds in one
    workgroup, from the second pass on) to hundreds.  Lists and counts are
    whole numbers: equal."""
    from gazpart_amd import contacts as CT
    from gazpart_amd import workload as W
    L = 2.0 * np.pi
    a = L / (4.0 * cells + 0.5)
    sp = W.species_spheroid(a, 2.0, 500.0)[None, :]
    sid = np.zeros(np_, dtype=np.int32)
    st = W.random_particles(np_, L, a, 5)
    st[3:6] = np.random.default_rng(np_).standard_normal((3, np_))
    ctx = G.Context(16, L, 0.01, 1.0, 1e-4, dpmax=2.0 * a)
    ctx.set_species(sp)
    ctx.bind_field(np.zeros((6, 20, 20, 16)))
    ctx.set_particles(st, sid)
    for rep in range(3):
        st = ctx.get_particles()
        home, near = ctx.collision_detection_connectivity()
        flag, e1, e2, cn, _ = ctx.ellipsoid_contact_detection(home, near)
        qd = CT.decision_quantities(st, sp, sid, L, home, near, e1, e2, cn)
        hit = CT.contact_of(flag, qd)
        used, want = np.zeros(np_ + 1, dtype=bool), []
        for h, n in zip(home[hit], near[hit]):
            want.append(not (used[h] or used[n]))
            if want[-1]:
                used[h] = used[n] = True
        ctx.collision()
        s = ctx.stats()
        assert s["nclose"] == len(home)
        h, n, r = ctx.contacts()
        np.testing.assert_array_equal(h, home[hit])
        np.testing.assert_array_equal(n, near[hit])
        np.testing.assert_array_equal(r, want)
        assert s["ncollision"] == sum(want)
        assert want or rep or np_ < 1_000
        after = ctx.get_particles()
        moved = (after != st).any(axis=0)
        np.testing.assert_array_equal(np.nonzero(moved)[0] + 1, np.nonzero(used)[0])
