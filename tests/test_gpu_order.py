"""The advance's layer order (every XCD through its own y block of the cell
layers), which takes cells of fewer than six particles and y blocks of four
workgroups or more: against the plain ranges, the same bits."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("n,scheme", [(24, 3), (33, 4)])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("np_,nz", [(335_872, 41), (341_007, 41), (353_000, 43)])
def test_layer_order_changes_no_result(n, scheme, prec, np_, nz):
    import gazpart_amd as G
    from gazpart_amd import workload as W
    wl = W.build_workload("order", n, np_, scheme=scheme, apr=2.0, emaj_dx=0.01, st=1.0, seed=np_)
    out = []
    for xcd in (0, 1):
        ctx = G.Context(wl.n, wl.L, wl.visc, wl.rhof, wl.dtime, scheme=scheme, precision=prec,
                        dpmax=wl.L / (2.0 * nz - 1.5), xcd_remap=xcd, graph=2)
        ctx.bind_field(wl.field)
        ctx.set_species(wl.species)
        ctx.set_particles(wl.state, wl.species_id)
        nb = ctx.collision_grid()[0]
        assert nb[2] == nz and (np_ + 255) // 256 >= 32 * nz and np_ < 6 * nb[3]
        ctx.step(4)
        out.append(ctx.get_particles())
    np.testing.assert_array_equal(out[0], out[1])
    assert not np.array_equal(out[0], wl.state)
