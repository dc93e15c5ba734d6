"""The contact solve over units of length: its norms are plain sums of squares
where every component is of intermediate magnitude and MINPACK's scaled sums
elsewhere, where the solve goes on out of line.  Lengths times a power of two
leave every quotient of the solve as it is and move the norms through the
three ranges.

Tolerances: points 1e-5 of the largest axis and normals 1e-4, those of the
comparison with the reference's own contact vectors (the solve stops at
sqrt(eps) = 1.5e-8 in the angles' step, whose paths differ by roundings).
Flags are equal except where a decision is within 1e-6 of its threshold."""
import numpy as np
import pytest

import oracle as O


@pytest.mark.gpu
# all norms plain; some from the middle of a solve on scaled (residuals
# (1e-6 .. 1e-1)^2 of the unit around 3.8e-20); all tiny; all huge
@pytest.mark.parametrize("exp2", [0, -20, -36, 40])
def test_contact_solve_in_any_unit(exp2):
    import gazpart_amd as G
    from gazpart_amd import contacts as CT
    from gazpart_amd import workload as W
    u, k = 2.0 ** exp2, 150
    g = np.random.default_rng(3)
    L = 2.0 * np.pi * u
    rows = np.stack([W.species_spheroid(0.2, 1.0 + 0.5 * c, 1000.0) for c in range(3)])
    rows[:, 0:3] *= u
    st = np.zeros((13, 2 * k))
    st[6:10] = g.standard_normal((4, 2 * k))
    st[6:10] /= np.sqrt((st[6:10] ** 2).sum(axis=0))
    d = g.standard_normal((3, k))
    d *= g.uniform(0.15, 0.4, k) / np.sqrt((d * d).sum(axis=0))
    st[0:3, 0::2] = g.uniform(1.0, 5.0, (3, k))
    st[0:3, 1::2] = st[0:3, 0::2] + d
    st[0:3] *= u
    sid = g.integers(0, 3, 2 * k).astype(np.int32)
    ctx = G.Context(16, L, 0.01, 1.0, 1e-3, dpmax=0.4 * u)
    ctx.set_species(rows)
    ctx.bind_field(np.zeros((6, 20, 20, 16)))
    ctx.set_particles(st, sid)
    home = np.arange(1, 2 * k, 2, dtype=np.int32)
    flag, e1, e2, cn, nfev = ctx.ellipsoid_contact_detection(home, home + 1)
    ref = [O.contact(rows[sid[i]], rows[sid[i + 1]], st[0:3, i], st[6:10, i], st[0:3, i + 1],
                     st[6:10, i + 1]) for i in range(0, 2 * k, 2)]
    rf, r1, r2, rn = (np.array([r[c] for r in ref]) for c in range(4))
    qd = CT.decision_quantities(st, rows, sid, L, home, home + 1, r1, r2, rn)
    clear = np.minimum.reduce([np.abs(qd["depth"]) / qd["scale"], np.abs(qd["fm1"] - 1.0),
                               np.abs(qd["fm2"] - 1.0)]) > 1e-6
    assert clear.sum() > 0.9 * k and 0 < rf.sum() < k
    np.testing.assert_array_equal(flag[clear], rf[clear])
    f = clear & (rf == 1)
    assert np.abs(e1[f] - r1[f]).max() < 1e-5 * 0.2 * u
    assert np.abs(e2[f] - r2[f]).max() < 1e-5 * 0.2 * u
    assert np.abs(cn[f] - rn[f]).max() < 1e-4
    assert (nfev > 0).all() and (nfev <= 300).all()
