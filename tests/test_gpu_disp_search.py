"""The dispersion search, whose bracketing steps are evaluated 64 at a time:
a root does not depend on how many steps lie before it.

A period's search starts 1.5 steps below the period before's root, so the
same period met with other periods in between is bracketed elsewhere and
refined to the same root within the refinement's relative bracket of 1e-6
(2e-6 between two of them; REAL(4) rounding is 6e-8).  Group velocities are
difference quotients over +-0.5% in period, which amplify that about 100-fold."""
import numpy as np
import pytest

import oracle as O
import satt

pytestmark = pytest.mark.gpu


def columns(nx, ny, nz, top, seed):
    rng = np.random.default_rng(seed)
    z = np.linspace(0.0, 60.0, nz)
    vs = top + (4.5 - top) * z / 60.0
    vs = vs[None, None] * (1 + 0.05 * rng.uniform(-1, 1, (nx, ny, 1)) * np.sin(z / 9.0)[None, None])
    return np.asfortranarray(vs), z


@pytest.mark.parametrize("iwave", [1, 2])
@pytest.mark.parametrize("igr", [0, 1])
@pytest.mark.parametrize("nz,top", [(12, 2.9), (31, 1.2), (65, 0.7)])
def test_roots_do_not_depend_on_the_steps_before_them(ctx, iwave, igr, nz, top):
    """Two periods far apart (hundreds of steps: several rounds of 64) against
    the same two with close ones between them (a few steps each)."""
    vs, z = columns(4, 3, nz, top, nz)
    dense = np.geomspace(2.0, 60.0, 80)
    far = ctx.fwdsurf3d(vs, z, dense[[0, -1]], iwave, igr)
    near = ctx.fwdsurf3d(vs, z, dense, iwave, igr)
    assert np.all(far > 0)
    if igr == 0:
        assert np.all(far[1] - far[0] > 0.35)   # 70 steps of 0.005 km/s or more
    tol = 2e-6 if igr == 0 else 2e-4
    np.testing.assert_allclose(far, near[[0, -1]], rtol=tol, atol=0)


def test_columns_without_a_root_are_still_reported(ctx):
    """A column of NaN, whose period equation never changes sign, with the
    columns beside it unaffected."""
    vs, z = columns(3, 2, 20, 3.0, 5)
    good = ctx.fwdsurf3d(vs, z, [5.0, 20.0])
    bad = vs.copy(order="F")
    bad[1, 1, :] = np.nan
    out, st = ctx.fwdsurf3d(bad, z, [5.0, 20.0], status=True)
    assert st[1, 1] == satt.E_DISPERSION and np.all(out[:, 1, 1] == 0)
    st[1, 1] = 0
    assert not st.any()
    keep = np.ones((3, 2), bool)
    keep[1, 1] = False
    assert np.array_equal(out[:, keep], good[:, keep])


def test_search_that_leaves_its_range_is_reported(ctx):
    """A homogeneous half-space carries no Love wave: at a wavelength of seven
    times the model's depth (past what the flattened earth's curvature traps)
    no step up to the largest Vs changes the sign.  The last step of the range
    lies among the first 64 (0.87 to 1.01 of Vs 1.5), or several rounds up."""
    for vs in (1.5, 4.0):
        out, good = {}, columns(3, 2, 20, 3.0, 5)[0]
        _, z = columns(1, 1, 20, 3.0, 5)
        mixed = good.copy(order="F")
        mixed[2, 0, :] = vs
        for p in ([5.0], [420.0 / vs]):
            ref = ctx.fwdsurf3d(good, z, p, 1, 0)
            out, st = ctx.fwdsurf3d(mixed, z, p, 1, 0, status=True)
            if p[0] > 5.0:
                assert st[2, 0] == satt.E_DISPERSION and out[0, 2, 0] == 0
            else:
                assert st[2, 0] == 0
            st[2, 0] = 0
            assert not st.any()
            keep = np.ones((3, 2), bool)
            keep[2, 0] = False
            assert np.array_equal(out[:, keep], ref[:, keep])


@pytest.mark.parametrize("vs", [1.5, 2.0, 4.0])
def test_root_and_limit_among_the_same_steps(ctx, vs):
    """The Rayleigh velocity of a homogeneous half-space, from its own equation
    (a tolerance of 1e-3 for the flattening of the earth, a wavelength over its
    radius): the search starts at 0.95 of it, and for the lower velocities the
    limit above Vs is among the 64 steps that bracket it, after it."""
    vp = float(O.brocher_vp_rho(np.float32(vs))[0])
    c = np.linspace(0.7, 0.9999, 200001) * vs
    f = (2 - (c / vs) ** 2) ** 2 - 4 * np.sqrt(1 - (c / vp) ** 2) * np.sqrt(1 - (c / vs) ** 2)
    root = c[np.argmax(np.sign(f) != np.sign(f[0]))]
    z = np.linspace(0.0, 60.0, 20)
    got = ctx.fwdsurf3d(np.full((2, 2, 20), vs, order="F"), z, [1.0, 2.0])
    assert np.all(np.abs(got - root) < 1e-3 * root)
