"""The batched FP64 sweeps, whose cell leaves out candidates that cannot be
accepted, against the one-solve-per-launch kernels, which evaluate every
candidate of the reference's update: the same bits and iteration counts, where
a candidate is left out by the narrowest margins or may not be left out."""
import numpy as np
import pytest

import oracle as O
import satt
import satt_workloads as W

pytestmark = pytest.mark.gpu


def model(kind, nx, ny, rng):
    """(velocity, m11, m12, m22)"""
    one, zero = np.ones((nx, ny)), np.zeros((nx, ny))
    if kind == "ties":          # every quadrant's gradient equal: roots on the current value
        return 3.0 * one, one, zero, one
    if kind == "rough":         # large jumps from cell to cell
        return np.exp(rng.uniform(np.log(0.8), np.log(8.0), (nx, ny))), one, zero, one
    if kind == "sheared":       # m12^2 within 2% of m11 m22, of either sign
        a, b = rng.uniform(0.5, 1, (nx, ny)), rng.uniform(0.5, 1, (nx, ny))
        return rng.uniform(2, 4, (nx, ny)), a, 0.99 * np.sqrt(a * b) * np.sign(rng.uniform(-1, 1, (nx, ny))), b
    if kind == "oblique":       # condition numbers to 1e7, the long axis across the cells' diagonals
        a, b = rng.uniform(0.5, 1, (nx, ny)), rng.uniform(0.5, 1, (nx, ny))
        eps = 10.0 ** rng.uniform(-6.5, -2, (nx, ny))
        return rng.uniform(2, 4, (nx, ny)), a, (1 - eps) * np.sqrt(a * b), b
    if kind == "indefinite":    # no metric at all: ea of either sign in some cells
        return rng.uniform(2, 4, (nx, ny)), one, np.where(rng.uniform(size=(nx, ny)) < 0.1, 1.2, 0.1), one
    if kind == "nan":
        v = rng.uniform(2, 4, (nx, ny))
        v[rng.integers(0, nx, 3), rng.integers(0, ny, 3)] = np.nan
        return v, one, zero, one
    return W.smooth_random_field(nx, ny, 5.0, rng, 2.5, 4.2), one, zero, one


@pytest.mark.parametrize("kind,nx,ny,d,lat", [
    ("ties", 41, 37, 0.05, 20.0), ("ties", 130, 20, 0.01, -1.0), ("smooth", 65, 64, 0.02, 60.0),
    ("smooth", 5, 70, 0.1, 0.0), ("smooth", 129, 6, 0.01, 10.0), ("rough", 64, 40, 0.01, 30.0),
    ("rough", 90, 35, 0.5, 40.0), ("sheared", 50, 66, 0.02, 20.0), ("sheared", 67, 31, 0.02, 20.0),
    ("oblique", 48, 45, 0.02, 0.0), ("oblique", 70, 35, 0.02, 50.0),
    ("indefinite", 40, 33, 0.02, 20.0), ("nan", 33, 40, 0.02, 20.0),
])
@pytest.mark.parametrize("waves", [1, 3])
def test_sweeps_equal_the_full_update(ctx, kind, nx, ny, d, lat, waves):
    rng = np.random.default_rng(nx * 1000 + ny)
    xg, yg = 100.0 + d * np.arange(nx), lat + d * np.arange(ny)
    v, m11, m12, m22 = model(kind, nx, ny, rng)
    b = W.random_receiver_batch(xg, yg, v, 4, rng, nrec=(1, 9), m11=m11, m12=m12, m22=m22)
    # one source on a node (T0 = 0 there), one on a grid line, two between nodes
    b["item_srcx"][0], b["item_srcy"][0] = xg[nx // 2], yg[ny // 2]
    b["item_srcx"][1] = xg[2]
    with ctx.plan(b) as p:
        p.set_waves(waves)
        out, T = [], []
        for launch in (satt.LAUNCH_BATCHED, satt.LAUNCH_PER_SOLVE):
            p.run(True, kind != "nan", launch)
            out.append(p.results())
            T.append([p.item_field(k) for k in range(4)] if launch == satt.LAUNCH_BATCHED else None)
    for k in ("iters", "tt_fwd", "chi", "item_status"):
        np.testing.assert_array_equal(out[0][k], out[1][k], err_msg=k)
    if kind != "nan":
        np.testing.assert_array_equal(out[0]["adj_s"], out[1]["adj_s"])
    for k in range(4):
        solve = (xg, yg, m11, m22, -m12, 1.0 / v, b["item_srcx"][k], b["item_srcy"][k])
        for entry in (ctx.fwd, ctx.fwd_noalloc):
            Tk, it, _ = entry(*solve)
            np.testing.assert_array_equal(T[0][k], Tk)
            assert it == out[0]["iters"][k, 0]


@pytest.mark.parametrize("nx,ny,nr", [(40, 33, 0), (65, 30, 1), (129, 3, 12), (3, 70, 5), (70, 41, 700)])
def test_adjoint_entry_point_equals_the_sequential_sweeps(ctx, nx, ny, nr):
    """satt_adj_lonlat, without receivers, with more of them than a workgroup's
    entries hold, several to a cell, on grids of one interior row or column."""
    rng = np.random.default_rng(nx + ny)
    xg, yg = 100.0 + 0.02 * np.arange(nx), 10.0 + 0.02 * np.arange(ny)
    one, zero = np.ones((nx, ny)), np.zeros((nx, ny))
    # times from a point inside (a grid of three rows has no forward solution)
    T = 37.0 * np.hypot(xg[:, None] - xg[nx // 2] - 0.003, yg[None] - yg[ny // 2] - 0.004)
    T = np.asfortranarray(T * (1 + 0.01 * rng.uniform(size=(nx, ny))))
    xr, yr = rng.uniform(xg[0], xg[-2], nr), rng.uniform(yg[0], yg[-2], nr)
    sa = rng.standard_normal(nr)
    a, b, c, delta = ctx.adj_setup_fields(xg, yg, one, one, zero, xr, yr, sa)
    want, it_o, _ = O.adj_pre(xg, yg, a, b, c, T, delta)
    got, it, _ = ctx.adj(xg, yg, one, one, zero, T, xr, yr, sa)
    assert it == it_o
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("nx,ny", [
    (3, 3), (15, 9), (16, 8), (17, 7), (32, 40), (33, 41), (4, 1231), (4, 1232), (1024, 5), (1025, 5)])
def test_solve_across_compute_units_at_its_edges(ctx, nx, ny):
    """satt_fwd_lonlat and satt_adj_lonlat on widths about a strip's 16 columns
    and the largest sizes of that route and the first past it."""
    rng = np.random.default_rng(nx + 7 * ny)
    xg, yg = 100.0 + 0.01 * np.arange(nx), 5.0 + 0.01 * np.arange(ny)
    one = np.ones((nx, ny))
    v = rng.uniform(2.5, 4.5, (nx, ny))
    c = rng.uniform(-0.3, 0.3, (nx, ny))
    sx, sy = xg[(nx - 1) // 2] + 0.003, yg[(ny - 1) // 2] + 0.004
    solve = (xg, yg, one, one, c, 1.0 / v, sx, sy)
    T = 37.0 * np.hypot(xg[:, None] - sx, yg[None] - sy)
    if min(nx, ny) > 3:
        T, it, _ = ctx.fwd(*solve)
        want, it_o, _ = ctx.fwd_noalloc(*solve)
        assert it == it_o
        np.testing.assert_array_equal(T, want)
    xr, yr = rng.uniform(xg[0], xg[-2], 5), rng.uniform(yg[0], yg[-2], 5)
    sa = rng.standard_normal(5)
    ga, gb, gc, delta = ctx.adj_setup_fields(xg, yg, one, one, c, xr, yr, sa)
    want, it_o, _ = O.adj_pre(xg, yg, ga, gb, gc, T, delta)
    got, it, _ = ctx.adj(xg, yg, one, one, c, T, xr, yr, sa)
    assert it == it_o
    np.testing.assert_array_equal(got, want)


def solve_pair(nx, ny, seed):
    """(arguments of Context.fwd, of Context.adj after its T)"""
    rng = np.random.default_rng(seed)
    xg, yg = 100.0 + 0.01 * np.arange(nx), 5.0 + 0.01 * np.arange(ny)
    one, c = np.ones((nx, ny)), rng.uniform(-0.3, 0.3, (nx, ny))
    fun = 1.0 / rng.uniform(2.5, 4.5, (nx, ny))
    xr, yr = rng.uniform(xg[0], xg[-2], 7), rng.uniform(yg[0], yg[-2], 7)
    return ((xg, yg, one, one, c, fun, xg[nx // 2] + 0.003, yg[ny // 2] + 0.004),
            (xr, yr, rng.standard_normal(7)))


def recovered(nx, ny, **fail):
    """Forward and adjoint with waits that run out, in a context whose scratch
    holds another solve: what a call without such waits gives."""
    solve, rec = solve_pair(nx, ny, nx)
    with satt.Context(0) as c:
        T, it, st = c.fwd(*solve)
        Ta, ita, sta = c.adj(*solve[:5], T, *rec)
        other, orec = solve_pair(nx, ny, nx + 1)
        c.adj(*other[:5], c.fwd(*other)[0], *orec)
        c.solve_fail_waits(**fail)
        for _ in range(2):
            got, it2, st2 = c.fwd(*solve)
            assert (it2, st2) == (it, st)
            np.testing.assert_array_equal(got, T)
            got, it2, st2 = c.adj(*solve[:5], T, *rec)
            assert (it2, st2) == (ita, sta)
            np.testing.assert_array_equal(got, Ta)


@pytest.mark.parametrize("nx,ny,strip", [(12, 9, 0), (70, 41, 0), (70, 41, 2), (70, 41, 4)])
def test_a_strip_that_gives_up_is_not_lost(ctx, nx, ny, strip):
    """The strip's columns are not written: the solve is done again on the
    batched sweeps, also where the other strips ended in order."""
    recovered(nx, ny, strip=strip)


@pytest.mark.parametrize("nx,ny,strip", [(70, 41, 1), (1025, 5, -1)])
def test_solves_whose_teams_give_up_too(ctx, nx, ny, strip):
    """The one-workgroup kernels, which wait for nothing, are the last resort,
    with and without a solve across compute units before."""
    recovered(nx, ny, strip=strip, team=True)


def test_solves_past_the_batched_row_limit(ctx):
    """More rows than the batched sweeps take: the one-workgroup kernels."""
    nx, ny = 4, 10250
    xg, yg = 100.0 + 0.002 * np.arange(nx), 0.002 * np.arange(ny)
    one, zero = np.ones((nx, ny)), np.zeros((nx, ny))
    sx, sy = xg[1] + 0.001, yg[5000] + 0.0007
    T, it, _ = ctx.fwd(xg, yg, one, one, zero, one / 3.0, sx, sy)
    To, it_o, _ = O.fwd(xg, yg, one, one, zero, one / 3.0, sx, sy)
    assert it == it_o
    assert np.max(np.abs(T - To)) <= 1e-9 * np.max(To)
    Ta, _, _ = ctx.adj(xg, yg, one, one, zero, To, [xg[2]], [yg[100] + 0.001], [1.0])
    Tao, _, _ = O.adj(xg, yg, one, one, zero, To, [xg[2]], [yg[100] + 0.001], [1.0])
    assert np.max(np.abs(Ta - Tao)) <= 1e-8 * np.max(np.abs(Tao))
