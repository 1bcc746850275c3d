"""The rule by which the batched FP64 sweep's cell (fwd_cell_r) leaves out the
lesser root of a quadrant, restated: a root that is left out may not pass the
causality tests as they round.  Random cells about the corner where it could,
near-double roots with a gradient across the neighbours' direction, for metrics
of condition numbers to 1e8."""
import numpy as np
import pytest


@pytest.mark.parametrize("small_time", [False, True])
@pytest.mark.parametrize("digits", [2, 5, 8])
def test_a_root_left_out_fails_the_causality_tests(digits, small_time):
    rng, n = np.random.default_rng(10 * digits + small_time), 1_000_000
    a, b = rng.uniform(0.5, 1, n), rng.uniform(0.5, 1, n)
    c = (1 - 10.0 ** rng.uniform(-digits, -0.5, n)) * np.sqrt(a * b) * rng.choice([-1, 1], n)
    ff = 1.0
    px, py = 10.0 ** rng.uniform(-12, 4, n), 10.0 ** rng.uniform(0, 4, n)
    # a gradient of length 1 in the metric, to rounding and more, orthogonal to p
    gx, gy = c * px - b * py, a * px - c * py
    g = rng.choice([-1, 1], n) / np.sqrt(a * gx * gx + b * gy * gy - 2 * c * gx * gy)
    g = g * (1 + rng.uniform(-1, 1, n) * 10.0 ** rng.uniform(-17, -4, n))
    t = 0.0 if small_time else 10.0 ** rng.uniform(-16, 1, n)
    qx, qy = g * gx - px * t, g * gy - py * t
    # the cell's expressions, in its order
    A1, A2, A3 = a * (px * px), 2 * a * px * qx, a * (qx * qx)
    B1, B2, B3 = b * (py * py), 2 * b * py * qy, b * (qy * qy)
    C1, C2 = 2 * c * px, 2 * c * qx
    ea = A1 + B1 - C1 * py
    eb = A2 + B2 - 2 * c * (px * qy + py * qx)
    ec = A3 + B3 - C2 * qy - ff
    ebb = eb * eb
    delta = ebb - 4 * ea * ec
    real = (ea > 0) & (delta >= 0)
    tt = (-eb - np.sqrt(np.where(real, delta, 0))) / (2 * ea)
    Tx, Ty = px * tt + qx, py * tt + qy
    accepted = real & (a * Tx - c * Ty >= 0) & (b * Ty - c * Tx >= 0)
    left_out = real & (delta > 1e-12 * (ea * ff + ebb))
    assert left_out.sum() > n / 10 and accepted.any()   # both are met here
    assert not (left_out & accepted).any()
