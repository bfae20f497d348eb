"""Cell and weights of positions at the conversion's limits: on nodes and next
to them, outside the grid, around 2^31 and 2^63 spacings, infinite and NaN.
The temperature and stress gathers bit for bit as the oracle (which truncates in 64 bits and divides by the spacing)."""
from __future__ import annotations

import numpy as np
import pytest

import cases
import ereb
from ereb import api
from ereb.constants import Geometry, Materials
from oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("xsize,ysize", [(3900.0, 3200.0), (1.0e5 / 3, 8.0e4 / 7)])
def test_gathers_at_extremes(xsize, ysize):
    g = Geometry(Nx=40, Ny=33, xsize=xsize, ysize=ysize)
    mat = Materials(marker_property_mode=1)
    rng = np.random.default_rng(8)
    k = np.concatenate([np.arange(-3, 44) / 2.0, [2.0**31 - 1, 2.0**31, 2.0**32 + 0.5, 1e12],
                        2.0**63 * np.array([0.99, 1.0, 1.01]), [1e250, np.inf, np.nan]])
    k = np.concatenate([k, -k])

    def axis(h):
        v = k * h
        return np.concatenate([v, np.nextafter(v, np.inf), np.nextafter(v, -np.inf)])

    with np.errstate(all="ignore"):
        ex, ey = axis(g.dx), axis(g.dy)
    n = ex.size
    x = np.concatenate([ex, g.xsize * rng.random(n), ex])
    y = np.concatenate([g.ysize * rng.random(n), ey, ey])
    M = x.size
    tkm, sxx, sxy = (200.0 + rng.random(M) for _ in range(3))
    S, B = (g.Ny1, g.Nx1), (g.Ny, g.Nx)
    DT, tk2 = cases.rand_grid(rng, S, -5, 5), cases.rand_grid(rng, S, 263, 310)
    DSXX, DSXY = cases.rand_grid(rng, S, -1e5, 1e5), cases.rand_grid(rng, B, -1e5, 1e5)
    orc = Oracle(g, mat)
    with np.errstate(all="ignore"):
        ref_t = orc.update_marker_temperature(x, y, tkm, DT, tk2, 2)
        ref_s = orc.update_marker_stress(x, y, sxx, sxy, DSXX, DSXY)
    t, a, b = tkm.copy(), sxx.copy(), sxy.copy()
    with ereb.Context(g, mat, ereb.FP64) as ctx:
        api.update_marker_temperature_(ctx, x, y, t, DT, tk2, 2, M)
        api.update_marker_stress_(ctx, x, y, a, b, DSXX, DSXY, M)
    np.testing.assert_array_equal(t, ref_t)
    np.testing.assert_array_equal(a, ref_s[0])
    np.testing.assert_array_equal(b, ref_s[1])
