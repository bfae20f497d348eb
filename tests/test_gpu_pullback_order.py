"""The grid cotangents of the pullbacks are integer sums: the same bits whatever
order the markers come in.  In lattice order a workgroup's markers share an LDS
window of nodes; shuffled over the box they do not fit one and add to the grid
directly; marker counts around a workgroup's 128 leave lanes without a marker.
Marker cotangents are each marker's own and move with it."""
from __future__ import annotations

import numpy as np
import pytest

import cases
import ereb
from ereb import Geometry, Materials, api

pytestmark = pytest.mark.gpu

DT = 3e11


@pytest.mark.parametrize("M", [1, 127, 128, 129, 12_000])
def test_any_marker_order_gives_the_same_bits(M):
    g = Geometry(Nx=41, Ny=37, xsize=40_000.0, ysize=36_000.0, Nxmc=3, Nymc=3)
    mat = Materials(marker_property_mode=1)
    rng = np.random.default_rng(M)
    mk = {k: v[:M].copy() for k, v in cases.ref_markers(g, mat, seed=3, extra=200).items()}
    S, B = g.stag_shape, g.basic_shape
    gr = {n: cases.rand_grid(rng, S, -1e-9, 1e-9) for n in ("vx", "vy", "vxf", "vyf")}
    gr.update(wyx=cases.rand_grid(rng, B, -1e-12, 1e-12), tk2=cases.rand_grid(rng, S, 200, 300),
              DT=cases.rand_grid(rng, S, -1, 1), DSXX=cases.rand_grid(rng, S, -1e3, 1e3),
              DSXY=cases.rand_grid(rng, B, -1e3, 1e3))
    bars = {k: rng.random(M) - 0.5 for k in ("xm", "ym", "tkm", "sxym", "sxxm")}

    def run(ctx, p):
        m = {k: v[p].copy() for k, v in mk.items()}
        b = {k: v[p].copy() for k, v in bars.items()}
        mo, go = api.move_markers_rk4_pullback(
            ctx, m["xm"], m["ym"], m["tm"], m["tkm"], m["phim"], m["sxym"], m["sxxm"], gr["vx"],
            gr["vy"], gr["vxf"], gr["vyf"], gr["wyx"], gr["tk2"], M, DT, 1, b)
        t = api.update_marker_temperature_pullback(ctx, m["xm"], m["ym"], gr["DT"], gr["tk2"], 2,
                                                   M, b["tkm"])
        s = api.update_marker_stress_pullback(ctx, m["xm"], m["ym"], gr["DSXX"], gr["DSXY"], M,
                                              b["sxxm"], b["sxym"])
        grids = {**go, "DT": t[1], "DSXX": s[0], "DSXY": s[1]}
        return grids, {**mo, "T tkm": t[0], "T xm": t[3], "T ym": t[4], "S xm": s[2], "S ym": s[3]}

    same, shuffled = np.arange(M), rng.permutation(M)
    with ereb.Context(g, mat, ereb.FP64) as ctx:
        ga, ma = run(ctx, same)
        gb, mb = run(ctx, shuffled)
    for n in ga:
        assert np.abs(ga[n]).max() > 0, n
        assert np.array_equal(ga[n], gb[n]), n
    for n in ma:
        assert np.array_equal(ma[n][shuffled], mb[n]), n
