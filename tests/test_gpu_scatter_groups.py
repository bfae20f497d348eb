"""The scatter's matrix-core groups against the oracle at the sizes where a
group, a chunk of four groups or a tile ends: fine cells (quarters of a basic
cell) of 0 to 65 markers side by side, grids whose cells fill no tile and whose
tiles are one cell wide, type-derived and free material vectors.

Bars: node sums within 1e-12 of the per-node sum of |terms| (the order of the
sum differs), in the Float64 form against the oracle, in the mixed form against
the sums of the property values it holds (its property vectors are float, its
weights and sums Float64); those against the oracle within 1e-6 of the field's
largest sum of |terms|."""
from __future__ import annotations

import numpy as np
import pytest

import cases
import ereb
from ereb import Geometry, Materials
from oracle import Oracle

pytestmark = pytest.mark.gpu

COUNTS = [0, 1, 2, 3, 4, 5, 8, 9, 12, 13, 15, 16, 17, 20, 33, 64, 65]


def _markers(g, mat, seed, typed):
    """COUNTS markers, in turn from a random start, in the quarters of the basic
    cells (so fine cells next to each other differ), and a few outside the box."""
    rng = np.random.default_rng(seed)
    nq = 4 * (g.Nx - 1) * (g.Ny - 1)
    cnt = np.array(COUNTS)[(np.arange(nq) * 7 + rng.integers(17)) % len(COUNTS)]
    cnt[rng.random(nq) < 0.15] = 0
    q = np.repeat(np.arange(nq), cnt)
    jq, iq = q // (2 * (g.Ny - 1)), q % (2 * (g.Ny - 1))
    x = (jq + rng.random(q.size)) * g.dx / 2
    y = (iq + rng.random(q.size)) * g.dy / 2
    x = np.concatenate([x, [-0.7 * g.dx, g.xsize + 0.4 * g.dx, 0.0, g.xsize]])
    y = np.concatenate([y, [0.3 * g.dy, g.ysize + 0.2 * g.dy, 0.0, g.ysize]])
    mk = cases.ref_markers(g, mat, seed=seed, extra=x.size)
    mk = {k: v[-x.size:].copy() for k, v in mk.items()}
    order = rng.permutation(x.size)
    mk["xm"], mk["ym"] = x[order], y[order]
    if typed:
        t = mk["tm"] - 1
        for f, tab in (("inv_gggtotalm", 1.0 / np.array(mat.gggsolidm)),
                       ("fricttotalm", mat.frictsolidm), ("cohestotalm", mat.cohessolidm),
                       ("tenstotalm", mat.tenssolidm), ("rhofluidcur", mat.rhofluidm),
                       ("alphasolidcur", mat.alphasolidm), ("alphafluidcur", mat.alphafluidm)):
            mk[f] = np.asarray(tab)[t]
    return mk


@pytest.mark.parametrize("form", [ereb.FP64, ereb.MIXED])
@pytest.mark.parametrize("typed", [True, False])
@pytest.mark.parametrize("Nx,Ny", [(3, 3), (7, 8), (8, 26), (14, 19)])
def test_groups(Nx, Ny, typed, form):
    g = Geometry(Nx=Nx, Ny=Ny, xsize=1000.0 * (Nx - 1), ysize=700.0 * (Ny - 1))
    mat = Materials(marker_property_mode=1)
    mk = _markers(g, mat, 10 * Nx + Ny + typed, typed)
    hrs, hrf = mat.radioactive_heating(7.1e13)
    props, sums = Oracle(g, mat).marker_to_nodes(mk, hrs, hrf, 1)
    scale = cases.abs_sums(g, mk, props)
    with ereb.Context(g, mat, form) as ctx:
        ctx.set_markers(mk)
        ctx.step_scatter(hrs, hrf, 1)
        got = [ctx.get_grid(n) for n in ereb.SUM_FIELDS]
        ctx.step_scatter(hrs, hrf, 1)
        again = [ctx.get_grid(n) for n in ereb.SUM_FIELDS]
        held = {n: ctx.get_marker(n) for n in cases.SCATTERED}
    if form == ereb.MIXED:
        own = cases.node_sums(g, mk, held)
        for n, a, b, c in zip(ereb.SUM_FIELDS, got, own, cases.abs_sums(g, mk, held)):
            assert np.all(np.abs(a - b) <= 1e-12 * c), n
    for n, a, b, c, d in zip(ereb.SUM_FIELDS, got, sums, scale, again):
        bar = 1e-12 * c if form == ereb.FP64 else 1e-6 * c.max()
        assert np.all(np.abs(a - b) <= bar), n
        assert np.array_equal(a, d), f"{n}: differs from run to run"
