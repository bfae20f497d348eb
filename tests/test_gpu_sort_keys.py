"""The sort's key starts and segment order at the sizes where its launches
change: up to 16,384 keys are scanned by one workgroup, more by several; a
workgroup of the ordering pass holds 1,024 keys, of which those with more than
48 markers are ordered by the whole workgroup.  Fine keys and sort order
bit-exact with the oracle's stable counting sort."""
from __future__ import annotations

import numpy as np
import pytest

import ereb
from ereb import Geometry, Materials
from oracle import Oracle

pytestmark = pytest.mark.gpu


# 144 keys a tile of 6 x 6 cells: 113 tiles 16,272 keys, 114 tiles 16,416, 1 tile 144
@pytest.mark.parametrize("Nx,Ny,crowd", [(679, 7, 0), (685, 7, 0), (679, 7, 60), (7, 7, 900)])
def test_key_counts(Nx, Ny, crowd):
    g = Geometry(Nx=Nx, Ny=Ny, xsize=100.0 * (Nx - 1), ysize=100.0 * (Ny - 1))
    mat = Materials(marker_property_mode=1)
    rng = np.random.default_rng(Nx + crowd)
    M = 20_011
    x, y = g.xsize * rng.random(M), g.ysize * rng.random(M)
    for c in range(crowd and 30):  # 30 crowded quarter cells, some of them neighbours
        k = slice(c * crowd, (c + 1) * crowd)
        x[k] = 50.0 * (c % (2 * (Nx - 1))) + 5 + 40 * rng.random(x[k].size)
        y[k] = 50.0 * (c % (2 * (Ny - 1))) + 5 + 40 * rng.random(x[k].size)
    p = rng.permutation(M)
    x, y = x[p].copy(), y[p].copy()
    perm_o, key_o, _ = Oracle(g, mat).fine_sort(x, y)
    if crowd:
        assert (np.bincount(np.asarray(key_o, dtype=np.int64)) > 48).sum() > 4
    one = np.ones(M)
    with ereb.Context(g, mat, ereb.FP64) as ctx:
        ctx.set_markers({"xm": x, "ym": y, "tm": np.full(M, 1), "tkm": 200 * one,
                         "phim": 0.1 * one})
        for _ in range(2):  # the second finds the counts cleared by the first
            ctx.step_scatter(np.zeros(3), np.zeros(3), 1)
            perm, key, nkeys = ctx.sort_order()
            assert np.array_equal(key, key_o)
            assert np.array_equal(perm, perm_o)


def test_segment_lengths():
    """Quarter cells of 1 to 50 markers each: the register networks of 16 and 32
    (padded), insertion to 48, the workgroup beyond."""
    g = Geometry(Nx=26, Ny=7, xsize=2500.0, ysize=600.0)
    mat = Materials(marker_property_mode=1)
    rng = np.random.default_rng(3)
    n = np.tile(np.arange(1, 51), 12)  # 50 x 12 quarter cells of 50 m
    q = np.repeat(np.arange(n.size), n)
    p = rng.permutation(q.size)
    q = q[p]
    x = 50.0 * (q % 50) + 5 + 40 * rng.random(q.size)
    y = 50.0 * (q // 50) + 5 + 40 * rng.random(q.size)
    perm_o, key_o, _ = Oracle(g, mat).fine_sort(x, y)
    lengths = np.bincount(np.asarray(key_o, dtype=np.int64))
    assert set(range(1, 51)) <= set(lengths[lengths > 0].tolist())
    one = np.ones(x.size)
    with ereb.Context(g, mat, ereb.FP64) as ctx:
        ctx.set_markers({"xm": x, "ym": y, "tm": np.full(x.size, 1), "tkm": 200 * one,
                         "phim": 0.1 * one})
        ctx.step_scatter(np.zeros(3), np.zeros(3), 1)
        perm, key, _ = ctx.sort_order()
    assert np.array_equal(key, key_o)
    assert np.array_equal(perm, perm_o)
