"""Where a walk enters the octree and goes from cell to cell (the start grid
and the neighbour table) against the oracle's descents from the root, bit for
bit: starts on walls of the cells, one unit in the last place beside them, near
the domain's faces, in domains far from the origin (where the grid gets coarser
and its margin wider) and of very uneven sides, and flights through many cells."""
import numpy as np
import pytest

from nebula_amd import api as A
from nebula_amd import workloads as W
from oracle import pyoracle as O
from tests.helpers import grating_tris, material, slab_tris

pytestmark = pytest.mark.gpu


def _rays(center, half, n, rng):
    """Positions whose coordinates are cell walls of some level (the roundings
    of a descent included), their neighbours in float32, or anything."""
    pos = np.empty((n, 3), np.float32)
    for a in range(3):
        c, h = np.float32(center[a]), np.float32(half[a])
        x = np.full(n, c, np.float32)
        hw = np.float32(0.5)
        stop = rng.integers(0, 8, n)
        for level in range(8):
            step = np.where(rng.random(n) < 0.5, hw * h, -(hw * h)).astype(np.float32)
            x = np.where(level < stop, (x + step).astype(np.float32), x)
            hw = np.float32(hw * np.float32(0.5))
        kind = rng.integers(0, 6, n)
        any_x = (c + (rng.random(n) * 2 - 1).astype(np.float32) * h * np.float32(0.999)).astype(np.float32)
        edge = (c + np.where(rng.random(n) < 0.5, -1, 1).astype(np.float32) * h * np.float32(0.99999)).astype(np.float32)
        x = np.where(kind == 0, np.nextafter(x, np.float32(1e30)), x)
        x = np.where(kind == 1, np.nextafter(x, np.float32(-1e30)), x)
        x = np.where(kind == 2, edge, x)
        x = np.where(kind >= 4, any_x, x)
        pos[:, a] = np.clip(x, np.nextafter(c - h, np.float32(1e30)), np.nextafter(c + h, np.float32(-1e30)))
    d = rng.standard_normal((n, 3)).astype(np.float32)
    d[rng.random(n) < 0.1, 0] = 0.0
    d[rng.random(n) < 0.1, 1] = -0.0
    s = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]).astype(np.float32)
    d = (d * (np.float32(1) / np.sqrt(s))[:, None]).astype(np.float32)
    dist = np.exp(rng.uniform(np.log(1e-3), np.log(4.0 * float(np.max(half))), n)).astype(np.float32)
    return pos, d, dist


@pytest.mark.parametrize("shape,shift", [
    ("grating", (0.0, 0.0, 0.0)), ("grating", (1e5, -3e4, 777.0)), ("grating", (3e6, 0.0, 0.0)),
    ("holes", (0.0, 0.0, 0.0)), ("holes", (-4096.0, 8192.0, 1.0)), ("slab", (0.1, 0.2, 0.3)),
    ("wire", (0.0, 0.0, 0.0))])
def test_cells_equal_oracle(shape, shift):
    if shape == "holes":
        tris = A.mesh_to_triangles(W.contact_hole_geometry(3, 3, n_seg=12, layers=((40.0, 1), (40.0, 2))))
    else:
        tris = np.array(slab_tris() if shape == "slab" else grating_tris(), copy=True)
    if shape == "wire":   # sides of 1 : 1 : 1000
        for f in ("r0", "e1", "e2"):
            tris[f][:, 0] *= np.float32(1000.0)
    tris["r0"] += np.asarray(shift, np.float32)
    dev = A.Device(0)
    g = A.Geometry(dev, tris)
    ow = O.OracleWorld(tris, [material("si"), material("pmma"), material("si")])
    rng = np.random.default_rng(len(shape) + int(abs(shift[0])))
    n = 20011
    pos, d, dist = _rays(g.center, g.halfsize, n, rng)
    it = np.full(n, -1, np.int32)
    im = rng.choice(np.array([-123, 0, 1], np.int32), n)
    print(shape, shift, flush=True)
    t, dd = g.query(pos, d, dist, it, im)
    rt, rd = ow.queries(pos, d, dist, it, im)
    assert np.array_equal(t, rt)
    assert np.array_equal(dd.view(np.uint32), rd.view(np.uint32))
    dev.close()
