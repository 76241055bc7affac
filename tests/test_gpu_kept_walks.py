"""Walks that a launch leaves to the next one, in the scored, deposit and
several-world kernels and across a change of material parameters, against
drivers with too few slots to leave any (below 65 536, they finish every walk
in the launch that began it)."""
import numpy as np
import pytest

from nebula_amd import api as A
from nebula_amd import workloads as W
from tests.helpers import grating_tris, material, slab_tris

pytestmark = pytest.mark.gpu

SCORES = [(0, 0), (0, 1), (1, 1), (1, 2)]


@pytest.fixture(scope="module")
def world():
    dev = A.Device(0)
    mats = [A.Material(dev, A.HostMaterial(material(m))) for m in ("si", "pmma")]
    return dev, mats, A.Geometry(dev, grating_tris()), A.Geometry(dev, slab_tris())


def _rows(a):
    a = np.ascontiguousarray(a)
    return np.sort(a.view(np.dtype((np.void, a.dtype.itemsize))))


def _track(world, kind, pri, capacity, few):
    dev, mats, grating, slab = world
    n = len(pri)
    tags = np.arange(n, dtype=np.uint32)
    d = A.Driver(dev, capacity, grating, mats, seed=31, steps_per_launch=2)
    if few is not None:
        d.set_cascade(few)
    if kind == "scores":
        d.set_score_params(SCORES)
    if kind == "deposits":
        d.set_deposits(True)
    if kind == "worlds":
        d.push(pri[::2], tags[::2], sid_base=1 << 40, world=d.add_world(slab, mats))
        d.push(pri[1::2], tags[1::2])
    else:
        d.push(pri, tags)
    more = b""
    if kind == "scores":
        det, more = d.run_scores(4 * n)
        more = more[np.argsort(det["sid"])].tobytes()
    elif kind == "deposits":
        det, dep = d.run_with_deposits(0)
        more = _rows(dep).tobytes()
        assert len(dep) > n
    else:
        det = d.run(4 * n)
    steps = d.steps()
    d.close()
    assert len(det) > n // 20
    return np.sort(det, order="sid").tobytes(), more, steps


@pytest.mark.parametrize("kind,energy", [("scores", 200.0), ("deposits", 30.0), ("worlds", 200.0)])
def test_kept_walks_equal_finished_ones(world, kind, energy):
    pri = W.raster_scan(100, 100, 7, energy, -140.0, 140.0, -140.0, 140.0, 37.0, seed=6)
    print(kind, "finished", flush=True)
    want = _track(world, kind, pri, 4096, 0)
    for few in (0, None):
        print(kind, few, flush=True)
        assert _track(world, kind, pri, 1 << 17, few) == want


def test_parameters_change_while_walks_are_kept(world):
    """The first launch takes all electrons towards the sample (no parameter
    counts in the vacuum) and leaves many on their way; then the mean free
    paths change."""
    dev, mats, grating, _ = world
    n, part = 70000, 30000
    pri = W.raster_scan(100, 100, 7, 250.0, -140.0, 140.0, -140.0, 140.0, 37.0, seed=7)
    tags = np.arange(n, dtype=np.uint32)

    def track(lo, hi, capacity):
        d = A.Driver(dev, capacity, grating, mats, seed=12, steps_per_launch=1)
        d.set_cascade(0)
        d.push(pri[lo:hi], tags[lo:hi], sid_base=lo)
        d.do_iteration(1)
        ended = d.steps()
        for m in (0, 1):
            d.set_material_params(m, el_mfp_scale=1.5, in_mfp_scale=0.75)
        det = d.run(4 * n)
        steps = d.steps()
        d.close()
        return det, steps, ended

    print("finished", flush=True)
    parts = [track(lo, min(lo + part, n), part) for lo in range(0, n, part)]
    assert sum(p[2] for p in parts) == n
    print("kept", flush=True)
    det, steps, ended = track(0, n, 1 << 17)
    assert ended < n // 2                      # the others' walks were kept
    assert steps == sum(p[1] for p in parts)
    assert np.sort(det, order="sid").tobytes() == np.sort(np.concatenate([p[0] for p in parts]), order="sid").tobytes()
