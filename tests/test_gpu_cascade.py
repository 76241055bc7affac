"""Launches with few particles in flight (k_cascade: waves keep their
particles and secondaries) against the oracle: records and step counts, bit
for bit, at populations around the edges of a wave, of the waves a launch
spreads particles over, and with a particle buffer too small for them."""
import numpy as np
import pytest

from nebula_amd import api as A
from nebula_amd import workloads as W
from oracle import pyoracle as O
from tests.helpers import grating_tris, material, slab_tris

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def world():
    dev = A.Device(0)
    raw = [material("si"), material("pmma")]
    mats = [A.Material(dev, A.HostMaterial(m)) for m in raw]
    tris = {"grating": grating_tris(), "slab": slab_tris()}
    return dev, mats, {k: A.Geometry(dev, t) for k, t in tris.items()}, \
        {k: O.OracleWorld(t, raw) for k, t in tris.items()}


@pytest.mark.parametrize("sample,energy,n,capacity", [
    ("grating", 300.0, 1, 64), ("grating", 300.0, 63, 4096), ("grating", 300.0, 64, 64), ("grating", 300.0, 65, 64),
    ("grating", 300.0, 2048, 65536), ("grating", 300.0, 2049, 65536), ("grating", 300.0, 4097, 4096),
    ("slab", 4000.0, 7, 4096), ("slab", 4000.0, 130, 64)])
def test_few_particles_equal_oracle(world, sample, energy, n, capacity):
    dev, mats, geoms, oracles = world
    pri = W.raster_scan(n, 1, 1, energy, -60.0, 60.0, -60.0, 60.0, 37.0 if sample == "grating" else 5.0, seed=n)
    print(sample, energy, n, capacity, flush=True)
    d = A.Driver(dev, capacity, geoms[sample], mats, seed=3, steps_per_launch=5)
    tags = np.arange(n, dtype=np.uint32)
    d.push(pri, tags, sid_base=9)
    det = d.run(100 * n + 100)
    ref, steps = oracles[sample].run_philox(pri, 3, 100 * n + 100, threads=8, sid_base=9)
    assert d.steps() == steps
    assert np.sort(det, order="sid").tobytes() == np.sort(ref.astype(det.dtype), order="sid").tobytes()
    # the same through iterations of the caller's own
    d.push(pri, tags, sid_base=9)
    got = []
    while True:
        d.do_iteration(1)
        running, found, queued = d.counts()
        if found:
            got.append(d.flush_detected())
        if running == 0 and queued == 0:
            break
    assert d.steps() == 2 * steps
    assert np.sort(np.concatenate(got or [det[:0]]), order="sid").tobytes() == np.sort(det, order="sid").tobytes()
    d.close()


@pytest.mark.parametrize("few", [0, 500])
@pytest.mark.parametrize("kind", ["plain", "scores", "deposits", "worlds"])
def test_both_routes_give_the_same(world, kind, few):
    """Populations that grow past `few` and shrink below it again change
    route on the way; 0 keeps them in k_step and k_inel."""
    dev, mats, geoms, _ = world
    pri = W.raster_scan(20, 20, 1, 700.0, -60.0, 60.0, -60.0, 60.0, 37.0, seed=5)
    tags = np.arange(len(pri), dtype=np.uint32)

    def track(limit):
        d = A.Driver(dev, 2048, geoms["grating"], mats, seed=11, steps_per_launch=6)
        if limit is not None:
            d.set_cascade(limit)
        if kind == "worlds":
            d.push(pri[:150], tags[:150], sid_base=1 << 40, world=d.add_world(geoms["slab"], mats))
        if kind == "scores":
            d.set_score_params([(0, 0), (0, 1), (1, 1), (1, 2)])
        if kind == "deposits":
            d.set_deposits(True)
        d.push(pri, tags)
        if kind == "scores":
            det, more = d.run_scores(20000)
            order = np.argsort(det["sid"])
            more = more[order].tobytes()
        elif kind == "deposits":
            det, dep = d.run_with_deposits(20000)
            more = np.sort(dep.view(np.dtype((np.void, dep.dtype.itemsize)))).tobytes()
        else:
            det, more = d.run(20000), b""
        steps = d.steps()
        d.close()
        return np.sort(det, order="sid").tobytes(), more, steps

    assert track(few) == track(None)


@pytest.mark.parametrize("few", [0, None])
def test_walks_kept_between_launches(world, few):
    """With many particles in flight a launch leaves unfinished walks to the
    next one: records and step counts equal the oracle's."""
    dev, mats, geoms, oracles = world
    n = 70000
    pri = W.raster_scan(100, 100, 7, 260.0, -140.0, 140.0, -140.0, 140.0, 37.0, seed=6)
    d = A.Driver(dev, 1 << 18, geoms["grating"], mats, seed=21, steps_per_launch=3)
    if few is not None:
        d.set_cascade(few)
    d.push(pri, np.arange(n, dtype=np.uint32), sid_base=5)
    det = d.run(4 * n)
    ref, steps = oracles["grating"].run_philox(pri, 21, 4 * n, threads=16, sid_base=5)
    assert d.steps() == steps
    assert np.sort(det, order="sid").tobytes() == np.sort(ref.astype(det.dtype), order="sid").tobytes()
    d.close()
