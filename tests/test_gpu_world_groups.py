"""Grouping of a launch's particles by world at the numbers of worlds where its
kernels change: a wave's lanes, the worlds counted in LDS (1024) and one more,
with enough particles for every block to have some.  All worlds are the same,
so the records equal those of one world, stream id for stream id."""
import numpy as np
import pytest

from nebula_amd import api as A
from nebula_amd import workloads as W
from tests.helpers import material, slab_tris

pytestmark = pytest.mark.gpu

N = 24000


@pytest.fixture(scope="module")
def setup():
    dev = A.Device(0)
    g = A.Geometry(dev, slab_tris())
    m = [A.Material(dev, A.HostMaterial(material("si")))]
    pri = W.raster_scan(N, 1, 1, 300.0, -60.0, 60.0, -60.0, 60.0, 5.0, seed=3)
    d = A.Driver(dev, 65536, g, m, seed=5, steps_per_launch=4)
    d.push(pri, np.arange(N, dtype=np.uint32))
    ref = np.sort(d.run(40 * N), order="sid").tobytes()
    d.close()
    return dev, g, m, pri, ref


@pytest.mark.parametrize("worlds", [2, 63, 65, 1023, 1024, 1025])
@pytest.mark.parametrize("few", [0, None])
def test_grouped_equals_one_world(setup, worlds, few):
    dev, g, m, pri, ref = setup
    d = A.Driver(dev, 65536, g, m, seed=5, steps_per_launch=4)
    if few is not None:
        d.set_cascade(few)
    ids = [0] + [d.add_world(g, m) for _ in range(worlds - 1)]
    # uneven shares, some worlds without particles
    cuts = np.sort(np.random.default_rng(worlds).integers(0, N + 1, worlds - 1))
    cuts = np.concatenate([[0], cuts, [N]])
    tags = np.arange(N, dtype=np.uint32)
    print(worlds, few, flush=True)
    for w, a, b in zip(ids, cuts, cuts[1:]):
        if b > a:
            d.push(pri[a:b], tags[a:b], sid_base=int(a), world=w)
    assert np.sort(d.run(40 * N), order="sid").tobytes() == ref
    d.close()
