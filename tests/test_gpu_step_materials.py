"""Materials as the step kernels keep them (a copy in LDS, the two mean free
path tables side by side where they share their energies): tables with energies
of their own, one and several materials, the most that LDS holds (64) and one
more (the general kernels read them from global memory), with scores, deposits
and several worlds, against the oracle or the plain driver, bit for bit."""
import copy

import numpy as np
import pytest

from nebula_amd import api as A
from nebula_amd import workloads as W
from oracle import pyoracle as O
from tests.helpers import grating_tris

pytestmark = pytest.mark.gpu


def _mixed(spec, model="penn"):
    """Elastic tables on another energy grid than the inelastic ones."""
    raw = copy.copy(W.make_material(spec, model))
    other = W.make_material(spec, model, nK=77, Kmin=7.0)
    raw.datasets = {k: (other if k.startswith("/elastic") else raw).datasets[k] for k in raw.datasets}
    return raw


def _raws(kind, n):
    two = [_mixed(W.SI), _mixed(W.PMMA)] if kind == "mixed" else \
        [W.make_material(W.SI), _mixed(W.PMMA)] if kind == "one_mixed" else \
        [W.make_material(W.SI), W.make_material(W.PMMA)]
    return two + [two[0]] * (n - 2)


@pytest.mark.parametrize("few", [0, 100000])
@pytest.mark.parametrize("kind,n", [("plain", 3), ("mixed", 2), ("one_mixed", 2), ("plain", 64), ("mixed", 65)])
def test_materials_equal_oracle(kind, n, few):
    dev = A.Device(0)
    raws = _raws(kind, n)
    uploaded = {id(r): A.Material(dev, A.HostMaterial(r)) for r in raws}
    mats = [uploaded[id(r)] for r in raws]
    tris = grating_tris()
    geom = A.Geometry(dev, tris)
    d = A.Driver(dev, 4096, geom, mats, seed=11, steps_per_launch=5)
    d.set_cascade(few)
    m = 300
    pri = W.raster_scan(m, 1, 1, 500.0, -60.0, 60.0, -60.0, 60.0, 37.0, seed=6)
    tags = np.arange(m, dtype=np.uint32)
    print(kind, n, few, flush=True)
    d.push(pri, tags)
    det = np.sort(d.run(100 * m), order="sid")
    ref, steps = O.OracleWorld(tris, raws).run_philox(pri, 11, 100 * m, threads=8)
    assert d.steps() == steps
    assert det.tobytes() == np.sort(ref.astype(det.dtype), order="sid").tobytes()
    # the same electrons with scores, with deposits and in a second world
    d.set_score_params([(0, 0), (1, 1)])
    d.push(pri, tags)
    scored, _ = d.run_scores(100 * m)
    assert np.sort(scored, order="sid").tobytes() == det.tobytes()
    d.set_score_params([])
    d.set_deposits(True)
    d.push(pri, tags)
    with_dep, _ = d.run_with_deposits(0)
    assert np.sort(with_dep, order="sid").tobytes() == det.tobytes()
    d.set_deposits(False)
    w = d.add_world(geom, mats)
    d.push(pri, tags, world=w)
    assert np.sort(d.run(100 * m), order="sid").tobytes() == det.tobytes()
    dev.close()
