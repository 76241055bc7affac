"""Launches in which no walk ends of itself, and launches that run far more
steps than they were asked for: what the checks for a run without progress and
the callers that count iterations make of them."""
import numpy as np
import pytest

from nebula_amd import api as A
from nebula_amd import workloads as W
from oracle import pyoracle as O
from tests.helpers import grating_tris, material

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def world():
    dev = A.Device(0)
    raw = [material("si"), material("pmma")]
    return dev, [A.Material(dev, A.HostMaterial(m)) for m in raw], A.Geometry(dev, grating_tris()), \
        O.OracleWorld(grating_tris(), raw)


def _spot(n, x, y):
    pri = W.pencil_beam(n, 120.0, 37.0)
    pri["pos"][:, 0], pri["pos"][:, 1] = x, y
    return pri


def _equal(det, ref):
    return np.sort(det, order="sid").tobytes() == np.sort(ref.astype(det.dtype), order="sid").tobytes()


@pytest.mark.parametrize("x,y", [(0.3, 5.7), (-32.2, 1.9), (0.1, -20.3)])
@pytest.mark.parametrize("tally", [False, True])
def test_a_first_flight_of_many_cells_is_progress(world, x, y, tally):
    """70 000 electrons that all start in one point and cross the cells of a
    trench together, a step a launch and a launch a frame."""
    dev, mats, geom, oracle = world
    n = 70000
    pri = _spot(n, x, y)
    print(x, y, tally, flush=True)
    d = A.Driver(dev, 1 << 17, geom, mats, seed=8, steps_per_launch=1)
    d.set_cascade(0)
    d.push(pri, np.arange(n, dtype=np.uint32))
    ref, steps = oracle.run_philox(pri, 8, 4 * n, threads=16)
    if tally:
        got = d.run_tally(np.arange(n) % 7, 7, frame=1)
        assert np.array_equal(got.sum(axis=1), np.bincount(ref["tag"] % 7, minlength=7))
    else:
        rec = []
        d.run_frames(1, lambda r, running, queued: rec.append(r))
        assert _equal(np.concatenate(rec), ref)
    assert d.steps() == steps
    d.close()


def _frames(launches, first, most):
    """The frames of `launches` iterations, of `first` growing to `most`."""
    out = []
    while launches > 0:
        out.append(min(first, most))
        launches -= out[-1]
        first *= 2
    return out if launches == 0 else None


@pytest.mark.parametrize("why", ["off", "deposits"])
@pytest.mark.parametrize("entry", ["tally", "run"])
def test_frames_stay_long_where_launches_are_short(world, why, entry):
    """A frame is cut to two iterations where these run many steps each, and
    not where the caller, or deposits, keep them at steps_per_launch."""
    dev, mats, geom, _ = world
    n = 2000
    pri = W.raster_scan(n, 1, 1, 300.0, -60.0, 60.0, -60.0, 60.0, 37.0, seed=2)
    print(why, entry, flush=True)
    d = A.Driver(dev, 4096, geom, mats, seed=8, steps_per_launch=4)
    d.set_timing(True)
    if why == "deposits":
        d.set_deposits(True)
    else:
        d.set_cascade(0)
    d.push(pri, np.arange(n, dtype=np.uint32))
    if entry == "tally":
        d.run_tally(np.zeros(n, np.int64), 1, frame=32)
        launches = d.timing()[1]
        assert launches == 32 * sum(d.k_frames.values())
    else:
        d.run(40 * n)
        launches = d.timing()[1]
        assert _frames(launches, 4, 32), launches
    assert launches > 28
    d.close()


def test_the_tuner_measures_short_launches(world):
    """All electrons fly after the first trial, which ends the search: two
    trials of one launch of four steps."""
    dev, mats, geom, oracle = world
    n = 3000
    pri = W.raster_scan(n, 1, 1, 300.0, -60.0, 60.0, -60.0, 60.0, 37.0, seed=3)
    d = A.Driver(dev, 4096, geom, mats, seed=9, steps_per_launch=4)
    d.push(pri, np.arange(n, dtype=np.uint32))
    assert d.autotune(iters_per_trial=1)["trials"] == 2
    assert n <= d.steps() <= 2 * 4 * d.info()["slots"]
    det = d.run(40 * n)
    ref, steps = oracle.run_philox(pri, 9, 40 * n, threads=8)
    assert _equal(det, ref) and d.steps() == steps
    d.close()
