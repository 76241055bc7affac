"""The short quotients, roots and logarithms of a step where their operands
leave the range they are short for (direction components that are zero, tiny or
denormal, directions that are not unit vectors, energies from denormal to
10^30 eV, table look-ups beyond their ends): the events and paths of the oracle,
bit for bit."""
import numpy as np
import pytest

from nebula_amd import api as A
from nebula_amd import workloads as W
from oracle import pyoracle as O
from tests.helpers import material, slab_tris
from tests.test_gpu_parity import _to_oracle_states

pytestmark = pytest.mark.gpu

SMALL = np.array([0.0, -0.0, 1e-45, -1e-38, 1e-30, -1e-20, 1e-16, -3e-8, 0.3, -0.7, 1.0], np.float32)


@pytest.mark.parametrize("model", ["penn", "kieft"])
@pytest.mark.parametrize("scale", [1.0, 1e-12, 3e4])
def test_steps_off_the_usual_range(model, scale):
    dev = A.Device(0)
    tris, raw = slab_tris(), [material("si", model), material("pmma", model)]
    d = A.Driver(dev, 64, A.Geometry(dev, tris), [A.Material(dev, A.HostMaterial(m)) for m in raw], seed=5)
    ow = O.OracleWorld(tris, raw)
    rng = np.random.default_rng(3)
    n = 8001
    st = np.zeros(n, A.STATE_DTYPE)
    st["pos"] = rng.uniform(-40.0, 40.0, (n, 3)).astype(np.float32)
    st["pos"][:, 2] = -rng.uniform(0.01, 50.0, n)
    for a in range(3):
        st["dir"][:, a] = SMALL[rng.integers(0, len(SMALL), n)] * np.float32(scale)
    zero = ~np.any(np.abs(st["dir"]) > 1e-18, axis=1)
    st["dir"][zero, 2] = -1.0      # a direction all of whose squares vanish has no normal
    st["E"] = np.exp(rng.uniform(np.log(12.0), np.log(2e4), n)).astype(np.float32)
    st["E"][::97] = np.float32(1e30)
    st["E"][1::97] = np.float32(1e-40)
    st["mat"] = rng.choice(np.array([-123, 0, 1], np.int32), n)
    st["last_tri"] = -1
    st["sid"] = np.arange(n)
    print(model, scale, flush=True)
    g_st, g_ev, g_oc, _, g_made = d.step_states(st)
    o_st, o_ev, o_oc, _, o_made = ow.step_states(_to_oracle_states(st), 5)
    assert np.array_equal(g_ev, o_ev)
    assert np.array_equal(g_oc, o_oc)
    assert np.array_equal(g_made, o_made)
    for k in ("pos", "dir", "E"):
        a, b = g_st[k].reshape(n, -1), o_st[k].reshape(n, -1)
        same = (a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))
        assert same.all(), (k, int((~same).any(axis=1).sum()))
    dev.close()


@pytest.mark.parametrize("scale", [1.0, 1e-12, 3e4])
@pytest.mark.parametrize("few", [0, None])
def test_tracks_off_the_usual_range(scale, few):
    """Primaries of such directions and energies through the step kernels."""
    dev = A.Device(0)
    tris, raw = slab_tris(), [material("si"), material("pmma")]
    ow = O.OracleWorld(tris, raw)
    d = A.Driver(dev, 4096, A.Geometry(dev, tris), [A.Material(dev, A.HostMaterial(m)) for m in raw], seed=7)
    if few is not None:
        d.set_cascade(few)
    rng = np.random.default_rng(4)
    n = 700
    pri = W.raster_scan(n, 1, 1, 300.0, -60.0, 60.0, -60.0, 60.0, 5.0, seed=1)
    for a in range(3):
        pri["dir"][:, a] = SMALL[rng.integers(0, len(SMALL), n)] * np.float32(scale)
    pri["dir"][:, 2] = -np.abs(pri["dir"][:, 2])
    zero = ~np.any(np.abs(pri["dir"]) > 1e-18, axis=1)
    pri["dir"][zero, 2] = -1.0
    pri["E"] = np.exp(rng.uniform(np.log(12.0), np.log(900.0), n)).astype(np.float32)
    pri["E"][::53] = np.float32(1e-40)
    pri["E"][1::53] = np.float32(1.0)
    tags = np.arange(n, dtype=np.uint32)
    print(scale, few, flush=True)
    d.push(pri, tags)
    det = np.sort(d.run(100 * n), order="sid")
    ref, steps = ow.run_philox(pri, 7, 100 * n, threads=8)
    ref = np.sort(ref.astype(det.dtype), order="sid")
    assert d.steps() == steps
    assert len(det) == len(ref) > n // 10
    for k in ("pos", "dir", "E"):
        a, b = det[k].reshape(len(det), -1), ref[k].reshape(len(ref), -1)
        same = (a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))
        assert same.all(), (k, int((~same).any(axis=1).sum()))
    dev.close()
