"""Driver.run_tally on the GPU and on the host against numpy's bincount of the
records that Driver.run returns: bins that a block counts in LDS (2048 at most)
and that it does not, types and strides of the table, cutoffs that a record's
energy meets exactly, a table that is too long for the GPU route, and tables
that name no bin for a record."""
import numpy as np
import pytest

from nebula_amd import _lib, api as A
from nebula_amd import workloads as W
from tests.helpers import grating_tris, material

pytestmark = pytest.mark.gpu

N = 3000


@pytest.fixture(scope="module")
def setup():
    dev = A.Device(0)
    d = A.Driver(dev, 4096, A.Geometry(dev, grating_tris()),
                 [A.Material(dev, A.HostMaterial(material(m))) for m in ("si", "pmma")], seed=4)
    pri = W.raster_scan(N, 1, 1, 400.0, -60.0, 60.0, -60.0, 60.0, 37.0, seed=2)
    tags = np.arange(N, dtype=np.uint32)
    d.push(pri, tags)
    rec = d.run(40 * N)
    assert len(rec) > N // 4
    return d, pri, tags, rec


def _want(rec, table, n_bins, cutoff):
    b, se = table[rec["tag"]], rec["E"] < cutoff
    return np.stack([np.bincount(b[se], minlength=n_bins), np.bincount(b[~se], minlength=n_bins)], axis=1)


@pytest.mark.parametrize("n_bins,dtype,stride", [
    (1, np.int64, 1), (6, np.int32, 1), (2047, np.uint16, 1), (2048, np.int64, 1), (2049, np.int64, 2),
    (3000, np.uint32, 1), (200000, np.int64, 1)])
@pytest.mark.parametrize("long", [False, True])
def test_tally_equals_bincount(setup, n_bins, dtype, stride, long):
    d, pri, tags, rec = setup
    rng = np.random.default_rng(n_bins)
    size = N + (4 * N + 65536 if long else 0)
    table = rng.integers(0, n_bins, stride * size).astype(dtype)[::stride]
    on_energy = rec["E"][len(rec) // 2]
    for cutoff in (50.0, on_energy, float(on_energy), np.float64(on_energy) + 1e-9, 0):
        d.push(pri, tags)
        got = d.run_tally(table, n_bins, frame=4, se_cutoff=cutoff)
        assert np.array_equal(got, _want(rec, table, n_bins, cutoff)), (n_bins, dtype, cutoff)


@pytest.mark.parametrize("what,error", [("tag", IndexError), ("bin", ValueError), ("negative", ValueError)])
def test_tally_refuses_records_without_a_bin(setup, what, error):
    d, pri, tags, rec = setup
    last = int(rec["tag"].max())
    table = np.zeros(N if what != "tag" else last, np.int64)
    if what != "tag":
        table[last] = 5 if what == "bin" else -1
    d.push(pri, tags)
    with pytest.raises(error):
        d.run_tally(table, 5)
    # and the driver goes on
    while d.counts()[0] or d.counts()[2]:
        d.do_iteration(4)
    d.flush_detected()
    d.push(pri, tags)
    assert d.run_tally(np.zeros(N, np.int64), 1).sum() == len(rec)


def test_tally_of_no_bins():
    """No bins are enough for a beam of which nothing is detected (on a new
    driver, whose tally has no memory yet); a detected record has none."""
    dev = A.Device(0)
    mats = [A.Material(dev, A.HostMaterial(material(m))) for m in ("si", "pmma")]
    d = A.Driver(dev, 4096, A.Geometry(dev, grating_tris()), mats, seed=4)
    pri = W.raster_scan(50, 1, 1, 400.0, -60.0, 60.0, -60.0, 60.0, 37.0, seed=2)
    tags = np.arange(len(pri), dtype=np.uint32)
    out = pri.copy()
    out["pos"][:, 2] = 1e6             # outside the domain: ended by their first step
    for _ in range(2):
        d.push(out, tags)
        assert d.run_tally(np.zeros(len(pri), np.int64), 0).shape == (0, 2)
    d.push(pri, tags)
    with pytest.raises(ValueError):
        d.run_tally(np.zeros(len(pri), np.int64), 0)
    d.push(pri, tags)
    assert d.run_tally(np.zeros(len(pri), np.int64), 1).sum() > 0
    d.close()


def test_tally_without_memory_for_it_is_done_on_the_host(setup, monkeypatch):
    d, pri, tags, rec = setup
    monkeypatch.setattr(A.lib(), "nbl_driver_tally_begin", lambda *a: _lib.NBL_ERR_ALLOC)
    table = np.arange(N) % 5
    d.push(pri, tags)
    assert np.array_equal(d.run_tally(table, 5), _want(rec, table, 5, 50.0))
