"""Energy-deposit records of few particles: a wave gathers them and writes them
together.  The multiset equals the oracle's bit for bit, also where the
launches stop at the room left for records many times over."""
import numpy as np
import pytest

from nebula_amd import api as A
from nebula_amd import workloads as W
from oracle import pyoracle as O
from tests.helpers import grating_tris, material
from tests.test_gpu_deposits import _sorted_bytes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, energy, capacity", [(1, 300.0, 4096), (21, 800.0, 4096), (65, 500.0, 4096),
                                                 (200, 1000.0, 8192), (260, 600.0, 4096)])
def test_gathered_records_equal_oracle(n, energy, capacity):
    dev = A.Device(0)
    si, pmma = material("si"), material("pmma")
    g = A.Geometry(dev, grating_tris())
    d = A.Driver(dev, capacity, g, [A.Material(dev, A.HostMaterial(m)) for m in (si, pmma)], seed=11,
                 steps_per_launch=8)
    d.set_deposits(True)
    pri = W.raster_scan(1, 1, n, energy, -32.0, 32.0, -32.0, 32.0, 37.0, seed=6)
    d.push(pri, np.arange(n, dtype=np.uint32))
    det, dep = d.run_with_deposits(0)
    det_o, dep_o, _ = O.OracleWorld(grating_tris(), [si, pmma]).run_philox_deposits(pri, 11, 100000, 2000000,
                                                                                    threads=8)
    assert len(det) == len(det_o)
    assert len(dep) == len(dep_o) > 0
    assert np.array_equal(_sorted_bytes(dep), _sorted_bytes(dep_o.astype(dep.dtype)))
