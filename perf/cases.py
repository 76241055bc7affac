"""Timed cases of the electron-tracking path, through its public entry points.

What a user of this library runs: scans of a meshed sample (a slab, a line
grating, an array of contact holes) with primaries of some energy, from a
handful of electrons to a full raster, and what comes back: the detected
electrons' records, per-pixel secondary and backscattered counts, a yield
and its gradient with respect to material parameters, a dose map, or the
counts of several scans tracked together.

A state holds the open device, the uploaded sample and materials and the
driver, as a program does that tracks scan after scan; one pass queues the
primaries and tracks them and their cascades to the end.  Records come in the
order in which electrons happen to arrive, so passes that return records
order them by stream id, as a program does that compares or stores runs.

A trajectory is a chain of hundreds of random choices, each of which a
rounding can turn, so no 64-bit evaluation exists to compare records with:
`exact` has none.
"""
import functools
import math

import numpy as np
import torch

from nebula_amd import api as A
from nebula_amd import grad as G
from nebula_amd import workloads as W

# ------------------------------------------------------------------ cases --
# sample: "slab" (1 um Si, 14 triangles), "grating" (PMMA lines on Si, about
# 2.2e4 triangles at dy = 3.2 nm; `detail` is 10 dy), "holes" (`detail` x
# `detail` contact holes through PMMA on Si).  nx x ny pixels with per_pixel
# primaries each.


def _case(name, kind, sample, energy, nx, ny, per_pixel, capacity, steps, model="penn", detail=0):
    return {"name": name, "kind": kind, "sample": sample, "detail": detail, "model": model, "energy": energy,
            "nx": nx, "ny": ny, "per_pixel": per_pixel, "capacity": capacity, "steps": steps}


def listed():
    return [
        # a first look at a material: a hundred electrons into a flat slab
        _case("beam_100", "records", "slab", 1000.0, 1, 1, 100, 4096, 4),
        # a caller that cannot allocate tracks a few thousand electrons that
        # are on the GPU already
        _case("noalloc_grating", "noalloc", "grating", 300.0, 31, 33, 2, 65536, 4, detail=32),
        # a quick preview of a grating: one electron a pixel, all records kept
        _case("preview_grating", "records", "grating", 500.0, 64, 64, 1, 200000, 4, detail=32),
        # few electrons of high energy, deep cascades: the backscatter
        # coefficient of a bulk sample
        _case("beam_10kev", "tally", "slab", 10000.0, 1, 1, 1003, 200000, 8),
        # an ordinary low-dose image: odd pixel counts, the command line's
        # default capacity
        _case("image_500ev", "tally", "grating", 500.0, 97, 111, 9, 1000000, 4, detail=32),
        # contact holes at 1 keV
        _case("holes_1kev", "tally", "holes", 1000.0, 80, 80, 25, 1000000, 8, detail=8),
        # the other inelastic model on a grating
        _case("kieft_800ev", "frames", "grating", 800.0, 64, 64, 20, 1000000, 6, model="kieft", detail=32),
        # per-pixel yield and its gradient for five material parameters
        _case("yield_gradient", "grad", "grating", 300.0, 64, 64, 61, 1 << 20, 8, detail=32),
        # where the energy goes: deposit records of a small area
        _case("dose_1kev", "deposits", "grating", 1000.0, 16, 16, 8, 65536, 8, detail=32),
        # six scans of uneven size tracked together
        _case("batch_scans", "batch", "mixed", 600.0, 48, 40, 30, 1 << 20, 8, detail=6),
        # a full image: 256 x 256 pixels, 100 electrons each at 300 eV
        _case("scan_full", "tally", "grating", 300.0, 256, 256, 100, 1 << 22, 6, detail=32),
    ]


def _steps_per_primary(energy):
    """Particle-steps of one primary and its cascade, about (615 at 300 eV on
    a grating, 1550 at 1 keV in a slab)."""
    return 615.0 * (energy / 300.0) ** 0.8


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["records", "noalloc", "tally", "tally", "frames", "grad", "deposits", "batch"])
    sample = {"batch": "mixed"}.get(kind) or rng.choice(["slab", "grating", "grating", "holes"])
    energy = round(math.exp(rng.uniform(math.log(250.0), math.log(10000.0))), 1)
    model = rng.choice(["penn", "penn", "kieft"]) if kind in ("tally", "frames", "records") else "penn"
    most = {"records": 20000, "noalloc": 20000, "tally": 3000000, "frames": 1000000, "grad": 300000,
            "deposits": 3000, "batch": 300000}[kind]
    # a drawn pass stays well below the largest listed one
    budget = {"records": 1.5e8, "noalloc": 5e7, "deposits": 8e6, "grad": 2e8}.get(kind, 1.5e9)
    n = min(_log_int(rng, 60, most), max(40, int(budget / _steps_per_primary(energy))))
    per_pixel = max(1, min(n, _log_int(rng, 1, 100)))
    side = max(1, int(math.sqrt(n / per_pixel)))
    nx = max(1, side + rng.randint(-2, 2))
    ny = max(1, int(n / per_pixel / nx))
    capacity = 65536 if kind in ("noalloc", "deposits") else rng.choice([1 << 18, 1000000, 1 << 20])
    detail = {"mixed": rng.randint(2, 8), "holes": rng.choice([4, 6, 8]), "grating": rng.choice([32, 50, 20]),
              "slab": 0}[sample]
    c = _case("", kind, sample, energy, nx, ny, per_pixel, capacity, rng.choice([4, 5, 6, 8]), model, detail)
    del c["name"]
    return c


# ------------------------------------------------------- samples and inputs --
@functools.lru_cache(maxsize=None)
def _device():
    return A.Device(0)


@functools.lru_cache(maxsize=None)
def _materials(model):
    """Si and PMMA, uploaded."""
    dev = _device()
    return [A.Material(dev, A.HostMaterial(W.make_material(s, model))) for s in (W.SI, W.PMMA)]


@functools.lru_cache(maxsize=None)
def _sample(sample, detail):
    """(uploaded geometry, half side of the scanned field, beam start height)."""
    dev = _device()
    if sample == "slab":
        return A.Geometry(dev, W.slab_geometry()), 100.0, 5.0
    if sample == "grating":
        return A.Geometry(dev, W.grating_geometry(dy=detail / 10.0)), 128.0, 37.0
    mesh = W.contact_hole_geometry(detail, detail, layers=((80.0, 1),), n_seg=48, nz=2, radius_sigma=1.0, seed=5)
    return A.Geometry(dev, mesh), 0.8 * 40.0 * detail, 5.0


def _beam(case, seed, half, top, scale=1.0):
    nx, ny = max(1, int(case["nx"] * scale)), max(1, int(case["ny"] * scale))
    if nx * ny == 1:
        half = 0.0
    return W.raster_scan(nx, ny, case["per_pixel"], case["energy"], -half, half, -half, half, top, seed=seed)


def _pinned(dev, pri):
    """The primaries as the 28-byte particles of a push, in page-locked memory."""
    p = dev.host_array(len(pri))
    p["pos"], p["dir"], p["E"] = pri["pos"], pri["dir"], pri["E"]
    return p


def _batch_worlds(case):
    """The samples of a batch: gratings and contact holes in turn, with
    another raster size for each."""
    for i in range(case["detail"]):
        sample, detail = (("grating", 32), ("holes", 4), ("grating", 50), ("holes", 6))[i % 4]
        yield sample, detail, (1.0, 0.35, 1.6, 0.6)[i % 4]


def prepare(case, seed):
    dev = _device()
    kind = case["kind"]
    mats = _materials(case["model"])
    s = {"case": case, "dev": dev, "seed": seed}
    if kind == "batch":
        worlds, pris = [], []
        for i, (sample, detail, scale) in enumerate(_batch_worlds(case)):
            geom, half, top = _sample(sample, detail)
            worlds.append(geom)
            pris.append(_pinned(dev, _beam(case, seed * 64 + i, half, top, scale)))
        d = A.Driver(dev, case["capacity"], worlds[0], mats, seed=seed, steps_per_launch=case["steps"])
        s["worlds"] = [0] + [d.add_world(g, mats) for g in worlds[1:]]
        d.set_graph(True)
        offs = np.concatenate([[0], np.cumsum([len(p) for p in pris])])
        # one image after the other, a bin a pixel
        n = int(offs[-1])
        s.update(driver=d, particles=pris, tags=[np.arange(a, b, dtype=np.uint32) for a, b in zip(offs, offs[1:])],
                 bin=np.arange(n) // case["per_pixel"], bins=n // case["per_pixel"])
        return s
    geom, half, top = _sample(case["sample"], case["detail"])
    pri = _beam(case, seed, half, top)
    n = len(pri)
    s["n"] = n
    if kind == "noalloc":
        s.update(geom=geom, mats=mats, cap=4 * n + 1024,
                 particles=torch.from_numpy(A.to_particles(pri).view(np.float32).reshape(n, 7).copy()).cuda(),
                 out=torch.zeros((4 * n + 1024, 5), dtype=torch.int64, device="cuda"))
        return s
    d = A.Driver(dev, case["capacity"], geom, mats, seed=seed, steps_per_launch=case["steps"])
    s["driver"] = d
    if kind == "grad":
        s["scan"] = G.DifferentiableScan(d, pri, [(0, 0), (0, 1), (1, 0), (1, 1), (1, 2)])
        s["theta"] = s["scan"].theta0()
        return s
    s["particles"] = _pinned(dev, pri)
    s["tags"] = np.arange(n, dtype=np.uint32)
    s["bin"] = pri["py"].astype(np.int64) * case["nx"] + pri["px"]
    s["bins"] = case["nx"] * case["ny"]
    if kind == "deposits":
        d.set_deposits(True)
    return s


# ----------------------------------------------------------------- a pass --
def _records(det, n):
    """Detected electrons by stream id, a plain array for each field of a
    table with room for four a primary (what is not used stays zero)."""
    out = np.zeros(4 * n + 1024, det.dtype)
    out[:len(det)] = det[np.argsort(det["sid"])]
    return {"count": len(det), "pos": out["pos"], "dir": out["dir"], "E": out["E"], "tag": out["tag"].astype(np.int64),
            "sid": out["sid"].view(np.int64)}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "noalloc":
        out = s["out"]
        n, steps = A.track_noalloc(s["dev"], s["geom"], s["mats"], s["particles"].data_ptr(), s["n"],
                                   out.data_ptr(), s["cap"], seed=s["seed"], capacity=case["capacity"],
                                   steps_per_launch=case["steps"])
        # by stream id, in the caller's own table
        out[:n] = out[:n][torch.argsort(out[:n, 4])]
        out[n:] = 0
        return {"records": out, "count": n, "steps": steps}
    d = s["driver"]
    if kind == "grad":
        return {"yield": s["scan"].forward(s["theta"]), "jacobian": s["scan"].jacobian(s["theta"])}
    if kind == "batch":
        for i, p in enumerate(s["particles"]):
            d.push(p, s["tags"][i], sid_base=i << 40, world=s["worlds"][i])
        return d.run_tally(s["bin"], s["bins"], adapt_k=True)
    d.push(s["particles"], s["tags"])
    if kind == "records":
        return _records(d.run(40 * s["n"] + 4096), s["n"])
    if kind == "tally":
        return d.run_tally(s["bin"], s["bins"])
    if kind == "frames":
        image = np.zeros((s["bins"], 2), np.int64)

        def on_records(rec, running, queued):
            b, se = s["bin"][rec["tag"]], rec["E"] < 50.0
            image[:, 0] += np.bincount(b[se], minlength=s["bins"])
            image[:, 1] += np.bincount(b[~se], minlength=s["bins"])

        d.run_frames(16, on_records)
        return image
    det, dep = d.run_with_deposits(0)
    # the dose in 5 nm layers below the tops of the lines, and by primary
    layer = np.clip(((40.0 - dep["pos"][:, 2]) / 5.0).astype(np.int64), 0, 63)
    return {"records": _records(det, s["n"]), "events": np.bincount(dep["tag"], minlength=s["n"]),
            "by_primary": np.bincount(dep["tag"], weights=dep["deposit"], minlength=s["n"]),
            "by_layer": np.bincount(layer, weights=dep["deposit"], minlength=64)}


def exact(case, seed):
    return None


def work(case):
    """A step's arithmetic (two free paths: logarithms, exponentials and two
    table lookups; ray against cell and triangles; a scattering event) is
    about 400 float operations.  Primaries (28 bytes) are read and records
    (40 bytes, about one a primary) written once."""
    scales = [sc for _, _, sc in _batch_worlds(case)] if case["kind"] == "batch" else [1.0]
    n = sum(max(1, int(case["nx"] * sc)) * max(1, int(case["ny"] * sc)) for sc in scales) * case["per_pixel"]
    steps = n * _steps_per_primary(case["energy"]) * (2.0 if case["kind"] == "grad" else 1.0)
    return {"bytes": 68.0 * n + (32.0 * 0.8 * steps if case["kind"] == "deposits" else 0.0), "flops": 400.0 * steps}
