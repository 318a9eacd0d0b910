"""The work that users of this package have it do, as cases to measure.

Every case runs electron transport through the public entry points: the host
API's MonteCarloSS.runPixels (the drop-in for the reference's own loop), the
asynchronous engine (Engine.submit / Engine.result, for images, batches and
request streams) and the allocation-free Engine.run(static=True).  A pass is
one whole call: the jobs go in, their tallies come back to the host.

A job's tallies are integer counts (and sums of whole numbers of fixed-point
units): they depend on the job and its seed alone, not on launch shape, job
mix or scheduling.  They are the outcome of one FP32 random walk per electron,
so there is no 64-bit value of the same outputs to compare with (`exact`).
"""
import json
import math
import os

import numpy as np

from cudamonsel_amd import DATA_DIR, scenes, serving
from cudamonsel_amd.abi import Engine

BEAM_SIGMA_M = 0.5e-9

# electron steps per primary and eV of beam energy (0.8 to 2.3 over the
# materials and geometries here) and arithmetic operations one step cannot do
# without: three elements' cross-sections, the stopping power, one deflection,
# the move, and eight uniforms
STEPS_PER_EV = 1.5
OPS_PER_STEP = 200.0
# one Mott element's tables (61 + 61 x 201 FP32), the part of a scene that is
# read; a scene here holds up to four elements
SCENE_BYTES = 4 * (61 + 61 * 201) * 4


def listed():
    return [
        # the reference's own pattern, one call per pixel of a line scan with
        # 100 primaries (the LinesOnLayers driver): a call's latency is all
        dict(name="pixel_layers_100", kind="pixel", geometry="layers", compat=True, beam_eV=500.0, primaries=100,
             nbins=50),
        # one pixel in a caller that cannot allocate device memory
        dict(name="pixel_static_1500", kind="static", geometry="flat:PMMA", compat=True, beam_eV=300.0,
             primaries=1500, nbins=50),
        # one pixel of a contact hole with the reference's defects corrected
        # (barrier normals are used), an odd count
        dict(name="pixel_hole_fixed_367", kind="pixel", geometry="holes", compat=False, beam_eV=800.0, primaries=367,
             nbins=80),
        # a yield measurement on bulk Si with the tabulated inelastic model
        dict(name="bulk_si_tables_20000", kind="pixel", geometry="flat:Si-dielectric", compat=True, beam_eV=1000.0,
             primaries=20000, nbins=200),
        # the upper end of the yield energies, long cascades in a metal
        dict(name="bulk_cu_tables_3001", kind="pixel", geometry="flat:Cu-dielectric", compat=False, beam_eV=5000.0,
             primaries=3001, nbins=100),
        # the line scan: 128 pixels at 1 nm across one trapezoidal line
        dict(name="scan_line_128x2000", kind="scan", geometry="line", compat=True, beam_eV=500.0, pixels=128,
             per_pixel=2000, nbins=50, jobs=1),
        # a ragged scan over three different lines, defects corrected
        dict(name="scan_lines_fixed_131x517", kind="scan", geometry="lines:3", compat=False, beam_eV=1300.0,
             pixels=131, per_pixel=517, nbins=50, jobs=1),
        # a scan service: several scans on the device at once, on the shipped
        # line-scan tuning
        dict(name="scans_in_flight_4", kind="scan", geometry="line", compat=True, beam_eV=500.0, pixels=128,
             per_pixel=2000, nbins=50, jobs=4),
        # a small image of a contact hole
        dict(name="image_hole_64x275", kind="image", geometry="holes", compat=True, beam_eV=1100.0, side=64,
             per_pixel=275, nbins=50),
        # the SEM image of three seeded lines, the largest single job
        dict(name="image_lines_256x300", kind="image", geometry="lines:3", compat=True, beam_eV=500.0, side=256,
             per_pixel=300, nbins=50),
        # yield jobs of uneven size and energy, submitted together on the
        # shipped batch tuning
        dict(name="batch_512", kind="batch", jobs=512, workload_seed=4),
        # image requests of different sizes and geometries served at once
        dict(name="requests_6", kind="requests", jobs=6, workload_seed=10, sides="32,64,128", max_primaries=6000000),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """One more case over the ranges of the listed ones: beam energies of 0.2
    to 5 keV, 100 to 20,000 primaries for a single pixel, scans of 16 to 256
    pixels, images of 16 to 160 pixels a side, batches of 16 to 360 jobs,
    2 to 8 requests at once; never more electron steps than the largest image."""
    kind = rng.choice(["pixel", "pixel", "static", "scan", "scan", "image", "batch", "requests"])
    if kind in ("pixel", "static"):
        geometry = rng.choice(["layers", "holes", "line", "flat:PMMA", "flat:Si", "flat:Cu", "flat:Si-dielectric",
                               "flat:Cu-dielectric", "step:Si", "step:Cu"])
        return dict(kind=kind, geometry=geometry, compat=rng.random() < 0.5,
                    beam_eV=round(_log_uniform(rng, 200.0, 5000.0), 1), primaries=int(_log_uniform(rng, 100, 20000)),
                    nbins=rng.randrange(20, 201))
    if kind == "scan":
        pixels = int(_log_uniform(rng, 16, 256))
        return dict(kind=kind, geometry=rng.choice(["line", "holes", f"lines:{rng.randrange(100)}"]),
                    compat=rng.random() < 0.5, beam_eV=round(rng.uniform(300.0, 2000.0), 1), pixels=pixels,
                    per_pixel=int(_log_uniform(rng, 50, 2000)), nbins=50, jobs=rng.choice([1, 1, 2, 3, 5]))
    if kind == "image":
        beam_eV = round(rng.uniform(300.0, 2000.0), 1)
        side = int(_log_uniform(rng, 16, 160))
        most = 256 * 256 * 300 * 500.0 / beam_eV / (side * side)
        return dict(kind=kind, geometry=rng.choice(["holes", f"lines:{rng.randrange(100)}"]),
                    compat=rng.random() < 0.5, beam_eV=beam_eV, side=side,
                    per_pixel=max(1, min(int(_log_uniform(rng, 50, 500)), int(most))), nbins=50)
    if kind == "batch":
        return dict(kind=kind, jobs=int(_log_uniform(rng, 16, 360)), workload_seed=rng.randrange(1000))
    return dict(kind=kind, jobs=rng.randrange(2, 9), workload_seed=rng.randrange(1000), sides="32,64",
                max_primaries=3000000)


def _scene(geometry, compat, beam_eV):
    name, _, arg = geometry.partition(":")
    if name == "layers":
        return scenes.lines_on_layers(beam_eV=beam_eV, compat=compat)
    if name == "line":
        return scenes.line_on_substrate(beam_eV=beam_eV, compat=compat)
    if name == "lines":
        return scenes.random_lines(seed=int(arg), beam_eV=beam_eV, compat=compat)
    if name == "holes":
        return scenes.contact_holes(beam_eV=beam_eV, compat=compat)
    if name == "step":
        return scenes.step_edge(arg, beam_eV=beam_eV, compat=compat)
    return scenes.flat(arg, beam_eV=beam_eV, compat=compat)


def _workload(case):
    """The jobs of a batch or the image requests of a stream."""
    if case["kind"] == "batch":
        return serving.batch_workload(case["jobs"], seed=case["workload_seed"])
    sides = [int(s) for s in case["sides"].split(",")]
    reqs = serving.request_stream(rate_per_s=100.0, duration_s=1.0, seed=case["workload_seed"], sides=sides)
    keep, total = [], 0
    for r in reqs:
        if len(keep) < case["jobs"] and total + r.primaries <= case["max_primaries"]:
            keep.append(r)
            total += r.primaries
    return keep


# A program keeps one engine per tuning for as long as it runs.
_engines = {}


def _engine(tuning=""):
    if tuning not in _engines:
        kw = dict(admission_order=1) if tuning == "serving" else {}
        if tuning in ("linescan", "batch"):
            kw = json.load(open(os.path.join(DATA_DIR, f"tuning_{tuning}.json")))["tuning"]
        _engines[tuning] = Engine(**kw)
    return _engines[tuning]


def prepare(case, seed):
    """The scene (built with the reference's classes, uploaded where the
    engine is used), the beam positions and the job's seed."""
    rng = np.random.default_rng(seed)
    job_seed = int(rng.integers(1, 2 ** 62))
    offset_nm = rng.uniform(-0.5, 0.5, 2)
    kind = case["kind"]
    st = dict(kind=kind)
    if kind in ("batch", "requests"):
        eng = _engine("batch" if kind == "batch" else "serving")
        cache = serving.SceneCache(eng)
        jobs = []
        for k, j in enumerate(_workload(case)):
            if kind == "batch":
                sc, _, sid = serving._yield_scene(cache, j)
                jobs.append((sid, np.array([[0.0, 0.0, sc.beam_z]]), j.primaries, j.beam_eV, job_seed + k, 50))
            else:
                sc, _, sid = serving._request_scene(cache, j)
                cen = serving.raster_centers(j.side, sc.beam_z)
                cen[:, :2] += offset_nm * 1e-9
                jobs.append((sid, cen, j.per_pixel, j.beam_eV, job_seed + k, 50))
        st.update(engine=eng, cache=cache, jobs=jobs)
        return st
    sc = _scene(case["geometry"], case["compat"], case["beam_eV"])
    if kind in ("pixel", "static"):
        centers, per = np.array([[0.0, 0.0, sc.beam_z]]), case["primaries"]
    elif kind == "scan":
        xs = np.arange(case["pixels"]) - case["pixels"] // 2
        centers, per = scenes.scan_centers(xs, [0.0], sc.beam_z), case["per_pixel"]
    else:
        centers, per = serving.raster_centers(case["side"], sc.beam_z), case["per_pixel"]
    centers[:, :2] += offset_nm * 1e-9
    st.update(scene=sc, centers=centers, per=per, nbins=case["nbins"], beam_eV=case["beam_eV"], seed=job_seed)
    if kind == "pixel" or (kind == "scan" and case["jobs"] == 1):
        st["kind"] = "host"
        sc.monte.setSeed(job_seed)
        return st
    eng = _engine("linescan" if kind == "scan" else "")
    cs = sc.monte.compileScene()
    sid = eng.upload(cs)
    st.update(engine=eng, compiled=cs, sid=sid)
    if kind != "static":
        st["jobs"] = [(sid, centers, per, case["beam_eV"], job_seed + k, case["nbins"])
                      for k in range(case.get("jobs", 1))]
    return st


_COUNTS = ("primaries", "electrons", "steps", "escapes", "watchdog_drops", "queue_overflow")


def _tallies(r):
    """A job's tallies and its counters (not its timings)."""
    out = {k: v for k, v in r.items() if k != "stats"}
    out.update({k: r["stats"][k] for k in _COUNTS})
    return out


def run(state):
    if state["kind"] == "host":
        r = state["scene"].monte.runPixels(state["centers"], state["per"], state["nbins"], 50.0)
        out = dict(back=r.back, fwd=r.fwd, se=r.se, se_sq=r.seSq, bse_sq=r.bseSq, back_energy=r.backEnergy,
                   back_energy_hist=r.backEnergyHist, fwd_energy_hist=r.fwdEnergyHist,
                   elevation_hist=r.elevationHist, azimuth_hist=r.azimuthHist)
        out.update({k: getattr(r.stats, k) for k in _COUNTS})
        return out
    eng = state["engine"]
    if state["kind"] == "static":
        return _tallies(eng.run(state["sid"], state["centers"], state["per"], state["beam_eV"], BEAM_SIGMA_M,
                                state["seed"], nbins=state["nbins"], static=True))
    ids = [eng.submit(sid, cen, per, beam_eV, BEAM_SIGMA_M, seed, nbins=nbins)
           for sid, cen, per, beam_eV, seed, nbins in state["jobs"]]
    results = [_tallies(eng.result(i)) for i in ids]
    return {k: np.concatenate([np.atleast_1d(r[k]) for r in results]) for k in results[0]}


def work(case):
    """Beam positions in, tallies out (6 sums of 8 bytes per pixel and the
    histograms) and one read of the scene; the electron steps' arithmetic."""
    kind = case["kind"]
    if kind == "batch":
        jobs = [(1, j.primaries, j.beam_eV, 50) for j in _workload(case)]
    elif kind == "requests":
        jobs = [(r.side * r.side, r.primaries, r.beam_eV, 50) for r in _workload(case)]
    else:
        if kind in ("pixel", "static"):
            px, prim = 1, case["primaries"]
        else:
            px = case["pixels"] if kind == "scan" else case["side"] ** 2
            prim = px * case["per_pixel"]
        jobs = [(px, prim, case["beam_eV"], case["nbins"])] * case.get("jobs", 1)
    nbytes = SCENE_BYTES + sum(px * (24 + 48) + 8 * (2 * (nb + 2) + 182 + 362) for px, _, _, nb in jobs)
    flops = sum(prim * eV * STEPS_PER_EV * OPS_PER_STEP for _, prim, eV, _ in jobs)
    return {"bytes": float(nbytes), "flops": float(flops)}


def exact(case, seed):
    """None: the outputs are counts of one pseudo-random FP32 walk (see the
    module's description), for which there is no 64-bit value."""
    return None
