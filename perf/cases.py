"""What a user of this framework has it do, through its public entry points.

A case is one of four kinds of work:

  track   the per-track loop on one track already on the host: upload, begin,
          n_os x (score, sort-reduce-bin), end, and the last oversample's
          (sphere key, lineal energy) pairs read back
  loop    the same loop over a run of tracks (run_plain), one oversample at a
          time or with each track's oversamples queued
  batch   one pass over a resident track library, as a serving or sweep
          program repeats it: run, sync, counts back on the host
  job     what a program with new tracks pays in all: library layout and
          upload, batch set-up, one pass, counts back

Tracks come from the synthetic generator that the benchmark and the tests use
(straight primaries with delta-ray clusters, lognormal energies), with their
point counts fixed by the case (a logarithmic ladder from n_min to n_max) so
that the work does not depend on the seed.  "broad" tracks are dense sheets
of points across the voxel, which the batched form scores on its exact
per-segment path.
"""
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np

import supertrack_amd as st
from supertrack_amd import workloads as W

HISTS = {
    "lin3000": [("lin", 3000, 0.01, 300.0)],
    "log1000": [("log", 1000, 1e-2, 1e3)],
    "both": [("lin", 3000, 0.01, 300.0), ("log", 1000, 1e-2, 1e3)],
}
# (half-length, sphere diameter) in nm of the benchmark's workloads; "mixed"
# cycles through the last three of them, as the mixed-geometry workload does
GEOMETRIES = {
    "2500/10": [(2.5e3, 10.0)],
    "2500/2": [(2.5e3, 2.0)],
    "1000/1": [(1e3, 1.0)],
    "5000/100": [(5e3, 100.0)],
    "mixed": [(1e3, 1.0), (2.5e3, 10.0), (5e3, 100.0)],
}


def _case(name, kind, geometry, hists, n_tracks, n_min, n_max, n_os, precision="f64", queued=False, shift_z=True,
          broad=0):
    c = dict(kind=kind, geometry=geometry, hists=hists, n_tracks=n_tracks, n_min=n_min, n_max=n_max, n_os=n_os,
             precision=precision, queued=queued, shift_z=shift_z, broad=broad)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: one 10 um track, 10 oversamples (the quick check of a macro)
        _case("track-5k", "track", "2500/10", "lin3000", 1, 4901, 4901, 10),
        # a dense track of the drop-in path, beyond the one-workgroup sort
        _case("track-150k-2nm", "track", "2500/2", "log1000", 1, 150001, 150001, 20),
        # the reference's own loop: ordinary tracks, 100 oversamples each, x/y shifts only
        _case("loop-24", "loop", "2500/10", "lin3000", 24, 2000, 10000, 100, shift_z=False),
        # the same loop with the driver's QueueOversamples option
        _case("loop-24-queued", "loop", "2500/10", "lin3000", 24, 2000, 10000, 100, queued=True, shift_z=False),
        # batched double precision, 10 nm spheres, uneven tracks
        _case("batch-f64-10nm", "batch", "2500/10", "log1000", 256, 1000, 1000000, 100),
        # the same library in single precision
        _case("batch-f32-10nm", "batch", "2500/10", "log1000", 256, 1000, 1000000, 100, "f32"),
        # the headline: 2 nm spheres, 1000 oversamples
        _case("batch-f32-2nm", "batch", "2500/2", "log1000", 256, 1000, 1000000, 1000, "f32"),
        # three geometries and two histograms in one pass
        _case("batch-f32-mixed", "batch", "mixed", "both", 96, 1000, 2000000, 1000, "f32"),
        # a small resident library scored again and again (latency)
        _case("batch-f32-small", "batch", "2500/10", "log1000", 16, 1000, 10000, 100, "f32"),
        # a library with tracks of broad, dense sheets next to ordinary ones
        _case("batch-f64-broad", "batch", "2500/10", "lin3000", 16, 2000, 60000, 20, broad=2),
        # new tracks: layout, upload, one pass
        _case("job-f32-2nm", "job", "2500/2", "log1000", 128, 1000, 1000000, 100, "f32"),
        # a small job, double precision
        _case("job-f64-small", "job", "2500/10", "lin3000", 24, 2001, 10001, 100),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["track", "loop", "batch", "batch", "batch", "job"])
    geometry = rng.choice(["2500/10", "2500/2", "1000/1", "5000/100"])
    hists = rng.choice(["lin3000", "log1000"])
    shift_z = rng.random() < 0.7
    if kind == "track":
        n = _log_int(rng, 700, 200000)
        return _case(None, kind, geometry, hists, 1, n, n, rng.randint(1, 25), shift_z=shift_z)
    if kind == "loop":
        return _case(None, kind, geometry, hists, rng.randint(2, 24), _log_int(rng, 500, 3000),
                     _log_int(rng, 3000, 14000), rng.randint(5, 100), queued=rng.random() < 0.5, shift_z=shift_z)
    precision = rng.choice(["f32", "f32", "f64"])
    if rng.random() < 0.25:
        geometry, hists = "mixed", "both"
    n_tracks = _log_int(rng, 3, 200)
    n_max = _log_int(rng, 5000, 1000000)
    n_os = _log_int(rng, 10, 1000 if kind == "batch" else 200)
    broad = 1 if rng.random() < 0.1 and n_os <= 50 else 0
    return _case(None, kind, geometry, hists, n_tracks, _log_int(rng, 300, 3000), n_max, n_os, precision,
                 shift_z=shift_z, broad=broad)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _sizes(case):
    """Point counts: a logarithmic ladder, its rungs spread over the library."""
    t = case["n_tracks"]
    lo, hi = math.log(case["n_min"]), math.log(max(case["n_max"], case["n_min"]))
    if t == 1:
        return [case["n_max"]]
    rungs = [int(round(math.exp(lo + (k + 0.5) / t * (hi - lo)))) for k in range(t)]
    step = next(s for s in range(int(t * 0.618) + 1, 2 * t + 2) if math.gcd(s, t) == 1)
    return [rungs[(k * step + t // 2) % t] for k in range(t)]


def _geom_of_track(case):
    n = len(GEOMETRIES[case["geometry"]])
    chunk = max(1, case["n_tracks"] // (2 * n))
    return ((np.arange(case["n_tracks"]) // chunk) % n).astype(np.int32)


def _one_track(case, seed, k, n, half_length):
    if k < case["broad"]:
        # a sheet of points across the voxel, 40 nm deep, over its first half
        rng = np.random.default_rng([seed, k])
        x = rng.uniform(-half_length, half_length, n)
        y = rng.uniform(-half_length, half_length, n)
        z = -half_length + rng.uniform(-20.0, 20.0, n)
        e = np.clip(15.0 * np.exp(0.8 * rng.standard_normal(n)), 1.0, 1000.0)
        return x, y, z, e
    spec = dict(W.workload("cfg2")["synth"], voxel_half_length=half_length, entry_half_length=half_length,
                p_cluster=0.1, p_cluster_max=0.6, n_min=n, n_max=n, stream_id=(17 + 7919 * int(seed)) & 0xFFFFFFFF)
    return st.synth_library(spec, 1, k)[:4]


def _tracks(case, seed):
    sizes = _sizes(case)
    geoms = GEOMETRIES[case["geometry"]]
    g_of_t = _geom_of_track(case)
    with ThreadPoolExecutor(12) as pool:
        parts = list(pool.map(lambda k: _one_track(case, seed, k, sizes[k], geoms[g_of_t[k]][0]), range(len(sizes))))
    off = np.zeros(len(parts) + 1, np.int64)
    np.cumsum([len(p[0]) for p in parts], out=off[1:])
    x, y, z, e = (np.concatenate([p[a] for p in parts]) for a in range(4))
    return x, y, z, e, off, g_of_t


def _shift_seed(seed):
    return (W.SEED + 1000003 * int(seed)) & 0xFFFFFFFFFFFF


def prepare(case, seed):
    x, y, z, e, off, g_of_t = _tracks(case, seed)
    s = dict(case=case, seed=_shift_seed(seed), geoms=[st.SphericalGeometry(h, d) for h, d in GEOMETRIES[case["geometry"]]],
             hists=[st.Histogram(nb, lo, hi, kind) for kind, nb, lo, hi in HISTS[case["hists"]]])
    kind = case["kind"]
    if kind in ("track", "loop", "job"):
        s["host"] = (x, y, z, e, off, g_of_t)
    if kind == "track":
        s["track"] = st.Track(x, y, z, e)
        s["pairs"] = st.VolumeEdepPair(len(x))
        s["method"] = st.VoxelConstrainedSphereMethod(s["geoms"][0], True, case["shift_z"])
    if kind == "batch":
        s["lib"], s["batch"] = _library_and_batch(s, (x, y, z, e, off, g_of_t))
    return s


def _library_and_batch(s, host):
    case = s["case"]
    x, y, z, e, off, g_of_t = host
    lib = st.TrackLibrary(x, y, z, e, off, s["geoms"], g_of_t, st.ST_F32 if case["precision"] == "f32" else st.ST_F64)
    return lib, st.BatchRun(lib, s["hists"], case["n_os"], s["seed"], True, case["shift_z"])


def _pairs_of(n, keys, lineal):
    """The pairs in arrays of the track's length, zeros after the last."""
    out = {"keys": np.zeros(n, np.int64), "lineal": np.zeros(n)}
    out["keys"][:len(keys)] = keys.view(np.int64)
    out["lineal"][:len(lineal)] = lineal
    return out


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "track":
        x, y, z, e = s["host"][:4]
        track, pairs, method, hist = s["track"], s["pairs"], s["method"], s["hists"][0]
        hist.cpu[:] = 0.0
        track.upload(x, y, z, e)
        method.allocate_track_process(track, s["seed"], 0, case["n_os"])
        hist.allocate_track_process(pairs)
        for _ in range(case["n_os"]):
            method.process_track(track, pairs)
            hist.sort_reduce_and_add_to_histogram(pairs)
        method.free_track_process()
        hist.free_track_process()
        return {"counts": hist.counts(), **_pairs_of(len(x), *pairs.download())}
    if kind == "loop":
        x, y, z, e, off, _ = s["host"]
        hist = s["hists"][0]
        hist.cpu[:] = 0.0
        st.run_plain(x, y, z, e, off, s["geoms"][0], hist, case["n_os"], s["seed"], True, case["shift_z"],
                     queued=case["queued"])
        return {"counts": hist.counts()}
    if kind == "batch":
        b = s["batch"]
        b.run()
        b.sync()
        return [h.fetch(reset=True).view(np.int64) for h in s["hists"]]
    lib, b = _library_and_batch(s, s["host"])
    b.run()
    b.sync()
    counts = [h.fetch(reset=True).view(np.int64) for h in s["hists"]]
    b.free()
    lib.free()
    return counts


def work(case):
    """Each point read once in the form that the kind of work holds it in, each bin written once; per deposit that can
    lie in the voxel (9/16 of the oversamples pass the x/y shift, about half of a track lies inside along z, half of
    that again with z shifts) three shifts, three nearest-centre steps, a squared distance and a sum: about 30
    operations."""
    points = sum(_sizes(case))
    per_point = 32 if case["kind"] != "batch" or case["precision"] == "f64" else 16
    bins = sum(nb for _, nb, _, _ in HISTS[case["hists"]])
    scored = 0.5625 * 0.45 * (0.5 if case["shift_z"] else 1.0)
    out = 8 * bins + (16 * points * scored * 0.5 if case["kind"] == "track" else 0)
    return {"bytes": per_point * points + out, "flops": 30.0 * points * case["n_os"] * scored}


# ---------------------------------------------------------------------------
# the per-track loop in numpy (64 bits)
# ---------------------------------------------------------------------------
def _philox(c0, c1, c2, c3, k0, k1):
    c = [np.asarray(v, np.uint64) for v in np.broadcast_arrays(c0, c1, c2, c3)]
    m = np.uint64(0xFFFFFFFF)
    for _ in range(10):
        p0 = np.uint64(0xD2511F53) * c[0]
        p1 = np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & m, (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & m]
        k0 = (k0 + 0x9E3779B9) & 0xFFFFFFFF
        k1 = (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return c


def _shifts(seed, track, n_os, shift_z, length, half):
    r = _philox(np.arange(n_os, dtype=np.uint64), np.uint64(track), np.uint64(0x53484654), np.uint64(0),
                seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF)
    u = [((v >> np.uint64(8)) + np.uint64(1)).astype(np.float64) / 16777216.0 for v in r[:3]]
    s = [v * length - half for v in u]
    return s[0], s[1], s[2] if shift_z else np.zeros(n_os)


def _edges(kind, nb, lo, hi):
    lo, hi = np.float32(lo), np.float32(hi)
    if kind == "lin":
        return float(lo) + np.arange(nb + 1) * float((hi - lo) / np.float32(nb))
    bo, to = np.float32(np.log10(float(lo))), np.float32(np.log10(float(hi)))
    return 10.0 ** (float(bo) + np.arange(nb + 1) * float((to - bo) / np.float32(nb)))


def exact(case, seed):
    """The counts of the per-track loop, and for one track the last oversample's pairs; the batched kinds return whole
    numbers only."""
    if case["kind"] not in ("track", "loop"):
        return None
    x, y, z, e, off, _ = _tracks(case, seed)
    half, d = GEOMETRIES[case["geometry"]][0]
    n = int(math.floor(2 * half / d))
    length = n * d
    half, r = length / 2, d / 2
    origin = -half + r
    kind, nb, lo, hi = HISTS[case["hists"]][0]
    edges = _edges(kind, nb, lo, hi)
    counts = np.zeros(nb)
    keys = lineal = None
    for t in range(len(off) - 1):
        p = slice(int(off[t]), int(off[t + 1]))
        xt, yt, zt = x[p], y[p], z[p] + half
        lin = e[p] / ((2.0 / 3.0) * d)
        for sx, sy, sz in zip(*_shifts(_shift_seed(seed), t, case["n_os"], case["shift_z"], length, half)):
            if xt.max() + sx <= -half or xt.min() + sx >= half or yt.max() + sy <= -half or yt.min() + sy >= half:
                keys, lineal = np.zeros(0, np.int64), np.zeros(0)
                continue
            a = [xt + sx, yt + sy, zt + sz]
            i = np.nonzero((np.abs(a[0]) < half) & (np.abs(a[1]) < half) & (np.abs(a[2]) < half))[0]
            a = [v[i] - origin for v in a]
            k = [np.rint(v / d) for v in a]
            q = [kk * d - v for kk, v in zip(k, a)]
            hit = ((q[0] * q[0]) + (q[1] * q[1])) + (q[2] * q[2]) <= r * r
            k = [v[hit].astype(np.int64) for v in k]
            keys, lineal = k[0] + k[1] * n + k[2] * n * n, lin[i[hit]]
            sums = np.bincount(np.unique(keys, return_inverse=True)[1], lineal) if len(keys) else np.zeros(0)
            b = np.searchsorted(edges, sums, side="right") - 1
            np.add.at(counts, b[(b >= 0) & (b < nb)], 1.0)
    if case["kind"] == "loop":
        return {"counts": counts}
    return {"counts": counts, **_pairs_of(len(x), keys, lineal)}
