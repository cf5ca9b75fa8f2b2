"""Benchmark of the MI355X spectral path tracer on the 1080p mixed-material terrain scene.

Workload: benchmark configuration 2 -- 1920x1080, max depth 16, a 1000 x 500 fBm terrain
(997 002 triangles) with 200 level-4 icospheres (1 024 000 triangles; 40% Lambertian, 30% rough
anisotropic GGX conductors, 30% rough BK7 with Sellmeier dispersion) and 64 blackbody quad lights
sampled through the light BVH. Synthetic, seeded scene generated by the host library.

A step is one call of the plugin's render entry point: `--spp-per-step` passes over the whole
image (camera rays -> wavefront bounces -> film), accumulated into the FP64 film resident in HBM.
The default, 16 spp (33.2 M camera samples), is one batch at the plugin's default queue capacity
of 32 M paths in flight; the configuration's 1024 spp are 64 such steps (the host batch loop grows
its calls further, doubling them while a call takes under 0.15 s). The value is camera samples per
second over exactly --steps timed steps (Msamples/s).

Prints one JSON line. `roofline` covers the dominant kernel of the timed steps, its duration
measured with HIP events on the plugin's own stream; `cpu_baseline` times the oracle (the C++
restatement of the reference CPU path tracer) on this host's cores over a bounded sample;
`relmse` is the metric's second part: equal-time relMSE of the guided and the plain path tracer
on the indoor configuration at the same resolution, against a high-spp plain reference.
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "ar-renderer_amd"))

HBM_PEAK_GBS = 8000.0  # MI355X HBM3E
# HBM bytes per launch of the traversal, from rocprofv3 FETCH_SIZE / WRITE_SIZE counter runs scaled by a
# copy kernel of known size, and its VALU issue and lane counters; written by hand from the runs. They are
# of the kernels as they were then: a change to the traversal takes new runs.
TRAFFIC_FILE = os.path.join(ROOT, "profiles", "trace_bounce_terrain_1080p_traffic.md")
METRIC = "Msamples/s and equal-time relMSE, guided vs plain PT, 1080p on one MI355X"


NODE_READ = 80  # bytes of a wide node that the traversal loads; its line in memory has stats["nodeBytes"]


def kernel_bytes(name, stats, items, fused=False):
    """Algorithmic HBM bytes of one kind of launch, from its item count and the traversal counters.

    intersect: per ray 32 B ray in (origin, direction) + 4 B queue entry + 16 B hit out, plus
      the bytes of the wide nodes fetched and of the leaf records tested.
    shadow: per shadow ray a 48 B record in and 32 B radiance read-modify-write in the fused launch;
      with media or interfaces 80 B record + 32 B wavelengths in and 64 B read-modify-write; plus the
      same node and record bytes.
    surface: per path the 64 B ray record read, the 128 B primitive, the 64 B vertex record written,
      8 B of queue entries. material: per path 160 B read, 112 B written, the 88 B material and a
      48 B shadow record.
    """
    nb, rb = NODE_READ, stats["recBytes"]
    if name == "intersect" and fused:
        # one launch per bounce traces the bounce's closest rays and the previous bounce's shadow
        # rays: its items are both, and the bytes per item their mix
        rc, rs = stats["closestRays"], stats["shadowRays"]
        per = ((52 * rc + nb * stats["closestNodes"] + rb * stats["closestRecs"]) +
               (80 * rs + nb * stats["shadowNodes"] + rb * stats["shadowRecs"])) / max(1, rc + rs)
        return per * items, per
    if name == "intersect":
        rays = max(1, stats["closestRays"])
        per = 52 + nb * stats["closestNodes"] / rays + rb * stats["closestRecs"] / rays
        return per * items, per
    if name == "shadow":
        rays = max(1, stats["shadowRays"])
        per = 176 + nb * stats["shadowNodes"] / rays + rb * stats["shadowRecs"] / rays
        return per * items, per
    if name == "surface":
        # the ray record (ray, hit, state) in, the 128 B primitive, the vertex record out, 8 B of
        # queue entries
        per = 64 + 128 + 64 + 8
        return per * items, per
    if name == "material":
        # direction, state, path and vertex record in, 112 B state out, the 88 B material, and a 48 B
        # shadow record
        per = 160 + 112 + 88 + 48
        return per * items, per
    return None, None


def measured_traffic(kernel):
    """`traffic_bytes_per_launch <kernel> <bytes>` line of the committed counter summary, if any."""
    if not os.path.exists(TRAFFIC_FILE):
        return None
    for line in open(TRAFFIC_FILE):
        f = line.strip().strip("`").split()
        if len(f) == 3 and f[0] == "traffic_bytes_per_launch" and f[1] == kernel:
            return float(f[2])
    return None


def copy_calibration(nbytes=1 << 30, reps=3):
    """A plain device copy of known size (read nbytes, write nbytes), for scaling the HBM counters."""
    import torch
    x = torch.ones(nbytes // 4, dtype=torch.float32, device="cuda")
    y = torch.empty_like(x)
    for _ in range(reps):
        torch.mul(x, 1.0, out=y)
    torch.cuda.synchronize()
    print(json.dumps({"copy_calibration": {"bytes_read": nbytes, "bytes_written": nbytes, "launches": reps}}),
          flush=True)


def relmse(a, r):
    """Mean over pixels and channels of (a - r)^2 / (r^2 + 1e-2), linear sRGB (reference
    tests/test_quality.cpp:241-248)."""
    d = a.astype(np.float64) - r
    return float(np.mean(d * d / (r * r + 1e-2)))


def equal_time_relmse(plugin, host, width, height, seconds, ref_spp, spp_per_call=4):
    """Equal-time relMSE of the guided and the plain path tracer on the indoor configuration
    (sun through a window, indirect light everywhere) against a high-spp plain reference.

    Guided time includes inference at the guided bounces and training after every call (the
    model starts from its initial parameters). Sample ranges of the four renders (two reference
    halves, plain, guided) are disjoint."""
    import prender_amd as pa
    scene = host.generate(4, width, height)

    def render(first, flags, budget=None, spp=None):
        plugin.film_reset(width, height)
        done, k = 0, 0
        t0 = time.perf_counter()
        while True:
            f = flags | (pa.RENDER_GUIDE_RESET if (k == 0 and flags) else 0)
            plugin.render_resident(scene, pa.render_params(spp=spp_per_call, first_sample=first + done, seed=1,
                                                           max_depth=32, rr_start=1, flags=f))
            done += spp_per_call
            k += 1
            el = time.perf_counter() - t0
            if (budget is not None and el >= budget) or (spp is not None and done >= spp):
                break
        film, _ = plugin.film_read(width, height, variance=False)
        rgb = host.resolve_srgb(film.reshape(-1, 3), 1.0 / done).reshape(height, width, 3)
        return rgb, done, el

    # The reference is rendered as two independent halves: their difference estimates the
    # reference's own noise, which adds to the relMSE of both renders alike.
    ref_a, ras, rat = render(0, 0, spp=ref_spp // 2)
    ref_b, rbs, rbt = render(1 << 23, 0, spp=ref_spp // 2)
    ref = 0.5 * (ref_a + ref_b)
    rs, rt = ras + rbs, rat + rbt
    plain, ps, pt = render(1 << 24, 0, budget=seconds)
    guide_flags = pa.RENDER_GUIDE | pa.RENDER_GUIDE_TRAIN
    guided, gs, gt = render(2 << 24, guide_flags, budget=seconds)
    ep, eg = relmse(plain, ref), relmse(guided, ref)
    # E[(a - r)^2] = E[(a - truth)^2] + Var(r); Var(r) per pixel and channel = E[(r_a - r_b)^2] / 4.
    d = ref_a.astype(np.float64) - ref_b
    noise = float(np.mean(d * d / 4 / (ref * ref + 1e-2)))
    return {"plain": round(ep, 5), "guided": round(eg, 5), "guided_over_plain": round(eg / ep, 4),
            "reference_noise": round(noise, 5),
            "guided_over_plain_noise_corrected": round((eg - noise) / (ep - noise), 4) if ep > noise else None,
            "seconds": {"plain": round(pt, 2), "guided": round(gt, 2)}, "spp": {"plain": ps, "guided": gs},
            "reference": f"plain path tracer, {rs} spp in two independent halves ({rt:.1f} s)",
            "workload": f"configuration 4 (indoor room, 520k triangles, sun through a 1 x 1 window) at "
                        f"{width}x{height}, max depth 32"}


# The oracle against the reference's own CPU path tracer on the same 8 cores of the build container:
# reference_s is the reference's recorded time for its sample scene scenes/sphere-pyramid at
# 480x270, 16 spp, max depth 64 (measured outside this repository); the oracle renders the scene as
# the loader flattens it (tests/golden/sample_scene.npz, studio rig) with 8 threads.
CPU_CALIBRATION = {"scene": "reference scenes/sphere-pyramid, 480x270, 16 spp, 8 threads (build container)",
                   "reference_s": 1.20, "oracle_s": [1.17, 1.075, 1.073, 1.104], "oracle_time_over_reference_time": 0.91}


def cpu_baseline(scene, target_seconds, spp_cap):
    """Times the oracle on a bounded sample of the same workload (render time only)."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle
    import prender_amd as pa

    threads = os.cpu_count() or 1
    if os.environ.get("OMP_NUM_THREADS", "").isdigit():
        threads = min(threads, int(os.environ["OMP_NUM_THREADS"]))
    o = oracle.OracleScene(scene)
    p = pa.render_params(spp=1, first_sample=0, seed=1, max_depth=16, rr_start=1)
    _, _, first = o.render(p, variance=False, threads=threads)
    passes = int(max(1, min(spp_cap, round(target_seconds / max(first, 1e-3)))))
    p = pa.render_params(spp=passes, first_sample=1, seed=1, max_depth=16, rr_start=1)
    _, _, secs = o.render(p, variance=False, threads=threads)
    samples = scene.width * scene.height * passes
    model = ""
    try:
        with open("/proc/cpuinfo") as f:
            model = next((l.split(":", 1)[1].strip() for l in f if l.startswith("model name")), "")
    except OSError:
        pass
    return {"value": samples / secs / 1e6, "unit": "Msamples/s", "cores": threads, "kind": "port", "cpu": model,
            "calibration": CPU_CALIBRATION,
            "sample": f"configuration 2 at {scene.width}x{scene.height}, {passes} spp ({secs:.1f} s render time, "
                      f"oracle C++ restatement of the reference PathIntegrator, {threads} threads)"}


# The reference's published GPU times for its sample scene at 960x540 (ms per sample per pixel,
# startup excluded; Arc A770, docs/acceleration-investigation.md:202-206).
SAMPLE_SCENE_PUBLISHED_MS = {"studio": 31.0, "studio_fog": 62.0}
# ... and at 1920x1080 with the materials the plugin had then (glass, metals, dispersion; coats,
# sheen and subsurface approximated), 16.5 ms per spp (docs/acceleration-investigation.md:150-152).
# This build renders the full materials at that size: more work than the published run.
SAMPLE_SCENE_PUBLISHED_1080P_MS = 16.5


def sample_scene(pa, plugin, spp=256, batch=16, only=None):
    """ms per spp of the reference's sample scene (scenes/sphere-pyramid as this build's loader
    flattens it, every material family: glass, dispersion, metals, subsurface, coats, sheen, an
    emissive sphere; studio rig, and studio + fog) at its own 960 x 540 film and max depth, rendered
    into the resident film, startup excluded, next to the reference's published A770 times."""
    g = np.load(os.path.join(ROOT, "tests", "golden", "sample_scene.npz"))
    rows = {}
    runs = [(name, name, published, None) for name, published in SAMPLE_SCENE_PUBLISHED_MS.items()]
    runs.append(("studio_1920x1080_full_materials", "studio", SAMPLE_SCENE_PUBLISHED_1080P_MS, (1920, 1080)))
    runs.append(("studio_1920x1080_subset_materials", "studio", SAMPLE_SCENE_PUBLISHED_1080P_MS, (1920, 1080)))
    if only:
        unknown = set(only) - {r[0] for r in runs}
        if unknown:
            raise SystemExit(f"--sample-scene-runs: unknown {sorted(unknown)}; choose from {[r[0] for r in runs]}")
        runs = [r for r in runs if r[0] in only]
    for label, name, published, size in runs:
        scene = pa.flat_scene(g, name)
        if size:
            cam = pa.CameraEx.from_buffer_copy(bytes(scene.camera))
            cam.width, cam.height = size
            prims, mats, spectra = scene.prims.copy(), scene.materials.copy(), scene.spectra.copy()
            cam_medium = scene.desc.cameraMedium
            if label.endswith("subset_materials"):
                # the materials of the plugin's first version, as its exporter fell back for the rest
                # (gpu_path.cpp:249-253): coated materials as grey diffuse, no sheen, no media
                grey = np.zeros(1, pa.SPECTRUM_DTYPE)
                grey["kind"], grey["scale"], grey["p"][0][0] = pa.SPEC_CONSTANT, 1.0, 0.5
                spectra = np.concatenate([spectra, grey])
                coated = np.isin(mats["type"], [pa.MAT_COATED_DIFFUSE, pa.MAT_COATED_CONDUCTOR])
                mats["type"][coated] = pa.MAT_DIFFUSE
                mats["albedo"][coated] = len(spectra) - 1
                mats["albedoB"][coated] = -1
                mats["sheenWeight"] = 0
                prims["mediumInside"] = prims["mediumOutside"] = -1
                cam_medium = -1
            scene = pa.Scene(prims, mats, spectra, scene.knots, scene.lights, scene.media, scene.grid, cam, cam_medium,
                             scene.defaults)
        w, h = scene.width, scene.height
        prm = lambda first, n: pa.render_params(spp=n, first_sample=first, seed=scene.defaults["seed"],  # noqa: E731
                                                max_depth=scene.defaults["maxDepth"], rr_start=1)
        plugin.film_reset(w, h)
        plugin.render_resident(scene, prm(0, batch))  # scene upload, BVH, first batch (calls block)
        t0 = time.perf_counter()
        done = 0
        while done < spp:
            plugin.render_resident(scene, prm(batch + done, batch))
            done += batch
        el = time.perf_counter() - t0
        film, _ = plugin.film_read(w, h, variance=False)
        if not np.all(np.isfinite(film)) or not film.any():
            raise RuntimeError(f"sample scene {label}: empty or non-finite film")
        ms = el * 1e3 / spp
        rows[label] = {"ms_per_spp": round(ms, 3), "Msamples_per_s": round(w * h / ms / 1e3, 1),
                      "published_a770_ms_per_spp": published, "speedup_vs_published": round(published / ms, 1),
                      "width": w, "height": h, "max_depth": scene.defaults["maxDepth"], "spp": spp}
    print(json.dumps({"sample_scene": rows, "scene": "reference scenes/sphere-pyramid (flattened, "
                      "tests/golden/sample_scene.npz)"}), flush=True)


# The reference's published relMSE of its plain GPU path tracer on the sample scene (960x540,
# studio rig) against a 16 384-spp reference: spp -> (relMSE, seconds on an Arc A770)
# (docs/denoising-investigation.md:64-69).
SAMPLE_SCENE_PUBLISHED_RELMSE = {16: (18.4, 0.6), 64: (6.0, 1.8), 256: (1.8, 6.7), 1024: (0.36, 26.0)}


def sample_scene_relmse(pa, host, plugin, ref_spp=16384, batch=16):
    """relMSE on the reference's sample scene (studio rig, 960x540, max depth 64) against a
    16 384-spp reference of this renderer, rendered in two independent halves. Two ladders: at
    the reference's published sample counts (the same unbiased estimator should give the same error,
    up to noise) and at the reference's published times (this renderer's samples in that time).
    Sample ranges of every render are disjoint. Progress goes to stderr."""
    g = np.load(os.path.join(ROOT, "tests", "golden", "sample_scene.npz"))
    scene = pa.flat_scene(g, "studio")
    w, h = scene.width, scene.height
    prm = lambda first, n: pa.render_params(spp=n, first_sample=first, seed=scene.defaults["seed"],  # noqa: E731
                                            max_depth=scene.defaults["maxDepth"], rr_start=1)
    plugin.film_reset(w, h)
    plugin.render_resident(scene, prm(1 << 30, 1))  # upload and BVH build outside every clock

    def render(first, spp=None, seconds=None):
        plugin.film_reset(w, h)
        done, t0 = 0, time.perf_counter()
        while True:
            n = batch if spp is None else min(batch * 4, spp - done)
            plugin.render_resident(scene, prm(first + done, n))
            done += n
            el = time.perf_counter() - t0
            if (spp is not None and done >= spp) or (seconds is not None and el >= seconds):
                break
        film, _ = plugin.film_read(w, h, variance=False)
        return host.resolve_srgb(film.reshape(-1, 3), 1.0 / done).reshape(h, w, 3), done, el

    ref_a, _, ta = render(0, spp=ref_spp // 2)
    print(f"reference half 1: {ref_spp // 2} spp in {ta:.1f} s", file=sys.stderr, flush=True)
    ref_b, _, tb = render(1 << 24, spp=ref_spp // 2)
    print(f"reference half 2: {ref_spp // 2} spp in {tb:.1f} s", file=sys.stderr, flush=True)
    ref = 0.5 * (ref_a + ref_b)
    d = ref_a.astype(np.float64) - ref_b
    noise = float(np.mean(d * d / 4 / (ref * ref + 1e-2)))
    by_spp, by_time = {}, {}
    first = 2 << 24
    for spp, (pub, secs) in SAMPLE_SCENE_PUBLISHED_RELMSE.items():
        img, done, el = render(first, spp=spp)
        first += 1 << 22
        by_spp[spp] = {"relmse": round(relmse(img, ref), 4), "seconds": round(el, 3), "published_relmse": pub,
                       "published_seconds": secs}
        img, done, el = render(first, seconds=secs)
        first += 1 << 22
        by_time[secs] = {"relmse": round(relmse(img, ref), 4), "spp": done, "published_relmse": pub,
                         "published_spp": spp}
        print(f"{spp} spp / {secs} s done", file=sys.stderr, flush=True)
    print(json.dumps({"sample_scene_relmse": {"at_published_spp": by_spp, "at_published_seconds": by_time,
                                              "reference": f"{ref_spp} spp of this renderer in two halves "
                                                           f"({ta + tb:.1f} s)",
                                              "reference_noise": round(noise, 5),
                                              "scene": "reference scenes/sphere-pyramid, studio rig, 960x540, "
                                                       "max depth 64"}}), flush=True)


def traversal_counts(pa, host, plugin):
    """Per-ray work of closest-hit queries on configuration 2 at 1920x1080 for the two batches of
    prender_amd.measurement_rays(scene, 8192, 7): this build's 8-wide quantised BVH (wide nodes
    fetched and 48 B leaf records tested, counted by the ray-query kernel in profile mode 2) next to
    the reference's binary BVH (32 B nodes and 128 B primitives tested), whose counts were recorded
    from the reference's own BVH on the same rays (tests/golden/ref_components.npz)."""
    import hashlib
    g = np.load(os.path.join(ROOT, "tests", "golden", "ref_components.npz"))
    scene = host.generate(2)
    rows = {}
    for name, rays, ref, sha in zip(("primary", "random"), pa.measurement_rays(scene, 8192, 7), g["refbvh_counts"],
                                    g["refbvh_ray_sha1"]):
        if hashlib.sha1(rays.tobytes()).hexdigest() != str(sha):
            raise RuntimeError("measurement rays differ from those of the recorded reference counts")
        plugin.trace(scene, rays[:64])  # upload the geometry outside the counted call
        plugin.profile(2)
        plugin.profile_read(reset=True)
        hits = plugin.trace(scene, rays)
        st = plugin.profile_read(reset=True)
        plugin.profile(0)
        n = st["closestRays"]
        nodes, recs = st["closestNodes"] / n, st["closestRecs"] / n
        rows[name] = {
            "rays": int(n), "hit_rate": round(float((hits["prim"] >= 0).mean()), 4),
            "wide_bvh": {"nodes_per_ray": round(nodes, 3), "records_per_ray": round(recs, 3),
                         "bytes_per_ray": round(nodes * NODE_READ + recs * st["recBytes"] + 52, 1)},
            "reference_bvh": {"nodes_per_ray": round(float(ref[0]), 3), "primitives_per_ray": round(float(ref[1]), 3),
                              "hit_rate": round(float(ref[2]), 4),
                              "bytes_per_ray": round(float(ref[0]) * 32 + float(ref[1]) * 128 + 48, 1)}}
    print(json.dumps({"traversal_counts": rows, "scene": "configuration 2 at 1920x1080",
                      "bytes": "wide: 80 B node + 48 B record + 32 B ray + 4 B queue + 16 B hit; "
                               "reference: 32 B node + 128 B primitive + 32 B ray + 16 B hit"}), flush=True)


# The other benchmark configurations at their own sizes, for the throughput table beside the
# headline (configuration 2): (config, width, height, detail, max depth, rr start, spp per call, calls).
# (configuration, width, height, detail, max depth, roulette start, spp per call, timed calls): a call
# is at most one batch at the default queue capacity (32 M paths).
OTHER_CONFIGS = {
    "c1": (1, 256, 256, 1.0, 8, 3, 64, 2),
    "c3": (3, 1280, 720, 1.0, 256, 1, 32, 2),
    "c5": (5, 3840, 2160, 1.0, 16, 1, 4, 2),
}
OTHER_CONFIG_NAMES = {
    "c1": "sphere pyramid (28.8k triangles), 256x256, max depth 8, roulette from depth 3",
    "c3": "256^3 fBm grid medium (spectral + ratio tracking) behind an interface box, subsurface sphere, distant "
          "light, 1280x720, max depth 256",
    "c5": "150 brilliant-cut gems (diamond Sellmeier) on rough silver, thin lens f/2.8, 3840x2160, max depth 16",
}


def other_configs(pa, host, plugin, names):
    """ms per spp and Msamples/s of the other configurations at their full sizes (resident film,
    production bounce loop, scene generation and the first call's upload excluded)."""
    rows = {}
    for name in names:
        cfg, w, h, detail, depth, rr_start, spp, calls = OTHER_CONFIGS[name]
        scene = host.generate(cfg, w, h, detail)
        prm = lambda first: pa.render_params(spp=spp, first_sample=first, seed=1, max_depth=depth,  # noqa: E731
                                             rr_start=rr_start)
        plugin.film_reset(w, h)
        plugin.render_resident(scene, prm(0))
        t0 = time.perf_counter()
        for k in range(calls):
            plugin.render_resident(scene, prm(spp * (k + 1)))
        el = time.perf_counter() - t0
        film, _ = plugin.film_read(w, h, variance=False)
        if not np.all(np.isfinite(film)) or not film.any():
            raise RuntimeError(f"{name}: empty or non-finite film")
        ms = el * 1e3 / (spp * calls)
        rows[name] = {"workload": OTHER_CONFIG_NAMES[name], "ms_per_spp": round(ms, 3),
                      "Msamples_per_s": round(w * h / ms / 1e3, 1), "spp_timed": spp * calls,
                      "triangles": len(scene.prims)}
        print(f"{name}: {ms:.2f} ms per spp", file=sys.stderr, flush=True)
    return rows


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=8)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--spp-per-step", type=int, default=16)
    ap.add_argument("--width", type=int, default=1920)
    ap.add_argument("--height", type=int, default=1080)
    ap.add_argument("--cpu-seconds", type=float, default=15.0)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-counters", action="store_true")
    ap.add_argument("--other-configs", default="c1,c3,c5",
                    help="comma-separated configurations timed beside the headline ('' skips them)")
    ap.add_argument("--relmse-seconds", type=float, default=3.0,
                    help="equal time budget of the guided and the plain render (0 skips the comparison)")
    ap.add_argument("--relmse-ref-spp", type=int, default=1024)
    ap.add_argument("--copy-calibration", action="store_true",
                    help="run only a 1 GiB device copy (for scaling rocprofv3 FETCH_SIZE/WRITE_SIZE)")
    ap.add_argument("--sample-scene", action="store_true",
                    help="only time the reference's sample scene (sphere pyramid, 960x540) in ms per spp")
    ap.add_argument("--sample-scene-runs", default="",
                    help="with --sample-scene: a comma-separated subset of its runs (studio, studio_fog, "
                         "studio_1920x1080_full_materials, studio_1920x1080_subset_materials)")
    ap.add_argument("--sample-scene-spp", type=int, default=256,
                    help="with --sample-scene: timed samples per pixel of each run (a multiple of 16)")
    ap.add_argument("--sample-scene-relmse", action="store_true",
                    help="only measure relMSE on the reference's sample scene at its published spp and times")
    ap.add_argument("--traversal-counts", action="store_true",
                    help="only compare per-ray traversal work of the wide BVH with the reference's binary BVH")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU: this build runs the path tracer on a single MI355X "
              "(multi-GPU sharding is a design note only); use --gpus 1", file=sys.stderr)
        sys.exit(2)

    if args.copy_calibration:
        copy_calibration()
        return

    import prender_amd as pa

    host = pa.Host()
    plugin = pa.Plugin()
    if not plugin.devices():
        raise RuntimeError("no HIP device visible")
    if args.traversal_counts:
        traversal_counts(pa, host, plugin)
        return
    if args.sample_scene:
        sample_scene(pa, plugin, spp=max(16, args.sample_scene_spp // 16 * 16),
                     only=[r for r in args.sample_scene_runs.split(",") if r] or None)
        return
    if args.sample_scene_relmse:
        sample_scene_relmse(pa, host, plugin)
        return
    t0 = time.perf_counter()
    scene = host.generate(2, args.width, args.height)
    gen_s = time.perf_counter() - t0
    W, H, S = scene.width, scene.height, args.spp_per_step

    def params(step):
        return pa.render_params(spp=S, first_sample=step * S, seed=1, max_depth=16, rr_start=1)

    plugin.film_reset(W, H)
    t0 = time.perf_counter()
    plugin.render_resident(scene, params(0))  # first call: BVH build + upload + one step
    setup_s = time.perf_counter() - t0
    for w in range(1, args.warmup):
        plugin.render_resident(scene, params(w))
    # The timed steps run the production bounce loop (profile mode 0: queued one round ahead of
    # the path-count read-back, no per-kernel events). The plugin's calls are synchronous on its
    # stream: each returns after its work completes.
    plugin.profile(0)
    t0 = time.perf_counter()
    for k in range(args.steps):
        plugin.render_resident(scene, params(args.warmup + k))
    t1 = time.perf_counter()
    elapsed = t1 - t0
    samples = W * H * S * args.steps
    value = samples / elapsed / 1e6
    # Per-kernel durations from the same number of further steps with HIP events around every
    # launch (profile mode 1, which also waits for each bounce's path count); not part of `value`.
    plugin.profile(1)
    plugin.profile_read(reset=True)
    tp = time.perf_counter()
    for k in range(args.steps):
        plugin.render_resident(scene, params(args.warmup + args.steps + k))
    profiled_elapsed = time.perf_counter() - tp
    timed = plugin.profile_read(reset=True)
    extra_steps = args.steps

    # Traversal counters from a counting run of one more step (outside the timed region).
    counters = None
    if not args.no_counters:
        plugin.profile(2)
        plugin.render_resident(scene, params(args.warmup + 2 * args.steps))
        counters = plugin.profile_read(reset=True)
        extra_steps += 1
    plugin.profile(0)
    film, _ = plugin.film_read(W, H)

    kernels = timed["kernels"]
    dominant = max(kernels, key=lambda k: kernels[k]["ms"])
    roofline = None
    if counters is not None:
        fused = kernels["shadow"]["launches"] == 0 and counters["shadowRays"] > 0
        total, per = kernel_bytes(dominant, counters, kernels[dominant]["items"], fused)
        if total is not None and kernels[dominant]["ms"] > 0:
            achieved = total / (kernels[dominant]["ms"] * 1e-3) / 1e9
            traffic = measured_traffic(dominant)
            avg_ms = kernels[dominant]["ms"] / max(1, kernels[dominant]["launches"])
            # `frac` prices the algorithmic bytes (every node and record fetch counted as if it came
            # from HBM) against the HBM peak; `frac_hbm_traffic` prices the counter-measured HBM bytes
            # of one launch. Most node and record re-reads hit L2 / MALL. What bounds the traversal is VALU
            # issue: the counters of the same file find the SIMDs' issue slots full.
            trav_bound = dominant == "intersect" and traffic is not None
            roofline = {"bound": "valu" if trav_bound else "hbm", "kernel": dominant, "achieved": round(achieved, 1),
                        "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBS, 4),
                        "frac_of": "HBM peak, every fetch priced as if from HBM",
                        "traffic": traffic,
                        "frac_hbm_traffic": (round(traffic / (avg_ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4)
                                             if traffic else None),
                        "limited_by": ("VALU issue (slots full, 58 % of lanes active in the counter run); nodes and "
                                       "records come from L2 / MALL" if trav_bound else None),
                        "algorithmic_bytes_per_item": round(per, 1),
                        "items_per_launch": round(kernels[dominant]["items"] / max(1, kernels[dominant]["launches"]), 1),
                        "avg_launch_ms": round(kernels[dominant]["ms"] / max(1, kernels[dominant]["launches"]), 4)}
    trav = None
    if counters is not None:
        cr, sr = max(1, counters["closestRays"]), max(1, counters["shadowRays"])
        trav = {"closest_nodes_per_ray": round(counters["closestNodes"] / cr, 2),
                "closest_records_per_ray": round(counters["closestRecs"] / cr, 2),
                "shadow_nodes_per_ray": round(counters["shadowNodes"] / sr, 2),
                "shadow_records_per_ray": round(counters["shadowRecs"] / sr, 2),
                "rays_per_sample": round((counters["closestRays"] + counters["shadowRays"]) / (W * H * S), 3)}
    rays = kernels["intersect"]["items"] + kernels["shadow"]["items"]

    guided = None
    if args.relmse_seconds > 0:
        guided = equal_time_relmse(plugin, host, args.width, args.height, args.relmse_seconds, args.relmse_ref_spp)

    others = None
    if args.other_configs:
        others = other_configs(pa, host, plugin, [n for n in args.other_configs.split(",") if n])

    cpu = None
    if not args.no_cpu:
        cpu = cpu_baseline(scene, args.cpu_seconds, 16)

    out = {
        "metric": METRIC, "value": round(value, 3), "unit": "Msamples/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(elapsed / args.steps * 1e3, 3), "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": "configuration 2: 1920x1080 fBm terrain (997k triangles) + 200 icospheres (1.02M "
                               "triangles), 40/30/30 Lambert/GGX conductor/BK7, 64 blackbody quad lights, light-BVH "
                               "NEE, max depth 16, plain path tracer",
                   "width": W, "height": H, "spp_per_step": S, "max_depth": 16, "triangles": len(scene.prims),
                   "parallelism": "1 GPU",
                   "guided_vs_plain_relMSE": guided["guided_over_plain"] if guided else None},
        "relmse": guided,
        "other_configs": others,
        "rays_per_s": round(rays / elapsed / 1e6, 2), "rays_unit": "Mrays/s",
        "kernels_ms_per_step": {k: round(v["ms"] / args.steps, 3) for k, v in kernels.items()},
        "traversal": trav, "roofline": roofline, "cpu_baseline": cpu,
        "tuning": plugin.tuning(),
        "setup_s": {"scene_generation": round(gen_s, 2), "first_call_bvh_upload_and_step": round(setup_s, 2)},
        "profiled_ms_per_step": round(profiled_elapsed / args.steps * 1e3, 3),
        "timing": "value: production bounce loop (profile mode 0); kernels_ms_per_step and roofline: the same "
                  "number of further steps with HIP events around every launch (profile mode 1)",
        "film_mean_Y": float(film[..., 1].mean() / (S * (args.warmup + args.steps + extra_steps))),
    }
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
