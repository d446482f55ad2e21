#!/usr/bin/env python3
"""Benchmark of the MI355X LEE + porous-ground time step (one GPU).

Workload (deck.config_c1): the 512x256x128 air grid at 0.04 m, terrain-following over a
Gaussian hill (2 m high, sigma 5 m), over a 16-point Zwikker-Kosten porous layer, 20-point
PML on the sides and top, logarithmic wind u(z) = (0.4/0.41) ln(z/0.02), moving frame on,
Gaussian pulse of half-width 3 dx at 0.5 m, 32 receivers at 1.2 m, classical RK4 at CFL 0.5
for 10000 steps.  One "step" is one RK4 time step of the whole domain (four stages: air,
porous layer, faces).  FP32 (compensated accumulation) is the headline `value`; FP64 runs the
same workload and is the reference for the accuracy figures.

Timing: W untimed warm-up steps, then exactly K timed steps with a device synchronisation on
both sides; inputs are resident in HBM.  The receiver series of the whole run (W + K steps)
give the accuracy of FP32 against FP64: relative L2 and the largest insertion-loss
difference |20 log10 |P32(f)| - 20 log10 |P64(f)|| over 50-1000 Hz (the reference spectrum
of IL cancels in the difference).

`roofline`: the dominant kernel's compulsory HBM bytes per launch over its mean launch time
(HIP events on the solver stream); `traffic` comes from rocprofv3 FETCH_SIZE / WRITE_SIZE
runs when a JSON of them is given.  `cpu_baseline`: the FP64 C oracle of the same step on the host's
OpenMP threads (and on one thread beside it) over a bounded sample (the first step(s) of the
same workload).

`--workload c3` runs the batched ensemble: 64 seeded uneven domains (deck.config_c3) advanced
together by the ensemble runner, FP32 (and FP64 for the accuracy figures), 3000 steps.

`--workload c4` runs the learned ground: the training pipeline on the GPU, the judge, then the
1024x512x160 FB_p_v domain FP32 over the full porous layer and air-only with the learned
impedance (speed-up and IL difference between the two).

`--workload c2` runs the precision study instead: 768x384x192 at 0.04 m over a 24-point
porous layer and a seeded random terrain of 6 Gaussian hills, RK4, 2000 steps, FP32 against
FP64 (deck.config_c2).

    python bench.py [--gpus 1] [--workload c1|c2|c3|c4] [--steps K] [--warmup W] [--no-cpu] [--no-fb]
                    [--traffic-json F]
"""
from __future__ import annotations

import argparse
import importlib
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0  # MI355X HBM3E
# launch shapes of the RK4 air stage (lee_options.rk_tile 1..11), as the autotuner reports them
RK_TILES = ["whole domain in one launch a stage"] * 5 + ["interior two stages a launch, the rest one"] * 6
# launch forms of the FB_p_v air passes (lee_options.fb_form 1..7), as the autotuner reports them
FB_FORMS = ["split", "split, padded tile lists", "fused, 2 blocks/CU", "fused, 4 blocks/CU", "fused, 8 blocks/CU",
            "fused, 16 blocks/CU", "split, one point per lane"]


RK_TILE = 0  # --rk-tile: RK4 air-stage launch shape, 0 = the autotuner's choice
STREAMS = (12, 8)  # arrays read and written by the many-stream reference kernel (lee_stream_bench)
# launch forms of the ensemble's air and porous stages (lee_ensemble_set_launch), index = form
ENS_FORMS = [None, "a block per 256-column tile", "tiles padded per plane to multiples of 8", "persistent grid"]


def run_gpu(lee, deck, receivers, precision, steps, warmup, record=True):
    """Run warmup + steps steps of `deck`, frames moving as the reference schedules them.
    Returns timing, kernel statistics and the receiver series of the whole run."""
    s = lee.Solver(deck, precision=precision, receivers=receivers, rk_tile=RK_TILE)
    npts = s.nx * s.ny * s.nz + s.pnx * s.pny * s.pnz
    state = {"mf": 0, "temp": 0, "left": 0}

    def setup_frame():
        state["left"] = s.frame_steps(state["mf"], state["temp"])
        s.frame_setup(state["mf"])

    def advance(n):
        out = []
        while n > 0:
            if state["left"] <= 0:
                state["mf"] += 1
                setup_frame()
            k = min(n, state["left"])
            out.append(s.step(k, record=record))
            state["left"] -= k
            state["temp"] += k
            n -= k
        return out

    def kernel_stats():
        stats = (lee.LeeKstat * 16)()
        n = lee.lib().lee_kernel_stats(s.h, stats, 16)
        return [dict(name=k.name.decode(), launches=k.launches, total_ms=k.total_ms,
                     bytes_per_launch=k.bytes_per_launch, points=k.points_per_launch)
                for k in stats[:n] if k.launches]

    setup_frame()
    # every kernel kind carries timing marks over the warm-up steps (the kernel tables); over
    # the timed steps only the air stencil launches do, the dominant kernels the roofline
    # needs, measured live over the timed region (each mark is a packet between launches:
    # marking every kind costs 4 % of an RK4 step, marking the air launches 1 %)
    lee.lib().lee_profile(s.h, 1)
    series = advance(warmup)
    kall = kernel_stats()
    lee.lib().lee_profile(s.h, 2)
    t0 = time.perf_counter()
    series += advance(steps)
    t1 = time.perf_counter()
    kst = kernel_stats()
    tile, form = s.info().rk_tile, s.info().fb_form
    copy_ms = lee.lib().lee_copy_bench(s.h, 1 << 28, 10)  # 1 GiB read + 1 GiB write
    # a kernel with as many streams as an RK4 stage's average (12 read, 8 written, 64 MiB each)
    stream_ms = lee.lib().lee_stream_bench(s.h, 1 << 24, STREAMS[0], STREAMS[1], 10)
    rec = np.concatenate([x for x in series if x is not None], axis=0) if record else None
    info = dict(points=npts, wall=t1 - t0, kernels=kst, kernels_all=kall or kst, copy_ms=copy_ms, stream_ms=stream_ms,
                frames=state["mf"] + 1, series=rec,
                rk_tile=RK_TILES[tile - 1] if tile > 0 else None, fb_form=FB_FORMS[form - 1] if form > 0 else None)
    s.close()
    return info


def run_series(lee, deck, receivers, precision, nsteps):
    """Receiver series of nsteps steps of `deck` (frames moving as the reference schedules
    them), untimed: the accuracy pass."""
    s = lee.Solver(deck, precision=precision, receivers=receivers)
    out, mf, temp = [], 0, 0
    left = s.frame_steps(mf, temp)
    s.frame_setup(mf)
    n = nsteps
    while n > 0:
        if left <= 0:
            mf += 1
            left = s.frame_steps(mf, temp)
            s.frame_setup(mf)
        k = min(n, left)
        out.append(s.step(k))
        left -= k
        temp += k
        n -= k
    s.close()
    return np.concatenate(out, axis=0)


def accuracy(a, b, dt, fmin=50.0, fmax=1000.0):
    """Relative L2 of series b against a, and the largest |IL_b - IL_a| in dB over
    [fmin, fmax] on receivers that carry signal (bins 60 dB below the band peak skipped).
    None when no receiver carries signal (nothing was measured)."""
    energy = (a ** 2).sum(axis=0)
    if not energy.max() > 0:
        return None
    rel = float(np.linalg.norm(b - a) / max(np.linalg.norm(a), 1e-300))
    use = energy > 1e-6 * energy.max()
    n = 1 << int(np.ceil(np.log2(a.shape[0])))
    f = np.fft.rfftfreq(n, dt)
    band = (f >= fmin) & (f <= fmax)
    worst = 0.0
    for r in np.nonzero(use)[0]:
        A = np.abs(np.fft.rfft(a[:, r], n))[band]
        B = np.abs(np.fft.rfft(b[:, r], n))[band]
        ok = A > 1e-3 * A.max()
        if ok.any():
            worst = max(worst, float(np.abs(20 * np.log10(B[ok] / A[ok])).max()))
    return rel, worst, int(use.sum())


def cpu_model():
    try:
        with open("/proc/cpuinfo") as fh:
            for line in fh:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline(deck, receivers, budget_s=20.0, threads=None, max_steps=10):
    """The FP64 oracle of the same step on the host: the first step(s) of the workload within
    about `budget_s` seconds (at most max_steps), on `threads` host threads (default:
    OpenMP's count, which OMP_NUM_THREADS sets)."""
    from oracle import oracle as orc

    if threads:
        orc.set_threads(threads)
    used = orc.get_threads()
    o = orc.Oracle(deck, receivers=receivers)
    o.frame_setup(0)
    npts = o.nx * o.ny * o.nz + o.pnx * o.pny * o.pnz
    t0 = time.perf_counter()
    o.step(1)
    first = time.perf_counter() - t0
    more = max(0, min(max_steps - 1, int(budget_s / max(first, 1e-3)) - 1))
    t2 = time.perf_counter()
    if more:
        o.step(more)
    sec = first + (time.perf_counter() - t2)
    return dict(value=npts * (1 + more) / sec, steps=1 + more, seconds=sec, points=npts, threads=used)


def run_c3(lee, a):
    """C3 ensemble: every member advanced by one launch per kernel kind per RK4 stage
    (lee_ensemble_*), captured in graphs.  `value` sums the grid-point updates of all members.
    The roofline figure is the whole step's compulsory bytes (the byte model of each member's
    kernels, summed) over the step time."""
    decks, recs = lee.deck.config_c3(time_domain=a.warmup + a.steps)
    prec = [int(x) for x in a.precisions.split(",")]
    out = {}
    for p in prec:
        print(f"[bench] C3 ensemble fp{p}: {len(decks)} domains, {a.warmup} warm-up + {a.steps} timed steps",
              file=sys.stderr, flush=True)
        e = lee.Ensemble(decks, precision=p, receivers=recs, use_graph=True)
        npts = e.points()
        ser = [e.step(a.warmup)]
        t0 = time.perf_counter()
        ser.append(e.step(a.steps))
        wall = time.perf_counter() - t0
        bytes_step = 0
        for m in e.members:
            stats = (lee.LeeKstat * 16)()
            n = lee.lib().lee_kernel_stats(m.h, stats, 16)
            for i in range(n):
                if stats[i].name.decode() in ("rk_air", "rk_pore", "rk_bnd"):
                    bytes_step += 4 * stats[i].bytes_per_launch
        series = [np.concatenate([ser[0][d], ser[1][d]]) for d in range(len(decks))]
        out[p] = dict(points=npts, wall=wall, bytes_step=bytes_step, series=series,
                      launch={"air": ENS_FORMS[e.launch()], "porous": ENS_FORMS[e.launch(porous=True)]})
        print(f"[bench] C3 fp{p}: {npts * a.steps / wall / 1e9:.2f} G pt-updates/s ({1e3 * wall / a.steps:.3f} ms/step)",
              file=sys.stderr, flush=True)
        e.close()
    head = 32 if 32 in out else prec[0]
    r = out[head]
    ms = 1e3 * r["wall"] / a.steps
    achieved = r["bytes_step"] / (ms / 1e3) / 1e9
    acc = None
    if 32 in out and 64 in out:
        worst_l2, worst_il = 0.0, 0.0
        measured = 0
        for d in range(len(decks)):
            m = accuracy(out[64]["series"][d], out[32]["series"][d], decks[d].dt)
            if m is None:
                continue
            measured += 1
            worst_l2, worst_il = max(worst_l2, m[0]), max(worst_il, m[1])
        if measured:
            acc = {"fp32_vs_fp64_worst_member_rel_l2": worst_l2,
                   "worst_member_max_dIL_dB_50_1000Hz": round(worst_il, 5), "members_with_signal": measured}
    line = {
        "metric": "grid-pt updates/s + %HBM BW, FP32 vs FP64; learned-ground speedup @<=0.2 dB",
        "value": round(r["points"] * a.steps / r["wall"], 1),
        "unit": "grid-pt updates/s",
        "n_gpus": 1, "steps": a.steps, "warmup": a.warmup, "ms_per_step": round(ms, 4),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": f"f{head}", "data": "synthetic",
        "config": {"workload": "C3: 64 seeded domains {64..128}x{48..96}x{48..64} at 0.05 m, porous layers 4-16 pts "
                               "(sigma log-U 10-2000 kPa s/m^2, porosity U[0.2,0.5], tortuosity U[1.5,4]), source "
                               "U[0.3,2] m, log wind u* U[0,0.5] m/s, 10-pt PML sides+top, RK4 CFL 0.5, one launch per "
                               "kernel kind per stage, graph-replayed",
                   "points": r["points"], "domains": len(decks), "parallelism": "single GPU",
                   "launch_form": r["launch"]},
        "roofline": {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": None,
                     "kernel": "whole RK4 step (rk_air + rk_pore + rk_bnd, all members)",
                     "bytes_per_step": r["bytes_step"]},
        "cpu_baseline": None,
        "accuracy": acc,
    }
    for p, rr in out.items():
        line[f"fp{p}_pt_updates_per_s"] = rr["points"] * a.steps / rr["wall"]
        line[f"fp{p}_ms_per_step"] = 1e3 * rr["wall"] / a.steps
    print(json.dumps(line))


def run_c4(lee, a):
    """C4 learned ground.  The pipeline end to end on the GPU: column runs of the full air +
    porous solve for 256 seeded grounds inside the hull (reflection data and the closure's
    calibration), residue fits, the network trained by the BF16-MFMA kernels, then the draws of
    the C3 distribution (seed 20261202) in order, each judged by the full porous solve (column
    reflection error and the one-third-octave IL in the judge box).  The
    timed runs are the 1024x512x160 domain over the full porous layer and air-only with the
    learned impedance, FP32, FB_p_v; `value` is the learned run's grid-point updates per second
    of the air domain and `learned_speedup` the porous run's step time over the learned run's.
    Draws the judge rejects (outside the hull, or above its bounds) keep the full porous layer;
    the timed comparison runs on the first accepted draw, and `judge` lists every draw tried."""
    G = lee.ground
    if a.eager:
        G.USE_GRAPH = False
    t0 = time.perf_counter()
    cols = G.Columns()
    train = [gd for gd in G.sample_grounds(2048, 20261203) if G.in_hull(gd)][:256]
    def progress(n, gd, e):
        if (n + 1) % 16 == 0:
            print(f"[bench] C4 training data: {n + 1}/{len(train)} grounds, {time.perf_counter() - t0:.1f} s",
                  file=sys.stderr, flush=True)

    X, A, E = G.training_set(train, cols, progress=progress)
    t_data = time.perf_counter() - t0
    keep = E <= G.HULL_FIT_R
    lg = G.LearnedGround(seed=1)
    t1 = time.perf_counter()
    mse = lg.train(X[keep], A[keep], epochs=600, batch=32, lr=2e-3)
    t_train = time.perf_counter() - t1
    print(f"[bench] C4 training data: {len(train)} grounds in {t_data:.1f} s (fit error median {np.median(E):.4f}, "
          f"max {E.max():.4f}); network trained in {t_train:.2f} s (mse {mse:.2e})", file=sys.stderr, flush=True)
    # the C4 ground: the draws of the C3 distribution (seed 20261202) in order; each is judged,
    # the first one the judge accepts runs learned (the ones before it fall back to the porous
    # layer and are reported)
    draws = G.sample_grounds(16, 20261202)
    # how much of the sweep distribution the learned model may serve (the rest keeps the layer)
    hull_fraction = float(np.mean([G.in_hull(gd) for gd in G.sample_grounds(4096, 7)]))
    judged = []
    g = a_pred = None
    for n, gd in enumerate(draws):
        res, rep = lg.decide(gd, cols)
        rep = {k: (round(v, 5) if isinstance(v, float) else v) for k, v in rep.items()}
        judged.append({"draw": n, "ground": vars(gd), **rep, "learned": res is not None})
        print(f"[bench] C4 draw {n} {gd}: judge {rep}", file=sys.stderr, flush=True)
        if res is not None:
            g, a_pred = gd, res
            break
    lg.close()
    if g is None:
        raise SystemExit("no C4 draw passed the judge: every ground keeps the full porous layer")
    total = a.warmup + a.steps
    rec = lee.deck.receivers_c4()
    runs = {}
    for kind in ("porous", "impedance"):
        deck = lee.deck.config_c4(g, kind, a_pred, time_domain=total)
        print(f"[bench] C4 {kind} fp32: {a.warmup} warm-up + {a.steps} timed steps", file=sys.stderr, flush=True)
        runs[kind] = run_gpu(lee, deck, rec, 32, a.steps, a.warmup)
        r = runs[kind]
        print(f"[bench] C4 {kind}: {r['points'] * a.steps / r['wall'] / 1e9:.2f} G pt-updates/s "
              f"({1e3 * r['wall'] / a.steps:.3f} ms/step)", file=sys.stderr, flush=True)
    lp, li = runs["porous"], runs["impedance"]
    rep = judged[-1]
    narrow, third = G.il_errors(lp["series"], li["series"], deck.dt)
    per_rec = [round(G.il_errors(lp["series"][:, n:n + 1], li["series"][:, n:n + 1], deck.dt)[1], 3)
               for n in range(lp["series"].shape[1])]
    rl2 = float(np.linalg.norm(li["series"] - lp["series"]) / np.linalg.norm(lp["series"]))
    speedup = lp["wall"] / li["wall"]
    dom = max(li["kernels"], key=lambda k: k["total_ms"])
    avg_s = dom["total_ms"] / dom["launches"] / 1e3
    achieved = dom["bytes_per_launch"] / avg_s / 1e9
    air = int(np.prod(deck.shape))
    line = {
        "metric": "grid-pt updates/s + %HBM BW, FP32 vs FP64; learned-ground speedup @<=0.2 dB",
        "value": round(li["points"] * a.steps / li["wall"], 1),
        "unit": "grid-pt updates/s",
        "n_gpus": 1, "steps": a.steps, "warmup": a.warmup, "ms_per_step": round(1e3 * li["wall"] / a.steps, 4),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": "C4: 1024x512x160 air at 0.04 m, terrain-following over a Gaussian hill (1 m, sigma "
                               "5 m, y = 12 m), 20-pt PML sides+top, FB_p_v CFL 0.5, "
                               "ground: the first draw of the C3 distribution (seed 20261202) the judge accepts; "
                               "learned 8-pole impedance on the ground interface plane vs the full porous layer",
                   "air_points": air, "ground": vars(g), "porous_points": lp["points"] - air,
                   "parallelism": "single GPU"},
        "roofline": {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": None, "kernel": dom["name"],
                     "bytes_per_launch": dom["bytes_per_launch"], "avg_launch_ms": round(avg_s * 1e3, 4)},
        "cpu_baseline": None,
        "learned_speedup": round(speedup, 3),
        "porous_pt_updates_per_s": lp["points"] * a.steps / lp["wall"],
        "porous_ms_per_step": 1e3 * lp["wall"] / a.steps,
        "accuracy": {"learned_vs_porous_rel_l2": rl2, "max_dIL_dB_50_1000Hz": round(narrow, 4),
                     "bound_dB": 0.2, "narrow_band_within_bound": bool(narrow <= 0.2),
                     "max_dIL_third_octave_dB_50_1000Hz": round(third, 4), "steps": total,
                     "third_octave_dB_per_receiver": dict(zip([f"{r[1] - 3.0:g} m @ {r[2]:g} m" for r in rec], per_rec))},
        "hull": {"sigma_min_Pa_s_m2": G.HULL_SIGMA_MIN,
                 "fraction_of_sweep_draws_inside": hull_fraction,
                 "draws_counted": 4096},
        "judge": judged,
        "training": {"grounds": len(train), "data_s": round(t_data, 2), "train_s": round(t_train, 3),
                     "fit_error_median": float(np.median(E)), "fit_error_max": float(E.max()), "mse": mse},
        "impedance_kernels": kernel_table(li["kernels_all"]),
        "porous_kernels": kernel_table(lp["kernels_all"]),
    }
    print(f"[bench] C4 learned vs porous: speedup {speedup:.3f}, rel-L2 {rl2:.3e}, max dIL {narrow:.3f} dB "
          f"(one-third octave {third:.3f} dB)", file=sys.stderr, flush=True)
    print(json.dumps(line))


def kernel_table(kernels):
    return [{k: (round(v, 4) if isinstance(v, float) else v) for k, v in kk.items()} for kk in kernels]


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--workload", choices=("c1", "c2", "c3", "c4"), default="c1")
    ap.add_argument("--steps", type=int, default=None, help="timed steps (C1: 10000, C2: 2000, C3: 3000, C4: 8000)")
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-fb", action="store_true", help="skip the reference-scheme (FB_p_v, flat) lines")
    ap.add_argument("--precisions", default="32,64")
    ap.add_argument("--eager", action="store_true", help="C4: launch the column and judge runs eagerly (no graphs)")
    ap.add_argument("--accuracy-steps", type=int, default=None,
                    help="C1/C2: steps of the untimed FP32-vs-FP64 accuracy pass when the timed run is shorter "
                         "(default: the whole workload, 10000 / 2000; 0 skips it)")
    ap.add_argument("--rk-tile", type=int, default=0,
                    help="RK4 air-stage launch shape 1..11 (lee_options.rk_tile; default 0: autotuned), for "
                         "profiling runs that should not time the tuner's trials")
    ap.add_argument("--traffic-json", default=os.path.join(ROOT, "profiles", "rk4_air_c1_traffic.json"),
                    help="JSON {kernel: HBM bytes per launch} from rocprofv3 FETCH_SIZE/WRITE_SIZE runs")
    a = ap.parse_args()
    global RK_TILE
    RK_TILE = a.rk_tile
    if a.gpus != 1:
        print(f"bench.py runs on one GPU only (asked for --gpus {a.gpus}): the domain lives in one "
              "GPU's HBM and no multi-GPU path is built", file=sys.stderr)
        sys.exit(2)
    lee = importlib.import_module("3d_mpi_test_amd")
    if a.steps is None:
        a.steps = {"c1": 10000, "c2": 2000, "c3": 3000, "c4": 8000}[a.workload]
    if a.workload == "c3":
        run_c3(lee, a)
        return
    if a.workload == "c4":
        run_c4(lee, a)
        return
    total = a.warmup + a.steps
    if a.workload == "c1":
        deck = lee.deck.config_c1(time_domain=total)
        rec = lee.deck.receivers_c1()
        workload = ("C1: 512x256x128 air at 0.04 m, terrain-following over a Gaussian hill (2 m, sigma 5 m), "
                    "16-point porous ground (200 kPa s/m^2, 0.3, 3), 20-pt PML sides+top, log wind u*=0.4 m/s "
                    "z0=0.02 m, moving frame, 32 receivers at 1.2 m, RK4 CFL 0.5")
    else:
        deck = lee.deck.config_c2(time_domain=total)
        rec = lee.deck.receivers_c2()
        workload = ("C2: 768x384x192 air at 0.04 m, terrain-following over 6 seeded random Gaussian hills "
                    "(heights U[0,1.5] m, widths U[3,10] m), 24-point porous ground, 20-pt PML sides+top, no wind, "
                    "32 receivers at 1.2 m, RK4 CFL 0.5")
    wl = a.workload.upper()
    res = {}
    for p in [int(x) for x in a.precisions.split(",")]:
        print(f"[bench] {wl} RK4 fp{p}: {a.warmup} warm-up + {a.steps} timed steps", file=sys.stderr, flush=True)
        res[p] = run_gpu(lee, deck, rec, p, a.steps, a.warmup)
        r = res[p]
        print(f"[bench] {wl} RK4 fp{p}: {r['points'] * a.steps / r['wall'] / 1e9:.2f} G pt-updates/s "
              f"({1e3 * r['wall'] / a.steps:.3f} ms/step, {r['frames']} frames)", file=sys.stderr, flush=True)
    head = 32 if 32 in res else list(res)[0]
    r = res[head]
    value = r["points"] * a.steps / r["wall"]
    dom = max(r["kernels"], key=lambda k: k["total_ms"])
    avg_s = dom["total_ms"] / dom["launches"] / 1e3
    achieved = dom["bytes_per_launch"] / avg_s / 1e9
    traffic = traffic_src = None
    if a.traffic_json and os.path.exists(a.traffic_json) and a.workload == "c1":
        # HBM bytes per launch of the launch shape this run's autotuner kept (the profiles
        # measure each shape; null for a shape they do not hold)
        with open(a.traffic_json) as fh:
            tj = json.load(fh)
        per_shape = tj.get(f"{dom['name']}_fp{head}") or {}
        traffic = per_shape.get(r["rk_tile"]) if isinstance(per_shape, dict) else None
        traffic_src = tj.get("_source") if traffic is not None else None
    roof = {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
            "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": traffic, "traffic_source": traffic_src,
            "kernel": dom["name"], "launch_shape": r["rk_tile"],
            "bytes_per_launch": dom["bytes_per_launch"], "avg_launch_ms": round(avg_s * 1e3, 4),
            "copy_kernel_GBs": round(2 * (1 << 30) / (r["copy_ms"] / 1e3) / 1e9, 1) if r["copy_ms"] > 0 else None}
    if r["stream_ms"] > 0:
        sgb = sum(STREAMS) * (1 << 26) / (r["stream_ms"] / 1e3) / 1e9
        roof["stream_kernel"] = {"reads": STREAMS[0], "writes": STREAMS[1], "GB/s": round(sgb, 1),
                                 "achieved_over_it": round(achieved / sgb, 4)}
    acc = None
    if 32 in res and 64 in res:
        full = {"c1": 10000, "c2": 2000}[a.workload] if a.accuracy_steps is None else a.accuracy_steps
        ser, steps_acc, src = {p: res[p]["series"] for p in (32, 64)}, total, "the timed runs"
        if total < full:
            # the timed run is shorter than the workload: the accuracy comes from an untimed
            # pass of the whole workload, so the figure is the same whatever --steps is
            adeck = (lee.deck.config_c1 if a.workload == "c1" else lee.deck.config_c2)(time_domain=full)
            for p in (32, 64):
                print(f"[bench] accuracy pass {wl} RK4 fp{p}: {full} untimed steps", file=sys.stderr, flush=True)
                ser[p] = run_series(lee, adeck, rec, p, full)
            steps_acc, src = full, "an untimed pass of the whole workload"
        m = accuracy(ser[64], ser[32], deck.dt)
        if m is not None:
            rl2, dil, nrec = m
            acc = {"fp32_vs_fp64_rel_l2": rl2, "max_dIL_dB_50_1000Hz": round(dil, 5), "receivers_with_signal": nrec,
                   "receivers": len(rec), "steps": steps_acc, "series_from": src}
            print(f"[bench] FP32 vs FP64 ({steps_acc} steps, {nrec} receivers with signal): rel-L2 {rl2:.3e}, "
                  f"max |dIL| {dil:.4f} dB over 50-1000 Hz", file=sys.stderr, flush=True)
    fb = {}
    if not a.no_fb and a.workload == "c1":
        # the reference's own scheme on the same grid: FB_p_v, flat ground, no wind
        fdeck = lee.deck.config_c1(time_domain=220, reference_scheme=True)
        for p in (32, 64):
            print(f"[bench] C1 reference scheme FB_p_v fp{p}", file=sys.stderr, flush=True)
            rr = run_gpu(lee, fdeck, rec, p, 200, 20, record=False)
            fb[f"fb_fp{p}_pt_updates_per_s"] = rr["points"] * 200 / rr["wall"]
            fb[f"fb_fp{p}_ms_per_step"] = 1e3 * rr["wall"] / 200
            fb[f"fb_fp{p}_kernels"] = kernel_table(rr["kernels_all"])
            fb[f"fb_fp{p}_launch_form"] = rr["fb_form"]
    cpu = cpu_ref = None
    if not a.no_cpu:
        from oracle import oracle as orc
        nthr = orc.get_threads()
        model = cpu_model()
        print(f"[bench] cpu baseline (oracle, {nthr} threads, then 1; {model})", file=sys.stderr, flush=True)
        c = cpu_baseline(deck, rec, threads=nthr)
        c1 = cpu_baseline(deck, rec, budget_s=15.0, threads=1)
        cpu = {"value": round(c["value"], 1), "unit": "grid-pt updates/s", "cores": c["threads"], "kind": "port",
               "sample": f"{wl} (RK4, terrain, porous ground) FP64, first {c['steps']} step(s) "
                         f"({c['seconds']:.1f} s) on {c['threads']} OpenMP threads of {model}",
               "single_thread_value": round(c1["value"], 1),
               "single_thread_sample": f"first {c1['steps']} step(s) ({c1['seconds']:.1f} s), one thread"}
        if a.workload == "c1" and not a.no_fb:
            # the reference's own scheme (FB_p_v) on the CPU, beside the GPU FB lines: the C1
            # grid flat (a bounded sample), and the 96x64x48 workload in full (2000 steps) on
            # every thread and a sample of it on one
            print("[bench] cpu baseline, reference scheme FB_p_v (C1 grid; 96x64x48 x 2000 steps)", file=sys.stderr,
                  flush=True)
            fdeck = lee.deck.config_c1(time_domain=220, reference_scheme=True)
            f_all = cpu_baseline(fdeck, rec, budget_s=12.0, threads=nthr)
            f_one = cpu_baseline(fdeck, rec, budget_s=10.0, threads=1, max_steps=2)
            c0 = lee.deck.config_c0(time_domain=2000, reference_scheme=True)
            c0_all = cpu_baseline(c0, lee.deck.receivers_c0(), budget_s=1e9, threads=nthr, max_steps=2000)
            c0_one = cpu_baseline(c0, lee.deck.receivers_c0(), budget_s=12.0, threads=1, max_steps=2000)
            cpu_ref = {"cpu": model, "unit": "grid-pt updates/s", "kind": "port",
                       "c1_grid_fb": {"threads": f_all["threads"], "value": round(f_all["value"], 1),
                                      "sample": f"first {f_all['steps']} step(s) ({f_all['seconds']:.1f} s)",
                                      "single_thread_value": round(f_one["value"], 1),
                                      "single_thread_sample": f"first {f_one['steps']} step(s) "
                                                              f"({f_one['seconds']:.1f} s)"},
                       "c0_fb": {"threads": c0_all["threads"], "value": round(c0_all["value"], 1),
                                 "steps": c0_all["steps"], "seconds": round(c0_all["seconds"], 2),
                                 "single_thread_value": round(c0_one["value"], 1),
                                 "single_thread_sample": f"first {c0_one['steps']} step(s) "
                                                         f"({c0_one['seconds']:.1f} s)"}}
        orc.set_threads(nthr)
    extra = {}
    for p, rr in res.items():
        extra[f"fp{p}_pt_updates_per_s"] = rr["points"] * a.steps / rr["wall"]
        extra[f"fp{p}_ms_per_step"] = 1e3 * rr["wall"] / a.steps
        extra[f"fp{p}_kernels"] = kernel_table(rr["kernels_all"])
    if 32 in res and 64 in res:
        extra["fp32_over_fp64"] = round(extra["fp32_pt_updates_per_s"] / extra["fp64_pt_updates_per_s"], 3)
    line = {
        "metric": "grid-pt updates/s + %HBM BW, FP32 vs FP64; learned-ground speedup @<=0.2 dB",
        "value": round(value, 1),
        "unit": "grid-pt updates/s",
        "n_gpus": 1,
        "steps": a.steps,
        "warmup": a.warmup,
        "ms_per_step": round(1e3 * r["wall"] / a.steps, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": f"f{head}",
        "data": "synthetic",
        "config": {"workload": workload,
                   "air_points": int(np.prod(deck.shape)), "porous_points": r["points"] - int(np.prod(deck.shape)),
                   "frames_in_run": r["frames"], "integrator": "RK4 (FP32: compensated accumulation)",
                   "rk_air_launch": r["rk_tile"],
                   "parallelism": "single GPU"},
        "roofline": roof,
        "cpu_baseline": cpu,
        "cpu_baseline_reference_scheme": cpu_ref,
        "accuracy": acc,
        **extra,
        **fb,
    }
    print(json.dumps(line))


if __name__ == "__main__":
    main()
