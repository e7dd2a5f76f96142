"""Times the walking kernels and every configuration of the two matrix kernels on a set of layers, and checks the time models that
the library chooses between them with, or fits them (csrc/matrix_conv.hip).

    make fit                                                  the library with the entry points used here
    TETRIS_SPCONV2D_LIB=$PWD/build_fit/libtetris_spconv2d.so python -m tetris_amd.kernel_times --measure FILE     (GPU)
    TETRIS_SPCONV2D_LIB=... python -m tetris_amd.kernel_times --fit FILE      (CPU: the models' constants, fitted)
    TETRIS_SPCONV2D_LIB=... python -m tetris_amd.kernel_times --check FILE    (CPU: how far the built-in models are off)

FILE: one line per layer -- N C H W K ks stride pad nnz, the walking tile (six numbers), its microseconds, then per matrix
configuration the microseconds with 1, 2, 3, 4, 6 and 8 slices ("-": cannot be run).  Layers: those of the benchmark's
suites at batch 1, 4 and 16, and random ones.  Every time is the mean of back-to-back launches, the better of two.
"""
import argparse
import ctypes as C
import math
import random
import sys

import numpy as np

import tetris_amd as T
from tetris_amd import workloads as W

# kMatShapes in csrc/matrix.h: a team's waves along the channels and along the pixels, pixel blocks of a wave, teams; those of
# matrix_kernel, then those of half_kernel, four with long and eight with short chunks of channels
CONFIGS = [(4, 1, 4, 1), (4, 1, 4, 2), (4, 1, 2, 1), (4, 1, 2, 2), (4, 1, 2, 4), (2, 2, 2, 1), (2, 2, 2, 2), (2, 2, 2, 4),
           (2, 2, 1, 1), (2, 2, 1, 2), (2, 2, 1, 4),
           (8, 1, 2, 1), (8, 1, 3, 1), (4, 1, 2, 2), (2, 2, 1, 2),
           (8, 1, 2, 1), (8, 1, 3, 1), (8, 1, 4, 1), (4, 2, 3, 1), (4, 2, 4, 1), (4, 1, 2, 2), (2, 2, 1, 1), (2, 2, 1, 2)]
# half_kernel is taken where it is predicted to be faster than matrix_kernel by this, and its margin to the walking kernel is larger
# by that (choose_mat_geom)
BIAS, MORE = 1.05, 0.09
SLICES = (1, 2, 3, 4, 6, 8)
I16 = C.c_int * 16


def layers(count, seed):
    seen = set()
    for suite in ("single", "vgg19", "resnet50", "mobilenet", "yolov3"):
        for L in W.SUITES[suite]():
            for n in (1, 4, 16):
                key = (n, L.C, L.H, L.W, L.K, L.ks, L.stride, L.pad)
                if L.C >= 16 and key + (L.sparsity,) not in seen:
                    seen.add(key + (L.sparsity,))
                    yield key, L.sparsity
    rnd = random.Random(seed)
    spread = lambda lo, hi: int(round(math.exp(rnd.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    while count:
        ks, stride = rnd.choice([(1, 1), (1, 1), (3, 1), (3, 1), (3, 1), (1, 2), (3, 2), (5, 1)])
        n, c, k, h = spread(1, 16), spread(16, 1024), spread(16, 1024), spread(7, 224)
        w = h if rnd.random() < 0.6 else max(7, int(h * rnd.uniform(0.6, 1.4)))
        if 2.0 * n * k * c * (ks * h / stride) * (ks * w / stride) > 6e11 or n * max(c, k) * h * w > 1 << 27 or c * k * ks * ks > 5 << 19:
            continue
        count -= 1
        yield (n, c, h, w, k, ks, stride, ks // 2), round(rnd.uniform(0.70, 0.95), 3)


def measure(path, count):
    import torch

    time = T._lib.tetris_fit_time
    time.argtypes = [C.c_void_p] * 3 + [C.c_int] * 5 + [C.POINTER(T.Tile)] + [C.c_int] * 4 + [C.POINTER(C.c_float)]
    with open(path, "w") as f:
        f.write("# N C H W K ks stride pad nnz  lanes_w quads oc_per_wave waves tile_ic csplit  walk  us per configuration %s "
                "with %s slices\n" % (CONFIGS, SLICES))
        for i, (key, sparsity) in enumerate(layers(count, 1)):
            n, c, h, w, k, ks, stride, pad = key
            rng = np.random.default_rng(i)
            filt = (rng.standard_normal((k, c, ks, ks)) * 0.05 * (rng.random((k, c, ks, ks)) >= sparsity)).astype(np.float32)
            nnz = int(np.count_nonzero(filt))
            tile = T.tile_select(n, h, w, c, k, ks, stride, pad)
            pk = T.G950Filter.for_tile(filt, tile, oc_order="balanced")
            x = torch.rand((n, c, h, w), device="cuda").sub_(0.5).clamp_(min=0)
            y = torch.empty((n, k, T.out_extent(h, pad, ks, stride), T.out_extent(w, pad, ks, stride)), device="cuda")
            torch.cuda.synchronize()
            us = C.c_float()

            def run(cfg, slices, warm, repeat):
                rc = time(pk._h, x.data_ptr(), y.data_ptr(), n, h, w, stride, pad, C.byref(tile), cfg, slices, warm, repeat,
                          C.byref(us))
                return us.value if rc == 0 else None

            out, info, pred = [], I16(), C.c_double()
            run(-1, 1, int(4e4 / run(-1, 1, 3, 5)), 1)  # after the pause for the filter the shader clock needs some 30 ms of work
            best = walk = min(run(-1, 1, 3, 10), run(-1, 1, 1, 10))
            for cfg in range(len(CONFIGS)):
                row = []
                for s in SLICES:
                    ok = T._lib.tetris_fit_matrix_geom(n, c, h, w, k, ks, stride, pad, cfg, s, info, C.c_longlong(nnz), C.byref(pred)) == 0
                    first = run(cfg, s, 2, 5) if ok else None
                    if first is None or first > 3 * best:
                        row.append("-")
                    else:
                        first = min(first, run(cfg, s, 1, 10))
                        best = min(best, first)
                        row.append("%.1f" % first)
                out.append("|".join(row))
            t = [tile.lanes_w, tile.quads, tile.oc_per_wave, tile.waves, tile.tile_ic, tile.csplit]
            f.write(" ".join(map(str, list(key) + [nnz] + t)) + " %.1f " % walk + " ".join(out) + "\n")
            f.flush()
            print(i, key, sparsity, "walk %.1f best %.1f" % (walk, best), flush=True)
            pk.close()


def read(path):
    """-> per layer (walk features, walk us, walk prediction, [(matrix features, us, prediction), ...])"""
    out, info, pred = [], I16(), C.c_double()
    for line in open(path):
        if line.startswith("#"):
            continue
        v = line.split()
        key, nnz, tile = [int(a) for a in v[:8]], int(v[8]), T.Tile(*[int(a) for a in v[9:15]])
        n, c, h, w, k, ks, stride, pad = key
        order = (n, c, h, w, k, ks, stride, pad)
        T._check(T._lib.tetris_fit_walk_geom(*order, C.byref(tile), C.c_longlong(nnz), info, C.byref(pred)))
        layer = dict(zip("N C H W K ks".split(), key[:6]), nnz=nnz)
        names = "ugroups kblocks csplit stages waves nq g ver OH OW one".split()
        walk = (dict(layer, **dict(zip(names, info))), float(v[15]), pred.value)
        rows = []
        for cfg, field in enumerate(v[16:]):
            for s, us in zip(SLICES, field.split("|")):
                if us != "-":
                    T._check(T._lib.tetris_fit_matrix_geom(*order, cfg, s, info, C.c_longlong(nnz), C.byref(pred)))
                    names = "ptiles mtiles csplit chunks kgs lpad OH OW lds mblocks half".split()
                    rows.append((dict(layer, cfg=cfg, **dict(zip(names, info))), float(us), pred.value))
        out.append((walk, rows))
    return out


def columns(features):
    return {k: np.array([f[k] for f in features], np.float64) for k in features[0]}


def filled(wgs, fit, cycles):
    """cycles of whole rounds of 256 * fit workgroups and of the rest, which is spread over the CUs"""
    full, rest = np.floor(wgs / (256 * fit)), wgs % (256 * fit)
    last = np.ceil(rest / 256)
    return full * cycles(fit) + np.where(last > 0, cycles(last), 0)


PLAIN0 = dict(start=3214, team=733, round1=1213, round3=2935, staging=293, step=469, product=1.08, launch=2.06,
              reread=0.72, rate=4.26, weights=2.9, add=2.37, add_rate=3.95)


def plain_model(p, f):
    wm, wn, nb, kw = (np.array([CONFIGS[int(c)][i] for c in f["cfg"]]) for i in range(4))
    regs = np.select([nb == 4, nb == 2, kw == 1, kw == 2], [2 // kw, np.maximum(1, 3 // kw), 5, 2], 1)
    fit = np.maximum(1, np.minimum(regs, np.floor(160 * 1024 / f["lds"])))
    rounds = np.ceil(np.ceil(f["chunks"] / f["csplit"]) / kw)
    steps, staging = f["ks"] ** 2 * f["kgs"] / 2, np.ceil(f["kgs"] * f["lpad"] / 256)
    one = f["ks"] == 1

    def cycles(n):
        step = np.maximum(np.where(one, 0, p["step"]), p["product"] * 256 * nb * kw * n)
        return (p["start"] + p["team"] * nb * n * kw +
                rounds * (np.where(one, p["round1"], p["round3"]) + p["staging"] * staging * kw * n + steps * step))

    compute = filled(f["ptiles"] * f["mtiles"] * f["csplit"], fit, cycles) / 2.2e3
    out = 4 * f["N"] * f["K"] * f["OH"] * f["OW"]
    inp = 4 * f["N"] * f["C"] * np.where(one, f["OH"], f["H"]) * f["W"]
    memory = (inp * (1 + p["reread"] * np.sqrt(f["mtiles"] - 1)) + out * f["csplit"] + p["weights"] * 3072 * f["mblocks"] * f["chunks"] * steps) / (p["rate"] * 1e6)
    return p["launch"] + np.maximum(compute, memory) + np.where(f["csplit"] > 1, p["add"] + out * (f["csplit"] + 1) / (p["add_rate"] * 1e6), 0)


HALF0 = dict(start=4973, team=1257, round1=221, round3=722, staging=681, step=165, issue=2.032, product=1.231, work=87,
             launch=1.67, add=2.48, add_rate=4.3)


def half_model(p, f):
    wm, wn, nb, kw = (np.array([CONFIGS[int(c)][i] for c in f["cfg"]], np.float64) for i in range(4))
    team = wm * wn
    waves = team * kw
    regs = np.maximum(1, np.floor(np.where(nb >= 2, 8, 12) / waves))
    fit = np.maximum(1, np.minimum(regs, np.floor(160 * 1024 / f["lds"])))
    rounds = np.ceil(np.ceil(f["chunks"] / f["csplit"]) / kw)
    density = np.minimum(1, f["nnz"] / (f["K"] * f["C"] * f["ks"] ** 2))
    more = density ** 3 * (4 - 3 * density)
    steps = np.ceil(f["C"] / 8) * f["ks"] ** 2 / f["chunks"] * (2 - (1 - more) ** 64) / 4 + 0.375
    staging = f["kgs"] * f["lpad"] / 64 / team
    one = f["ks"] == 1

    def cycles(n):
        w = n * waves / 4
        step = np.maximum(p["step"] + p["issue"] * 192 * nb, (p["work"] + p["product"] * 192 * nb) * w)
        return p["start"] + p["team"] * nb * w + rounds * (np.where(one, p["round1"], p["round3"]) + p["staging"] * staging * w + steps * step)

    out = 4 * f["N"] * f["K"] * f["OH"] * f["OW"]
    return p["launch"] + filled(f["ptiles"] * f["mtiles"] * f["csplit"], fit, cycles) / 2.3e3 + np.where(
        f["csplit"] > 1, p["add"] + out * (f["csplit"] + 1) / (p["add_rate"] * 1e6), 0)


WALK0 = dict(start2=9249, start3=10770, start4=8002, stage2=2913, stage3=5287, stage4=1239, busy2=1.55, busy3=0.905,
             busy4=1.415, alone2=65.4, alone3=104, alone4=59.4, rate=5.01, add=1.61, add_rate=2.96)


def walk_model(p, f):
    pick = lambda name: np.select([f["ver"] == 2, f["ver"] == 3], [p[name + "2"], p[name + "3"]], p[name + "4"])  # noqa: E731
    entry = np.select([f["nq"] == 1, f["nq"] == 2], [26.2, 43.5], 85.0)
    entries = (f["nnz"] / f["K"] * f["g"] + 1.05 * f["stages"]) / f["csplit"]
    fit = np.where(f["one"] > 0, 1, 2)

    def cycles(n):
        return pick("start") + pick("stage") * f["stages"] / f["csplit"] + np.maximum(
            entries * n * f["waves"] / 4 * entry * pick("busy"), entries * pick("alone") * np.sqrt(f["nq"]))

    compute = filled(f["ugroups"] * f["kblocks"] * f["csplit"], fit, cycles) / 2.3e3
    out, inp = 4 * f["N"] * f["K"] * f["OH"] * f["OW"], 4 * f["N"] * f["C"] * f["H"] * f["W"]
    return np.maximum(compute, (inp + out) / (p["rate"] * 1e6)) + np.where(
        f["csplit"] > 1, p["add"] + out * (f["csplit"] + 1) / (p["add_rate"] * 1e6), 0)


def fit(model, start, features, us, weight):
    from scipy.optimize import least_squares

    names, f, us = list(start), columns(features), np.array(us)
    x0 = np.log([start[k] for k in names])
    loss = lambda x: weight * np.log(model(dict(zip(names, np.exp(x))), f) / us)  # noqa: E731
    r = least_squares(loss, x0, loss="soft_l1", f_scale=0.2, diff_step=1e-3)
    return dict(zip(names, np.exp(r.x)))


def report(data, predict_matrix, predict_walk, margins):
    """what choosing by the two predictions gives over all layers, against the walk alone and the best of what was timed"""
    for half, name in ((0, "matrix_kernel"), (1, "half_kernel")):
        off = np.log([predict_matrix(f, p) / us for _, rows in data for f, us, p in rows if f["half"] == half])
        if len(off):
            print("%s: %d times, predictions %+.1f %% on average, standard deviation %.1f %%" % (name, len(off), 100 * off.mean(), 100 * off.std()))
    off_w = np.log([predict_walk(w[0], w[2]) / w[1] for w, _ in data])
    weighed = lambda f, p: predict_matrix(f, p) * (BIAS if f["half"] else 1)  # noqa: E731
    print("walking kernels: %d times, predictions %+.1f %% on average, standard deviation %.1f %%" % (len(off_w), 100 * off_w.mean(), 100 * off_w.std()))
    named = []
    for walk, rows in data:
        if rows:
            us, pred = np.array([r[1] for r in rows]), np.array([weighed(r[0], r[2]) for r in rows])
            named.append(us[pred.argmin()] / us.min())
    print("the configuration of least predicted time is %.1f %% slower than the fastest" % (100 * (np.exp(np.mean(np.log(named))) - 1)))
    for m in margins:
        lost, gain, taken, slower = [], [], [0, 0], []
        for walk, rows in data:
            pw = predict_walk(walk[0], walk[2])
            below = [r for r in rows if predict_matrix(r[0], r[2]) < (1 - m - (MORE if r[0]["half"] else 0)) * pw]
            use = min(below, key=lambda r: weighed(r[0], r[2]), default=None)
            us = use[1] if use else walk[1]
            lost.append(us / min([walk[1]] + [r[1] for r in rows]))
            gain.append(walk[1] / us)
            if use:
                taken[int(use[0]["half"])] += 1
            if us > 1.03 * walk[1]:
                slower.append(us / walk[1])
        print("margin %.2f: matrix_kernel on %d and half_kernel on %d of %d layers; %.3f x the walk on (geometric) average, %.1f %% from the best choice; "
              "%d layers more than 3 %% slower than the walk (worst %.2f x)" % (m, taken[0], taken[1], len(data), np.exp(np.mean(np.log(gain))),
              100 * (np.exp(np.mean(np.log(lost))) - 1), len(slower), max(slower, default=1)))


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--measure", metavar="FILE")
    ap.add_argument("--random", type=int, default=160, help="random layers to measure besides the suites'")
    ap.add_argument("--fit", metavar="FILE")
    ap.add_argument("--check", metavar="FILE")
    a = ap.parse_args()
    margins = (0, 0.03, 0.05, 0.07, 0.1, 0.15, 0.2)
    if a.measure:
        measure(a.measure, a.random)
    elif a.check:
        report(read(a.check), lambda f, p: p, lambda f, p: p, margins)
    elif a.fit:
        data = read(a.fit)
        # the fastest configurations of a layer decide, and are weighed accordingly
        models = {}
        for half, name, model, start in ((0, "plain_time", plain_model, PLAIN0), (1, "half_time", half_model, HALF0)):
            fm, um, wm = [], [], []
            for walk, rows in data:
                best = min([r[1] for r in rows], default=0)
                for f, us, _ in rows:
                    if f["half"] == half:
                        fm.append(f), um.append(us), wm.append((best / us) ** 2 / math.sqrt(len(rows)))
            models[half] = model, fit(model, start, fm, um, np.array(wm))
            print(name, ", ".join("%s %.4g" % kv for kv in models[half][1].items()))
        pw = fit(walk_model, WALK0, [w[0] for w, _ in data], [w[1] for w, _ in data], 1.0)
        print("walk_time", ", ".join("%s %.4g" % kv for kv in pw.items()))
        one = lambda model, p, f: float(model(p, columns([f]))[0])  # noqa: E731
        report(data, lambda f, _: one(*models[f["half"]], f), lambda f, _: one(walk_model, pw, f), margins)
    else:
        sys.exit("one of --measure, --fit, --check")


if __name__ == "__main__":
    main()
