"""Measure the best tile for every layer shape of the benchmark suites and write csrc/tuned_tiles.inc.

Timing alone:
    python -m tetris_amd.tune [--suites vgg19 resnet50 ...] [--batches 1 2 4 8 16] [--candidates 48] [--cold]

Timing first, then rocprofv3's HBM counters to choose among near ties (from the repository root, on the GPU the
table is meant for):
    python -m tetris_amd.tune --shortlist FILE.json [--cold] [--include TABLE.inc] ...
                                                  the four fastest tiles of every shape, timed (and TABLE's tile)
    rocprofv3 --pmc FETCH_SIZE --output-format csv -d DIR_F -- python3 -m tetris_amd.tune --replay FILE.json
    rocprofv3 --pmc WRITE_SIZE --output-format csv -d DIR_W -- python3 -m tetris_amd.tune --replay FILE.json
    rocprofv3 --pmc SQ_LDS_BANK_CONFLICT SQ_LDS_IDX_ACTIVE --output-format csv -d DIR_S -- python3 -m tetris_amd.tune --replay FILE.json
    python -m tetris_amd.tune --choose FILE.json --fetch DIR_F --write DIR_W [--lds DIR_S] [--within 0.02]
--replay launches every shortlisted tile once, in the order of the file; --choose reads the counters of those
dispatches back (FETCH_SIZE and WRITE_SIZE in KiB, scaled by --fetch-scale / --write-scale: what the same counters
read for a copy of known size), and takes, for a layer whose binding roof is HBM, among the tiles no more than
--within (2 %) slower than the fastest, the one that moved the fewest bytes; a layer bound by the vector units takes
its fastest tile unless --within-compute gives it slack too (on the VGG19-shaped stack at batch 16 three per cent of
slack took the bytes moved from 1.66 to 1.29 times the algorithmic ones and cost 2.2 % of the pass).  Every row of the table then carries the time, the bytes moved and
the LDS bank-conflict rate that chose it.

With --base TABLE, --choose keeps TABLE's tile for a shape unless it moves more than --waste (2) times the layer's
algorithmic bytes and a tile within --within of the fastest moves fewer: a rule against gross waste only.  (On the
VGG19 stack it switches the 28x28 and 14x14 layers to tiles that do not split the channel reduction and costs 2.1 %
of the pass at batch 16, 5.9 % at batch 1; the built-in table keeps the faster tiles.)

    python -m tetris_amd.tune --refine OLD.inc NEW.inc --out MERGED.inc [--cold-suites resnet50 mobilenet single]
times, for every shape on which two tables disagree, both tiles head to head (three alternating rounds of 30 launches;
from cold caches for the suites named) and keeps OLD's row unless NEW's tile is faster by more than --margin.

A table other than the built-in one is for tetris_tile_table_load, whose rows are obeyed: a layer that the library runs
faster on the matrix cores than the best walking tile does gets no row there.  All times of tiles are those of the
walking kernels.

Rebuild the library afterwards.  tetris_tile_select consults the table before its cycle model; a shape that is not
listed, or whose tile the kernel's checks refuse, falls back to the model.
"""
import argparse
import csv
import glob
import json
import os
import sys
import tempfile

import tetris_amd as T
from tetris_amd import workloads as W


BUILT_IN = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "csrc", "tuned_tiles.inc")


def own_choice_ms(w, L, n, cold):
    """Milliseconds per launch where the library runs the layer on the matrix cores, else None."""
    import torch

    tile = T.tile_select(n, L.H, L.W, L.C, L.K, L.ks, L.stride, L.pad)
    pk = T.G950Filter.for_tile(w, tile, oc_order="balanced")
    try:
        if pk.launch_shape(n, L.H, L.W, L.stride, L.pad, tile).kernel != 5:
            return None
        x = torch.zeros((n, L.C, L.H, L.W), device="cuda")
        y = torch.empty((n, L.K) + tuple(W.out_hw(L)), device="cuda")
        return pk.time(x.data_ptr(), y.data_ptr(), n, L.H, L.W, L.stride, L.pad, tile, warm=2 if cold else 5, repeat=10)
    finally:
        pk.close()


def shapes(args):
    """(key, layer, batch, suite) of every distinct layer shape; layers of one shape differ in sparsity and the table
    knows shapes only, so the densest (the slowest) is measured."""
    seen = set()
    for suite in args.suites:
        layers = {}
        for L in W.SUITES[suite]():
            k = (L.H, L.W, L.C, L.K, L.ks, L.stride, L.pad)
            if args.layers and not any(name in L.name for name in args.layers):
                continue
            if k not in layers or L.sparsity < layers[k].sparsity:
                layers[k] = L
        for L in layers.values():
            for n in args.batches:
                key = (n, L.H, L.W, L.C, L.K, L.ks, L.stride, L.pad)
                if key not in seen:
                    seen.add(key)
                    yield key, L, n, suite


ROW = (r"\s*\{(\d+), (\d+), (\d+), (\d+), (\d+), (\d+), (\d+), (\d+), "
       r"\{(\d+), (\d+), (\d+), (\d+), (\d+)(?:, (\d+))?\}\}")


def row_tile(groups):
    """The tile of a table row matched by ROW: five numbers, or six when the row fixes csplit."""
    v = [int(x) for x in groups[8:14] if x is not None]
    return tuple(v[:5] + ([v[5]] if len(v) > 5 and v[5] else []))


def tile_text(t):
    return "{" + ", ".join("%d" % v for v in t) + "}"


def write_table(path, rows):
    with open(path, "w") as f:
        f.write("// Generated by tetris_amd/tune.py -- {N, H, W, C, K, ks, stride, pad, {lanes_w, quads, oc_per_wave, "
                "waves, tile_ic[, csplit]}},\n")
        for key, t, note in rows:
            f.write("    {%d, %d, %d, %d, %d, %d, %d, %d, %s},  // %s\n" % (tuple(key) + (tile_text(t), note)))
    print("wrote %d shapes to %s" % (len(rows), path), file=sys.stderr)


def obey(key, tile):
    """From now on `tile` is a loaded row for this shape: its launches run the walking kernel it describes, not the matrix
    kernel that the library may predict to be faster where a tile is the one it would choose itself."""
    with tempfile.NamedTemporaryFile("w", suffix=".inc") as f:
        f.write("    {%d, %d, %d, %d, %d, %d, %d, %d, %s},\n" % (tuple(key) + (tile_text(tile),)))
        f.flush()
        T.tile_table_load(f.name)


def counter_sums(directory, names):
    """Per conv launch, in dispatch order: the sum of the named counters over the conv kernel and the kernel that may
    follow it to add the slices (reduce_kernel or add_kernel)."""
    files = glob.glob(os.path.join(directory, "**", "*counter_collection.csv"), recursive=True)
    if not files:
        sys.exit("no counter_collection.csv under %s" % directory)
    per = {}
    for r in csv.DictReader(open(files[0])):
        if r["Counter_Name"] in names:
            d = per.setdefault(int(r["Dispatch_Id"]), [r["Kernel_Name"], {}])
            d[1][r["Counter_Name"]] = d[1].get(r["Counter_Name"], 0.0) + float(r["Counter_Value"])
    out = []
    for did in sorted(per):
        name, vals = per[did]
        if "spconv2d_" in name:
            out.append(dict(vals))
        elif ("reduce_kernel" in name or "add_kernel" in name) and out:
            for k, v in vals.items():
                out[-1][k] = out[-1].get(k, 0.0) + v
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--suites", nargs="+", default=["single", "vgg19", "resnet50", "mobilenet", "yolov3"])
    ap.add_argument("--batches", nargs="+", type=int, default=[1, 2, 4, 8, 16])
    ap.add_argument("--layers", nargs="+", metavar="NAME", help="only layers whose name contains one of these")
    ap.add_argument("--candidates", type=int, default=48)
    ap.add_argument("--cold", action="store_true",
                    help="time every candidate from cold caches (TETRIS_OPT_COLD_TIMING): the conditions a layer meets in "
                         "the middle of a network, rather than those of back-to-back launches of one layer")
    ap.add_argument("--shortlist", metavar="FILE", help="write the four fastest tiles of every shape, with their times")
    ap.add_argument("--include", metavar="TABLE", help="with --shortlist: also time the tile an existing table holds for "
                    "each shape, so that the incumbent competes under the same rule")
    ap.add_argument("--replay", metavar="FILE", help="launch every tile of a shortlist once (run under rocprofv3 --pmc)")
    ap.add_argument("--choose", metavar="FILE", help="choose from a shortlist with the counters of its replays")
    ap.add_argument("--fetch", metavar="DIR", help="rocprofv3 output of the FETCH_SIZE replay")
    ap.add_argument("--write", metavar="DIR", help="rocprofv3 output of the WRITE_SIZE replay")
    ap.add_argument("--lds", metavar="DIR", help="rocprofv3 output of the SQ_LDS_BANK_CONFLICT SQ_LDS_IDX_ACTIVE replay")
    ap.add_argument("--fetch-scale", type=float, default=2.0, help="bytes per FETCH_SIZE KiB / 1024 (copy calibration)")
    ap.add_argument("--write-scale", type=float, default=1.0, help="bytes per WRITE_SIZE KiB / 1024 (copy calibration)")
    ap.add_argument("--refine", nargs=2, metavar=("OLD", "NEW"), help="two tables to reconcile by head-to-head timing")
    ap.add_argument("--margin", type=float, default=0.015, help="--refine keeps OLD's tile unless NEW's is faster by more")
    ap.add_argument("--cold-suites", nargs="*", default=["single", "resnet50", "mobilenet"],
                    help="suites whose rows --refine times from cold caches")
    ap.add_argument("--base", metavar="TABLE", help="with --choose: keep TABLE's tile for a shape (it must be on the "
                    "shortlist, see --include) unless it moves more than --waste times the layer's algorithmic bytes; "
                    "only then does the bytes rule apply")
    ap.add_argument("--waste", type=float, default=2.0)
    ap.add_argument("--within-compute", type=float, default=0.0, help="the same slack for layers whose binding roof is the "
                    "vector units (0: they take their fastest tile)")
    ap.add_argument("--within", type=float, default=0.02, help="how much slower than the fastest a tile may be and still "
                    "win on bytes moved")
    ap.add_argument("--out", default=BUILT_IN)
    args = ap.parse_args()

    if args.replay:
        import numpy as np
        import torch

        items = json.load(open(args.replay))
        for it in items:
            n, H, Wd, Cc, K, ks, stride, pad = it["key"]
            L = W.Layer(it["suite"], 0, it["name"], Cc, H, Wd, K, ks, stride, pad, it["sparsity"])
            w = W.make_weights(W.SUITES[it["suite"]]()[it["index"]])
            assert w.shape == (K, Cc, ks, ks)
            oh, ow = W.out_hw(L)
            x = torch.zeros((n, Cc, H, Wd), device="cuda")
            y = torch.empty((n, K, oh, ow), device="cuda")
            for c in it["candidates"]:
                tile = T.Tile(*c["tile"])
                obey(it["key"], c["tile"])
                pk = T.G950Filter.for_tile(w, tile, oc_order="balanced")
                pk.prepare(n, H, Wd, stride, pad, tile)
                pk.launch(x.data_ptr(), y.data_ptr(), n, H, Wd, stride, pad, tile)
                torch.cuda.synchronize()
                pk.close()
        return

    if args.choose:
        items = json.load(open(args.choose))
        fetch = counter_sums(args.fetch, ("FETCH_SIZE",))
        write = counter_sums(args.write, ("WRITE_SIZE",))
        lds = counter_sums(args.lds, ("SQ_LDS_BANK_CONFLICT", "SQ_LDS_IDX_ACTIVE")) if args.lds else None
        total = sum(len(it["candidates"]) for it in items)
        if len(fetch) != total or len(write) != total or (lds is not None and len(lds) != total):
            sys.exit("the replays hold %d / %d conv launches, the shortlist %d tiles" % (len(fetch), len(write), total))
        base = {}
        if args.base:
            import re

            row = re.compile(ROW + r",\s*// (.*)")
            for ln in open(args.base):
                m = row.match(ln)
                if m:
                    g = m.groups()
                    base[tuple(int(x) for x in g[:8])] = (list(row_tile(g)), g[14])
        rows, i, switched = [], 0, 0
        for it in items:
            best_ms = min(c["ms"] for c in it["candidates"])
            L = W.SUITES[it["suite"]]()[it["index"]]
            slack = args.within if W.work(L, it["key"][0])["bound"] == "hbm" else args.within_compute
            if args.base:
                slack = max(args.within, args.within_compute)
            for c in it["candidates"]:
                c["bytes"] = fetch[i]["FETCH_SIZE"] * 1024 * args.fetch_scale + write[i]["WRITE_SIZE"] * 1024 * args.write_scale
                if lds is not None:
                    act = lds[i].get("SQ_LDS_IDX_ACTIVE", 0.0)
                    c["lds_conflict_rate"] = lds[i].get("SQ_LDS_BANK_CONFLICT", 0.0) / act if act else 0.0
                i += 1
            fastest = min(it["candidates"], key=lambda c: c["ms"])
            pick = min((c for c in it["candidates"] if c["ms"] <= best_ms * (1.0 + slack)), key=lambda c: c["bytes"])
            if args.base:
                key = tuple(it["key"])
                held = [c for c in it["candidates"] if key in base and c["tile"] == base[key][0]]
                if held and not (held[0]["bytes"] > args.waste * W.work(L, key[0])["bytes"] and pick["bytes"] < held[0]["bytes"]):
                    rows.append((it["key"], held[0]["tile"], base[key][1]))  # the incumbent stays, with its note
                    continue
            switched += pick is not fastest
            note = "%s %s: %.1f us, %.2f MB moved" % (it["suite"], it["name"], pick["ms"] * 1e3, pick["bytes"] / 1e6)
            if "lds_conflict_rate" in pick:
                note += ", LDS conflict rate %.3f" % pick["lds_conflict_rate"]
            if pick is not fastest:
                f = fastest
                note += " (fastest: %s %.1f us, %.2f MB)" % (tile_text(f["tile"]), f["ms"] * 1e3, f["bytes"] / 1e6)
            rows.append((it["key"], pick["tile"], note))
        write_table(args.out, rows)
        print("%d of %d shapes took a tile other than the fastest, for fewer bytes" % (switched, len(items)), file=sys.stderr)
        return

    if args.refine:
        import re
        import torch

        row = re.compile(ROW + r",\s*// (.*)")

        def read(path):
            out = {}
            for ln in open(path):
                m = row.match(ln)
                if m:
                    g = m.groups()
                    out[tuple(int(x) for x in g[:8])] = (row_tile(g), g[14])
            return out

        old, new = read(args.refine[0]), read(args.refine[1])
        layer_of = {}
        for suite, make in W.SUITES.items():
            for L in make():
                k = (L.H, L.W, L.C, L.K, L.ks, L.stride, L.pad)
                if k not in layer_of or L.sparsity < layer_of[k].sparsity:
                    layer_of[k] = L
        rows, kept_old = [], 0
        for key, (tile_new, note_new) in new.items():
            if key not in old or old[key][0] == tile_new or key[1:] not in layer_of:
                rows.append((key, tile_new, note_new))
                continue
            tile_old, note_old = old[key]
            L, n = layer_of[key[1:]], key[0]
            cold = L.suite in args.cold_suites
            T.options_set((T.options_get() | T.OPT_COLD_TIMING) if cold else (T.options_get() & ~T.OPT_COLD_TIMING))
            w = W.make_weights(L)
            oh, ow = W.out_hw(L)
            x = torch.zeros((n, L.C, L.H, L.W), device="cuda")
            y = torch.empty((n, L.K, oh, ow), device="cuda")
            best = {}
            packs = {t: T.G950Filter.for_tile(w, T.Tile(*t), oc_order="balanced") for t in (tile_old, tile_new)}
            for _ in range(3):
                for t, pk in packs.items():
                    obey(key, t)
                    ms = pk.time(x.data_ptr(), y.data_ptr(), n, L.H, L.W, L.stride, L.pad, T.Tile(*t), warm=2 if cold else 5,
                                 repeat=10 if cold else 30)
                    best[t] = min(best.get(t, 1e9), ms)
            for pk in packs.values():
                pk.close()
            if best[tile_old] < best[tile_new] * (1.0 + args.margin):
                kept_old += 1
                rows.append((key, tile_old, "%s (head to head %.1f us against %s %.1f us)" % (
                    note_old.split(" (head to head")[0], best[tile_old] * 1e3, tile_text(tile_new), best[tile_new] * 1e3)))
            else:
                rows.append((key, tile_new, note_new))
            print("%s N=%d old %r %.1f us new %r %.1f us%s" % (L.name, n, tile_old, best[tile_old] * 1e3, tile_new,
                                                             best[tile_new] * 1e3, " (cold)" if cold else ""), file=sys.stderr, flush=True)
        write_table(args.out, rows)
        print("%d rows kept from %s" % (kept_old, args.refine[0]), file=sys.stderr)
        return

    if args.cold:
        T.options_set(T.options_get() | T.OPT_COLD_TIMING)
    incumbent = {}
    if args.include:
        import re
        import torch

        row = re.compile(ROW)
        for ln in open(args.include):
            m = row.match(ln)
            if m:
                g = m.groups()
                incumbent[tuple(int(x) for x in g[:8])] = row_tile(g)
    rows, items = [], []
    for key, L, n, suite in shapes(args):
        w = W.make_weights(L)
        if args.shortlist:
            cands = T.tile_autotune_list(w, n, L.H, L.W, L.stride, L.pad, args.candidates, 4)
            inc = incumbent.get(key)
            if inc and all(tuple(t.as_list()) != inc for t, _ in cands):
                try:  # the incumbent, timed like the tuner's second pass (2 + 10 launches)
                    tile = T.Tile(*inc)
                    obey(key, inc)
                    pk = T.G950Filter.for_tile(w, tile, oc_order="balanced")
                    oh, ow = W.out_hw(L)
                    x = torch.zeros((n, L.C, L.H, L.W), device="cuda")
                    y = torch.empty((n, L.K, oh, ow), device="cuda")
                    cands.append((tile, pk.time(x.data_ptr(), y.data_ptr(), n, L.H, L.W, L.stride, L.pad, tile, warm=2, repeat=10)))
                    pk.close()
                except T.TetrisError:
                    pass
            items.append({"key": list(key), "suite": suite, "name": L.name, "index": L.index, "sparsity": L.sparsity,
                          "candidates": [{"tile": t.as_list(), "ms": ms}
                                         for t, ms in cands]})
            tile, ms = cands[0]
        else:
            tile, ms = T.tile_autotune(w, n, L.H, L.W, L.stride, L.pad, args.candidates)
            own = own_choice_ms(w, L, n, args.cold) if args.out != BUILT_IN else None
            if own is not None and own < ms:
                print("%-10s %-26s N=%-2d %8.1f us  %r, left out: the library runs it in %.1f us on the matrix cores" % (
                    suite, L.name, n, ms * 1e3, tile, own * 1e3), file=sys.stderr, flush=True)
                continue
        rows.append((key, tuple(tile.as_list()),
                     "%s %s: %.1f us" % (suite, L.name, ms * 1e3)))
        print("%-10s %-26s N=%-2d %8.1f us  %r" % (suite, L.name, n, ms * 1e3, tile), file=sys.stderr, flush=True)
    if args.shortlist:
        with open(args.shortlist, "w") as f:
            json.dump(items, f)
        print("wrote %d shapes to %s" % (len(items), args.shortlist), file=sys.stderr)
    else:
        write_table(args.out, rows)


if __name__ == "__main__":
    main()
