"""The work that a user of this framework has it do: sparse convolutions called through tetris_amd, layer by layer and
network by network, the packing of their filters, and the launchers of the reference's call shapes.

A case is a dict of plain values.  `kind` says which entry points it goes through:
  layer   one convolution on device tensors: G950Filter.launch, or launch_act where an activation follows
  stack   every layer of a network of tetris_amd.workloads once, back to back, each on tensors of its own (what bench.py
          times): `side` is the network's input size, `shift` is added to every layer's sparsity
  chain   the VGG19-shaped network as one: every convolution reads the activation (ReLU, 2x2 max-pooling) of the last
  pack    a filter in host memory put into the balanced channel order, packed on the device and read back (model loading)
  raw     SparseConv2d on the five device arrays of a SparseFilter, the reference launcher's call shape
  host    CudaSparseConv2d, from host arrays to host arrays (its 30 + 100 launches are part of what it is asked for)
`prune`: "uniform" zeroes a random subset of the weights, as the benchmark's masks do; "magnitude" zeroes the smallest
weights of a filter whose output channels differ in scale, as global pruning does: channels then differ in density.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "tetris-artifact-evalution_amd"))
import tetris_amd as T  # noqa: E402
from tetris_amd import workloads as W  # noqa: E402


def _layer(name, N, C, H, W_, K, ks, stride, pad, sparsity, prune="uniform", act=0, kind="layer"):
    case = dict(kind=kind, N=N, C=C, H=H, W=W_, K=K, ks=ks, stride=stride, pad=pad, sparsity=sparsity, prune=prune)
    if kind == "layer":
        case["act"] = act
    return dict(case, name=name) if name else case


def _net(name, kind, suite, N, side, shift=0.0):
    case = dict(kind=kind, suite=suite, N=N, side=side, shift=shift)
    return dict(case, name=name) if name else case


def listed():
    return [
        # one image through one layer, the smallest call there is: latency of a launch
        _layer("layer_b1", 1, 64, 56, 56, 128, 3, 1, 1, 0.90),
        # one image through a pointwise layer of a mobile network: latency, few pixels, all of them reduced over 512 channels
        _layer("pointwise_b1", 1, 512, 14, 14, 512, 1, 1, 0, 0.85, act=1),
        # nothing is a multiple of anything: image of any size, stride 2, channels of unequal density
        _layer("ragged_b3", 3, 83, 61, 45, 70, 3, 2, 1, 0.80, prune="magnitude", act=1),
        # an ordinary layer in the middle of a network at batch 16
        _layer("conv_b16", 16, 256, 56, 56, 256, 3, 1, 1, 0.90, act=1),
        # one image through a whole network (interactive use), and the benchmark's batch through the same network
        _net("vgg19_b1", "chain", "vgg19", 1, 224),
        _net("vgg19_b16", "chain", "vgg19", 16, 224),
        # the other networks of the benchmark at its batch: many short layers, pointwise layers only, the largest images
        _net("resnet50_b16", "stack", "resnet50", 16, 224),
        _net("mobilenet_b16", "stack", "mobilenet", 16, 224),
        _net("yolov3_b16", "stack", "yolov3", 16, 416),
        # loading a model: one large filter packed
        _layer("pack_512", 8, 512, 28, 28, 512, 3, 1, 1, 0.90, kind="pack"),
        # programs written against the reference's launcher and against its host-to-host function
        _layer("raw_b4", 4, 256, 28, 28, 256, 3, 1, 1, 0.90, kind="raw"),
        _layer("host_b4", 4, 64, 56, 56, 64, 3, 1, 1, 0.90, kind="host"),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer"] * 6 + ["stack"] * 2 + ["chain", "pack", "raw", "host"])
    if kind in ("stack", "chain"):
        suite = "vgg19" if kind == "chain" else rng.choice(["resnet50", "mobilenet", "yolov3"])
        side = 32 * rng.randint(5, 7) if suite != "yolov3" else 32 * rng.randint(7, 13)
        return _net(None, kind, suite, _spread(rng, 1, 16), side, round(rng.uniform(-0.08, 0.04), 3))
    largest = {"layer": 6e11, "pack": 4e10, "raw": 5e10, "host": 1e10}[kind]  # dense multiply-adds of one launch, times two
    while True:
        ks, stride = rng.choice([(1, 1), (1, 1), (3, 1), (3, 1), (3, 1), (1, 2), (3, 2), (5, 1), (7, 2)])
        pad = ks // 2
        N, C, K = _spread(rng, 1, 16), _spread(rng, 16, 1024), _spread(rng, 16, 1024)
        if ks == 7 or rng.random() < 0.08:
            C = 3  # the first layer of a network
        H = _spread(rng, 7, 224)
        W_ = H if rng.random() < 0.6 else max(7, int(H * rng.uniform(0.6, 1.4)))
        dense = 2.0 * N * K * C * ks * ks * ((H + 2 * pad - ks) // stride + 1) * ((W_ + 2 * pad - ks) // stride + 1)
        if dense <= largest and N * max(C, K) * H * W_ <= 1 << 27 and C * K * ks * ks <= 5 << 19:
            break
    sparsity = round(rng.uniform(0.70, 0.95), 3) if C > 3 else 0.5
    return _layer(None, N, C, H, W_, K, ks, stride, pad, sparsity, rng.choice(["uniform", "magnitude"]),
                  rng.choice([0, 1, 1]), kind)


def _dims(case):
    """(N, C, H, W, K, ks, stride, pad) of a case of one layer."""
    return tuple(case[k] for k in ("N", "C", "H", "W", "K", "ks", "stride", "pad"))


def _layers(case):
    """The layers of a network case at its image size: one dict per layer, shaped like a case of one layer."""
    base = 416 if case["suite"] == "yolov3" else 224
    layers = W.SUITES[case["suite"]]()
    if case["suite"] == "yolov3":
        layers = layers[:52]  # the Darknet-53 backbone
    return [_layer(None, case["N"], L.C, L.H * case["side"] // base, L.W * case["side"] // base, L.K, L.ks, L.stride, L.pad,
                   L.sparsity if L.C == 3 else min(0.97, round(L.sparsity + case["shift"], 3))) for L in layers]


def _out_hw(case):
    N, C, H, W_, K, ks, stride, pad = _dims(case)
    return T.out_extent(H, pad, ks, stride), T.out_extent(W_, pad, ks, stride)


def _nnz(case):
    n = case["K"] * case["C"] * case["ks"] ** 2
    return n - int(round(case["sparsity"] * n))


def _weights(gen, case):
    """A pruned fp32 filter, OIHW, on the host (weights come from a file in a user's program)."""
    K, C, ks = case["K"], case["C"], case["ks"]
    n = K * C * ks * ks
    w = torch.randn(n, generator=gen, device="cuda") * 0.05
    w[w == 0] = 1e-6
    if case["prune"] == "magnitude":
        scale = torch.exp(0.35 * torch.randn(K, generator=gen, device="cuda"))
        w = (w.view(K, -1) * scale[:, None]).reshape(-1)
        drop = w.abs().argsort()[:n - _nnz(case)]
    else:
        drop = torch.randperm(n, generator=gen, device="cuda")[:n - _nnz(case)]
    w[drop] = 0.0
    return w.view(K, C, ks, ks).cpu().numpy()


def _activations(gen, shape):
    """The output of a ReLU: half of the elements zero, the others uniform in [0, 1)."""
    x = torch.rand(shape, generator=gen, device="cuda") * 2 - 1
    return x.clamp_(min=0.0)


def _pack_tile(case):
    """A tile of the caller's own, so that the packed arrays do not depend on what the library would choose."""
    return T.Tile(min(14, case["W"]), 1, 8, 8, min(8, case["C"]))


def _packed(gen, case):
    N, C, H, W_, K, ks, stride, pad = _dims(case)
    w = _weights(gen, case)
    tile = T.tile_select(N, H, W_, C, K, ks, stride, pad)
    pack = T.G950Filter.for_tile(w, tile, oc_order="balanced")
    pack.prepare(N, H, W_, stride, pad, tile)
    return pack, tile


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind in ("stack", "chain"):
        calls, outs, x = [], [], None
        layers = _layers(case)
        for i, L in enumerate(layers):
            N, C, H, W_, K, ks, stride, pad = _dims(L)
            pack, tile = _packed(gen, L)
            if x is None or kind == "stack":
                x = _activations(gen, (N, C, H, W_))
            oh, ow = _out_hw(L)
            act, y = 0, None
            if kind == "chain":  # pooled where the next layer's image is half as large, and at the end
                act = 2 if i + 1 == len(layers) or layers[i + 1]["H"] * 2 == oh else 1
                if act == 2 and not pack.act_supported(N, H, W_, stride, pad, tile, T.ACT_RELU_POOL2):
                    y = torch.empty((N, K, oh, ow), device="cuda")
            out = torch.empty((N, K, oh // 2, ow // 2) if act == 2 else (N, K, oh, ow), device="cuda")
            calls.append((pack, tile, x, y, out, act, L))
            outs.append(out)
            x = out
        torch.cuda.synchronize()
        return dict(case, calls=calls, outs=outs)
    N, C, H, W_, K, ks, stride, pad = _dims(case)
    if kind in ("pack", "host"):
        state = dict(case, w=_weights(gen, case))
        if kind == "host":
            state["x"] = _activations(gen, (N, C, H, W_)).cpu().numpy()
        else:  # where the program keeps the packed stream, for any zero pattern: streams are padded to eight entries
            tile = _pack_tile(case)
            streams = -(-K // 128) * 128 // tile.oc_per_wave * -(-C // tile.tile_ic)
            room = (_nnz(case) + 7 * streams,)
            state.update(position=np.zeros(room, np.int32), values=np.zeros(room, np.float32))
        return state
    x = _activations(gen, (N, C, H, W_))
    y = torch.empty((N, K) + _out_hw(case), device="cuda")
    if kind == "raw":
        sf = T.SparseFilter(_weights(gen, case), C, K, ks, TILE_IC=32, apply_reorder=True, flags=T.REORDER_OUT_CHANNEL)
        arrays = (sf.GetDeviceOffsets(), sf.GetDeviceStageLen(), sf.GetDeviceOCPermutation(), sf.GetDevicePosition(),
                  sf.GetDeviceValues())
        return dict(case, filter=sf, arrays=arrays, x=x, y=y)
    pack, tile = _packed(gen, case)
    return dict(case, pack=pack, tile=tile, x=x, y=y)


def _run_layer(pack, tile, x, y, act, L):
    N, C, H, W_, K, ks, stride, pad = _dims(L)
    if act:
        pack.launch_act(x.data_ptr(), y.data_ptr(), N, H, W_, stride, pad, tile, act)
    else:
        pack.launch(x.data_ptr(), y.data_ptr(), N, H, W_, stride, pad, tile)


def run(state):
    kind = state["kind"]
    if kind in ("stack", "chain"):
        for pack, tile, x, y, out, act, L in state["calls"]:
            if y is None:
                _run_layer(pack, tile, x, out, act, L)
            else:
                _run_layer(pack, tile, x, y, 1, L)
                T.relu_maxpool(y.data_ptr(), out.data_ptr(), L["N"], L["K"], y.shape[2], y.shape[3], 2)
        return state["outs"]
    N, C, H, W_, K, ks, stride, pad = _dims(state)
    if kind == "pack":
        arrays = T.G950Filter.for_tile(state["w"], _pack_tile(state), oc_order="balanced").host_arrays()
        for name in ("position", "values"):
            state[name][:len(arrays[name])] = arrays[name]
            arrays[name] = state[name]
        return arrays
    if kind == "host":
        return T.CudaSparseConv2d(state["x"], state["w"], N, H, W_, C, K, ks, stride, pad)[0]
    if kind == "raw":
        offsets, stage_len, perm, position, values = state["arrays"]
        T.SparseConv2d(state["x"].data_ptr(), offsets, stage_len, perm, position, values, state["y"].data_ptr(), N, H, W_, C,
                       K, ks, stride, pad)
        return state["y"]
    _run_layer(state["pack"], state["tile"], state["x"], state["y"], state["act"], state)
    return state["y"]


def work(case):
    if case["kind"] in ("stack", "chain"):
        total = {"bytes": 0, "flops": 0}
        layers = _layers(case)
        for i, L in enumerate(layers):
            w = work(L)
            oh, ow = _out_hw(L)
            if case["kind"] == "chain" and (i + 1 == len(layers) or layers[i + 1]["H"] * 2 == oh):
                w["bytes"] -= 4 * L["N"] * L["K"] * (oh * ow - (oh // 2) * (ow // 2))  # only the pooled tensor is written
            total = {k: total[k] + w[k] for k in total}
        return total
    N, C, H, W_, K, ks, stride, pad = _dims(case)
    if case["kind"] == "pack":  # the filter read, eight bytes written per non-zero
        return {"bytes": 4 * K * C * ks * ks + 8 * _nnz(case), "flops": 0}
    oh, ow = _out_hw(case)
    # a pointwise layer of stride 2 reads only the pixels its outputs depend on
    pixels = oh * ow if ks == 1 else H * W_
    return {"bytes": 4 * N * (C * pixels + K * oh * ow) + 8 * _nnz(case), "flops": 2 * N * _nnz(case) * oh * ow}


def tolerance(case):
    # packed arrays are whole numbers and copied floats; outputs are 32-bit sums in an order the library chooses
    return "exact" if case["kind"] == "pack" else {"rel": 1e-5}
