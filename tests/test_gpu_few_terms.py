"""Outputs that few products add up to are as exact as fp32 FMAs, whatever kernel the library picks: inputs that are nearly all zero, output
channels that pruning left few weights, on layers whose filters have many weights a channel."""
import numpy as np
import pytest

from test_gpu_half_kernel import conv64, filter_of

pytestmark = pytest.mark.gpu

LAYERS = [  # N, C, H, W, K, ks, stride, pad, density of the filter
    (11, 41, 8, 146, 3, 5, 2, 5, 0.15), (1, 49, 28, 122, 352, 4, 2, 1, 0.15), (7, 119, 100, 6, 70, 6, 1, 3, 0.15), (18, 197, 43, 43, 41, 2, 1, 1, 0.15),
    (4, 52, 143, 21, 158, 4, 1, 1, 0.2), (16, 96, 40, 40, 250, 3, 1, 1, 0.15), (16, 256, 56, 56, 256, 3, 1, 1, 0.1)]


@pytest.mark.parametrize("what", ["one term", "5 % of the inputs", "channels of few weights"])
@pytest.mark.parametrize("N,C,H,W,K,ks,stride,pad,density", LAYERS)
def test_few_terms(N, C, H, W, K, ks, stride, pad, density, what):
    import torch
    import tetris_amd as T

    rng = np.random.default_rng(N * C + K)
    w = filter_of(rng, K, C, ks, density)
    x = 1 + rng.random((N, C, H, W))
    if what == "one term":  # pixels a window apart, in a channel each
        at = np.zeros((H, W), bool)
        at[::ks, ::ks] = True
        x *= at & (np.arange(C).reshape(C, 1, 1) == rng.integers(0, C, (H, W)))
    elif what == "5 % of the inputs":
        x *= rng.random(x.shape) < 0.05
    else:
        for k in range(0, K, 8):
            w.reshape(K, -1)[k, rng.permutation(np.flatnonzero(w.reshape(K, -1)[k]))[1 + k % 5:]] = 0
    x = x.astype(np.float32)
    tile = T.tile_select(N, H, W, C, K, ks, stride, pad)
    pack = T.G950Filter.for_tile(w, tile, oc_order="balanced")
    dx = torch.from_numpy(x).cuda()
    y = torch.full((N, K, T.out_extent(H, pad, ks, stride), T.out_extent(W, pad, ks, stride)), float("nan"), device="cuda")
    pack.launch(dx.data_ptr(), y.data_ptr(), N, H, W, stride, pad, tile)
    torch.cuda.synchronize()
    ref, terms = conv64(x, w, stride, pad)
    count = np.round(conv64((x != 0).astype(np.float32), (w != 0).astype(np.float32), stride, pad)[0])
    # a rounding per product that is not zero, and one where two slices of the channels meet, each of the terms' magnitude at most (and of
    # what the roundings before have added)
    bound = (2 * count - 1).clip(0) * 2.0 ** -24 * (1 + 2.0 ** -10) * terms
    off = np.abs(y.cpu().numpy() - ref)
    few = (count > 0) & (count < 6)
    assert few.any()
    assert (off <= bound).all(), "%d of %d outputs of fewer than six terms, by up to %.2f times the bound" % (
        (off > bound)[few].sum(), few.sum(), (off / np.maximum(bound, 1e-300))[few].max())
    pack.close()
