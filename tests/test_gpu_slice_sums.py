"""Split layers whose slices' sums are added by a kernel of their own, on either side of the size that decides how they are
kept, against the CPU oracle: partly filled waves, padding slots, images side by side, outputs that are not 16-byte
aligned, and the activations the adder applies."""
import numpy as np
import pytest

from helpers import max_rel_err, relu_like, sparse_filter

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,C,H,W,K,ks,t5,slices", [
    (3, 40, 9, 11, 70, 3, (6, 2, 2, 4, 4), (2, 3, 5)),     # single-tile kernel, K over a slot padding, ragged rows
    (5, 64, 7, 7, 33, 3, (7, 1, 4, 16, 4), (2, 7, 8)),     # four images side by side
    (2, 48, 14, 14, 64, 3, (14, 2, 8, 8, 4), (6,)),        # 128 accumulators; the tile pools
    (3, 256, 13, 13, 40, 1, (64, 1, 2, 16, 16), (2, 8)),   # flat tile, H*W not a multiple of four
    (2, 128, 6, 10, 96, 1, (64, 2, 8, 8, 16), (4,)),       # flat tile, whole quads
    (16, 32, 28, 28, 128, 1, (28, 2, 4, 16, 4), (2, 4)),   # 14 and 28 MiB of sums
])
def test_slices_added_by_a_kernel(N, C, H, W, K, ks, t5, slices, oracle):
    import torch
    import tetris_amd as T

    assert torch.cuda.is_available()
    rng = np.random.default_rng(C + K)
    w, x = sparse_filter(rng, K, C, ks, 0.8), relu_like(rng, (N, C, H, W))
    pad = ks // 2
    ref = oracle.host_conv2d(x, w, 1, pad, threads=8)
    dx = torch.from_numpy(x).cuda()
    for cs in slices:
        tile = T.Tile(*t5, cs)
        pk = T.G950Filter.for_tile(w, tile, oc_order="balanced")
        assert pk.launch_shape(N, H, W, 1, pad, tile).csplit == cs
        for shift in (0, 1):  # the output 16-byte aligned, or not
            buf = torch.full((ref.size + 8,), float("nan"), device="cuda")
            y = buf[shift:shift + ref.size]
            pk.launch(dx.data_ptr(), y.data_ptr(), N, H, W, 1, pad, tile)
            torch.cuda.synchronize()
            got = y.cpu().numpy().reshape(ref.shape)
            assert max_rel_err(got, ref) <= 1e-4 and bool(torch.isnan(buf[shift + ref.size:]).all()), (cs, shift)
            pk.launch_act(dx.data_ptr(), y.data_ptr(), N, H, W, 1, pad, tile, T.ACT_RELU)
            torch.cuda.synchronize()
            assert y.cpu().numpy().tobytes() == np.maximum(got, 0).tobytes(), (cs, shift)
        ph, pw = ref.shape[2] // 2, ref.shape[3] // 2
        p = torch.full((N, K, ph, pw), float("nan"), device="cuda")
        pk.launch_act(dx.data_ptr(), p.data_ptr(), N, H, W, 1, pad, tile, T.ACT_RELU_POOL2)
        torch.cuda.synchronize()
        want = np.maximum(got, 0)[:, :, :2 * ph, :2 * pw].reshape(N, K, ph, 2, pw, 2).max(axis=(3, 5))
        assert p.cpu().numpy().tobytes() == want.tobytes(), cs
        pk.close()
