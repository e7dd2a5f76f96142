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


def test_room_for_the_sums_is_taken_where_they_are_kept(oracle):
    """33 of 128 channel slots used: the waves' order of the sums (51 MB) takes four times the room of the slices' copies
    of the output (13 MB), and beyond 16 MiB only TETRIS_OPT_ADD_IN_KERNEL keeps it."""
    import torch
    import tetris_amd as T

    N, C, H, K = 1024, 32, 7, 33
    rng = np.random.default_rng(9)
    w, x = sparse_filter(rng, K, C, 3, 0.8), relu_like(rng, (N, C, H, H))
    tile = T.Tile(7, 1, 8, 16, 4, 2)
    pk = T.G950Filter.for_tile(w, tile, oc_order="balanced")
    copies = pk.launch_shape(N, H, H, 1, 1, tile).scratch_bytes
    assert 13e6 < copies < 14e6
    dx, y = torch.from_numpy(x).cuda(), torch.empty((N, K, H, H), device="cuda")
    pk.prepare(1, H, H, 1, 1, tile)  # what any first plan on a device allocates
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    pk.prepare(N, H, H, 1, 1, tile)
    torch.cuda.synchronize()
    assert before - torch.cuda.mem_get_info()[0] < copies + (8 << 20)
    outs, options = [], T.options_get()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    pk.prepare(N, H, H, 1, 1, tile, stream=side.cuda_stream)
    try:
        pk.launch(dx.data_ptr(), y.data_ptr(), N, H, H, 1, 1, tile)
        torch.cuda.synchronize()
        outs.append(y.cpu().numpy())
        T.options_set(options | T.OPT_ADD_IN_KERNEL)
        with torch.cuda.graph(graph, stream=side):  # the buffer was made without the option: the copies are added instead
            pk.launch(dx.data_ptr(), y.data_ptr(), N, H, H, 1, 1, tile, stream=torch.cuda.current_stream().cuda_stream)
        for _ in range(2):
            y.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            outs.append(y.cpu().numpy())
        y.fill_(float("nan"))
        pk.launch(dx.data_ptr(), y.data_ptr(), N, H, H, 1, 1, tile)  # grows
        torch.cuda.synchronize()
        outs.append(y.cpu().numpy())
    finally:
        T.options_set(options)
    assert max_rel_err(outs[0][:32], oracle.host_conv2d(x[:32], w, 1, 1, threads=8)) <= 1e-4
    assert all(o.tobytes() == outs[0].tobytes() for o in outs)
    del graph
    pk.close()
