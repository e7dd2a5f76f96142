"""Layers that the library runs on the matrix cores (three bf16 parts of every fp32 number), against the CPU oracle: ragged
channels and pixels, images cut into strips, strided and padded windows, tiles that cross images, split channel
reductions, and the activations applied on the way out."""
import numpy as np
import pytest

from helpers import max_rel_err, relu_like, sparse_filter

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,C,H,W,K,ks,stride,pad", [
    (6, 25, 55, 77, 72, 1, 1, 0),      # pointwise, two strips, C and K over a multiple of 8 and 32
    (5, 163, 41, 54, 81, 3, 1, 1),     # 128 pixels a tile, slices
    (2, 23, 67, 45, 161, 5, 1, 2),     # 512 staged pixels; every slice of the input in one buffer
    (3, 38, 53, 25, 279, 2, 1, 1),     # four teams, more channel blocks than fill the last workgroup
    (7, 61, 31, 32, 5, 3, 1, 0),       # fewer output channels than lanes
    (2, 16, 38, 137, 11, 3, 2, 1),     # stride 2 in three strips
    (3, 72, 49, 67, 5, 2, 1, 1),       # even kernel, two teams, slices
    (1, 194, 46, 8, 10, 3, 1, 1),      # eight slices
    (1, 53, 14, 5, 105, 2, 1, 1),      # tiles of rows shorter than a quad
    (4, 17, 5, 7, 40, 1, 2, 0),        # strided pointwise, one tile over all images
    (3, 28, 7, 47, 5, 1, 1, 0),        # odd rows and columns to pool
])
def test_layer_on_the_matrix_cores(N, C, H, W, K, ks, stride, pad, oracle):
    import torch
    import tetris_amd as T

    rng = np.random.default_rng(N * C + K)
    w, x = sparse_filter(rng, K, C, ks, 0.7), relu_like(rng, (N, C, H, W)) - np.float32(0.25)
    ref = oracle.host_conv2d(x, w, stride, pad, threads=8)
    tile = T.tile_select(N, H, W, C, K, ks, stride, pad)
    pk = T.G950Filter.for_tile(w, tile, oc_order="balanced")
    assert pk.launch_shape(N, H, W, stride, pad, tile).kernel == 5
    dx = torch.from_numpy(x).cuda()
    buf = torch.full((ref.size + 8,), float("nan"), device="cuda")
    y = buf[1:1 + ref.size]
    outs = []
    for act in (T.ACT_NONE, T.ACT_RELU):
        pk.launch_act(dx.data_ptr(), y.data_ptr(), N, H, W, stride, pad, tile, act)
        torch.cuda.synchronize()
        outs.append(y.cpu().numpy().reshape(ref.shape))
        assert bool(torch.isnan(buf[:1]).all()) and bool(torch.isnan(buf[1 + ref.size:]).all())
    assert max_rel_err(outs[0], ref) <= 1e-4
    assert outs[1].tobytes() == np.maximum(outs[0], 0).tobytes()
    oh, ow = ref.shape[2] // 2, ref.shape[3] // 2
    if pk.act_supported(N, H, W, stride, pad, tile, T.ACT_RELU_POOL2):
        p = torch.full((N, K, oh, ow), float("nan"), device="cuda")
        pk.launch_act(dx.data_ptr(), p.data_ptr(), N, H, W, stride, pad, tile, T.ACT_RELU_POOL2)
        torch.cuda.synchronize()
        want = outs[1][:, :, :2 * oh, :2 * ow].reshape(N, K, oh, 2, ow, 2).max(axis=(3, 5))
        assert p.cpu().numpy().tobytes() == want.tobytes()
    # a tile that is not the library's own choice is obeyed
    other = T.Tile(tile.lanes_w, tile.quads, tile.oc_per_wave, tile.waves, tile.tile_ic, 1 if tile.csplit != 1 else 0)
    assert pk.launch_shape(N, H, W, stride, pad, other).kernel != 5
    pk.close()


def test_parts_keep_every_bit():
    """One weight of 1 per channel: the three parts of an input add up to the input itself, whatever its exponent."""
    import torch
    import tetris_amd as T

    N, C, H, K = 2, 64, 20, 96
    rng = np.random.default_rng(4)
    w = np.zeros((K, C, 1, 1), np.float32)
    w[np.arange(K), np.arange(K) % C] = 1.0
    x = (rng.standard_normal((N, C, H, H)) * np.exp2(rng.integers(-60, 60, (N, C, H, H)))).astype(np.float32)
    w[:, :, 0, 0] += (rng.random((K, C)) < 0.4) * np.float32(2.0 ** -149)  # dense enough; below every product that is kept
    tile = T.tile_select(N, H, H, C, K, 1, 1, 0)
    pk = T.G950Filter.for_tile(w, tile)
    assert pk.launch_shape(N, H, H, 1, 0, tile).kernel == 5
    dx, y = torch.from_numpy(x).cuda(), torch.empty((N, K, H, H), device="cuda")
    pk.launch(dx.data_ptr(), y.data_ptr(), N, H, H, 1, 0, tile)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy(), x[:, np.arange(K) % C])
    pk.close()


def test_loaded_row_is_obeyed(oracle, tmp_path):
    """A walking tile that the caller loaded runs as such, given or chosen, where the library would take the matrix cores."""
    import torch
    import tetris_amd as T

    N, C, H, W, K, ks = 3, 50, 22, 31, 90, 3
    rng = np.random.default_rng(12)
    w, x = sparse_filter(rng, K, C, ks, 0.7), relu_like(rng, (N, C, H, W))
    tile = T.tile_select(N, H, W, C, K, ks, 1, 1)
    before, after = (T.G950Filter.for_tile(w, tile, oc_order="balanced") for _ in range(2))
    dx = torch.from_numpy(x).cuda()

    def conv(pk, t):
        y = torch.full((N, K, H, W), float("nan"), device="cuda")
        pk.launch(dx.data_ptr(), y.data_ptr(), N, H, W, 1, 1, t)
        torch.cuda.synchronize()
        return y.cpu().numpy()

    assert before.launch_shape(N, H, W, 1, 1, tile).kernel == 5
    matrix = conv(before, tile)
    table = tmp_path / "tiles.inc"
    table.write_text("    {%d, %d, %d, %d, %d, %d, 1, 1, {%s}},\n" % (N, H, W, C, K, ks, ", ".join(map(str, tile.as_list()))))
    assert T.tile_table_load(str(table)) == 1
    shape = after.launch_shape(N, H, W, 1, 1, tile)
    assert shape.kernel != 5
    walk = conv(after, T.Tile(*tile.as_list()[:5], shape.csplit))
    assert walk.tobytes() != matrix.tobytes()  # sums in another order: tells the two kernels apart
    assert conv(after, tile).tobytes() == walk.tobytes() and conv(after, None).tobytes() == walk.tobytes()
    ref = oracle.host_conv2d(x, w, 1, 1, threads=8)
    assert max_rel_err(walk, ref) <= 1e-4 and max_rel_err(matrix, ref) <= 1e-4
    before.close()
    after.close()


@pytest.mark.parametrize("C,matrix", [(24, True), (15, False)])
def test_queries_tell_what_launches_run(C, matrix, oracle):
    """Options set after a plan was made change neither what the plan runs nor what the queries say of it; a shape that has
    no plan yet is answered for under the options in force."""
    import torch
    import tetris_amd as T

    N, H, W, K, ks = 2, 20, 26, 40, 3
    rng = np.random.default_rng(13)
    w, x = sparse_filter(rng, K, C, ks, 0.6), relu_like(rng, (N, C, H, W))
    tile = T.tile_select(N, H, W, C, K, ks, 1, 1)
    pk = T.G950Filter.for_tile(w, tile, oc_order="balanced")
    dx, y = torch.from_numpy(x).cuda(), torch.empty((N, K, H, W), device="cuda")

    def ask():
        s = pk.launch_shape(N, H, W, 1, 1, tile)
        acts = [pk.act_supported(N, H, W, 1, 1, tile, a) for a in (T.ACT_NONE, T.ACT_RELU, T.ACT_RELU_POOL2)]
        return [getattr(s, f) for f, _ in T.LaunchShape._fields_], acts

    def conv():
        y.fill_(float("nan"))
        pk.launch(dx.data_ptr(), y.data_ptr(), N, H, W, 1, 1, tile)
        torch.cuda.synchronize()
        return y.cpu().numpy()

    options = T.options_get()
    try:
        T.options_set(options | T.OPT_PAIRS)
        assert ask()[0][6] != 5  # the option picks a walking kernel, and no plan says otherwise
        T.options_set(options)
        before = ask()
        assert (before[0][6] == 5) == matrix
        out = conv()
        assert ask() == before
        T.options_set(options | T.OPT_PAIRS | T.OPT_NO_BANK_RULE)
        assert ask() == before and conv().tobytes() == out.tobytes()
    finally:
        T.options_set(options)
    assert max_rel_err(out, oracle.host_conv2d(x, w, 1, 1, threads=8)) <= 1e-4
    pk.close()
