"""Layers that the library runs on the matrix cores (three bf16 parts of every fp32 number), against the CPU oracle: ragged
channels and pixels, images cut into strips, strided and padded windows, tiles that cross images, split channel
reductions, and the activations applied on the way out."""
import numpy as np
import pytest

from helpers import max_rel_err, relu_like, sparse_filter

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,C,H,W,K,ks,stride,pad", [
    (6, 25, 55, 77, 72, 1, 1, 0),      # pointwise, two strips, C and K over a multiple of 8 and 32
    (5, 163, 41, 54, 81, 3, 1, 1),     # half_kernel: 192 pixels a tile, slices
    (2, 23, 67, 45, 161, 5, 1, 2),     # 512 staged pixels; every slice of the input in one buffer
    (3, 38, 53, 25, 279, 2, 1, 1),     # four teams, more channel blocks than fill the last workgroup
    (7, 61, 31, 32, 5, 3, 1, 0),       # fewer output channels than lanes
    (2, 16, 38, 137, 11, 3, 2, 1),     # stride 2 in three strips
    (3, 72, 49, 67, 5, 2, 1, 1),       # even kernel, two teams, slices
    (1, 194, 46, 8, 10, 3, 1, 1),      # eight slices
    (1, 53, 14, 5, 105, 2, 1, 1),      # tiles of rows shorter than a quad
    (4, 17, 5, 7, 40, 1, 2, 0),        # strided pointwise, one tile over all images
    (3, 28, 7, 47, 5, 1, 1, 0),        # odd rows and columns to pool
    # the remaining configurations of tile and teams, kernel sizes and strides
    (2, 44, 71, 53, 129, 1, 1, 0),     # 128 channels by 64 pixels, two teams
    (10, 120, 40, 32, 89, 3, 2, 1),    # ... in four slices
    (4, 80, 51, 42, 66, 3, 1, 1),      # 128 by 128, two teams, three slices
    (14, 56, 48, 7, 271, 2, 1, 1),     # 64 by 128, four teams
    (11, 152, 57, 18, 17, 2, 1, 0),    # ... in three slices
    (3, 200, 48, 21, 19, 1, 4, 0),     # every fourth pixel
    (15, 60, 22, 7, 130, 2, 3, 0),     # stride 3: pixels that are staged and not used
    (2, 196, 8, 11, 128, 4, 1, 0),
    (7, 169, 71, 12, 59, 4, 2, 0),
    (4, 143, 11, 9, 117, 6, 1, 0),
    (1, 82, 19, 18, 274, 6, 2, 0),
    (2, 95, 9, 27, 244, 7, 1, 3),
    (3, 60, 31, 7, 30, 7, 2, 3),
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
    w[np.arange(K), np.arange(K) % 48] = 1.0
    w[:, 48:] = sparse_filter(rng, K, 16, 1, 0.2, False)  # dense enough for the matrix cores, and x is zero there
    x = (rng.standard_normal((N, C, H, H)) * np.exp2(rng.integers(-145, 125, (N, C, H, H)))).astype(np.float32)
    x[:, 48:] = 0
    tile = T.tile_select(N, H, H, C, K, 1, 1, 0)
    pk = T.G950Filter.for_tile(w, tile)
    assert pk.launch_shape(N, H, H, 1, 0, tile).kernel == 5
    for each in (x, np.clip(x, -2.0 ** 60, 2.0 ** 60)):  # with numbers whose tiles are computed again, and without
        dx, y = torch.from_numpy(each).cuda(), torch.empty((N, K, H, H), device="cuda")
        pk.launch(dx.data_ptr(), y.data_ptr(), N, H, H, 1, 0, tile)
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy(), each[:, np.arange(K) % 48])
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


def conv64(x, w, stride, pad, terms=False):
    """float64 on the CPU; with `terms`: also the sum of the terms' magnitudes, which bounds what any order of sums can lose"""
    import torch

    f = lambda a, b: torch.nn.functional.conv2d(torch.from_numpy(a).double(), torch.from_numpy(b).double(),  # noqa: E731
                                                stride=stride, padding=pad).numpy()
    return (f(x, w), f(np.abs(x), np.abs(w))) if terms else f(x, w)


def run_both(w, x, stride, pad, act=0):
    """The layer as the library runs it, on the matrix cores, and on a walking tile of the same pack; None where one of the
    two cannot pool"""
    import torch
    import tetris_amd as T

    N, C, H, W = x.shape
    K, _, ks, _ = w.shape
    tile = T.tile_select(N, H, W, C, K, ks, stride, pad)
    pk = T.G950Filter.for_tile(w, tile, oc_order="balanced")
    assert pk.launch_shape(N, H, W, stride, pad, tile).kernel == 5
    other = T.Tile(tile.lanes_w, tile.quads, tile.oc_per_wave, tile.waves, tile.tile_ic, 1 if tile.csplit != 1 else 0)
    if not all(pk.act_supported(N, H, W, stride, pad, t, act) for t in (tile, other)):
        return None
    dx, outs, div = torch.from_numpy(x).cuda(), [], 2 if act == T.ACT_RELU_POOL2 else 1
    for t in (tile, other):
        y = torch.full((N, K, T.out_extent(H, pad, ks, stride) // div, T.out_extent(W, pad, ks, stride) // div), float("nan"),
                       device="cuda")
        pk.launch_act(dx.data_ptr(), y.data_ptr(), N, H, W, stride, pad, t, act)
        torch.cuda.synchronize()
        outs.append(y.cpu().numpy())
    pk.close()
    return outs


RANGE_LAYERS = [
    (6, 25, 55, 77, 72, 1, 1, 0), (5, 163, 41, 54, 81, 3, 1, 1), (2, 23, 67, 45, 161, 5, 1, 2), (3, 38, 53, 25, 279, 2, 1, 1),
    (2, 16, 38, 137, 11, 3, 2, 1), (1, 194, 46, 8, 10, 3, 1, 1), (4, 17, 5, 7, 40, 1, 2, 0), (3, 28, 7, 47, 5, 1, 1, 0)]


@pytest.mark.parametrize("N,C,H,W,K,ks,stride,pad", RANGE_LAYERS)
def test_values_out_of_range_give_what_the_walk_gives(N, C, H, W, K, ks, stride, pad):
    """Infinities, NaN, the largest numbers and sums that overflow, a few among ordinary values: they reach the outputs
    whose window holds them with a weight that is not zero, and no others."""
    rng = np.random.default_rng(C * K)
    w, x = sparse_filter(rng, K, C, ks, 0.7), relu_like(rng, (N, C, H, W)) - np.float32(0.25)
    odd = np.array([np.inf, -np.inf, np.nan, 3.4e38, -3.4e38, 2.0 ** 100, -2.0 ** 90, 1e-45], np.float32)
    at = rng.permutation(x.size)[:48]
    x.reshape(-1)[at] = np.tile(odd, 6)
    for act in (0, 1, 2):
        with np.errstate(all="ignore"):
            both = run_both(w, x, stride, pad, act)
            if both is None:
                continue
            matrix, walk = both
            assert np.array_equal(np.isnan(matrix), np.isnan(walk)) and np.array_equal(np.isinf(matrix), np.isinf(walk))
            assert act or (np.isnan(walk).any() and np.isinf(walk).any())
            ok = np.isfinite(walk)
            assert np.array_equal(np.sign(matrix[~ok]), np.sign(walk[~ok]), equal_nan=True)
            tame = np.where(np.isfinite(x), x, 0)
            _, terms = conv64(tame, w, stride, pad, True)
            if act == 2:  # of a maximum: the largest bound of the four
                k, oh, ow = walk.shape[1:]
                terms = terms[:, :, :2 * oh, :2 * ow].reshape(N, k, oh, 2, ow, 2).max(axis=(3, 5))
            n = C * ks * ks
            assert (np.abs(matrix[ok].astype(np.float64) - walk[ok]) <= 2 * n * 2.0 ** -24 * terms[ok]).all()


@pytest.mark.parametrize("scale_x,scale_w", [(-120, 0), (-140, 4), (0, -130), (-70, -60), (40, 20), (80, -100), (120, -10)])
def test_precision_at_any_scale(scale_x, scale_w):
    """Outputs of one term each, inputs and weights of full 24-bit significands at either end of fp32's exponents: as exact
    as one rounding of the product, and to the last bit of a subnormal one."""
    N, C, H, K = 2, 64, 20, 96
    rng = np.random.default_rng(5)
    w = np.zeros((K, C, 1, 1), np.float32)
    w[:, 48:] = sparse_filter(rng, K, 16, 1, 0.2, False)  # dense enough for the matrix cores, and x is zero there
    w[np.arange(K), np.arange(K) % 48, 0, 0] = np.ldexp(1 + rng.random(K, dtype=np.float32), scale_w)
    x = np.zeros((N, C, H, H), np.float32)
    x[:, :48] = np.ldexp((1 + rng.random((N, 48, H, H))).astype(np.float32), scale_x)
    matrix, walk = run_both(w, x, 1, 0)
    ref = conv64(x, w, 1, 0)
    # half a unit in the last place; for the matrix cores also the rounding of the smaller products' sum, which is 2^-8 of
    # the product, and of a subnormal output first that of the scaled sum and then its own
    normal = np.abs(ref) >= 2.0 ** -126
    half = np.where(normal, np.abs(ref) * 2.0 ** -24, 2.0 ** -150)
    assert (np.abs(walk - ref) <= half * 1.0001).all()
    assert (np.abs(matrix - ref) <= half * (1 + 2.0 ** -5) + np.where(normal, 0, np.abs(ref) * 2.0 ** -24)).all()


def test_weights_out_of_range_stay_with_the_walk(oracle):
    import torch
    import tetris_amd as T

    N, C, H, K = 2, 64, 20, 96
    for value, kernel5 in [(1.0, True), (2.0 ** 63, True), (2.0 ** -149, True), (2.0 ** 64, False), (np.inf, False), (np.nan, False)]:
        rng = np.random.default_rng(6)
        w, x = sparse_filter(rng, K, C, 1, 0.6), relu_like(rng, (N, C, H, H))
        w[5, 7] = value
        tile = T.tile_select(N, H, H, C, K, 1, 1, 0)
        pk = T.G950Filter.for_tile(w, tile, oc_order="balanced")
        assert (pk.launch_shape(N, H, H, 1, 0, tile).kernel == 5) == kernel5, value
        assert pk.host_arrays()["nnz"] == int((w != 0).sum())
        dx, y = torch.from_numpy(x).cuda(), torch.empty((N, K, H, H), device="cuda")
        pk.launch(dx.data_ptr(), y.data_ptr(), N, H, H, 1, 0, tile)
        torch.cuda.synchronize()
        got = y.cpu().numpy()
        if np.isfinite(value):
            ref, terms = conv64(x, w, 1, 0, True)
            assert (np.abs(got - ref) <= C * 2.0 ** -24 * terms).all(), value
        else:
            assert np.isfinite(np.delete(got, 5, 1)).all()
        pk.close()


# run on the matrix cores in slices: by half_kernel and by matrix_kernel (LDS: whole KiB of input, then what half_kernel alone keeps there)
SPLIT = [((5, 163, 41, 54, 81, 3, 1, 1), True), ((10, 120, 40, 32, 89, 3, 2, 1), False)]


def split_layer(seed, layer, half):
    import torch
    import tetris_amd as T

    N, C, H, W, K, ks, stride, pad = layer
    rng = np.random.default_rng(seed)
    w = sparse_filter(rng, K, C, ks, 0.7)
    tile = T.tile_select(N, H, W, C, K, ks, stride, pad)
    pk = T.G950Filter.for_tile(w, tile, oc_order="balanced")
    shape = pk.launch_shape(N, H, W, stride, pad, tile)
    assert shape.kernel == 5 and shape.csplit > 1 and (shape.lds_bytes % 1024 != 0) == half
    oh, ow = T.out_extent(H, pad, ks, stride), T.out_extent(W, pad, ks, stride)
    xs = [torch.from_numpy(relu_like(rng, (N, C, H, W))).cuda() for _ in range(2)]

    def launch(x, y, stream=0):
        pk.launch(x.data_ptr(), y.data_ptr(), N, H, W, stride, pad, tile, stream)

    want = []
    for x in xs:
        y = torch.full((N, K, oh, ow), float("nan"), device="cuda")
        launch(x, y)
        torch.cuda.synchronize()
        want.append(y.cpu().numpy())
    return pk, tile, launch, xs, want


@pytest.mark.parametrize("layer,half", SPLIT)
def test_graph_of_a_split_matrix_layer(layer, half):
    import torch

    N, C, H, W, K, ks, stride, pad = layer
    pk, tile, launch, xs, want = split_layer(21, layer, half)
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    pk.prepare(N, H, W, stride, pad, tile, side.cuda_stream)
    x, y, other = xs[0].clone(), torch.empty(want[0].shape, device="cuda"), torch.empty(want[0].shape, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        launch(x, y, torch.cuda.current_stream().cuda_stream)
    for i in range(6):
        x.copy_(xs[i % 2])
        y.fill_(float("nan"))
        graph.replay()
        launch(xs[1 - i % 2], other)  # eager, on another stream, with sums of its own
        torch.cuda.synchronize()
        assert y.cpu().numpy().tobytes() == want[i % 2].tobytes(), i
        assert other.cpu().numpy().tobytes() == want[1 - i % 2].tobytes(), i
    del graph
    pk.close()


@pytest.mark.parametrize("layer,half", SPLIT)
def test_two_streams_of_a_split_matrix_layer(layer, half):
    import torch

    pk, tile, launch, xs, want = split_layer(22, layer, half)
    streams = [torch.cuda.Stream() for _ in range(2)]
    ys = [[torch.full(want[0].shape, float("nan"), device="cuda") for _ in range(8)] for _ in streams]
    torch.cuda.synchronize()
    for i in range(8):
        for x, y, s in zip(xs, ys, streams):
            launch(x, y[i], s.cuda_stream)
    torch.cuda.synchronize()
    for each, ref in zip(ys, want):
        assert all(y.cpu().numpy().tobytes() == ref.tobytes() for y in each)
    pk.close()
