"""The kernel that writes filter and input as two fp16 parts and hands the staging of inputs on from tile to tile (csrc/matrix_relay.hip),
through the public entry points, on layers that the library gives to it."""
import numpy as np
import pytest

from test_gpu_half_kernel import conv64, filter_of

pytestmark = pytest.mark.gpu

LDS = 2 * 60 * 1024 + 1848 + 8 * 4096  # what this kernel alone asks for

# N, C, H, W, K, ks, stride, pad, density of the filter; workgroups along the pixels and the channels, slices
LAYERS = [
    (11, 41, 8, 146, 3, 5, 2, 5, 0.15, (85, 1, 3)),        # three channels; quads of columns outside of the image; two strips, stored in quads
    (6, 34, 33, 19, 100, 6, 2, 3, 0.2, (16, 1, 3)),        # 6 x 6, stride 2; ragged channels on both sides
    (1, 49, 28, 122, 352, 4, 2, 1, 0.15, (14, 2, 4)),      # eight waves along the channels
    (5, 108, 8, 91, 483, 5, 2, 0, 0.15, (7, 2, 8)),        # ... images of two rows
    (1, 103, 28, 28, 152, 7, 1, 0, 0.1, (2, 3, 8)),        # 7 x 7; two workgroups for an image
    (8, 95, 113, 113, 9, 3, 1, 0, 0.15, (256, 1, 1)),      # two waves along the channels; several tiles each
    (7, 55, 81, 143, 34, 5, 2, 2, 0.2, (256, 1, 1)),       # ... stride 2
    (5, 93, 124, 124, 24, 3, 1, 1, 0.2, (256, 1, 1)),      # ... stored in quads
    (14, 288, 69, 17, 8, 5, 1, 6, 0.15, (85, 1, 3)),       # the first row's quads begin before the tensor
    (18, 197, 43, 43, 41, 2, 1, 1, 0.15, (85, 1, 3)),      # 2 x 2
    (4, 52, 143, 21, 158, 4, 1, 1, 0.2, (89, 2, 1)),       # four waves along the channels
    (5, 23, 61, 61, 112, 6, 1, 3, 0.15, (155, 1, 1)),      # ... two chunks
    (13, 25, 6, 124, 204, 6, 1, 3, 0.15, (182, 1, 1)),     # eight; two strips
    (7, 119, 100, 6, 70, 6, 1, 3, 0.15, (32, 1, 8)),       # images of six columns
    (16, 96, 40, 40, 250, 3, 1, 1, 0.15, (256, 1, 1)),     # runs of 3 blocks, 64 pairs of which share one: tiles of 4, 3 for half of the waves
    (5, 96, 75, 71, 470, 3, 1, 1, 0.15, (128, 2, 1)),      # ... of 6, all of them; two channel blocks
    (16, 192, 46, 46, 250, 3, 1, 1, 0.07, (256, 1, 1)),    # ... of 4: the last tile has two blocks, of which half of the waves store one
]


class Layer:
    def __init__(self, w, shape, stride, pad, grid=None):
        import tetris_amd as T

        N, C, H, W = shape
        K, _, ks, _ = w.shape
        self.at = (N, H, W, stride, pad)
        self.out = (N, K, T.out_extent(H, pad, ks, stride), T.out_extent(W, pad, ks, stride))
        self.tile = t = T.tile_select(N, H, W, C, K, ks, stride, pad)
        self.pack = T.G950Filter.for_tile(w, t, oc_order="balanced")
        s = self.pack.launch_shape(*self.at, t)
        assert s.kernel == 5 and s.lds_bytes == LDS
        assert grid is None or (s.unit_groups, s.channel_blocks, s.csplit) == grid
        assert s.workgroups == s.unit_groups * s.channel_blocks * s.csplit
        # the walk, with as many slices as it would have here (by a tile that is not the library's)
        T.options_set(T.OPT_ADD_IN_KERNEL)
        slices = self.pack.launch_shape(*self.at, t).csplit
        T.options_set(0)
        self.walk = T.Tile(t.lanes_w, t.quads, t.oc_per_wave, t.waves, t.tile_ic, slices if t.csplit != slices else 0)

    def __call__(self, x, tile=None, act=0):
        import torch
        import tetris_amd as T

        (n, k, oh, ow), half = self.out, 2 if act == T.ACT_RELU_POOL2 else 1
        dx, y = torch.from_numpy(x).cuda(), torch.full((n, k, oh // half, ow // half), float("nan"), device="cuda")
        self.pack.launch_act(dx.data_ptr(), y.data_ptr(), *self.at, tile or self.tile, act)
        torch.cuda.synchronize()
        return y.cpu().numpy()


def pooled(a):
    n, k, oh, ow = a.shape
    return a[:, :, :oh // 2 * 2, :ow // 2 * 2].reshape(n, k, oh // 2, 2, ow // 2, 2).max((3, 5))


@pytest.mark.parametrize("N,C,H,W,K,ks,stride,pad,density,grid", LAYERS)
def test_layer(N, C, H, W, K, ks, stride, pad, density, grid):
    import tetris_amd as T

    rng = np.random.default_rng(N * C + K)
    w = filter_of(rng, K, C, ks, density)
    x = np.maximum(rng.standard_normal((N, C, H, W)), 0).astype(np.float32)
    layer = Layer(w, x.shape, stride, pad, grid)
    got, again, walk = layer(x), layer(x), layer(x, layer.walk)
    ref, terms = conv64(x, w, stride, pad)
    # in any order of fp32 sums an output is off by a rounding per term at most, each of the terms' magnitude; a term's own, of two
    # parts to a factor, 2^-23 each and 2^-22 for the product that is left out, are less than that many
    bound = (w != 0).reshape(K, -1).sum(1).reshape(1, K, 1, 1) * 2.0 ** -24 * terms
    assert np.array_equal(got, again)
    assert (np.abs(got - ref) <= bound).all()
    assert np.linalg.norm(got - ref) <= 1.05 * np.linalg.norm(walk - ref)
    assert np.array_equal(layer(x, act=T.ACT_RELU), np.maximum(got, 0))
    if layer.pack.act_supported(*layer.at, layer.tile, T.ACT_RELU_POOL2):
        assert (np.abs(layer(x, act=T.ACT_RELU_POOL2) - np.maximum(pooled(ref), 0)) <= pooled(bound)).all()
    layer.pack.close()


LAYER, SPLIT = LAYERS[10], LAYERS[2]


@pytest.mark.parametrize("what", ["2^40", "2^-60", "zero where it is looked at", "tiny beside ones", "2^120", "subnormal", "few out of range",
                                  "many out of range", "infinite"])
@pytest.mark.parametrize("at", [LAYERS[5], LAYER, SPLIT, LAYERS[12], LAYERS[14]])  # (2, 4, 8, 8 and 8 waves along the channels)
def test_inputs_of_any_scale(at, what):
    """Inputs are scaled by what some of them show; a few that fp16 parts then do not hold are added one by one, a tile with more of them is
    computed with bf16 parts, and sums that are not finite with FMAs."""
    N, C, H, W, K, ks, stride, pad, density, grid = at
    rng = np.random.default_rng(1)
    w = filter_of(rng, K, C, ks, density)
    x = rng.standard_normal((N, C, H, W)).astype(np.float32)
    scale = {"2^40": 40, "2^-60": -60, "2^120": 118, "subnormal": -130}
    if what in scale:
        x = np.ldexp(x, scale[what])
    elif what == "zero where it is looked at":
        x[:, :, ::2] = 0
        x[:, [C * i // 8 for i in range(8)]] = 0
    elif what == "tiny beside ones":
        x[:, :, :, W // 2:] *= np.float32(2.0 ** -80)
    elif what == "few out of range":
        for n, c, i, j, e in [(0, 0, 0, 0, -30), (0, C - 1, H - 1, 2, -50), (N - 1, C // 2, H // 2, W // 3, 8), (N - 1, C - 1, H - 1, W - 1, 25)]:
            x[n, c, i, j] = np.ldexp(1 + rng.random(), e)
    elif what == "many out of range":
        x.reshape(-1)[rng.permutation(x.size)[:x.size // 64]] *= np.float32(2.0 ** -40)
    odd = np.zeros(x.shape, bool)
    if what == "infinite":
        x[0, 20, 3, W // 2], x[N - 1, 3, H - 1, W - 1], x[N // 2, C - 1, 0, 0] = np.inf, np.nan, -np.inf
        odd = ~np.isfinite(x)
    layer = Layer(w, x.shape, stride, pad, grid)
    got, walk = layer(x), layer(x, layer.walk)
    ref, terms = conv64(np.where(odd, 0, x), w, stride, pad)
    reached = conv64(odd.astype(np.float32), (w != 0).astype(np.float32), stride, pad)[0] > 0
    assert np.array_equal(got[reached], walk[reached], equal_nan=True)
    # (a subnormal output is rounded as such, twice)
    off = np.abs(got - ref) <= C * ks * ks * 2.0 ** -24 * terms + 2.0 ** -149
    assert (off | reached).all()
    layer.pack.close()


@pytest.mark.parametrize("value,count", [(2.0 ** -20, 1), (2.0 ** -40, 60), (2.0 ** -40, 3000), (2.0 ** -149, 2), (2.0 ** 63, 1)])
def test_small_weights(value, count):
    """Weights far below the largest of their row: multiplied one by one; all with bf16 parts where they are many, or where their
    products would underflow."""
    N, C, H, W, K, ks, stride, pad, density, grid = LAYER
    rng = np.random.default_rng(2)
    w = filter_of(rng, K, C, ks, density)
    w.reshape(-1)[rng.permutation(np.flatnonzero(w))[:count]] = np.float32(value)
    x = rng.standard_normal((N, C, H, W)).astype(np.float32)
    layer = Layer(w, x.shape, stride, pad, grid)
    ref, terms = conv64(x, w, stride, pad)
    assert (np.abs(layer(x) - ref) <= C * ks * ks * 2.0 ** -24 * terms + 2.0 ** -149).all()
    layer.pack.close()


@pytest.mark.parametrize("at", [LAYER, SPLIT])
def test_graph_beside_eager_launches(at):
    import torch

    N, C, H, W, K, ks, stride, pad, density, grid = at
    rng = np.random.default_rng(3)
    w = filter_of(rng, K, C, ks, density)
    xs = [torch.from_numpy(rng.standard_normal((N, C, H, W)).astype(np.float32)).cuda() for _ in range(2)]
    layer = Layer(w, (N, C, H, W), stride, pad, grid)
    want = [layer(x.cpu().numpy()).tobytes() for x in xs]
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    layer.pack.prepare(*layer.at, layer.tile, side.cuda_stream)
    x, y, other = xs[0].clone(), torch.empty(layer.out, device="cuda"), torch.empty(layer.out, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        layer.pack.launch(x.data_ptr(), y.data_ptr(), *layer.at, layer.tile, torch.cuda.current_stream().cuda_stream)
    for i in range(4):
        x.copy_(xs[i % 2])
        y.fill_(float("nan"))
        graph.replay()
        layer.pack.launch(xs[1 - i % 2].data_ptr(), other.data_ptr(), *layer.at, layer.tile, 0)  # on another stream, with sums of its own
        torch.cuda.synchronize()
        assert y.cpu().numpy().tobytes() == want[i % 2] and other.cpu().numpy().tobytes() == want[1 - i % 2], i
    del graph
    layer.pack.close()
