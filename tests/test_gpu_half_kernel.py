"""The kernel that writes filter and input as three fp16 parts and multiplies them with the matrix cores' sparse instructions
(csrc/matrix_half.hip), through the public entry points, on layers that the library gives to it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def filter_of(rng, K, C, ks, density):
    """normally distributed weights, of which exactly `density` are not zero"""
    w = rng.standard_normal(K * C * ks * ks).astype(np.float32)
    w[rng.permutation(w.size)[int(density * w.size):]] = 0
    return w.reshape(K, C, ks, ks)


def conv64(x, w, stride, pad):
    """float64 on the CPU, and the sum of the terms' magnitudes"""
    import torch

    f = lambda a, b: torch.nn.functional.conv2d(torch.from_numpy(a).double(), torch.from_numpy(b).double(),  # noqa: E731
                                                stride=stride, padding=pad).numpy()
    return f(x, w), f(np.abs(x), np.abs(w))


class Layer:
    def __init__(self, w, shape, stride, pad):
        import tetris_amd as T

        N, C, H, W = shape
        K, _, ks, _ = w.shape
        self.at = (N, H, W, stride, pad)
        self.out = (N, K, T.out_extent(H, pad, ks, stride), T.out_extent(W, pad, ks, stride))
        self.tile = T.tile_select(N, H, W, C, K, ks, stride, pad)
        self.pack = T.G950Filter.for_tile(w, self.tile, oc_order="balanced")
        self.shape = self.pack.launch_shape(*self.at, self.tile)
        # (LDS: whole KiB of input, then what this kernel alone keeps there)
        assert self.shape.kernel == 5 and self.shape.lds_bytes % 1024

    def runs(self, channels, pixels, slices):
        """whether workgroups take tiles of this size (what the grid's numbers say)"""
        N, K, oh, ow = self.out
        strips = -(-ow // 64)
        columns = ow if strips == 1 else -(-ow // strips) + 1 & ~1
        return (self.shape.channel_blocks, self.shape.unit_groups, self.shape.csplit) == (
            -(--(-K // 32) // (channels // 32)), -(-N * strips * columns * oh // pixels), slices)

    def walk(self):
        import tetris_amd as T

        t = self.tile
        return T.Tile(t.lanes_w, t.quads, t.oc_per_wave, t.waves, t.tile_ic, 1 if t.csplit != 1 else 0)

    def __call__(self, x, tile=None):
        import torch

        dx, y = torch.from_numpy(x).cuda(), torch.full(self.out, float("nan"), device="cuda")
        self.pack.launch(dx.data_ptr(), y.data_ptr(), *self.at, tile or self.tile)
        torch.cuda.synchronize()
        return y.cpu().numpy()


LAYERS = [  # N, C, H, W, K, ks, stride, pad, density of the filter; channels, pixels and slices of the tiles it runs in
    (9, 16, 21, 21, 7, 2, 3, 0, 0.15, (256, 64, 1)),      # one chunk of channels; stride 3
    (15, 18, 21, 41, 131, 5, 1, 2, 0.3, (256, 64, 1)),    # chunks of 16 channels, the last of two; blocks that come twice
    (6, 39, 5, 9, 4, 7, 2, 3, 0.3, (256, 64, 3)),         # 7 x 7; four output channels
    (3, 42, 40, 77, 81, 3, 1, 1, 0.15, (128, 64, 1)),     # two teams, a chunk each and ten channels more; two strips
    (4, 17, 70, 26, 166, 6, 1, 0, 0.3, (128, 64, 1)),     # 6 x 6
    (12, 53, 27, 35, 7, 4, 1, 0, 0.15, (64, 64, 1)),      # two teams
    (1, 21, 8, 8, 3, 7, 1, 3, 0.3, (64, 64, 1)),          # an image of one tile
    (8, 33, 47, 63, 68, 5, 1, 0, 0.3, (256, 96, 1)),      # an odd number of blocks of pixels
    (11, 120, 18, 70, 11, 7, 2, 0, 0.2, (256, 96, 8)),    # ... 7 x 7
    (12, 111, 23, 78, 21, 3, 2, 1, 0.15, (256, 96, 4)),   # ... short chunks
    (8, 19, 79, 28, 275, 3, 1, 0, 0.3, (128, 192, 1)),
    (12, 17, 73, 24, 85, 2, 3, 1, 0.15, (256, 64, 1)),    # short chunks
    (3, 95, 9, 8, 3, 4, 3, 0, 0.3, (256, 64, 6)),
    (5, 17, 67, 31, 74, 4, 1, 2, 0.2, (128, 64, 1)),      # two teams
    (10, 17, 14, 6, 6, 2, 3, 0, 0.15, (64, 64, 1)),
    (1, 20, 28, 8, 10, 4, 1, 0, 0.3, (64, 64, 1)),        # two teams
    (8, 117, 38, 38, 183, 1, 1, 0, 0.15, (256, 64, 1)),   # pointwise
    (1, 2048, 4, 4, 1056, 2, 1, 0, 0.1, (64, 64, 8)),     # lists of steps too many to be added up where they are filled
    (4, 18, 69, 92, 175, 3, 1, 0, 0.15, (256, 128, 1)),   # four blocks of pixels a wave, which leave registers for two sets of weights
    (6, 19, 88, 50, 199, 3, 1, 0, 0.2, (256, 128, 1)),    # ... outputs four pixels at a time
    (3, 85, 45, 63, 228, 3, 1, 1, 0.3, (256, 128, 3)),
    (4, 17, 52, 80, 258, 3, 1, 1, 0.15, (128, 256, 1)),
    (8, 19, 79, 28, 275, 3, 1, 1, 0.3, (128, 256, 1)),
    (6, 68, 60, 57, 69, 3, 1, 1, 0.2, (128, 256, 3)),
]


@pytest.mark.parametrize("N,C,H,W,K,ks,stride,pad,density,tile", LAYERS)
def test_layer(N, C, H, W, K, ks, stride, pad, density, tile):
    rng = np.random.default_rng(N * C + K)
    w = filter_of(rng, K, C, ks, density)
    x = np.maximum(rng.standard_normal((N, C, H, W)), -0.25).astype(np.float32)
    layer = Layer(w, x.shape, stride, pad)
    assert layer.runs(*tile)
    got, walk = layer(x), layer(x, layer.walk())
    ref, terms = conv64(x, w, stride, pad)
    # in any order of fp32 sums an output is off by a rounding per term at most, each of the terms' magnitude; and the parts
    # lose no more than the walking kernel's FMAs do
    count = (w != 0).reshape(K, -1).sum(1).reshape(1, K, 1, 1)
    assert (np.abs(got - ref) <= count * 2.0 ** -24 * terms).all()
    assert np.linalg.norm(got - ref) <= 1.05 * np.linalg.norm(walk - ref)
    layer.pack.close()


@pytest.mark.parametrize("N,C,H,W,K,ks,stride,pad,density", [
    (3, 42, 40, 77, 81, 3, 1, 1, 0.15), (8, 33, 47, 63, 68, 5, 1, 0, 0.3), (11, 120, 18, 70, 11, 7, 2, 0, 0.2),
    (8, 19, 79, 28, 275, 3, 1, 0, 0.3), (1, 20, 28, 8, 10, 4, 1, 0, 0.3),
    (6, 19, 88, 50, 199, 3, 1, 0, 0.2), (4, 17, 52, 80, 258, 3, 1, 1, 0.15), (6, 68, 60, 57, 69, 3, 1, 1, 0.2)])
def test_activations(N, C, H, W, K, ks, stride, pad, density):
    import torch
    import tetris_amd as T

    rng = np.random.default_rng(K)
    w, x = filter_of(rng, K, C, ks, density), rng.standard_normal((N, C, H, W)).astype(np.float32)
    layer = Layer(w, x.shape, stride, pad)
    ref, terms = conv64(x, w, stride, pad)
    bound = C * ks * ks * 2.0 ** -24 * terms
    dx, (oh, ow) = torch.from_numpy(x).cuda(), layer.out[2:]
    y = torch.full(layer.out, float("nan"), device="cuda")
    layer.pack.launch_act(dx.data_ptr(), y.data_ptr(), *layer.at, layer.tile, T.ACT_RELU)
    torch.cuda.synchronize()
    assert (np.abs(y.cpu().numpy() - np.maximum(ref, 0)) <= bound).all()
    if layer.pack.act_supported(*layer.at, layer.tile, T.ACT_RELU_POOL2):
        pooled = torch.full((N, K, oh // 2, ow // 2), float("nan"), device="cuda")
        layer.pack.launch_act(dx.data_ptr(), pooled.data_ptr(), *layer.at, layer.tile, T.ACT_RELU_POOL2)
        torch.cuda.synchronize()
        most = lambda a: a[:, :, :oh // 2 * 2, :ow // 2 * 2].reshape(N, K, oh // 2, 2, ow // 2, 2).max((3, 5))  # noqa: E731
        assert (np.abs(pooled.cpu().numpy() - np.maximum(most(ref), 0)) <= most(bound)).all()
    layer.pack.close()


LAYER = (3, 42, 40, 77, 81, 3, 1, 1, 0.15)


@pytest.mark.parametrize("what", ["as it is", "2^40", "2^-60", "zero where it is looked at", "tiny beside ones", "2^120", "subnormal", "infinite"])
def test_inputs_of_any_scale(what):
    """Inputs are scaled by what some of them show; what fp16 parts do not hold then is computed with bf16 parts, and what those
    do not hold with FMAs."""
    N, C, H, W, K, ks, stride, pad, density = LAYER
    rng = np.random.default_rng(1)
    w = filter_of(rng, K, C, ks, density)
    x = rng.standard_normal((N, C, H, W)).astype(np.float32)
    if what == "2^40":
        x *= np.float32(2.0 ** 40)
    elif what == "2^-60":
        x *= np.float32(2.0 ** -60)
    elif what == "zero where it is looked at":
        x[:, :, ::2] = 0
        x[:, [C * i // 16 for i in range(16)]] = 0
    elif what == "tiny beside ones":
        x[:, :, :, 30:] *= np.float32(2.0 ** -80)
    elif what == "2^120":
        x *= np.float32(2.0 ** 120)
    elif what == "subnormal":
        x *= np.float32(2.0 ** -130)
    odd = None
    if what == "infinite":
        x[1, 20, 13, 50], x[2, 3, 30, 7] = np.inf, np.nan
        odd = ~np.isfinite(x)
    layer = Layer(w, x.shape, stride, pad)
    got = layer(x)
    ref, terms = conv64(np.where(np.isfinite(x), x, 0), w, stride, pad)
    # (a subnormal output is rounded as such, twice)
    off = np.abs(got - ref) <= C * ks * ks * 2.0 ** -24 * terms + 2.0 ** -149
    if odd is not None:
        reached = conv64(odd.astype(np.float32), np.abs(w), stride, pad)[0] > 0
        assert reached.any() and not np.isfinite(got[reached]).any()
        off |= reached
    assert off.all()
    layer.pack.close()


@pytest.mark.parametrize("what,large,small", [
    ("8 bits", 0, -38), ("8 bits", 0, -40), ("one bit", 0, -44), ("bf16", 0, -36),  # their parts add up to them, and are not enough
    ("24 bits", 0, -24), ("24 bits", 0, -27), ("24 bits", 0, -28), ("24 bits", 0, -29), ("24 bits", 0, -34),
    ("24 bits", 44, -126), ("24 bits", 60, -110), ("24 bits", 72, -100), ("24 bits", 110, -60), ("24 bits", 100, -130)])  # lost in its scale
@pytest.mark.parametrize("at", [LAYER, (8, 19, 79, 28, 275, 3, 1, 1, 0.3)])  # (tiles of 128 x 64 and of 128 x 256)
def test_small_inputs_beside_large_ones(at, what, large, small):
    """Stripes of small inputs between stripes of large ones, which the whole tile is scaled by: where an output is a sum of small ones
    alone, it is as exact as the walk's, whatever their size and their number of significant bits."""
    N, C, H, W, K, ks, stride, pad, density = at
    rng = np.random.default_rng(4)
    w = filter_of(rng, K, C, ks, density)
    x = rng.standard_normal((N, C, H, W)).astype(np.float32)
    tiny = {"8 bits": rng.integers(0, 256, x.shape) / 256, "one bit": rng.integers(0, 2, x.shape),
            "bf16": (x.view(np.uint32) & 0xffff0000).view(np.float32), "24 bits": x}[what].astype(np.float32)
    stripe = np.arange(W) // 6 % 2 == 1
    x = np.where(stripe, np.ldexp(tiny, small), np.ldexp(x, large)).astype(np.float32)
    layer = Layer(w, x.shape, stride, pad)
    got, walk = layer(x), layer(x, layer.walk())
    alone = conv64((x != 0) * ~stripe * np.float32(1), (w != 0).astype(np.float32), stride, pad)[0] == 0
    x[..., ~stripe] = 0
    ref, terms = conv64(x, w, stride, pad)
    assert alone.mean() > 0.2
    count = (w != 0).reshape(K, -1).sum(1).reshape(1, K, 1, 1)
    assert (np.abs(got - ref) <= count * 2.0 ** -24 * terms + 2.0 ** -149)[alone].all()
    if small > -120:  # (a subnormal output is rounded twice)
        assert np.linalg.norm((got - ref)[alone]) <= 1.05 * np.linalg.norm((walk - ref)[alone])
    layer.pack.close()


@pytest.mark.parametrize("tiny_weights", [False, True])
@pytest.mark.parametrize("N,C,H,W,K,ks,stride,pad,density", [
    (3, 42, 40, 77, 81, 3, 1, 1, 0.15), (8, 33, 47, 63, 68, 5, 1, 0, 0.3), (11, 120, 18, 70, 11, 7, 2, 0, 0.2), (12, 111, 23, 78, 21, 3, 2, 1, 0.15),
    (8, 117, 38, 38, 183, 1, 1, 0, 0.15), (1, 20, 28, 8, 10, 4, 1, 0, 0.3), (6, 19, 88, 50, 199, 3, 1, 0, 0.2), (4, 17, 52, 80, 258, 3, 1, 1, 0.15)])
def test_a_few_inputs_out_of_range(N, C, H, W, K, ks, stride, pad, density, tiny_weights):
    """Single inputs that fp16 parts do not hold, in the first and the last channels, at an edge and inside: the outputs that they do
    not reach keep the bits that they have without them (so nothing is computed again), and the others are as exact as any."""
    import torch
    import tetris_amd as T

    rng = np.random.default_rng(10)
    w = filter_of(rng, K, C, ks, density)
    if tiny_weights:  # the second of every eighth row, multiplied one by one too
        for k in range(0, K, 8):
            w.reshape(K, -1)[k, np.flatnonzero(w.reshape(K, -1)[k])[1]] *= np.float32(2.0 ** -22)
    without = rng.standard_normal((N, C, H, W)).astype(np.float32)
    at = [(0, C - 1, 5, W - 1, -30), (0, 0, H - 1, 2, -50), (N - 1, C // 2, H // 2, W // 3, 8), (N - 1, 1, H - 2, W // 2, 25)]
    # (The small ones alone.  A large one where a tile's scale is taken from, at the start of a row, would put more than itself out of range.)
    for n, c, y, x, e in at:
        without[n, c if e > 0 else slice(None), max(y - ks, 0):y + ks + 1, max(x - ks, 0):x + ks + 1] = 0
    few = without.copy()
    for n, c, y, x, e in at:
        few[n, c, y, x] = np.ldexp(1 + rng.random(), e)
    layer = Layer(w, few.shape, stride, pad)
    got, again, base = layer(few), layer(few), layer(without)
    reached = conv64((few != without).astype(np.float32), (w != 0).astype(np.float32), stride, pad)[0] != 0
    assert reached.any() and np.array_equal(got, again) and np.array_equal(got[~reached], base[~reached])
    ref, terms = conv64(few, w, stride, pad)
    bound = (w != 0).reshape(K, -1).sum(1).reshape(1, K, 1, 1) * 2.0 ** -24 * terms
    assert (np.abs(got - ref) <= bound).all()
    if layer.pack.act_supported(*layer.at, layer.tile, T.ACT_RELU_POOL2):
        n, k, oh, ow = layer.out
        dx, y = torch.from_numpy(few).cuda(), torch.full((n, k, oh // 2, ow // 2), float("nan"), device="cuda")
        layer.pack.launch_act(dx.data_ptr(), y.data_ptr(), *layer.at, layer.tile, T.ACT_RELU_POOL2)
        quads = lambda a: a[:, :, :oh // 2 * 2, :ow // 2 * 2].reshape(n, k, oh // 2, 2, ow // 2, 2).max((3, 5))  # noqa: E731
        assert (np.abs(y.cpu().numpy() - np.maximum(quads(ref), 0)) <= quads(bound)).all()
    layer.pack.close()


@pytest.mark.parametrize("scale_x,scale_w", [(0, 0), (-10, 3), (-120, 0), (-140, 4), (0, -130), (-70, -60), (40, 20), (80, -100), (120, -10)])
def test_outputs_of_one_term(scale_x, scale_w):
    """Inputs and weights of full 24-bit significands, one product an output: as exact as one rounding of it."""
    N, C, H, W, K, ks, stride, pad, density = 8, 117, 38, 38, 183, 1, 1, 0, 0.15
    rng = np.random.default_rng(8)
    w = np.zeros((K, C), np.float32)
    rest = np.zeros(K * (C - 48), np.float32)  # as many weights as make the library choose half_kernel, and x is zero there
    rest[rng.permutation(rest.size)[:int(density * K * C) - K]] = 1
    w[:, 48:] = rest.reshape(K, C - 48) * (1 + rng.random((K, C - 48)))
    w[np.arange(K), np.arange(K) % 48] = 1 + rng.random(K)
    w = np.ldexp(w, scale_w).astype(np.float32).reshape(K, C, 1, 1)
    x = np.zeros((N, C, H, W), np.float32)
    x[:, :48] = np.ldexp((1 + rng.random((N, 48, H, W))).astype(np.float32), scale_x)
    layer = Layer(w, x.shape, stride, pad)
    assert layer.runs(256, 64, 1)
    got = layer(x)
    ref = conv64(x, w, stride, pad)[0]
    # Half a unit in the last place, and what is left out, 2^-28, and the roundings of the smaller products' sum, which is 2^-8 of the
    # product; of a subnormal output first that of the scaled sum and then its own.
    normal = np.abs(ref) >= 2.0 ** -126
    half = np.where(normal, np.abs(ref) * 2.0 ** -24, 2.0 ** -150)
    assert (np.abs(got - ref) <= half * (1 + 2.0 ** -3) + np.where(normal, 0, np.abs(ref) * 2.0 ** -24)).all()
    layer.pack.close()


@pytest.mark.parametrize("N,C,H,W,K,ks,stride,pad,density", [
    (12, 53, 27, 35, 7, 4, 1, 0, 0.15), (8, 117, 38, 38, 183, 1, 1, 0, 0.15), (8, 19, 79, 28, 275, 3, 1, 1, 0.3),
    (6, 19, 88, 50, 199, 3, 1, 0, 0.2), (11, 120, 18, 70, 11, 7, 2, 0, 0.2), (5, 163, 41, 54, 81, 3, 1, 1, 0.3)])
def test_values_out_of_range_give_what_the_walk_gives(N, C, H, W, K, ks, stride, pad, density):
    """Infinities, NaN and the largest numbers reach the outputs whose window holds them with a weight that is not zero, and no others:
    a wave stores what its passes give over what the pass before has stored, also where that is four pixels at a time (all of these
    layers but the last)."""
    import torch
    import tetris_amd as T

    rng = np.random.default_rng(9)
    w = filter_of(rng, K, C, ks, density)
    x = rng.standard_normal((N, C, H, W)).astype(np.float32)
    x.reshape(-1)[rng.permutation(x.size)[:48]] = np.tile(np.array([np.inf, -np.inf, np.nan, 3.4e38, -3.4e38, 2.0 ** 100, -2.0 ** 90, 1e-45], np.float32), 6)
    layer = Layer(w, x.shape, stride, pad)
    assert (-(-layer.out[3] // 64) == 1 and layer.out[2] * layer.out[3] % 4 == 0) == (C != 163)
    dx = torch.from_numpy(x).cuda()
    terms = conv64(np.where(np.isfinite(x), x, 0), w, stride, pad)[1]
    count = (w != 0).reshape(K, -1).sum(1).reshape(1, K, 1, 1)
    for act in (T.ACT_NONE, T.ACT_RELU, T.ACT_RELU_POOL2):
        if not all(layer.pack.act_supported(*layer.at, t, act) for t in (layer.tile, layer.walk())):
            continue
        n, k, oh, ow = layer.out
        outs, half = [], 2 if act == T.ACT_RELU_POOL2 else 1
        for t in (layer.tile, layer.walk()):
            y = torch.full((n, k, oh // half, ow // half), float("nan"), device="cuda")
            layer.pack.launch_act(dx.data_ptr(), y.data_ptr(), *layer.at, t, act)
            torch.cuda.synchronize()
            outs.append(y.cpu().numpy())
        got, walk = outs
        assert np.array_equal(np.isnan(got), np.isnan(walk)) and np.array_equal(np.isinf(got), np.isinf(walk))
        assert act or (np.isnan(walk).any() and np.isinf(walk).any())
        ok = np.isfinite(walk)
        assert np.array_equal(np.sign(got[~ok]), np.sign(walk[~ok]), equal_nan=True)
        bound = 2 * count * 2.0 ** -24 * terms
        if half == 2:  # of a maximum: the largest bound of the four
            bound = bound[:, :, :oh // 2 * 2, :ow // 2 * 2].reshape(n, k, oh // 2, 2, ow // 2, 2).max((3, 5))
        with np.errstate(all="ignore"):
            assert (np.abs(got.astype(np.float64) - walk)[ok] <= bound[ok]).all()
    layer.pack.close()


@pytest.mark.parametrize("value,count", [(2.0 ** -20, 1), (2.0 ** -40, 60), (2.0 ** -40, 3000), (2.0 ** -100, 1), (2.0 ** -149, 2), (2.0 ** 63, 1)])
def test_small_weights(value, count):
    """Weights far below the largest of their row: multiplied one by one; all with bf16 parts where they are many, or where their
    products would underflow."""
    N, C, H, W, K, ks, stride, pad, density = LAYER
    rng = np.random.default_rng(2)
    w = filter_of(rng, K, C, ks, density)
    there = np.flatnonzero(w)
    w.reshape(-1)[rng.permutation(there)[:count]] = np.float32(value)
    only = np.zeros_like(x := rng.standard_normal((N, C, H, W)).astype(np.float32))
    layer = Layer(w, x.shape, stride, pad)
    for each in (x, only):
        if each is only:  # an input that meets nothing but small weights in a row of the filter
            k, c, r, s = np.argwhere(w == np.float32(value))[0]
            w2 = w[k:k + 1]
            keep = [i for i in range(C) if not (np.abs(w2[0, i]) > abs(value)).any()]
            each[:, keep] = x[:, keep]
        got = layer(each)
        ref, terms = conv64(each, w, stride, pad)
        assert (np.abs(got - ref) <= C * ks * ks * 2.0 ** -24 * terms + 2.0 ** -149).all(), value
    layer.pack.close()


def test_small_weights_of_more_channels_than_their_places_hold():
    """The library would give this layer to half_kernel, whose lists of small weights name channels below 2^20."""
    import torch
    import tetris_amd as T

    C, K, H = 2 ** 20 + 24, 4, 10
    rng = np.random.default_rng(5)
    w = np.zeros((K, C, 1, 1), np.float32)
    w.reshape(-1)[rng.permutation(K * C)[:K * C // 20]] = 1
    at = [7, 2 ** 19 + 3, 2 ** 20 - 1, 2 ** 20, C - 1]
    for k in range(K):
        w[k, at, 0, 0] = np.ldexp(1 + k + np.arange(5), -20).astype(np.float32)
    tile = T.tile_select(1, H, H, C, K, 1, 1, 0)
    pack = T.G950Filter.for_tile(w, tile, oc_order="balanced")
    x, y = torch.zeros((1, C, H, H), device="cuda"), torch.empty((1, K, H, H), device="cuda")
    for c in at:
        x[0, c] = 3
        pack.launch(x.data_ptr(), y.data_ptr(), 1, H, H, 1, 0, tile)
        torch.cuda.synchronize()
        x[0, c] = 0
        assert (y.cpu().numpy()[0] == 3 * w[:, c]).all(), c
    pack.close()


NO_ROOM = """
#include <dlfcn.h>
#include <stddef.h>
#include <stdio.h>
int hipMalloc(void** p, size_t n) {
  int (*real)(void**, size_t) = (int (*)(void**, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_NOLOAD | RTLD_LAZY), "hipMalloc");
  if (n > 4000000 && n < 4800000) { fprintf(stderr, "no room for %zu bytes\\n", n); return 2; }
  return real(p, n);
}
"""
CHILD = """
import ctypes, sys
ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
import numpy as np
import tetris_amd as T
a = np.load(sys.argv[2])
y = T.CudaSparseConv2d(a["x"], a["w"], 4, 28, 28, 128, 256, 3, 1, 1)[0]
np.save(sys.argv[3], y)
"""


def test_no_room_for_the_plan(tmp_path):
    """Where the weights in parts cannot be allocated the layer runs on the walk, which needs a tenth of their room.  (In a process of
    its own, where an allocation of 4 to 4.8 MB is refused: of this layer, the plan's alone.)"""
    import os
    import subprocess
    import sys

    import tetris_amd as T

    N, C, H, W, K, ks, stride, pad = 4, 128, 28, 28, 256, 3, 1, 1
    rng = np.random.default_rng(6)
    w, x = filter_of(rng, K, C, ks, 0.15), rng.standard_normal((N, C, H, W)).astype(np.float32)
    layer = Layer(w, x.shape, stride, pad)
    walk = layer(x, layer.walk())
    layer.pack.close()
    (tmp_path / "no_room.c").write_text(NO_ROOM)
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", tmp_path / "no_room.so", tmp_path / "no_room.c", "-ldl"])
    np.savez(tmp_path / "in.npz", x=x, w=w)
    run = subprocess.run([sys.executable, "-c", CHILD, tmp_path / "no_room.so", tmp_path / "in.npz", tmp_path / "out.npy"], timeout=100,
                         env=dict(os.environ, PYTHONPATH=os.path.dirname(os.path.dirname(T.__file__))), capture_output=True, text=True)
    assert run.returncode == 0 and "no room" in run.stderr, run.stderr
    assert np.linalg.norm(np.load(tmp_path / "out.npy") - walk) <= 1e-6 * np.linalg.norm(walk)


def test_outputs_that_do_not_lie_on_16_bytes():
    """Outputs go out four pixels at a time where they lie so in memory, one by one elsewhere: the same bits."""
    import torch

    N, C, H, W, K, ks, stride, pad, density = 12, 53, 27, 35, 7, 4, 1, 0, 0.15
    rng = np.random.default_rng(3)
    w, x = filter_of(rng, K, C, ks, density), rng.standard_normal((N, C, H, W)).astype(np.float32)
    layer = Layer(w, x.shape, stride, pad)
    count = int(np.prod(layer.out))
    dx, y = torch.from_numpy(x).cuda(), torch.full((2 * count + 16,), float("nan"), device="cuda")
    for first in (0, count + 1):
        layer.pack.launch(dx.data_ptr(), y.data_ptr() + 4 * first, *layer.at, layer.tile)
    torch.cuda.synchronize()
    y = y.cpu().numpy()
    assert count % 4 == 0 and y[:count].tobytes() == y[count + 1:2 * count + 1].tobytes()
    assert np.isnan(y[count]) and np.isnan(y[2 * count + 1:]).all()
    layer.pack.close()
