"""A pack made in the balanced order in one call (order and upload side by side) holds what the two calls give, byte for byte."""
import numpy as np
import pytest

from helpers import sparse_filter

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,C,ks,tile_ic,g,waves", [(1, 1, 1, 1, 1, 1), (33, 7, 3, 4, 8, 4), (160, 48, 3, 16, 4, 16),
                                                   (130, 900, 1, 64, 2, 16), (512, 256, 3, 8, 8, 8)])
def test_one_call_equals_order_then_pack(K, C, ks, tile_ic, g, waves, oracle):
    import torch
    import tetris_amd as T

    assert torch.cuda.is_available()
    w = sparse_filter(np.random.default_rng(K + C), K, C, ks, 0.85)
    tile = T.Tile(7, 1, g, waves, tile_ic)
    order = T.oc_order_balanced(w, tile)
    one, two = T.G950Filter.for_tile(w, tile, oc_order="balanced"), T.G950Filter(w, tile_ic, g, order)
    a, b = one.host_arrays(), two.host_arrays()
    ref = oracle.G950Pack(w, tile_ic, g, order)
    assert a["nnz"] == b["nnz"] == int((w != 0).sum())
    for name in ("grp_offsets", "grp_nnz", "position", "values", "oc_order"):
        assert a[name].tobytes() == b[name].tobytes(), name
    assert np.array_equal(a["oc_order"][:K], order) and np.array_equal(a["position"], ref.position)
    with pytest.raises(T.TetrisError):
        T.G950Filter.for_tile(w, T.Tile(7, 1, 0, waves, tile_ic), oc_order="balanced")


def test_refused_pack_has_let_go_of_the_filter():
    """A pack that is refused for its arguments returns only when the upload no longer reads the caller's (pinned) filter."""
    import torch
    import tetris_amd as T

    w = torch.zeros((4096, 4096, 2, 2), pin_memory=True)  # 256 MiB: some milliseconds of upload
    torch.cuda.synchronize()
    with pytest.raises(T.TetrisError) as e:
        T.G950Filter(w.numpy(), 8, 3)  # three channels to a wave
    assert torch.cuda.default_stream().query()
    assert e.value.code == T.EINVAL
