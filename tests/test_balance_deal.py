"""tetris_oc_order_balanced against a plain restatement of its deal: on a filter small enough for one thread, on one whose
non-zeros are counted by several, and where waves, slots and stages do not come out even."""
import numpy as np
import pytest

import tetris_amd as T


def deal(w, g, waves, tile_ic):
    K, C = w.shape[:2]
    S, B, nsimd = -(-C // tile_ic), g * waves, min(4, waves)
    per = np.stack([(w[:, s * tile_ic:(s + 1) * tile_ic] != 0).reshape(K, -1).sum(1) for s in range(S)], 1).astype(np.int64)
    nblocks = -(-K // B)
    blocks, b, d = [[] for _ in range(nblocks)], 0, 1

    def step(b, d):
        b += d
        return (b - d, -d) if b < 0 or b >= nblocks else (b, d)

    for k in np.argsort(-per.sum(1), kind="stable"):
        while len(blocks[b]) >= min(B, K - b * B):
            b, d = step(b, d)
        blocks[b].append(int(k))
        b, d = step(b, d)
    order = []
    for blk in blocks:
        load, simd = np.zeros((waves, S), np.int64), np.zeros((nsimd, S), np.int64)
        members = [[] for _ in range(waves)]
        for k in blk:
            def cost(v):
                return (int(np.maximum(simd.max(0), simd[v % nsimd] + per[k]).sum()),
                        int(np.maximum(load.max(0), load[v] + per[k]).sum()), int(load[v].sum()))
            free = [v for v in range(waves) if len(members[v]) < min(g, max(0, len(blk) - v * g))]
            v = min(free, key=cost)
            load[v] += per[k]
            simd[v % nsimd] += per[k]
            members[v].append(k)
        order += [k for m in members for k in m]

    def waits(o):
        total = 0
        for b in range(nblocks):
            sums = [per[o[b * B + v * g:min(b * B + (v + 1) * g, (b + 1) * B)]].sum(0) for v in range(waves)]
            total += int(np.max(sums, 0).sum())
        return total

    return list(range(K)) if waits(list(range(K))) <= waits(order) else order


@pytest.mark.parametrize("K,C,ks,g,waves,tile_ic", [(1, 1, 1, 1, 1, 1), (70, 83, 3, 8, 4, 8), (33, 3, 7, 4, 2, 3),
                                                   (256, 512, 3, 8, 16, 64), (1030, 1024, 1, 16, 8, 32)])
def test_order_is_the_stated_deal(K, C, ks, g, waves, tile_ic):
    rng = np.random.default_rng(K * C)
    density = np.clip(rng.lognormal(np.log(0.1), 0.7, K), 0, 0.9)
    density[rng.random(K) < 0.1] = 0
    w = (rng.random((K, C, ks, ks), dtype=np.float32) * (rng.random((K, C, ks, ks), dtype=np.float32) < density[:, None, None, None]))
    got = T.oc_order_balanced(w.astype(np.float32), T.Tile(7, 1, g, waves, tile_ic))
    assert got.tolist() == deal(w, g, waves, tile_ic)


def test_order_of_more_weights_than_32_bits_count():
    """2^31 weights and some (nearly all zero: pages that are never written take no memory) are ordered as any others."""
    K, C = 32769, 65540
    w = np.zeros((K, C, 1, 1), np.float32)
    dense = np.arange(K) // 64 < 128
    dense &= np.arange(K) % 64 < 8  # in file order one wave of a workgroup holds all that the workgroup has
    w[dense, :40, 0, 0] = 1.0
    got = T.oc_order_balanced(w, T.Tile(7, 1, 8, 8, 32768))
    assert np.array_equal(np.sort(got), np.arange(K))
    # 1024 channels dealt to 513 blocks of 64, forth and back, and there to different waves of eight
    waves = dense[got[:64 * 512]].reshape(512, 8, 8).sum(2)
    assert waves.max() == 1 and waves.sum(1).min() == 1 and waves.sum(1).max() == 2
