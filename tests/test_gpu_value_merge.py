"""Completely written bricks of different values that occur many times in a block, over every
kind of old node: nothing, a branch, a leaf above them, a leaf of their own (the reference's
panic) and a fill; beside partial, all-same and untouched bricks, with values that no leaf
holds yet, and with more different bricks than a block's set takes."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_helpers import assert_same, oracle_apply_dense

pytestmark = pytest.mark.gpu

MB = 1024 * 1024
NP = {1: np.uint8, 2: np.uint16, 4: np.uint32}


def _batch(rng, width, depth, step, patterns, kinds):
    """One tree's Batch buffers: a kind per brick of `kinds` (0 untouched, 1 a pattern over
    all eight voxels, 2 a pattern over some, 3 one value)."""
    n = 8 ** (depth - 1)
    kind = rng.choice(kinds, size=n)
    values = patterns[rng.integers(0, len(patterns), n)].copy()
    values[kind == 3] = values[kind == 3][:, :1]
    mask = np.where(kind == 0, 0, np.where(kind == 2, rng.integers(1, 255, n), 255)).astype(np.uint8)
    values[~np.unpackbits(mask[:, None], axis=1, bitorder="little").astype(bool)] = 0
    masks = np.zeros((n, 2), dtype=np.uint8)
    masks[:, 0] = mask
    return masks, np.ascontiguousarray(values.astype(NP[width]))


@pytest.mark.parametrize("brick_rounds", [1, 2, 4])
@pytest.mark.parametrize("width", [1, 2, 4])
@pytest.mark.parametrize("few", [True, False])
def test_full_bricks_over_every_old_node(few, width, brick_rounds):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api
    rng = np.random.default_rng(width)
    depths = [5, 2, 4, 2, 3, 4, 2, 5, 6, 3]
    it, it_o = api.VoxInterner(width, 64 * MB), O.Interner(width, 64 * MB)
    it.set_tuning(brick_rounds=brick_rounds)
    f, trees = api.Forest(it, depths), [O.Tree(d) for d in depths]
    seen = set()
    for step in range(5):
        # (every step's values are its own: a value written over a split leaf of that value
        # meets the reference's missing reference counts, whose outcome depends on the order)
        patterns = rng.integers(40 * step + 1, 40 * step + 41, (4 if few else 2000, 8)).astype(NP[width])
        ms, vs, fills, want = [], [], [], []
        for i, (t, d) in enumerate(zip(trees, depths)):
            # one tree in three becomes a leaf, or bricks that are leaves, for the next step
            kinds = [[1], [3], [0, 1, 2, 3], [1, 1, 1, 2]][(step + i) % 4]
            one = patterns[:1] if kinds == [3] and i % 3 == 0 else patterns
            m, v = _batch(rng, width, d, step, one, kinds)
            fill = 210 + step if (step + 2 * i) % 7 == 3 else None
            ms.append(m)
            vs.append(v)
            fills.append(fill)
            snap, before = O.lib().vxo_snapshot_take(it_o.h), t.root
            try:
                want.append(1 if oracle_apply_dense(it_o, t, m, v, fill=fill)[0] else 0)
            except O.OraclePanic:
                O.lib().vxo_snapshot_restore(it_o.h, snap)
                t.root = before
                want.append(-1)
            finally:
                O.lib().vxo_snapshot_free(snap)
        st = f.apply([api.to_device(m) for m in ms], [api.to_device(v) for v in vs], fills=fills)
        assert [min(int(s), 1) if s >= 0 else -1 for s in st] == want, (step, st, want)
        seen.update(want)
        assert_same(it, f, it_o, trees, full_reads=step == 4, what=f"step {step}")
    assert {-1, 1} <= seen
    assert it.stats()["brick_merged"] > 0 or not few
