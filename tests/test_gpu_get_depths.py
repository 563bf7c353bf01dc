"""Grouped reads whose last runs are cut by the depths of the trees: worlds of shallow trees, of
deep ones, of both, and of more trees than the kernel looks at, at query counts around the
sizes where the runs' length changes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WORLDS = {"one shallow": [5], "one deep": [6], "mixed": [5, 6, 2, 6, 4], "deep": [6, 6, 6],
          "many shallow": [3, 2, 4] * 100, "a few deep of many": [3] * 150 + [6] + [2] * 150 + [6]}


@pytest.mark.parametrize("world", sorted(WORLDS))
def test_every_query_is_answered(world):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api, workloads as W
    depths = WORLDS[world]
    rng = np.random.default_rng(len(depths))
    it = api.VoxInterner(2, 128 << 20)
    f = api.Forest(it, depths)
    dense = [np.where(rng.random((1 << d,) * 3) < 0.4, rng.integers(1, 60000, (1 << d,) * 3), 0).astype(np.uint16)
             for d in depths]
    for v in dense:
        v[0, 0, 0] = 1
    bat = [W.dense_to_batch(v, d) for v, d in zip(dense, depths)]
    assert (f.apply([api.to_device(m) for m, _ in bat], [api.to_device(v) for _, v in bat]) == 1).all()
    first = np.concatenate([[0], np.cumsum([v.size for v in dense])])
    flat = np.concatenate([v.reshape(-1) for v in dense])
    d = np.array(depths)
    for nq in (1, 511, 512 * 4 + 1, 512 * 4096 + 1, 768 * 4096 - 1, 1_024 * 4096 + 77, 2_560 * 4096 + 5):
        cuts = np.sort(rng.integers(0, nq + 1, len(depths) - 1))
        offsets = np.concatenate([[0], cuts, [nq]]).astype(np.uint64)
        tree = np.repeat(np.arange(len(depths)), np.diff(offsets.astype(np.int64)))
        xyz = (rng.integers(0, 64, (nq, 3), dtype=np.int32) & ((1 << d[tree]) - 1)[:, None]).astype(np.int32)
        side = 1 << d[tree].astype(np.int64)
        want = flat[first[tree] + (xyz[:, 1] * side + xyz[:, 2]) * side + xyz[:, 0]]
        values, present = f.get_grouped(offsets, xyz)
        assert np.array_equal(np.where(present == 1, values, 0), want), nq
        assert np.array_equal(present == 1, want != 0), nq
    it.close()
