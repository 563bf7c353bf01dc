"""Grouped reads of a batch that is cut into long runs and, at its end, shorter ones: the
values written, at sizes where the two kinds of runs meet and end at odd places."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq", [512 * 4096, 512 * 4096 + 1, 3_000_001, 4_194_303])
def test_grouped_reads_of_long_and_short_runs(nq):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api, workloads as W
    rng = np.random.default_rng(nq)
    depths = [5, 2, 6, 4, 5, 3]
    it = api.VoxInterner(2, 64 << 20)
    f = api.Forest(it, depths)
    dense = [np.where(rng.random((1 << d,) * 3) < 0.4, rng.integers(1, 60000, (1 << d,) * 3), 0).astype(np.uint16)
             for d in depths]
    bat = [W.dense_to_batch(v, d) for v, d in zip(dense, depths)]
    assert (f.apply([api.to_device(m) for m, _ in bat], [api.to_device(v) for _, v in bat]) == 1).all()
    cuts = np.sort(rng.integers(0, nq + 1, len(depths) - 1))
    offsets = np.concatenate([[0], cuts, [nq]]).astype(np.uint64)
    tree = np.repeat(np.arange(len(depths)), np.diff(offsets.astype(np.int64)))
    xyz = (rng.integers(0, 64, (nq, 3)) & ((1 << np.array(depths)[tree]) - 1)[:, None]).astype(np.int32)
    want = np.zeros(nq, dtype=np.uint64)
    for t in range(len(depths)):
        s = slice(int(offsets[t]), int(offsets[t + 1]))
        want[s] = dense[t][xyz[s, 1], xyz[s, 2], xyz[s, 0]]
    values, present = f.get_grouped(offsets, xyz)
    assert np.array_equal(np.where(present == 1, values, 0), want)
    assert np.array_equal(present == 1, want != 0)
