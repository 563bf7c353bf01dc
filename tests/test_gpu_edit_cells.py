"""Edit-list calls one after the other over one workspace: each finds the masks of its own edits
only, whatever the calls before it edited there (other voxels of the same cells, other cells,
more trees or fewer, trees of another depth in their place, lists that failed)."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_helpers import assert_same

pytestmark = pytest.mark.gpu

MB = 1024 * 1024


@pytest.mark.parametrize("width", [1, 4])
def test_calls_in_a_row(width):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api
    rng = np.random.default_rng(width)
    depths = [5, 2, 4, 6, 3, 5, 4, 2, 6, 3]
    it, it_o = api.VoxInterner(width, 128 * MB), O.Interner(width, 128 * MB)
    f, trees = api.Forest(it, depths), [O.Tree(d) for d in depths]
    dt = {1: np.uint8, 4: np.uint32}[width]
    calls = [(2, 4), (0, 1, 2, 3), (3,), (0, 3, 5, 8), (1, 9), tuple(range(10)), (6, 7), (8, 3), (0,), tuple(range(10))]
    for step, edited in enumerate(calls):
        counts = [int(rng.integers(1, 40)) if t in edited else 0 for t in range(10)]
        offs = np.concatenate([[0], np.cumsum(counts)])
        xyz = np.concatenate([rng.integers(0, 1 << d, (k, 3)) for d, k in zip(depths, counts)]).astype(np.int32)
        val = rng.integers(1, 250, len(xyz)).astype(dt)
        if step in (3, 6):  # one list fails as a whole
            bad = edited[0]
            xyz[int(offs[bad + 1]) - 1] = 99
        else:
            bad = -1
        st = f.apply_edits(offs, api.to_device(xyz), api.to_device(val))
        for t, tr in enumerate(trees):
            a, e = int(offs[t]), int(offs[t + 1])
            if e == a or t == bad:
                assert st[t] == (0 if e == a else -4)
                continue
            b = O.Batch(tr.depth)
            b.set_many(xyz[a:e], val[a:e].astype(np.uint64))
            assert st[t] == (1 if tr.apply_batch(it_o, b) else 0)
        assert_same(it, f, it_o, trees, full_reads=False, what=f"call {step}")
    assert_same(it, f, it_o, trees)
    it.close()
