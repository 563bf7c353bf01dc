"""Edit lists whose offsets begin above 0, a window into a longer list: the edits before the
window belong to no tree, whether or not the first tree has edits of its own."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_helpers import assert_same

pytestmark = pytest.mark.gpu

MB = 1024 * 1024


@pytest.mark.parametrize("width", [1, 2, 4])
@pytest.mark.parametrize("before", [1, 300, 70000])
@pytest.mark.parametrize("first_edited", [True, False])
def test_edits_before_the_window_are_of_no_tree(width, before, first_edited):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api
    rng = np.random.default_rng(before + width)
    depths = [4, 3, 5, 2, 4]
    counts = [int(first_edited) * 5, 0, 3000, 4, 1]
    offs = before + np.concatenate([[0], np.cumsum(counts)])
    total = int(offs[-1]) + 50  # and some behind it
    xyz = rng.integers(0, 4, (total, 3)).astype(np.int32)  # few places: many writes of a voxel
    val = rng.integers(0, 200, total).astype({1: np.uint8, 2: np.uint16, 4: np.uint32}[width])
    it, it_o = api.VoxInterner(width, 64 * MB), O.Interner(width, 64 * MB)
    f = api.Forest(it, depths)
    trees = [O.Tree(d) for d in depths]
    want = []
    for t, tr in enumerate(trees):
        b = O.Batch(tr.depth)
        a, e = int(offs[t]), int(offs[t + 1])
        if e > a:
            b.set_many(xyz[a:e], val[a:e].astype(np.uint64))
        want.append(1 if e > a and tr.apply_batch(it_o, b) else 0)
    for dry in (True, False):
        assert list(f.apply_edits(offs, api.to_device(xyz), api.to_device(val), dry_run=dry)) == want
    assert_same(it, f, it_o, trees)
    it.close()
