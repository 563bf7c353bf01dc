"""Dry runs whose fill leaves do not exist yet, over more trees than a wavefront or a block
holds: every missing leaf is counted once, and no request stays behind in the leaf table (an
entry left there would be waited for by the apply that needs the value)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1024 * 1024


@pytest.mark.parametrize("width", [1, 2, 4])
@pytest.mark.parametrize("trees", [1, 65, 257, 5000])
def test_new_fills_are_counted_and_leave_nothing(width, trees):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api
    it = api.VoxInterner(width, 64 * MB)
    f = api.Forest(it, [3] * trees)
    distinct = min(trees, 255 if width == 1 else 60000)
    for step in range(4):
        # as many values as the width has; the next step's are new again
        vals = [((t % distinct) * 2654435761 % (1 << 32) if width == 4 else t % distinct) + 1 + step % 2 * (width > 1)
                for t in range(trees)]
        new = len(set(vals) - (set(held) if step else set()))
        none = [None] * trees
        for _ in range(3):
            st = f.apply(none, none, fills=vals, has_patches=[False] * trees, dry_run=True, counts=True)
            same = [step > 0 and held[t] == vals[t] for t in range(trees)]
            assert (st == [-6 if s else 1 for s in same]).all()
            assert f.counts_host()[:2] == (0, new), (step, f.counts_host()[:2], new)
        st = f.apply(none, none, fills=vals, has_patches=[False] * trees)
        assert (st == [-6 if s else 1 for s in same]).all()
        held = vals
        assert it.counts() == (len(set(held)), 1)
        v, p = f.get(np.arange(trees, dtype=np.uint32), np.zeros((trees, 3), dtype=np.int32))
        assert (p == 1).all() and np.array_equal(v, np.asarray(vals, dtype=np.uint64))
    it.close()
