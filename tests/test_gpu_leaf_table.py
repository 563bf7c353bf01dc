"""The hashed leaf table of four-byte voxels is rebuilt when tombstones fill it, whoever left
them (dry runs, applies rolled back for their node limit, frees), and is not when the
tombstones that frees leave are taken again by the next values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BUDGET = 40000  # 487 nodes, a leaf table of 1024 slots
TREES = 100


def _forest(n):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api
    it = api.VoxInterner(4, BUDGET)
    return it, api.Forest(it, [3] * n)


def _fill(f, vals, **opts):
    none = [None] * f.n
    return f.apply(none, none, fills=[int(v) for v in vals], has_patches=[False] * f.n, **opts)


@pytest.mark.parametrize("kind", ["dry run", "rolled back"])
def test_table_full_of_tombstones_is_rebuilt(kind):
    it, f = _forest(TREES)
    rng = np.random.default_rng(1)
    # 4000 new values over 1024 slots: all but a few slots have held an entry
    for _ in range(40):
        vals = rng.integers(1, 1 << 31, TREES)
        st = _fill(f, vals, **({"dry_run": True} if kind == "dry run" else {"node_limit": 1}))
        assert (st == (1 if kind == "dry run" else -8)).all()
        assert it.counts() == (0, 1)
    if kind == "dry run":  # (a rolled back apply is a write call and has rebuilt it by then)
        assert it.table_stats()[2] == 0
    assert (_fill(f, vals) == 1).all()
    assert it.table_stats()[2] >= 1
    assert it.counts() == (TREES, 1)
    got, p = f.get(np.arange(TREES, dtype=np.uint32), np.zeros((TREES, 3), dtype=np.int32))
    assert (p == 1).all() and np.array_equal(got, vals.astype(np.uint64))
    it.close()


def test_tombstones_taken_again_are_not_counted():
    it, f = _forest(1)
    for i in range(2000):  # each apply frees the other value's leaf: one tombstone at a time
        f.apply([None], [None], fills=[7 + i % 2], has_patches=[False], sync=False)
    it.sync()
    assert it.counts() == (1, 1)
    assert it.table_stats()[2] == 0
    it.close()
