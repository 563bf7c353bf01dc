"""Edit-list calls of more voxels than one window of the winners' array (2^27) holds: the same
trees as the oracle's, on both sides of a window's end, with trees that are not edited or are
rejected between them, and no more memory than the winners of one window beside what the dense
batches take."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

MB = 1024 * 1024
WINDOW = 1 << 27


def test_calls_of_several_windows():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api
    rng = np.random.default_rng(5)
    # 64 trees of 128^3 fill a window exactly; smaller ones shift the later windows' ends
    depths = [7] * 64 + [7, 2, 5] + [7] * 70 + [1, 4] + [7] * 3
    n = len(depths)
    counts = rng.integers(1, 60, n)
    counts[[10, 64, 80]] = 0
    it, it_o = api.VoxInterner(1, 512 * MB), O.Interner(1, 512 * MB, extended_depth=True)
    f = api.Forest(it, depths)
    trees = {t: O.Tree(depths[t]) for t in (0, 9, 11, 62, 63, 65, 66, 67, 127, 128, 129, 130, 131, 138, n - 1)}
    offs = np.concatenate([[0], np.cumsum(counts)])
    for step in range(2):
        xyz = np.concatenate([rng.integers(0, 1 << d, (k, 3)) for d, k in zip(depths, counts)]).astype(np.int32)
        xyz[offs[1:][counts > 1] - 1] = xyz[offs[1:][counts > 1] - 2]  # the last two writes share a voxel
        val = rng.integers(1, 250, len(xyz)).astype(np.uint8)
        st = f.apply_edits(offs, api.to_device(xyz), api.to_device(val))
        for t in range(n):
            assert st[t] == (0 if counts[t] == 0 else -3 if depths[t] == 1 else 1), (t, st[t])
        for t, tr in trees.items():
            a, e = int(offs[t]), int(offs[t + 1])
            b = O.Batch(tr.depth)
            b.set_many(xyz[a:e], val[a:e].astype(np.uint64))
            assert tr.apply_batch(it_o, b)
        got = f.canonical_hashes()
        for t, tr in trees.items():
            assert got[t] == tr.canonical_hash(it_o), (step, t)
    it.close()


def test_memory_of_a_large_call():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api
    n, depth = 130, 7
    voxels = n * 8 ** depth
    masks = torch.zeros(8 ** (depth - 1), 2, dtype=torch.uint8, device="cuda")
    masks[0, 0] = 1
    values = torch.ones(8 ** (depth - 1), 8, dtype=torch.uint8, device="cuda")
    offs = np.arange(n + 1)
    xyz, val = api.to_device(np.zeros((n, 3), np.int32)), api.to_device(np.ones(n, np.uint8))

    def taken(call):
        it = api.VoxInterner(1, 64 * MB)
        f = api.Forest(it, [depth] * n)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        assert (call(f) == 1).all()
        used = free - torch.cuda.mem_get_info()[0]
        it.close()
        return used

    taken(lambda f: f.apply([masks] * n, [values] * n))  # (the runtime's own first allocations)
    dense = taken(lambda f: f.apply([masks] * n, [values] * n))
    edits = taken(lambda f: f.apply_edits(offs, xyz, val))
    # masks and values of every voxel, one window's winners and dirty cells, allocation granules
    assert edits - dense <= voxels * 5 // 4 + WINDOW * 4 + WINDOW // 512 + 32 * MB, (edits, dense)
