"""A destroyed interner gives back everything that its calls made it keep."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1024 * 1024


@pytest.mark.parametrize("kind", ["set", "apply", "edits", "fill"])
def test_nothing_is_left_behind(kind):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api
    n, depth = 60000, 4
    xyz = torch.zeros(n, 3, dtype=torch.int32, device="cuda")
    val = torch.full((n,), 3, dtype=torch.uint8, device="cuda")
    masks = torch.zeros(8 ** (depth - 1), 2, dtype=torch.uint8, device="cuda")
    masks[0, 0] = 1
    values = torch.full((8 ** (depth - 1), 8), 5, dtype=torch.uint8, device="cuda")

    def cycle():
        it = api.VoxInterner(1, 256 * MB)
        f = api.Forest(it, [depth] * n)
        if kind == "set":
            f.set_voxels(xyz, val)
        elif kind == "apply":
            f.apply([masks] * n, [values] * n)
        elif kind == "edits":
            f.apply_edits(np.arange(n + 1), xyz, val)
        else:
            f.fill([7] * n)
        it.close()
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info()[0]

    free = [cycle() for _ in range(7)]
    # the runtime keeps what its first calls need; a set keeps 14 words per tree, 6.7 MB here
    assert free[2] - free[6] < 4 * MB, free
