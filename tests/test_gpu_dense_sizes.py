"""Dense extractions on both sides of the size where cells take over from a lane per voxel, at
strides that are and are not the trees' own."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1024 * 1024
LINE = 25 << 15  # places


@pytest.mark.parametrize("width", [1, 2, 4])
@pytest.mark.parametrize("depth,stride", [(5, 32768), (5, 33001), (4, 4096), (3, 512), (3, 4096), (2, 65)])
def test_around_the_line(width, depth, stride):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api, lib
    from voxelis_amd import workloads as W
    from voxelis_amd._lib import check
    rng = np.random.default_rng(depth)
    side, some = 1 << depth, 7
    dt = {1: np.uint8, 2: np.uint16, 4: np.uint32}[width]
    dense = [np.where(rng.random((side,) * 3) < 0.3, rng.integers(1, 250, (side,) * 3), 0).astype(dt) for _ in range(some)]
    dense[1][:] = 9  # one leaf
    dense[2][: side // 2] = 0
    for k in range(some):
        dense[k][-1, -1, -1] = 1 + k
    at = LINE // stride
    for n in (at - 1, at, at + 1):
        it = api.VoxInterner(width, 64 * MB)
        base = api.Forest(it, [depth] * some)
        bat = [W.dense_to_batch(v, depth) for v in dense]
        assert (base.apply([api.to_device(m) for m, _ in bat], [api.to_device(v) for _, v in bat]) == 1).all()
        f = api.Forest(it, [depth] * n)
        pick = rng.integers(0, some, n)
        f.roots.copy_(base.roots[torch.from_numpy(pick).cuda()])
        out = torch.full((n * stride * width,), 0xAB, dtype=torch.uint8, device="cuda")
        check(lib().vx_trees_to_vec(it.h, n, f.roots.data_ptr(), f.depths.data_ptr(), 0, C.c_uint64(stride), out.data_ptr()), "to_vec")
        it.sync()
        got = out.cpu().numpy().view(dt).reshape(n, stride)
        want = np.stack([v.reshape(-1) for v in dense])
        assert np.array_equal(got[:, :side ** 3], want[pick])
        assert (got[:, side ** 3:] == np.frombuffer(b"\xab" * width, dt)[0]).all()
        it.close()
