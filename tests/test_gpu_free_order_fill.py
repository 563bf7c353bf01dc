"""The free stack after a world was cleared by one call: the next call's nodes lie together in
the pool, since the stack was put in index order first."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1024 * 1024
RUN = 8192  # nodes of one run of the ordered stack


@pytest.mark.parametrize("width", [2, 4])
@pytest.mark.parametrize("aborted", [False, True])
def test_nodes_after_a_clear_lie_together(width, aborted):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api
    rng = np.random.default_rng(width)
    trees, depth = 48, 6
    it = api.VoxInterner(width, 512 * MB)
    f = api.Forest(it, [depth] * trees)
    n = 8 ** (depth - 1)
    dt = np.uint16 if width == 2 else np.uint32
    for k in range(2):  # the second world's nodes come from what the first one's clear freed
        v = rng.integers(1, 60000, (trees, n, 8)).astype(dt)
        v[rng.random(v.shape) >= 0.1] = 0
        m = np.zeros((trees, n, 2), dtype=np.uint8)
        m[:, :, 0] = np.packbits(v != 0, axis=2, bitorder="little")[:, :, 0]
        assert (f.apply([api.to_device(x) for x in m], [api.to_device(x) for x in v]) == 1).all()
        assert it.alive_nodes() > 1 << 18
        f.fill([0] * trees)
        assert it.alive_nodes() == 1
    small = 64
    g = api.Forest(it, [2] * small)
    m = np.zeros((8, 2), dtype=np.uint8)
    m[0, 0] = 3  # two voxels of one brick
    v = np.zeros((small, 8, 8), dtype=dt)
    v[:, 0, 0] = np.arange(small) + 1
    v[:, 0, 1] = 7000
    args = ([api.to_device(m)] * small, [api.to_device(x) for x in v])
    if aborted:  # an apply rolled back on the ordered stack leaves it so
        assert (g.apply(*args, node_limit=5) == -8).all()
    assert (g.apply(*args) == 1).all()
    at = np.array([r & 0xFFFFFFFF for r in g.roots_host()])
    assert len(set(at.tolist())) == small
    assert len(set((at // RUN).tolist())) <= 2, sorted(set((at // RUN).tolist()))
    it.close()
