"""changaBuildMoments over leaves without particles, the first of them before
the first particle and the last behind the last one: such a leaf reads no
particle. Its record is that of an empty sum (mass 0, centre of mass 0 / 0,
box inside out), its sibling's is bit for bit the record of the same bucket in
a tree without empty leaves, and a node above carries the empty leaf's NaN."""
import ctypes

import numpy as np
import pytest

from changa_amd import gpu

pytestmark = pytest.mark.gpu


def _moments(device, levels, first, count, child, pos, mass, soft):
    """node64 of a tree given by its arrays."""
    import torch
    t = lambda a, d: torch.from_numpy(np.ascontiguousarray(a, dtype=d)).to(device)
    nn = len(first)
    lo = np.asarray(levels, dtype=np.int32)
    ints = [t(a, np.int32) for a in (first, count, child)]
    reals = [t(a, np.float64) for a in (np.full(nn, 0.25), pos, mass, soft)]
    moments = torch.zeros((nn, 27), dtype=torch.float32, device=device)
    node64 = torch.zeros((nn, 34), dtype=torch.float64, device=device)
    p = lambda a: ctypes.c_void_p(a.data_ptr())
    rc = gpu.lib().changaBuildMoments(nn, len(lo) - 1, lo.ctypes.data_as(ctypes.c_void_p),
                                      *map(p, ints), *map(p, reals), p(moments), p(node64), None,
                                      ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    gpu.check(rc, "changaBuildMoments")
    torch.cuda.synchronize()
    return node64.cpu().numpy()


@pytest.mark.parametrize("n", [1, 4, 16, 21])
def test_gpu_moment_empty_leaves(device, n):
    rng = np.random.default_rng(n)
    pos, mass, soft = rng.normal(size=(n, 3)), rng.uniform(0.5, 1.0, n), rng.uniform(0.1, 0.2, n)
    alone = _moments(device, [0, 1], [0], [n], [-1, -1], pos, mass, soft)
    # root -> (empty leaf, node); node -> (bucket, empty leaf)
    g = _moments(device, [0, 1, 3, 5], [0, 0, 0, 0, n], [n, 0, n, n, 0],
                 [1, 2, -1, -1, 3, 4, -1, -1, -1, -1], pos, mass, soft)
    np.testing.assert_array_equal(g[3], alone[0])
    for nd in (1, 4):
        assert g[nd, 5] == 0.0 and np.isnan(g[nd, 0:3]).all()
        assert (g[nd, 6:9] == np.inf).all() and (g[nd, 9:12] == -np.inf).all()
    for nd in (0, 2):
        assert np.isnan(g[nd, 0:3]).all() and g[nd, 5] == alone[0, 5]
