"""The multipole build over trees whose depths go into shared launches, into
launches of their own, or both: one bucket, two levels, a few thousand nodes
in all, depths beyond the shared launches' node limit, and buckets of one to
more particles than a lane holds, against the FP64 oracle.

Bars as in test_gpu_parity's moment test, and for the same reasons: the
geometry is a few FP64 operations (1e-12), a node's moments carry at most its
depth's shift-and-project steps of FP64 rounding (1e-10 of the node's
largest)."""
import numpy as np
import pytest

from changa_amd import configs, engine
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,bucket", [(5, 16), (17, 16), (40, 3), (700, 1), (4097, 9),
                                      (30000, 16), (30000, 100), (150000, 8)])
def test_gpu_moment_depths(device, n, bucket):
    import torch
    w = configs.plummer(n=n, bucket=bucket)
    w["mass"] = w["mass"] * (0.5 + np.random.default_rng(n).uniform(size=n))
    ev = engine.Evaluation(w, device=device, tree="gpu", lists="none")
    torch.cuda.synchronize()
    g = ev.node64()
    geo, mom = O.build_moments(ev.tree, ev.pos, ev.mass, ev.soft)
    print(f"n {n} bucket {bucket}: {ev.tree['n_nodes']} nodes, {ev.tree['n_depths']} depths, "
          f"widest {np.diff(ev.tree['level_offsets']).max()}", flush=True)
    np.testing.assert_allclose(g[:, 0:12], geo, rtol=1e-12, atol=1e-14)
    scale = np.abs(mom).max(axis=1, keepdims=True)
    assert (np.abs(g[:, 12:] - mom) / scale).max() < 1e-10
