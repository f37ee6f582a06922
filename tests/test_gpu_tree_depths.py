"""The depths of a GPU-built tree against the host builder, every array equal:
trees with fewer nodes than one block of the depth kernels, with depths of
several groups of blocks, with one particle per bucket, and with more depths
than are queued at a time (up to one split per key bit)."""
import numpy as np
import pytest

from changa_amd import configs, engine, host
from tests.helpers import deep_chain_workload

pytestmark = pytest.mark.gpu

KEYS = ("perm", "node_first", "node_count", "node_child", "node_depth", "node_box_radius",
        "level_offsets", "bucket_node", "bucket_start", "bucket_size")


def _bit_chain():
    """Two particles that differ in each key bit alone, from the highest to
    the lowest: a chain of 63 splits."""
    pos = [np.zeros(3)]
    for bit in range(21):
        for axis in range(3):
            p = np.zeros(3)
            p[axis] = 0.5 ** (bit + 1)
            pos.append(p)
    return np.array(pos)


def _uniform(n):
    return np.random.default_rng(n).random((n, 3))


CASES = {
    "one": (_uniform(1), 1),
    "two": (_uniform(2), 1),
    "257_single": (_uniform(257), 1),
    "40000_single": (_uniform(40000), 1),
    "200000_single": (_uniform(200000), 1),
    "200000_bucket_7": (_uniform(200000), 7),
    "bucket_over_n": (_uniform(300), 400),
    "deep_chain": (deep_chain_workload()["pos"], 12),
    "deep_chain_single": (deep_chain_workload()["pos"], 1),
    "bit_chain": (_bit_chain(), 1),
    "clustered": (configs.plummer(n=70000)["pos"], 2),
}


@pytest.mark.parametrize("case", list(CASES))
def test_gpu_tree_depths(device, case):
    pos, bucket = CASES[case]
    kw = dict(box_lo=np.zeros(3), box_size=1.0) if case == "bit_chain" else {}
    th = host.build_tree(pos, bucket, **kw)
    tg = engine.gpu_build_tree(pos, bucket, device=device, **kw)
    print(f"tree {case}: {th['n_nodes']} nodes, {th['n_depths']} depths, widest "
          f"{np.diff(th['level_offsets']).max()}", flush=True)
    for k in ("n", "n_nodes", "n_buckets", "n_depths"):
        assert tg[k] == th[k], k
    for k in KEYS:
        np.testing.assert_array_equal(tg[k], th[k], err_msg=k)
