"""The adjoint's sort of a cell list beyond 512 tiles (8,192 entries each),
where the tiles' counters are summed in rows before the scan, with a last row
that is not full; and at the widest digits of two passes and in three passes
(trees of 2^22 nodes and one more: the same tree with unused nodes behind it).

Compared per cell with the FP64 sum over the same lists; bar and reasons as in
test_gpu_transpose. The gradient does not depend on how the keys are cut into
digits but for the order of FP64 atomic sums: 1e-12 of the largest component."""
import numpy as np
import pytest

from changa_amd import configs, engine
from tests.test_gpu_transpose import _cell_sums

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def case(device):
    ev = engine.Evaluation(configs.plummer(n=60000, bucket=8), precise=True, device=device)
    tiles = -(-int(ev.t_lists["cell_marks"][-1]) // 8192)
    per = -(-tiles // 512)
    assert per > 1 and tiles % per
    w = np.random.default_rng(5).normal(size=(ev.n_targets, 3)).astype(np.float32)
    return ev, w, _cell_sums(ev, w, ev.node64()[:, 0:3]), ev.adjoint(w).cpu().numpy()


@pytest.mark.parametrize("nodes", [0, 1 << 22, (1 << 22) + 1])
def test_gpu_adjoint_transpose_long(case, nodes, monkeypatch):
    import torch
    ev, w, (d0, scale), grad = case
    nn = ev.tree["n_nodes"]
    if nodes:
        pad = lambda t, v, per: torch.cat([t.reshape(-1), torch.full(((nodes - nn) * per,), v,
                                                                     dtype=t.dtype,
                                                                     device=t.device)])
        for k, v, per in (("d_first", 0, 1), ("d_count", 0, 1), ("d_child", -1, 2),
                          ("d_node64", 1.0, 34)):
            monkeypatch.setattr(ev, k, pad(getattr(ev, k), v, per))
        monkeypatch.setattr(ev, "tree", dict(ev.tree, n_nodes=nodes))
    for k in ("d_node_work", "d_list_work"):
        monkeypatch.setattr(ev, k, None)
    g = ev.adjoint(w).cpu().numpy()
    got = ev.d_node_work[:nn, 0].cpu().numpy()
    off, used = np.abs(got - d0), scale > 0
    d = (np.abs(g - grad) / np.abs(grad).max(axis=0)).max()
    print(f"{nodes or nn} nodes: {ev.t_lists['cell_marks'][-1]} entries, max off "
          f"{(off[used] / scale[used]).max():.1e}, gradient {d:.1e}", flush=True)
    assert (off <= 1e-5 * scale).all()
    assert d <= 1e-12
