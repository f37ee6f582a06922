"""The adjoint's sort of the cell list (transpose.h) at sizes where it can go
wrong: lists of less than a wavefront, of part of a tile and of several
tiles, keys of one and of two digit passes, buckets without cells, a rung in
a periodic box.

After an adjoint the caller's node scratch holds, per cell, the order-0
tensor D_0 = -sum_i w_i . r_i / r_i^3 over the targets of every bucket that
lists the cell: it is compared with that sum in FP64 over the same lists. Bar
per cell: 1e-5 of sum_i |w_i| / r_i^2. A term's FP32 evaluation is at most
about 15 roundings of 6e-8 off relative to |w| / r^2, and the sums add at most
100 in FP32 one after another (then FP64). A lost, doubled or misplaced entry
changes D_0 by whole terms."""
import numpy as np
import pytest

from changa_amd import configs, engine

pytestmark = pytest.mark.gpu


def _cell_sums(ev, w, cm):
    """(D_0, sum of |w| / r^2) per node, FP64, from the target buckets' lists."""
    L = ev.t_lists if "cells" in ev.t_lists else ev.lists
    cells = np.asarray(L["cells"]).reshape(-1, 2)
    marks = np.asarray(L["cell_marks"], dtype=np.int64)
    pos = ev.pos if ev.t_index is None else ev.pos[ev.t_index]
    d0, scale = np.zeros(ev.tree["n_nodes"]), np.zeros(ev.tree["n_nodes"])
    for b in range(len(marks) - 1):
        c = cells[marks[b]:marks[b + 1]]
        oid = c[:, 1].astype(np.int64) & 0xffffffff
        off = np.stack([((oid >> s) & 7) - 3 for s in (22, 25, 28)], axis=1) * ev.L
        assert not (oid >> 31).any()  # no softened cells here
        i = slice(ev.t_starts[b], ev.t_starts[b] + ev.t_sizes[b])
        r = pos[i][:, None, :] - (cm[c[:, 0]] + off)[None, :, :]
        ir = 1.0 / np.sqrt((r ** 2).sum(axis=2))
        wi = w[i][:, None, :].astype(np.float64)
        np.add.at(d0, c[:, 0], -((wi * r).sum(axis=2) * ir ** 3).sum(axis=0))
        np.add.at(scale, c[:, 0], (np.linalg.norm(wi, axis=2) * ir ** 2).sum(axis=0))
    return d0, scale


@pytest.mark.parametrize("n,bucket,ng", [(40, 4, 0), (300, 2, 0), (1500, 16, 0), (6000, 1, 0),
                                         (20000, 16, 0), (0, 8, 20)])
def test_gpu_adjoint_transpose(device, n, bucket, ng):
    import torch
    w = (configs.zeldovich(ng=ng, bucket=bucket, active_frac=0.3) if ng
         else configs.plummer(n=n, bucket=bucket))
    ev = engine.Evaluation(w, precise=True, device=device)
    wt = np.random.default_rng(5).normal(size=(ev.n_targets, 3)).astype(np.float32)
    ev.adjoint(wt, ewald=False)
    torch.cuda.synchronize()
    got = ev.d_node_work[:, 0].cpu().numpy()
    d0, scale = _cell_sums(ev, wt, ev.node64()[:, 0:3])
    off = np.abs(got - d0)
    used = scale > 0
    print(f"n {ev.n} bucket {bucket}: {ev.lists['cell_marks'][-1]} entries, {used.sum()} of "
          f"{ev.tree['n_nodes']} nodes used, max off {(off[used] / scale[used]).max(initial=0):.1e}",
          flush=True)
    assert (off <= 1e-5 * scale).all()
