"""The k-space sum of the Ewald kernel over h-tables of several kinds: the
usual table (h and -h with the same hC and opposite hS, summed as a half),
tables that are not of that kind (one of each pair, one sign changed, a
single entry, random weights), entries beyond the product form's cube, and an
empty table. The difference between a run with the table and one without is
compared with the FP64 sum over the table.

Bar per particle: a term is at most about 30 roundings off (the powers of
e^(2 pi i u) are products of up to nine factors), 2e-6 of |hC| + |hS|, times
|k| for the acceleration; the results are FP32 sums that both runs round once
more, 1e-7 of their magnitude each."""
import numpy as np
import pytest

from changa_amd import configs, engine

pytestmark = pytest.mark.gpu


def _table(kind, base):
    t = base.astype(np.float64).copy()
    rng = np.random.default_rng(3)
    if kind == "half":
        h = np.rint(t[:, 0:3] / (2 * np.pi))
        t = t[(h[:, 0] > 0) | ((h[:, 0] == 0) & ((h[:, 1] > 0) | ((h[:, 1] == 0) & (h[:, 2] > 0))))]
    elif kind == "sign":
        t[7, 4] = -t[7, 4] + 1e-4
    elif kind == "single":
        t = t[5:6]
    elif kind == "random":
        t[:, 3:5] = 1e-3 * rng.normal(size=(len(t), 2))
    elif kind == "outside":
        t = np.concatenate([t, [[2 * np.pi * 4, 0.0, -2 * np.pi, 2e-4, 3e-4],
                                [0.0, 2 * np.pi * 5, 0.0, -1e-4, 1e-4]]])
    return np.ascontiguousarray(t.astype(np.float32))


@pytest.mark.parametrize("kind", ["usual", "half", "sign", "single", "random", "outside"])
def test_gpu_ewald_tables(device, kind):
    import torch
    ev = engine.Evaluation(configs.zeldovich(ng=10, rms=0.08), precise=True, device=device)
    base = ev.ewt64
    out = []
    table = _table(kind, base)
    for t in (table, np.zeros((0, 5), dtype=np.float32)):
        ev.d_ewt = torch.from_numpy(t.copy() if len(t) else np.zeros((1, 5), np.float32)).to(device)
        ev.ewald_ro.nEwhLoop = len(t)
        ev.zero()
        ev.run_ewald(host_record=True)
        torch.cuda.synchronize()
        out.append(ev.d_vars.cpu().numpy().astype(np.float64))
    got = out[0] - out[1]
    t = table.astype(np.float64)
    # k as the kernel takes it on the cube: 2 pi h / L
    k = 2 * np.pi * np.rint(t[:, 0:3] * ev.L / (2 * np.pi)) / ev.L
    ph = (ev.pos - ev.root_cm64) @ k.T
    pot = np.cos(ph) @ t[:, 3] + np.sin(ph) @ t[:, 4]
    acc = (t[:, 3] * np.sin(ph) - t[:, 4] * np.cos(ph)) @ k
    w = np.abs(t[:, 3]) + np.abs(t[:, 4])
    bar_p = 2e-6 * w.sum() + 1e-7 * (np.abs(out[0][:, 3]) + np.abs(out[1][:, 3]))
    bar_a = (2e-6 * (w * np.linalg.norm(k, axis=1)).sum()
             + 1e-7 * (np.abs(out[0][:, 0:3]) + np.abs(out[1][:, 0:3])))
    ep, ea = np.abs(got[:, 3] - pot), np.abs(got[:, 0:3] - acc)
    print(f"{kind}: {len(t)} entries, pot {np.max(ep / bar_p):.2f}, acc {np.max(ea / bar_a):.2f} "
          "of the bar", flush=True)
    assert (ep <= bar_p).all() and (ea <= bar_a).all()
