"""The longest k-space table the Ewald kernel takes (it is staged in LDS beside
the kernel's own 24,704 bytes: 4,348 entries in 160 KB), with the most and with
few candidate lattice vectors, and longer ones, which are refused on the host
before any launch.

The difference between a run with the table and one without is compared with
the FP64 sum over the table. Bar per particle, as for the shorter tables: a
term is at most about 30 roundings off (its phase h.u, |h| up to 14
revolutions in FP32, 2 pi 14 6e-8 = 5e-6 on top), so 8e-6 of |hC| + |hS|,
times |k| for the acceleration; the results are FP32 sums that both runs round
once more, 1e-7 of their magnitude each."""
import numpy as np
import pytest

from changa_amd import configs, engine

pytestmark = pytest.mark.gpu


def _run(ev, table, device):
    import torch
    ev.d_ewt = torch.from_numpy(table if len(table) else np.zeros((1, 5), np.float32)).to(device)
    ev.ewald_ro.nEwhLoop = len(table)
    ev.zero()
    ev.run_ewald(host_record=True)
    torch.cuda.synchronize()
    return ev.d_vars.cpu().numpy().astype(np.float64)


def _table(ev, n):
    """The usual table and n - len more entries off the cube |h_i| <= 3."""
    g = np.arange(-8, 9)
    h = np.stack(np.meshgrid(g, g, g, indexing="ij"), axis=-1).reshape(-1, 3)
    h = h[np.abs(h).max(axis=1) > 3][:n - len(ev.ewt64)]
    c = 1e-5 * np.random.default_rng(9).normal(size=(len(h), 2))
    t = np.concatenate([ev.ewt64, np.concatenate([2 * np.pi * h / ev.L, c], axis=1)])
    assert len(t) == n
    return np.ascontiguousarray(t.astype(np.float32))


@pytest.mark.parametrize("reps", [3, 1])
def test_gpu_ewald_longest_table(device, reps):
    ev = engine.Evaluation(configs.zeldovich(ng=10, rms=0.08), precise=True, device=device)
    ev.ewald_ro.nEwReps = reps  # 343 or 27 candidate lattice vectors
    table = _table(ev, 4347)
    got, none = _run(ev, table, device), _run(ev, table[:0], device)
    t = table.astype(np.float64)
    k = 2 * np.pi * np.rint(t[:, 0:3] * ev.L / (2 * np.pi)) / ev.L
    ph = (ev.pos - ev.root_cm64) @ k.T
    pot = np.cos(ph) @ t[:, 3] + np.sin(ph) @ t[:, 4]
    acc = (t[:, 3] * np.sin(ph) - t[:, 4] * np.cos(ph)) @ k
    w = np.abs(t[:, 3]) + np.abs(t[:, 4])
    bar_p = 8e-6 * w.sum() + 1e-7 * (np.abs(got[:, 3]) + np.abs(none[:, 3]))
    bar_a = (8e-6 * (w * np.linalg.norm(k, axis=1)).sum()
             + 1e-7 * (np.abs(got[:, 0:3]) + np.abs(none[:, 0:3])))
    ep = np.abs(got[:, 3] - none[:, 3] - pot)
    ea = np.abs(got[:, 0:3] - none[:, 0:3] - acc)
    print(f"{reps} shells: pot {np.max(ep / bar_p):.2f}, acc {np.max(ea / bar_a):.2f} of the bar",
          flush=True)
    assert (ep <= bar_p).all() and (ea <= bar_a).all()


def test_gpu_ewald_table_too_long(device):
    ev = engine.Evaluation(configs.zeldovich(ng=10, rms=0.08), precise=True, device=device)
    table = _table(ev, 146)
    before = _run(ev, table, device)
    for n in (4349, 1 << 20):
        with pytest.raises(RuntimeError, match="nEwhLoop too large"):
            _run(ev, np.zeros((n, 5), dtype=np.float32), device)
    np.testing.assert_array_equal(_run(ev, table, device), before)
