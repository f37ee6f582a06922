"""The adjoint's target side on cell records and on wire moments: records,
none, and records that are not line-aligned (taken as none) stage the same
FP32 values, so each target's tidal terms are the same bits. What differs from
run to run is the order of the FP64 atomic sums over cells and source
particles: bar 1e-12 of the largest component (a few thousand roundings of
1.1e-16, most of them of terms far below it)."""
import numpy as np
import pytest

from changa_amd import configs, engine

pytestmark = pytest.mark.gpu

CASES = {
    "compact": (lambda: configs.plummer(n=4000), True),
    "per_particle": (lambda: configs.plummer(n=3000), False),
    "softened": (lambda: configs.plummer(n=3000, eps=0.4), True),
    "softened_per_particle": (lambda: configs.plummer(n=2000, eps=0.4), False),
    "periodic_rung": (lambda: configs.zeldovich(ng=14, rms=0.1, active_frac=0.3), True),
}


@pytest.mark.parametrize("case", list(CASES))
def test_gpu_adjoint_cell_sources(device, case, monkeypatch):
    import torch
    make, compact = CASES[case]
    ev = engine.Evaluation(make(), precise=True, pp_compact=compact, device=device)
    assert ev.d_cellrec is not None
    w = np.random.default_rng(8).normal(size=(ev.n_targets, 3)).astype(np.float32)
    launch, out = ev._launch, {}
    for name, shift in (("records", 0), ("wire", None), ("unaligned", 64)):
        def with_cells(pc, shift=shift):
            a = launch(pc)
            if pc:
                a.cellRecords = None if shift is None else a.cellRecords + shift
            return a
        monkeypatch.setattr(ev, "_launch", with_cells)
        out[name] = ev.adjoint(w).cpu().numpy()
        torch.cuda.synchronize()
    scale = np.abs(out["records"]).max(axis=0)
    for name in ("wire", "unaligned"):
        d = (np.abs(out[name] - out["records"]) / scale).max()
        print(f"{case} {name}: {d:.1e} of the largest component", flush=True)
        assert d <= 1e-12
