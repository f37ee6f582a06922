"""Several wavefronts per bucket: launches over the first m buckets of a tree,
m on both sides of each line of the wavefront rules (one, two or four per
bucket; lists shorter than the wavefronts included), through the per-bucket
kernels and the batched form, against the FP64 oracle on the same lists.
Targets of the other buckets stay zero.

Tolerance: a pair's FP32 evaluation is off by at most about 20 roundings
(1.2e-6 of the term), sums run in FP64 across tiles and wavefronts, and in a
Plummer sphere the terms' magnitudes add up to at most about ten times the net
force outside the very centre: 2e-5 for every particle, and a tenth of that in
the median."""
import numpy as np
import pytest

from changa_amd import configs, engine
from tests.helpers import oracle_forces, rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def case(device):
    ev = engine.Evaluation(configs.plummer(n=14000, bucket=2), precise=True, device=device)
    assert len(ev.t_sizes) > 8193
    return ev, oracle_forces(ev)


@pytest.mark.parametrize("m", [1, 3, 1024, 1025, 2048, 2049, 8192, 8193])
def test_gpu_list_teams(case, m, monkeypatch):
    import torch
    ev, (oa, op, _) = case
    launch = ev._launch

    def first(pc):
        a = launch(pc)
        a.numBuckets = m
        return a
    monkeypatch.setattr(ev, "_launch", first)

    def batched():
        ev.batch_plan(64, 256, 1, 1, targets_per_lane=3, cell_source=1)
        ev.step_batched()
    end = int(np.asarray(ev.t_sizes)[:m].sum())
    for name, run in (("step", ev.step), ("batched", batched)):
        run()
        torch.cuda.synchronize()
        acc, pot, _ = ev.results()
        ea, ep = rel_err(acc[:end], oa[:end]), rel_err(pot[:end], op[:end])
        print(f"{m} buckets {name}: acc max {ea.max():.1e} median {np.median(ea):.1e}, "
              f"pot max {ep.max():.1e}", flush=True)
        assert ea.max() < 2e-5 and np.median(ea) < 2e-6 and ep.max() < 2e-5, name
        assert not np.any(acc[end:]) and not np.any(pot[end:]), name
