"""Scratch of a local-tree-walk request: a full slice (16,384 cells, 8,192
particle runs) per 64 particles, an eighth of one per wavefront's claim, and a
second launch for the runs whose lists do not fit there.

Runs of lists below, at and beyond an eighth of a slice are compared bit for
bit with a request of so many copies of the same particles (targets on the
same tree) that every wavefront has a full slice: a run's walk and lanes depend
on the run only."""
import numpy as np
import pytest

from changa_amd import configs, engine, gpu, ltw

pytestmark = pytest.mark.gpu

SLICE = 16384 * 8 + 8192 * 12
CASES = {
    # particle runs beyond 1,024 in about half the buckets
    "runs": lambda: (dict(configs.plummer(n=3000, bucket=2), theta=0.3), 0),
    # cells (2,048) and runs beyond in some or all
    "cells": lambda: (dict(configs.zeldovich(ng=8, rms=0.05, bucket=2), theta=0.24), 3),
    "all": lambda: (dict(configs.zeldovich(ng=8, rms=0.05, bucket=2), theta=0.2), 3),
    "softened": lambda: (dict(configs.plummer(n=3000, bucket=2, eps=0.5), theta=0.3), 0),
}


@pytest.mark.parametrize("case", list(CASES))
def test_ltw_lists_beyond_a_share(device, case):
    import torch
    w, R = CASES[case]()
    ev = engine.Evaluation(dict(w, n_replicas=R), precise=False, device=device,
                           cell_records=False)
    torch.cuda.synchronize()
    cells, runs = np.diff(ev.lists["cell_marks"]), np.diff(ev.lists["part_marks"])
    over = (cells > 2048) | (runs > 1024)
    print(f"ltw scratch {case}: {ev.n} particles, {over.sum()} of {len(over)} buckets beyond a "
          f"share (cells {cells.max()}, runs {runs.max()})", flush=True)
    assert over.any()
    nodes, parts = ltw.serialize_evaluation(ev)
    period = float(w["L"]) if w["periodic"] else 0.0
    v = ltw.walk(nodes, parts, float(w["theta"]), R, period)
    # 2^19 targets: more 64s than the card holds wavefronts
    k = -(-(1 << 19) // len(parts))
    many = ltw.walk(nodes, np.tile(parts, k), float(w["theta"]), R, period)
    for c in (0, k // 2, k - 1):
        np.testing.assert_array_equal(many[c * len(parts):(c + 1) * len(parts)], v)
    assert (np.abs(v[:, 0:3]).sum(axis=1) > 0).all()


@pytest.mark.parametrize("n", [1, 64, 65, 4096, 32768])
def test_ltw_scratch_of_a_request(device, n):
    """Device memory a request leaves in its stream's pool: its slices, 4
    bytes a particle and the counters, a quarter more as the pool grows, in
    2 MiB steps (two of them allowed)."""
    import torch
    ev = engine.Evaluation(configs.plummer(n=32768), precise=False, device=device,
                           cell_records=False)
    nodes, parts = ltw.serialize_evaluation(ev)
    L = gpu.lib_ltw()
    walk = ltw.LocalWalk(nodes, parts, 0.7, last=n - 1, device=device)
    warm = ltw.LocalWalk(nodes, parts, 0.7, last=0, device=device)
    warm.run()
    warm.results()
    torch.cuda.synchronize()
    L.changaGpuReleasePools()
    before = torch.cuda.mem_get_info(device)[0]
    walk.run()
    walk.results()
    took = before - torch.cuda.mem_get_info(device)[0]
    bound = 1.25 * (-(-n // 64) * SLICE + 4 * n + 4096) + (4 << 20)
    print(f"ltw request of {n}: {took} bytes, bound {bound:.0f}", flush=True)
    assert took <= bound
