"""Particle ranges of a local-tree-walk request around the claims of its
wavefronts (8 particles): a few particles from different first ones, so that
runs of one nodeId begin before a claim, in its last particle, or span several.
Particles of runs that lie inside the range get the whole request's results
bit for bit (a run's walk and lanes depend on the run only); those of a run
that the range cuts get the same terms over fewer targets per wavefront: at
most 2^-23 of the largest component per rounding, a few roundings in the FP64
sums' FP32 tiles, so 2e-6 (dtGrav, a max, bit for bit). The others stay
zero."""
import numpy as np
import pytest

from changa_amd import configs, engine, ltw

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[1, 5, 40])
def case(request, device):
    import torch
    ev = engine.Evaluation(configs.plummer(n=3000, bucket=request.param), precise=False,
                           device=device, cell_records=False)
    torch.cuda.synchronize()
    nodes, parts = ltw.serialize_evaluation(ev)
    theta = float(ev.w["theta"])
    return nodes, parts, theta, ltw.walk(nodes, parts, theta)


@pytest.mark.parametrize("first", [0, 1, 7, 8, 1003, 2983])
@pytest.mark.parametrize("count", [1, 7, 8, 9, 16, 17])
def test_ltw_claims(case, first, count):
    nodes, parts, theta, full = case
    last = first + count - 1
    sub = ltw.walk(nodes, parts, theta, first=first, last=last)
    nid = parts["nodeId"]
    inside = np.zeros(len(parts), dtype=bool)
    inside[first:last + 1] = True
    cut = np.isin(nid, nid[~inside])
    whole, part = inside & ~cut, inside & cut
    np.testing.assert_array_equal(sub[whole], full[whole])
    scale = np.abs(full[:, :4]).max(axis=0)
    if part.any():
        d = np.abs(sub[part, :4].astype(np.float64) - full[part, :4]) / scale
        assert d.max() <= 2e-6
    np.testing.assert_array_equal(sub[inside, 4], full[inside, 4])
    assert not sub[~inside].any()
