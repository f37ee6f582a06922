"""Several buckets' walks in one wavefront (changaBuildListsCount / Fill): a
small tree's buckets repeated up to and past the lines at which a wavefront
takes 2, 4, ... 64 of them, with a last group that is not full; every copy's
lists are the host walk's entry for entry, with the copy's own number."""
import numpy as np
import pytest

from changa_amd import configs, engine, host

pytestmark = pytest.mark.gpu

CASES = {
    "softened": lambda: configs.plummer(n=400, eps=0.3),
    "periodic": lambda: configs.zeldovich(ng=8, rms=0.1),
}


@pytest.fixture(scope="module", params=list(CASES))
def case(request, device):
    ev = engine.Evaluation(CASES[request.param](), precise=True, device=device, lists="gpu")
    geo = np.ascontiguousarray(ev.node64()[:, :12])
    w = ev.w
    h = host.walk(ev.tree, geo, w["theta"], w["n_replicas"], ev.L if w["periodic"] else 1.0)
    return ev, h


@pytest.mark.parametrize("nb", [1, 3799, 3800, 7601, 15203, 30405, 60807, 121605])
def test_gpu_walk_groups(case, nb, monkeypatch):
    ev, h = case
    nb0 = len(ev.t_keep)
    keep = np.resize(np.arange(nb0), nb)
    for k, v in dict(t_keep=keep, t_sizes=np.resize(ev.t_sizes, nb), t_lists=None, counts=None,
                     d_cells=None, d_plist=None, d_cmarks=None, d_pmarks=None, d_soft_start=None,
                     d_bucket_node=None).items():
        monkeypatch.setattr(ev, k, v)
    ev._gpu_lists()
    cm, pm = np.asarray(h["cell_marks"]), np.asarray(h["part_marks"])
    ncell, nrun = np.diff(cm)[keep], np.diff(pm)[keep]
    gm = ev.t_lists["cell_marks"]
    np.testing.assert_array_equal(np.diff(gm), ncell)
    np.testing.assert_array_equal(np.diff(ev.t_lists["part_marks"]), nrun)
    np.testing.assert_array_equal(ev.t_lists["soft_start"] - gm[:-1],
                                  (np.asarray(h["soft_start"]) - cm[:-1])[keep])

    def copies(entries, marks, n):
        """Every copy's entries, in order."""
        at = np.repeat(marks[:-1][keep] - np.concatenate([[0], np.cumsum(n)[:-1]]), n)
        return entries[at + np.arange(n.sum())]
    hc = copies(h["cells"].reshape(-1, 2), cm, ncell)
    hp = copies(h["parts"].reshape(-1, 3), pm, nrun)
    gc = ev.d_cells.cpu().numpy()[:len(hc)]
    field = (1 << 22) - 1  # the bucket number of an encoded offset
    np.testing.assert_array_equal(gc[:, 0], hc[:, 0])
    np.testing.assert_array_equal(gc[:, 1] & ~field, hc[:, 1] & ~field)
    np.testing.assert_array_equal(gc[:, 1] & field, np.repeat(np.arange(nb), ncell))
    np.testing.assert_array_equal(ev.d_plist.cpu().numpy()[:len(hp)], hp)
