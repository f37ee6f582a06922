"""Building lists takes no stream from the framework's pool (32 of them, given
out in turn): a caller's streams stay the ones that the build does not touch,
and on the hardware queues that they had."""
import numpy as np
import pytest

from changa_amd import configs, engine

pytestmark = pytest.mark.gpu


def test_list_build_takes_no_pool_stream(device):
    import torch
    ev = engine.Evaluation(configs.plummer(n=2000), precise=True, device=device, lists="gpu")
    cells = ev.d_cells.cpu().numpy()
    turn = [torch.cuda.Stream(device).cuda_stream for _ in range(64)]
    size = len(set(turn))
    assert turn[:size] == turn[size:2 * size]
    for _ in range(3):
        before = turn.index(torch.cuda.Stream(device).cuda_stream)
        ev.build_lists()
        after = turn.index(torch.cuda.Stream(device).cuda_stream)
        assert after == (before + 1) % size
    torch.cuda.synchronize()
    np.testing.assert_array_equal(ev.d_cells.cpu().numpy(), cells)
