"""The top-k search starts from the smallest of the lanes' largest keys: expert counts around a wave's 64 lanes, where
that bound sits on the last candidates, and rows whose keys are all equal, all NaN or one far above the rest, must
select what the oracle selects, bit for bit."""
import numpy as np
import pytest
import torch

from oracle import routing as orr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,k", [(1, 1), (8, 8), (16, 16), (63, 8), (64, 8), (65, 16), (128, 8), (200, 8), (256, 8),
                                 (257, 16), (1000, 16)])
def test_selection_from_the_keys_own_range(rng, E, k):
    from mimo_stream import select_from_logits
    rows = (rng.standard_normal((10, E)) * 2).astype(np.float32)
    rows[1] = 0.25                                             # every key equal
    rows[2, E - 1] = 90.0                                      # one key far above the rest
    rows[3] = -200.0                                           # every sigmoid 0
    rows[4, ::2] = np.nan
    rows[5] = np.nan
    rows[6] = np.sort(rows[6])                                 # the last lanes' keys largest
    rows[7] = np.sort(rows[7])[::-1]
    rows[8, :] = np.where(np.arange(E) % 64 < k // 2, 3.0, 1.0)   # the k largest spread over few lanes
    rows[9, ::3] = -np.inf
    bias = np.zeros(E, np.float32)
    if E > 3:
        bias[3] = -2.0                                         # a negative key
    inds, w = select_from_logits(torch.from_numpy(rows).cuda(), torch.from_numpy(bias).cuda(), k)
    oi, ow = orr.select_topk(rows, bias, k)
    np.testing.assert_array_equal(inds.cpu().numpy(), oi)
    np.testing.assert_array_equal(w.cpu().numpy(), ow)
