"""The prefill chunk's routing launches at the sizes where their shape changes: logits as partial sums (up to 640
tokens) or whole, the dispatch counting in its own blocks (up to 16384 routes) or after a histogram launch."""
import numpy as np
import pytest
import torch

from oracle import routing as orr
from helpers import rand_bf16, to_dev_bf16, zipf_routes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [9, 31, 33, 639, 640, 641])
@pytest.mark.parametrize("H,E,k", [(256, 8, 2), (768, 70, 3), (1024, 300, 5)])
def test_block_routes_are_the_routers(rng, T, H, E, k):
    """The block's routes and weights equal the router entry point's (whole logits) bit for bit."""
    from mimo_stream import MoEBlock, Router, pools
    r = Router(H, E, k)
    r.weight.copy_(to_dev_bf16(rand_bf16(rng, (E, H), 0.05)))
    r.e_score_correction_bias.copy_(torch.from_numpy((rng.standard_normal(E) * 0.01).astype(np.float32)))
    blk = MoEBlock(r, pools.random_bank(E, seed=3, hidden=H, inter=128))
    x = to_dev_bf16(rand_bf16(rng, (T, H)))
    _, inds, w = blk(x, return_routes=True)
    logits, ri, rw = r.logits_and_routes(x)
    assert torch.equal(inds, ri) and torch.equal(w, rw)
    oi, ow = orr.select_topk(logits.cpu().numpy(), r.e_score_correction_bias.cpu().numpy(), k)
    np.testing.assert_array_equal(inds.cpu().numpy(), oi)
    np.testing.assert_array_equal(w.cpu().numpy(), ow)


@pytest.mark.parametrize("T,k,S", [(1, 1, 1), (128, 8, 256), (129, 8, 256), (1023, 8, 1024), (1024, 8, 256),
                                   (1025, 8, 256), (2049, 4, 7),
                                   (2048, 8, 256), (2049, 8, 256)])
def test_dispatch_against_oracle(rng, T, k, S):
    from mimo_stream import prefill_dispatch
    inds = zipf_routes(rng, T, max(S, k), k) % S
    got = prefill_dispatch(torch.from_numpy(inds.astype(np.int32)).cuda(), S)
    want = orr.prefill_dispatch(inds, S)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g.cpu().numpy(), np.asarray(w))
