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


@pytest.mark.parametrize("E,k", [(1024, 1), (300, 5)])
def test_short_chunk_in_the_longest_chunks_workspace(rng, E, k):
    """One workspace, sized for 650 tokens and filled with NaN bytes, serves shorter chunks on both sides of the 640
    tokens at which the logits' form changes.  The logits share the room of h and Y: the outputs are those of the
    router and the expert entry points called apart."""
    from mimo_stream import Router, _lib, pools
    H, I = 256, 128
    r = Router(H, E, k)
    r.weight.copy_(to_dev_bf16(rand_bf16(rng, (E, H), 0.05)))
    weights = pools.random_bank(E, seed=3, hidden=H, inter=I)   # outlives the calls
    bank = pools.bank_struct(weights)
    lib = _lib.load()
    n = lib.mimo_moe_prefill_block_workspace_size(650, E, k, E, H, I)
    ws = torch.full((n,), 255, dtype=torch.uint8, device="cuda")
    for T in (640, 641, 9, 650):
        x = to_dev_bf16(rand_bf16(rng, (T, H)))
        y, y2 = torch.empty_like(x), torch.empty_like(x)
        stream = _lib.stream_ptr(x.device)
        _lib.call("mimo_moe_prefill_block", _lib.ptr(x), T, _lib.ptr(r.weight), _lib.ptr(r.e_score_correction_bias), None,
                  E, k, bank, _lib.ptr(y), None, None, None, _lib.ptr(ws), n, stream)
        inds, w = r(x)
        n2 = lib.mimo_moe_prefill_workspace_size(T, k, E, H, I)
        ws2 = torch.empty(n2, dtype=torch.uint8, device="cuda")
        _lib.call("mimo_moe_prefill", _lib.ptr(x), T, _lib.ptr(inds), _lib.ptr(w), k, bank, _lib.ptr(y2), None,
                  _lib.ptr(ws2), n2, stream)
        assert torch.isfinite(y).all() and torch.equal(y, y2), T


@pytest.mark.parametrize("T,k,S", [(2048, 8, 1), (2048, 8, 2), (2047, 8, 3), (2048, 8, 512), (2048, 8, 513), (2048, 8, 1024),
                                   (1, 1, 1024), (2049, 8, 2)])
@pytest.mark.parametrize("slots", ["one", "last two"])
def test_dispatch_of_crowded_slots(T, k, S, slots):
    """Every route on one slot or two: the counters' largest counts, at the slot counts where their copies change."""
    from mimo_stream import prefill_dispatch
    inds = np.full((T, k), S - 1, np.int32)
    if slots == "last two":
        inds[::3] = max(S - 2, 0)
    got = prefill_dispatch(torch.from_numpy(inds).cuda(), S)
    want = orr.prefill_dispatch(inds, S)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g.cpu().numpy(), np.asarray(w))
