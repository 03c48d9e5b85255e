"""The prefill GEMMs' streaming configuration (few routes per slot) cuts popular slots into tiles of up to 64 routes: slots
at and beside each of its chunk counts and tile ends, at the average on both sides of the line to the other
configuration (which needs 256 blocks of 128 routes times 128 outputs as well: only I = 5376 passes the line), against
the oracle."""
import numpy as np
import pytest
import torch

from oracle import experts as ox
from helpers import assert_bf16_close, bf16_np, pool_np, rand_bf16, to_dev_bf16

pytestmark = pytest.mark.gpu

EDGES = [32, 33, 47, 48, 49, 63, 64, 65, 97, 128, 129]


@pytest.mark.parametrize("slots,last", [(40, 0), (33, 37), (33, 38)], ids=["streaming", "at_the_line", "past_it"])
@pytest.mark.parametrize("H,I", [(256, 128), (512, 640), (1024, 384), (256, 5376)])
def test_streaming_tile_edges(rng, H, I, slots, last):
    from mimo_stream import MoEBlock, Router, pools
    counts = EDGES + [0] * (slots - len(EDGES) - 1) + [last]
    assert (sum(counts) <= 24 * slots) == (last != 38)
    bank = pools.random_bank(slots, seed=H + I, hidden=H, inter=I)
    blk = MoEBlock(Router(H, slots, 1), bank)
    inds = np.repeat(np.arange(slots), counts)[:, None].astype(np.int32)
    rng.shuffle(inds)
    x = rand_bf16(rng, (len(inds), H), 1.0)
    w = (0.5 + rng.random((len(inds), 1))).astype(np.float32)
    y = blk._moe_prefill(to_dev_bf16(x), torch.from_numpy(inds).cuda(), torch.from_numpy(w).cuda())
    assert_bf16_close(bf16_np(y), ox.moe_prefill(x, pool_np(bank), inds, w), what=f"H={H} I={I} slots={slots}")
