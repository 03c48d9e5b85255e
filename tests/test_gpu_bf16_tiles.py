"""The expert products on bf16 MFMA at the edges of their tilings, against the oracle.

Prefill: routes per slot at and beside every chunk count a row tile can have (1 to 128 routes, then a second tile), in
the streaming configuration (few routes per slot, or few blocks) and in the wide one, at reduction lengths of 1 to 33
K-steps that do and do not fill a round of the K loop, with scale rows that can and cannot be copied 16 bytes at a time.  Decode: rows per expert
at and beside the number staged at once.  Both: E8M0 bytes 253 and 254, whose weights (up to 6 * 2^127) do not fit
bf16.  The bar is the parity tests' own."""
import numpy as np
import pytest
import torch

from oracle import experts as ox, routing as orr
from helpers import assert_bf16_close, bf16_np, pool_np, rand_bf16, to_dev_bf16

pytestmark = pytest.mark.gpu


def _block(H, I, S, seed, patch=None):
    from mimo_stream import MoEBlock, Router, pools
    bank = pools.random_bank(S, seed=seed, hidden=H, inter=I)
    if patch:
        patch(bank)
    return MoEBlock(Router(H, S, 1), bank), bank


def _prefill(rng, blk, bank, counts, scale=1.0):
    H = bank["gate_w"].shape[2] * 8
    inds = np.repeat(np.arange(len(counts)), counts)[:, None].astype(np.int32)
    rng.shuffle(inds)
    x = rand_bf16(rng, (len(inds), H), scale)
    w = (0.5 + rng.random((len(inds), 1))).astype(np.float32)
    y = blk._moe_prefill(to_dev_bf16(x), torch.from_numpy(inds).cuda(), torch.from_numpy(w).cuda())
    with np.errstate(over="ignore", invalid="ignore"):
        return bf16_np(y), ox.moe_prefill(x, pool_np(bank), inds, w)


FEW = [1, 15, 16, 17, 31, 32, 33, 0, 3, 2, 1, 5]            # at most 18 routes per slot on average
MANY = [1, 32, 33, 48, 64, 65, 96, 97, 128, 129, 257, 0]


@pytest.mark.parametrize("counts", [FEW, MANY], ids=["few", "many"])
@pytest.mark.parametrize("H,I", [(256, 128), (512, 640), (768, 384), (1024, 1152), (4096, 512)])
def test_prefill_tile_edges(rng, H, I, counts):
    blk, bank = _block(H, I, len(counts), seed=H + I)
    y, oy = _prefill(rng, blk, bank, counts)
    assert_bf16_close(y, oy, what=f"H={H} I={I}")


def test_prefill_scales_of_unaligned_pools(rng):
    """Scale pools at addresses that are a multiple of 4 bytes only (the 4-byte copies) give the aligned pools' bits."""
    H, I, S = 512, 512, 12
    blk, bank = _block(H, I, S, seed=9)
    moved = dict(bank)
    for p in ("gate", "up", "down"):
        t = bank[p + "_s"]
        buf = torch.empty(t.numel() + 4, dtype=torch.uint8, device="cuda")
        moved[p + "_s"] = buf[4:].view(t.shape)
        moved[p + "_s"].copy_(t)
    from mimo_stream import MoEBlock
    for counts in (FEW, MANY):
        state = rng.bit_generator.state
        y, _ = _prefill(rng, blk, bank, counts)
        rng.bit_generator.state = state
        y2, _ = _prefill(rng, MoEBlock(blk.router, moved), moved, counts)
        np.testing.assert_array_equal(y, y2)


def _many_blocks(I):
    """MANY and one more slot, crowded enough that the wide tiles are as many blocks as the chip has CUs (256 blocks of
    128 routes times 128 outputs of I); with fewer, or up to 24 routes a slot, the streaming configuration runs."""
    return MANY + [256 * 128 * 128 // I + 1 - sum(MANY)]


@pytest.mark.parametrize("H,I", [(256, 128), (512, 640), (768, 384), (1024, 1152), (256, 4224)])
def test_prefill_wide_tile_edges(rng, H, I):
    """The tile edges in the wide configuration, and its scales from pools whose rows cannot be copied 16 bytes at a
    time: the same bits."""
    from mimo_stream import MoEBlock
    counts = _many_blocks(I)
    blk, bank = _block(H, I, len(counts), seed=H + I)
    state = rng.bit_generator.state
    y, oy = _prefill(rng, blk, bank, counts)
    assert_bf16_close(y, oy, what=f"H={H} I={I}")
    moved = dict(bank)
    for p in ("gate_s", "up_s", "down_s"):
        moved[p] = torch.empty(bank[p].numel() + 4, dtype=torch.uint8, device="cuda")[4:].view(bank[p].shape)
        moved[p].copy_(bank[p])
    rng.bit_generator.state = state
    inds = np.repeat(np.arange(len(counts)), counts)[:, None].astype(np.int32)      # the same rows, routes and weights
    rng.shuffle(inds)
    x = rand_bf16(rng, (len(inds), H))
    w = (0.5 + rng.random((len(inds), 1))).astype(np.float32)
    y2 = MoEBlock(blk.router, moved)._moe_prefill(to_dev_bf16(x), torch.from_numpy(inds).cuda(), torch.from_numpy(w).cuda())
    np.testing.assert_array_equal(y, bf16_np(y2))


@pytest.mark.parametrize("M,same", [(3, 3), (4, 4), (5, 5), (8, 1), (8, 4), (8, 5), (8, 8)])
def test_decode_rows_per_expert(rng, M, same):
    """`same` of the M rows share their first expert; more than four rows of one expert take a second pass."""
    from mimo_stream import kernels, pools
    H, I, S, k = 1024, 512, 64, 4
    bank = pools.random_bank(S, seed=M + same, hidden=H, inter=I)
    inds = (1 + np.stack([rng.permutation(S - 1)[:k] for _ in range(M)])).astype(np.int32)
    inds[:same, 0] = 0
    w = rng.random((M, k)).astype(np.float32)
    x = rand_bf16(rng, (M, H))
    u = orr.group_routes(inds, w, R=8)
    y = kernels.moe_experts(to_dev_bf16(x), bank, *u[:4], R=8, gather_idx=u[4])
    oy, _, _ = ox.moe_experts(x, pool_np(bank), *u, k, R=8)
    assert_bf16_close(bf16_np(y), oy, what=f"{M} rows, {same} on one expert")


HUGE = {"gate253": ("gate_s", 253), "gate254": ("gate_s", 254), "up254": ("up_s", 254), "down253": ("down_s", 253)}


@pytest.mark.parametrize("case", list(HUGE))
def test_weights_past_the_bf16_range(rng, case):
    """One weight row of expert 1 with a scale byte of 253 or 254 in every block, rows small enough for finite sums:
    the products are the reference's (unit codes times activations, then the scale), not infinities."""
    from mimo_stream import kernels
    name, byte = HUGE[case]

    def patch(b):
        b[name][1, 7] = byte
    H, I, S = 512, 512, 12
    blk, bank = _block(H, I, S, seed=31, patch=patch)
    for counts in (FEW, MANY):
        y, oy = _prefill(rng, blk, bank, counts, scale=2.0 ** -24)
        assert np.isfinite(oy).all() and np.abs(oy).max() > 1e15
        assert_bf16_close(y, oy, what=f"prefill {case}")
    for M in (2, 8):
        inds = np.tile(np.array([[1, 2]], np.int32), (M, 1))
        w = rng.random((M, 2)).astype(np.float32)
        x = rand_bf16(rng, (M, H), 2.0 ** -24)
        x[1] = -x[0]                 # a gate of either sign: the SwiGLU of a huge negative one is 0
        u = orr.group_routes(inds, w, R=8)
        y = kernels.moe_experts(to_dev_bf16(x), bank, *u[:4], R=8, gather_idx=u[4])
        oy, _, _ = ox.moe_experts(x, pool_np(bank), *u, 2, R=8)
        assert np.isfinite(oy).all() and np.abs(oy).max() > 1e15
        assert_bf16_close(bf16_np(y), oy, what=f"decode {case} {M} rows")
