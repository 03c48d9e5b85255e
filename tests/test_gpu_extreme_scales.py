"""Scale bytes from one end of E8M0 to the other inside one weight tile: 253 and 254 (weights up to 6 * 2^127, which do
not fit bf16) beside 0 and 1 (2^-127 and 2^-126).

Every other block of 32 codes meets activations of about 2^122 under small scales, the ones between activations of about
2^-126 under large ones, so both add sums of ordinary size to every result and each must come out at its own scale.
Against the oracle at the parity bar, each kind of weight row held to its own magnitude; decode through the fused block
(1 to 8 rows, up to 8 of one expert, more than are staged at once), prefill in both of its tile configurations (the wide
one from 2731 rows)."""
import numpy as np
import pytest
import torch

from oracle import experts as ox, mxfp4 as oq, routing as orr
from helpers import assert_bf16_close, bf16_np, pool_np, to_dev_bf16

pytestmark = pytest.mark.gpu

H, I, E, K = 512, 512, 8, 3


def _pick(rng, values, shape):
    return torch.from_numpy(rng.choice(np.array(values, np.uint8), shape)).cuda()


def _block(rng, seed):
    from mimo_stream import MoEBlock, Router, pools
    bank = pools.random_bank(E, seed=seed, hidden=H, inter=I)
    r = Router(H, E, K)                     # zero weights: the bias alone routes every row to experts 0, 1 and 2
    r.weight.zero_()
    r.e_score_correction_bias.copy_(torch.tensor([3.0, 2.0, 1.0] + [0.0] * (E - 3)))
    return MoEBlock(r, bank), bank


def _gate_up(rng, bank):
    """Expert 0: every row mixed (gate small and up large, or the other way); expert 2: row 7 alone; expert 1: none."""
    nb = H // 32 // 2
    for p in ("gate_s", "up_s"):
        s = bank[p]
        s[:, :, 0::2] = _pick(rng, [4, 5, 6], (E, I, nb))
        s[:, :, 1::2] = _pick(rng, [247, 248, 250], (E, I, nb))
    for e, rows in ((0, slice(0, I, 2)), (0, slice(1, I, 2)), (2, slice(7, 8))):
        small, large = ("gate_s", "up_s") if rows.start != 1 else ("up_s", "gate_s")
        n = bank[small][e, rows].shape[0]
        bank[small][e, rows, 0::2] = _pick(rng, [0, 1], (n, nb))
        bank[large][e, rows, 1::2] = _pick(rng, [253, 254], (n, nb))


def _down(rng, bank):
    """Down rows mixed likewise: h is about 2^122 in its even blocks and 2^-123 in its odd ones (through the up scales);
    few and small codes in the odd blocks keep their sums near the even ones'."""
    nb = I // 32 // 2
    up = bank["up_s"].view(E, nb, 2, 32, H // 32)
    up[:, :, 0] = _pick(rng, [245], (E, nb, 32, H // 32))
    up[:, :, 1] = _pick(rng, [0, 1, 2], (E, nb, 32, H // 32))
    bank["down_w"].view(E, H, nb, 2, 4)[:, :, :, 1] &= 0x00000009    # the first of every 8 codes, 0 or +-0.5
    s = bank["down_s"]
    s[:, :, 0::2] = _pick(rng, [4, 5, 6], (E, H, nb))
    s[:, :, 1::2] = _pick(rng, [247, 248, 250], (E, H, nb))
    for e, rows in ((0, slice(0, H, 2)), (2, slice(7, 8))):
        n = s[e, rows].shape[0]
        s[e, rows, 0::2] = _pick(rng, [0, 1], (n, nb))
        s[e, rows, 1::2] = _pick(rng, [253, 254], (n, nb))
    s[0, 10, 1] = 255                       # NaN beside 253 and 254: this output alone


def _rows(rng, case, T):
    x = rng.standard_normal((T, H)).astype(np.float32)
    if case == "gate_up":
        x = x * np.where(np.arange(H) // 32 % 2, 2.0 ** -126, 2.0 ** 122).astype(np.float32)
    return oq.round_bf16(x)


def _check(case, got, ref, what):
    """Columns apart by the magnitude of their reference: each within the bar for its own scale."""
    nan = np.isnan(ref)
    np.testing.assert_array_equal(np.isnan(got), nan)
    assert nan.any() == (case == "down") and np.isfinite(ref[~nan]).all()
    cols = ~nan.any(0)
    size = np.abs(ref[:, cols]).max(0)
    order = np.argsort(size)
    for part in np.array_split(order, 8):
        assert_bf16_close(got[:, cols][:, part], ref[:, cols][:, part], what=what)


@pytest.mark.parametrize("case", ["gate_up", "down"])
@pytest.mark.parametrize("T", [1, 2, 3, 5, 8, 20, 100, 150, 2750])
def test_block(rng, case, T):
    blk, bank = _block(rng, seed=71)
    {"gate_up": _gate_up, "down": _down}[case](rng, bank)
    pool = pool_np(bank)
    x = _rows(rng, case, T)
    y, inds, w = blk(to_dev_bf16(x), return_routes=True)
    gi, gw = inds.cpu().numpy(), w.cpu().numpy()
    assert sorted(set(gi.ravel())) == [0, 1, 2]
    with np.errstate(over="ignore", invalid="ignore"):
        if T == 1:
            ref = ox.gather_m1(x[0], pool, gi[0], gw[0])[None]
        elif T <= 8:
            ref = ox.moe_experts(x, pool, *orr.group_routes(gi, gw, R=8), K, R=8)[0]
        else:
            ref = ox.moe_prefill(x, pool, gi, gw)
    _check(case, bf16_np(y), ref, f"{case} {T} rows")


@pytest.mark.parametrize("M", [2, 8])
def test_intermediates(rng, M):
    """h column by column: rows of the tile without such a scale are not touched by the ones that have it."""
    from mimo_stream import kernels
    _, bank = _block(rng, seed=72)
    _gate_up(rng, bank)
    x = _rows(rng, "gate_up", M)
    u = orr.group_routes(np.tile(np.arange(K, dtype=np.int32), (M, 1)), rng.random((M, K)).astype(np.float32), R=8)
    _, h, _ = kernels.moe_experts(to_dev_bf16(x), bank, *u[:4], R=8, gather_idx=u[4], return_intermediates=True)
    oh = ox.moe_experts(x, pool_np(bank), *u, K, R=8)[1]
    got = bf16_np(h)[:, :M]
    for e in range(K):
        assert np.isfinite(oh[e]).all()
        assert_bf16_close(got[e], oh[e, :M], what=f"h of expert {e}")
    assert_bf16_close(got[2, :, 7], oh[2, :M, 7], what="the one mixed row")
    assert_bf16_close(got[2, :, 8:16], oh[2, :M, 8:16], what="its tile")
