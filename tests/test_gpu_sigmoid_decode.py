"""The decode epilogue's in-register bf16 sigmoid over every finite bf16 gate value.

Gate row n picks column n of the activation row (one code 1.0 with scale 1, every other code 0), every up row picks the
last column, which holds 1: g is the activation itself and u is 1, so h = bf16(g * sigmoid(g)), compared bit for bit
with the oracle's SwiGLU (the specified sigmoid)."""
import numpy as np
import torch
import pytest

from oracle import experts as ox, mxfp4 as oq
from helpers import bf16_bits, to_dev_bf16

pytestmark = pytest.mark.gpu


def test_every_finite_gate_value():
    from mimo_stream import kernels, pools
    H, I, M = 4096, 2048, 8
    bank = pools.alloc_bank(1, hidden=H, inter=I)
    for p in ("gate", "up", "down"):
        bank[p + "_s"].fill_(127)
    n = torch.arange(I, device="cuda")
    bank["gate_w"][0, n, n // 8] = (2 << (4 * (n % 8))).to(torch.int32)      # code 2 is 1.0
    bank["up_w"][0, :, H // 8 - 1] = 2 << 28
    bits = np.arange(65536, dtype=np.uint16)
    vals = oq.bf16_bits_to_f32(bits[((bits & 0x7F80) != 0x7F80) & (bits != 0x8000)])   # a sum of zeros is +0
    vals = np.concatenate([vals, np.zeros(-len(vals) % (M * I), np.float32)]).reshape(-1, M, I)
    rows = np.arange(M, dtype=np.int32)
    for v in vals:
        x = np.zeros((M, H), np.float32)
        x[:, :I] = v
        x[:, H - 1] = 1.0
        _, h, _ = kernels.moe_experts(to_dev_bf16(x), bank, [0], rows[None], [M], np.ones((1, M), np.float32), R=M,
                                      gather_idx=rows, return_intermediates=True)
        with np.errstate(over="ignore"):
            ref = ox.swiglu_bf16(v, np.ones_like(v))
        np.testing.assert_array_equal(bf16_bits(h)[0], oq.f32_to_bf16_bits(ref))
