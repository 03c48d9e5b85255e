"""MXFP4 codec at the sizes its kernels cut into pieces (threads with several pieces in flight, groups of 4 lanes per
block) and over every finite bf16 value and every code and scale byte, bit-exact against the oracle."""
import numpy as np
import pytest
import torch

from oracle import mxfp4 as oq

pytestmark = pytest.mark.gpu


def _dev(w):
    return torch.from_numpy(w).to(torch.bfloat16).cuda()


@pytest.mark.parametrize("rows,cols", [(1, 32), (3, 96), (7, 992), (8, 1024), (33, 1056), (257, 256)])
def test_sizes(rng, rows, cols):
    from mimo_stream import kernels
    w = oq.round_bf16((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
    q, s = kernels.quantize_mxfp4(_dev(w))
    qo, so = oq.quantize_mxfp4(w)
    np.testing.assert_array_equal(q.cpu().numpy().view(np.uint32), qo)
    np.testing.assert_array_equal(s.cpu().numpy(), so)
    np.testing.assert_array_equal(kernels.dequantize_mxfp4(q, s).cpu().numpy(), oq.dequantize_mxfp4(qo, so))


def test_every_finite_bf16(rng):
    """Shuffled (wide ranges inside a block) and in order (one exponent per block: every rounding case)."""
    from mimo_stream import kernels
    bits = np.arange(65536, dtype=np.uint16)
    bits = bits[(bits & 0x7F80) != 0x7F80]
    for v in (bits, rng.permutation(bits), rng.permutation(bits)):
        w = oq.bf16_bits_to_f32(v).reshape(-1, 1024 if v.size % 1024 == 0 else 32)
        q, s = kernels.quantize_mxfp4(_dev(w))
        qo, so = oq.quantize_mxfp4(w)
        np.testing.assert_array_equal(s.cpu().numpy(), so)
        np.testing.assert_array_equal(q.cpu().numpy().view(np.uint32), qo)


def test_every_code_and_scale():
    from mimo_stream import kernels
    q = np.tile(np.array([0x76543210, 0xFEDCBA98, 0x01234567, 0x89ABCDEF], np.uint32), (256, 1))
    s = np.arange(256, dtype=np.uint8)[:, None]
    got = kernels.dequantize_mxfp4(torch.from_numpy(q.view(np.int32)).cuda(), torch.from_numpy(s).cuda()).cpu().numpy()
    with np.errstate(over="ignore"):
        ref = oq.dequantize_mxfp4(q, s)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    fine = ~np.isnan(ref)
    np.testing.assert_array_equal(got[fine].view(np.uint32), ref[fine].view(np.uint32))
