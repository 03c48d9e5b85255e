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


QNAN, SNAN, INF = 0x7FC1, 0x7F81, 0x7F80


def _quantize_nonfinite(bits):
    """The quantiser's arithmetic on blocks that hold a NaN or an infinity, which the OCP rule leaves open: the maximum is
    taken in element order with IEEE fmax (a quiet NaN is passed over, a signalling one restarts it), an infinity counts
    and saturates at 6, a NaN's code is 0.  bits uint16 [blocks, 32] -> codes uint8 [blocks, 32], scale bytes."""
    v = oq.bf16_bits_to_f32(bits).astype(np.float64)
    mag = (bits & 0x7FFF).astype(np.int64)
    nan, quiet = mag > INF, (bits & 0x40) != 0
    run = np.zeros(len(bits))
    for j in range(32):
        a = np.where(mag[:, j] == INF, 2.0 ** 128, np.abs(v[:, j]))     # an exponent field of 255
        run = np.where(nan[:, j], np.where(quiet[:, j], run, np.nan), np.fmax(run, a))
    run = np.where(np.isnan(run), 2.0 ** 128, run)                      # nothing after the last signalling NaN
    X = np.clip(np.where(run > 0, np.frexp(run)[1] - 3, -127), -127, 127)
    y = np.where(nan, 0.0, np.abs(v)) / np.ldexp(1.0, X)[:, None]
    code = oq._e2m1_round(y)
    return code | np.where((code > 0) & (bits >= 0x8000), 8, 0).astype(np.uint8), (X + 127).astype(np.uint8)


def test_quantize_nonfinite(rng):
    """Each kind of non-finite value at each of a block's 32 places (8 to a lane, 4 lanes to a block), alone, among
    ordinary, huge and tiny neighbours of both signs, and many at once; in rows that end inside a wave's pieces."""
    from mimo_stream import kernels
    blocks = []
    for scale in (0.0, 0.02, 2.0 ** 125, 2.0 ** -130):
        for at in range(32):
            for k in (INF, INF | 0x8000, QNAN, QNAN | 0x8000, SNAN, SNAN | 0x8000):
                b = (oq.round_bf16((rng.standard_normal(32) * scale).astype(np.float32)).view(np.uint32) >> 16).astype(np.uint16)
                b[at] = k
                blocks.append(b)
    for share in (0.1, 0.5, 1.0):
        for _ in range(200):
            b = (oq.round_bf16(rng.standard_normal(32).astype(np.float32)).view(np.uint32) >> 16).astype(np.uint16)
            some = rng.random(32) < share
            b[some] = rng.choice(np.array([INF, INF | 0x8000, QNAN, SNAN, SNAN | 0x8000], np.uint16), some.sum())
            blocks.append(b)
    bits = np.stack(blocks)
    bits = bits[:len(bits) // 3 * 3].reshape(-1, 96)                     # rows of three blocks
    with np.errstate(invalid="ignore", over="ignore"):
        code, scale = _quantize_nonfinite(bits.reshape(-1, 32))
    w = torch.from_numpy(bits.view(np.int16)).cuda().view(torch.bfloat16)
    q, s = kernels.quantize_mxfp4(w)
    np.testing.assert_array_equal(s.cpu().numpy().reshape(-1), scale)
    np.testing.assert_array_equal(oq.unpack_nibbles(q.cpu().numpy().view(np.uint32)).reshape(-1, 32), code)
