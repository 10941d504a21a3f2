"""Bitwise parity of the conversion kernels where their fast paths hand over:
quotients on and next to a rounding tie, scales whose reciprocal is not a
normal number, values on the fp4 midpoints, shared exponents past the fast
range, row counts around a workgroup's share of words (against the oracle's
restatement of the reference's quantizers and dequantizers)."""
import ctypes

import numpy as np
import pytest
import torch

import mlxcel_amd as mq
import oracle as orc
from mlxcel_amd import _lib
from mlxcel_amd.ops import _arr, _ref
from helpers import announce, dev_bf16, dev_u8, dev_u32, host_u16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("bits", [1, 2, 3, 4, 5, 6, 8])
@pytest.mark.parametrize("gs", [32, 64, 128])
def test_affine_quantize_ties_and_extreme_scales(dtype, bits, gs):
    announce("quantize ties", dtype, bits, gs)
    rng = np.random.default_rng(50000 + bits + gs)
    top = (1 << bits) - 1
    # groups on the half-step grid of their own range, then nudged by one ulp
    grid = rng.integers(0, 2 * top + 1, size=(24, 3 * gs)).astype(np.float32) / 2 - top / 2
    grid.reshape(24, 3, gs)[..., 0] = -top / 2
    grid.reshape(24, 3, gs)[..., 1] = top / 2
    grid[8:16] = np.nextafter(grid[8:16], np.float32(1e9)) * np.float32(0.37)
    big, small = (2.0 ** 14, 2.0 ** -14) if dtype == "float16" else (1e36, 1e-36)
    w = np.concatenate([grid, grid[:4] * np.float32(small), grid[:4] * np.float32(big / (top + 1))])
    t = torch.from_numpy(w).to(getattr(torch, dtype))
    host = {"bfloat16": lambda: t.view(torch.int16).numpy().astype(np.uint16), "float16": t.numpy, "float32": t.numpy}[dtype]()
    ewq, es, eb = orc.affine_quantize_t(host, dtype, gs, bits)
    wq, s, b = mq.quantize(t.cuda(), gs, bits)
    np.testing.assert_array_equal(wq.cpu().view(torch.int32).numpy().view(np.uint32), ewq)
    for got, want in ((s, es), (b, eb)):
        g = got.cpu()
        g = g.view(torch.int16).numpy().view(np.uint16) if dtype == "bfloat16" else g.numpy()
        assert g.tobytes() == np.ascontiguousarray(want).tobytes()


def test_mxfp4_quantize_midpoints_and_exponents():
    announce("quantize mxfp4 midpoints")
    rng = np.random.default_rng(51000)
    mids = np.array([0, 0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5, 6], np.float32)
    w = rng.choice(np.concatenate([mids, -mids]), size=(64, 96)).astype(np.float32)
    w[:, ::32] = 6
    w[32:] *= np.float32(1) + rng.integers(-1, 2, size=(32, 96)).astype(np.float32) * np.float32(2 ** -7)
    e = np.repeat(np.tile(np.array([0, -3, 40, -40, 119, -119, 123, -125], np.int32), 8), 96).reshape(64, 96)
    bits = orc.f32_to_bf16(np.ldexp(w, e))
    ewq, esc = orc.mxfp4_quantize(bits)
    wq, sc = mq.quantize(dev_bf16(bits), 32, 4, "mxfp4")
    np.testing.assert_array_equal(wq.cpu().view(torch.int32).numpy().view(np.uint32), ewq)
    np.testing.assert_array_equal(sc.cpu().numpy(), esc)


@pytest.mark.parametrize("scale", [1.0, 2.0 ** 122, 2.0 ** -124])
def test_mxfp4_quantize_nan_and_infinity_among_finite_values(scale):
    announce("quantize mxfp4 nonfinite", scale)
    rng = np.random.default_rng(51500)
    w = rng.standard_normal((6, 96)).astype(np.float32) * np.float32(scale)
    w[0, ::7], w[1, 5], w[2] = np.nan, -np.nan, np.nan
    w[3, 40], w[4, 70] = np.inf, -np.inf
    w[4, 71] = np.nan
    bits = orc.f32_to_bf16(w)
    ewq, esc = orc.mxfp4_quantize(bits)
    wq, sc = mq.quantize(dev_bf16(bits), 32, 4, "mxfp4")
    finite = ~np.isinf(w).reshape(6, 3, 32).any(-1)
    # (a group with an infinity has no scale the reference defines)
    np.testing.assert_array_equal(wq.cpu().view(torch.int32).numpy().view(np.uint32).reshape(6, 3, 4)[finite],
                                  ewq.reshape(6, 3, 4)[finite])
    np.testing.assert_array_equal(sc.cpu().numpy()[finite], esc.reshape(6, 3)[finite])


@pytest.mark.parametrize("bits", [2, 4, 8])
@pytest.mark.parametrize("rows,K", [(1, 128), (7, 256), (33, 1152), (65, 128)])
def test_affine_dequantize_words_and_nonfinite(bits, rows, K):
    announce("dequantize words", bits, rows, K)
    rng = np.random.default_rng(52000 + bits + rows)
    wq = rng.integers(0, 1 << 32, size=(rows, K * bits // 32), dtype=np.uint32)
    s = orc.f32_to_bf16(rng.standard_normal((rows, K // 64)).astype(np.float32) * np.float32(1e-38))
    b = orc.f32_to_bf16(rng.standard_normal((rows, K // 64)).astype(np.float32))
    s.reshape(-1)[::5], b.reshape(-1)[::7] = 0x7F80, 0xFF80  # infinities: NaN where they meet
    s.reshape(-1)[1::6] = 0x7F7F
    got = host_u16(mq.dequantize(dev_u32(wq), dev_bf16(s), dev_bf16(b), 64, bits))
    np.testing.assert_array_equal(got, orc.affine_dequantize(wq, s, b, 64, bits, 2))


@pytest.mark.parametrize("scale", [0, 1, 2, 127, 251, 252, 254, 255])
def test_mxfp4_dequantize_uniform_scales(scale):
    announce("dequantize mxfp4", scale)
    wq = np.random.default_rng(53000).integers(0, 1 << 32, size=(40, 32), dtype=np.uint32)
    sc = np.full((40, 8), scale, np.uint8)
    got = host_u16(mq.dequantize(dev_u32(wq), dev_u8(sc), None, 32, 4, "mxfp4"))
    np.testing.assert_array_equal(got, orc.mxfp4_dequantize(wq, sc))


@pytest.mark.parametrize("bits", [1, 2, 3, 4, 5, 6, 8])
def test_affine_quantize_into_words_aligned_as_words(bits):
    # a caller of the C ABI may give any uint32 array for the codes
    announce("quantize offset words", bits)
    lib = _lib.load()
    w = (torch.randn(9, 192, generator=torch.Generator().manual_seed(bits)) * 0.02).to(torch.bfloat16).cuda()
    want, s, b = mq.quantize(w, 64, bits)
    n = want.numel()
    buf = torch.zeros(n + 8, dtype=torch.int32, device="cuda")
    for off in (1, 2, 3):
        wq = buf[off:off + n].view(want.shape).view(torch.uint32)
        assert wq.data_ptr() % 16 == 4 * off
        buf.zero_()
        args = [_arr(t) for t in (w, wq, s, b)]
        st = lib.mlxq_quantize(_ref(args[0]), 64, bits, b"affine", *[_ref(a) for a in args[1:]],
                               ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert st == _lib.OK, _lib.last_error()
        assert torch.equal(wq.view(torch.int32), want.view(torch.int32))
        assert not buf[:off].any() and not buf[off + n:].any()
