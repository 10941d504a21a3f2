"""GPU parity of the strip kernel (qmm_strip.hpp): weights dequantized in
registers into MFMA operands, 5-128 dense rows and expert-sorted gathers of
affine codes, against the float64 numpy restatement of MLX's CPU kernels
(oracle/generic.py).

The sizes sit at the kernel's edges: the 16-row activation tiles (16/17,
32/33, 64/65, 128), the 16-64-row weight blocks, the 128-position windows and
the steps of several of them (K below one window, one past it, an odd number
of groups), K ranges with their partial sums.  Tolerance: max|y - y_ref| /
max|y_ref| <= 1e-2, the bound of every 16-bit result here (weights rounded to
the 16-bit type, one rounding of the result).
"""
import numpy as np
import pytest
import torch

import mlxcel_amd as mq
from oracle import generic as og
from helpers import announce, dev_u32, kernels_of, setknob

pytestmark = pytest.mark.gpu

TD = {"bfloat16": torch.bfloat16, "float16": torch.float16}


def _dev(vals, dt):
    t = torch.from_numpy(np.asarray(vals, dtype=np.float32)).to(TD[dt]).cuda()
    return t, t.float().cpu().numpy().astype(np.float64)


def _weights(rng, shape, K, bits, gs, dt):
    wqn = og.pack_codes(rng.integers(0, 1 << bits, size=shape + (K,)), bits)
    s, sv = _dev(rng.uniform(0.002, 0.02, size=shape + (K // gs,)), dt)
    b, bv = _dev(rng.uniform(-0.1, 0.1, size=shape + (K // gs,)), dt)
    return (dev_u32(wqn), s, b), (wqn, sv, bv)


def _rel(y, want, dt):
    got = y.float().cpu().numpy().astype(np.float64)
    want = og.round_to(want, dt)
    return float(np.abs(got - want).max() / max(np.abs(want).max(), 1e-30))


@pytest.mark.parametrize("bits", [2, 3, 4, 5, 6, 8])
@pytest.mark.parametrize("dt", ["bfloat16", "float16"])
@pytest.mark.parametrize("M,N,K,gs,nwn,ks", [
    (5, 33, 32, 32, 4, 1), (16, 64, 160, 32, 2, 1), (16, 17, 1056, 32, 1, 2), (17, 65, 4096, 128, 4, 3),
    (32, 1, 192, 64, 1, 1), (33, 130, 2112, 64, 2, 2), (64, 100, 640, 128, 4, 1), (65, 48, 1088, 64, 4, 2), (48, 80, 1088, 64, 2, 2), (35, 65, 416, 32, 4, 1),
    (128, 70, 576, 64, 4, 1), (300, 40, 256, 32, 4, 1)])
def test_dense_edges(monkeypatch, bits, dt, M, N, K, gs, nwn, ks):
    setknob(monkeypatch, "MLXQ_STRIP", "2")
    setknob(monkeypatch, "MLXQ_STRIP_NWN", str(nwn))
    setknob(monkeypatch, "MLXQ_STRIP_KS", str(ks))
    rng = np.random.default_rng(41000 + 100 * bits + M)
    announce("strip", bits, dt, M, N, K, gs, nwn, ks)
    x, xv = _dev(rng.standard_normal((M, K)), dt)
    (wq, s, b), (wqn, sv, bv) = _weights(rng, (N,), K, bits, gs, dt)
    y = mq.quantized_matmul(x, wq, s, b, True, gs, bits)
    assert _rel(y, og.qmm(xv, wqn, sv, bv, True, gs, bits), dt) <= 1e-2


@pytest.mark.parametrize("bits,M", [(3, 5), (6, 128), (4, 17), (8, 64), (4, 100), (5, 40)])
def test_default_route_matches_other_kernels(monkeypatch, bits, M):
    rng = np.random.default_rng(42000 + bits)
    N, K, gs = 513, 4096, 64
    announce("strip default", bits, M)
    x, xv = _dev(rng.standard_normal((M, K)), "bfloat16")
    (wq, s, b), (wqn, sv, bv) = _weights(rng, (N,), K, bits, gs, "bfloat16")
    y = mq.quantized_matmul(x, wq, s, b, True, gs, bits)
    again = mq.quantized_matmul(x, wq, s, b, True, gs, bits)
    setknob(monkeypatch, "MLXQ_STRIP", "0")
    other = mq.quantized_matmul(x, wq, s, b, True, gs, bits)
    want = og.qmm(xv, wqn, sv, bv, True, gs, bits)
    assert torch.equal(y, again)
    assert _rel(y, want, "bfloat16") <= 1e-2 and _rel(other, want, "bfloat16") <= 1e-2


@pytest.mark.parametrize("value", [float("nan"), float("inf"), 3e38, 2.0 ** 101])
def test_extreme_scales_stay_in_their_row(monkeypatch, value):
    # scales past 2^100 take the slower conversion; a row's NaN or infinity
    # must not reach its neighbours through the positions past K
    setknob(monkeypatch, "MLXQ_STRIP", "2")
    rng = np.random.default_rng(43000)
    M, N, K, gs, bits = 9, 40, 96, 32, 4
    announce("strip extreme scales", value)
    x, xv = _dev(rng.standard_normal((M, K)), "bfloat16")
    (wq, s, b), (wqn, sv, bv) = _weights(rng, (N,), K, bits, gs, "bfloat16")
    s[5] = value
    y = mq.quantized_matmul(x, wq, s, b, True, gs, bits).float().cpu().numpy().astype(np.float64)
    setknob(monkeypatch, "MLXQ_STRIP", "0")
    y0 = mq.quantized_matmul(x, wq, s, b, True, gs, bits).float().cpu().numpy().astype(np.float64)
    want = og.round_to(og.qmm(xv, wqn, sv, bv, True, gs, bits), "bfloat16")
    rest = [n for n in range(N) if n != 5]
    assert np.abs(y[:, rest] - want[:, rest]).max() <= 1e-2 * np.abs(want[:, rest]).max()
    if value == 2.0 ** 101:  # finite sums: the other kernel's values up to the summation order
        assert np.abs(y[:, 5] - y0[:, 5]).max() <= 1e-2 * np.abs(y0[:, 5]).max()
    elif value == value and value < 1e39:
        assert np.isfinite(y[:, rest]).all()
    else:
        assert np.isnan(y[:, 5]).all()


def test_mxfp4_special_scales(monkeypatch):
    setknob(monkeypatch, "MLXQ_STRIP", "2")
    rng = np.random.default_rng(44000)
    M, N, K = 18, 37, 224
    announce("strip mxfp4 scales")
    x, xv = _dev(rng.standard_normal((M, K)), "bfloat16")
    wqn = og.pack_codes(rng.integers(0, 16, size=(N, K)), 4)
    sc = rng.integers(120, 130, size=(N, K // 32)).astype(np.uint8)
    sc[3], sc[4], sc[7, 0] = 0, 230, 255  # 2^-127, 2^103 (254 would overflow the sums), NaN
    y = mq.quantized_matmul(x, dev_u32(wqn), torch.from_numpy(sc).cuda(), None, True, 32, 4, "mxfp4")
    got = y.float().cpu().numpy().astype(np.float64)
    want = og.round_to(og.qmm(xv, wqn, sc, None, True, 32, 4, "mxfp4"), "bfloat16")
    assert np.isnan(got[:, 7]).all()
    for n in range(N):
        if n != 7:
            ok = np.isclose(got[:, n], want[:, n], rtol=1e-2, atol=1e-2 * np.nanmax(np.abs(want[:, n])))
            assert ok.all(), n


@pytest.mark.parametrize("bits,gs", [(4, 64), (8, 32), (4, 128)])
@pytest.mark.parametrize("counts", [[8, 8, 8, 8], [0, 40, 1, 0, 33, 16], [0, 0, 130, 0, 300], [64, 0], [30, 49, 20, 96]])
@pytest.mark.parametrize("idx", [torch.int32, torch.int64])
def test_sorted_gather(bits, gs, counts, idx):
    rng = np.random.default_rng(45000 + bits + sum(counts))
    E, N, K = len(counts), 100, gs * 5
    ids = np.repeat(np.arange(E), counts)
    announce("strip gather", bits, gs, counts, idx)
    x, xv = _dev(rng.standard_normal((len(ids), 1, K)), "bfloat16")
    (wq, s, b), (wqn, sv, bv) = _weights(rng, (E, N), K, bits, gs, "bfloat16")
    y = mq.gather_qmm(x, wq, s, b, None, torch.from_numpy(ids).to(idx).cuda(), True, gs, bits, "affine", True)
    want = np.stack([og.qmm(xv[i], wqn[e], sv[e], bv[e], True, gs, bits) for i, e in enumerate(ids)])
    assert _rel(y, want, "bfloat16") <= 1e-2


@pytest.mark.parametrize("bits,dt", [(6, "bfloat16"), (3, "float16")])
def test_rows_in_passes(bits, dt):
    # more than 128 rows of an odd width whose K the prefill tiles do not take
    rng = np.random.default_rng(46500 + bits)
    M, N, K, gs = 200, 2080, 4128, 32
    announce("strip passes", bits, dt)
    x, xv = _dev(rng.standard_normal((M, K)), dt)
    (wq, s, b), (wqn, sv, bv) = _weights(rng, (N,), K, bits, gs, dt)
    y = mq.quantized_matmul(x, wq, s, b, True, gs, bits)
    assert _rel(y, og.qmm(xv, wqn, sv, bv, True, gs, bits), dt) <= 1e-2


@pytest.mark.parametrize("bits,gs,K", [(8, 64, 320), (8, 32, 192), (8, 128, 640), (4, 64, 320)])
@pytest.mark.parametrize("counts", [[110, 128, 120], [140, 1, 129, 0, 260], [16, 40, 1, 0, 33, 16], [8, 9, 10, 11]])
def test_sorted_gather_runs_here(monkeypatch, bits, gs, K, counts):
    # 8-bit codes, and passes of 128 rows with tails; forced, so that no other
    # kernel can stand in
    setknob(monkeypatch, "MLXQ_STRIP", "2")
    rng = np.random.default_rng(45300 + bits + sum(counts))
    E, N = len(counts), 100
    ids = np.repeat(np.arange(E), counts)
    announce("strip gather forced", bits, gs, counts)
    x, xv = _dev(rng.standard_normal((len(ids), 1, K)), "bfloat16")
    (wq, s, b), (wqn, sv, bv) = _weights(rng, (E, N), K, bits, gs, "bfloat16")
    i = torch.from_numpy(ids).cuda()
    out = []
    names = kernels_of(lambda: out.append(mq.gather_qmm(x, wq, s, b, None, i, True, gs, bits, "affine", True)))
    assert len(names) == 1 and "qmm_strip" in names[0], names
    want = np.stack([og.qmm(xv[i], wqn[e], sv[e], bv[e], True, gs, bits) for i, e in enumerate(ids)])
    assert _rel(out[0], want, "bfloat16") <= 1e-2


# counts of entries per expert: one long run among short ones, all on one
# expert (the first, the last), several long runs, as many experts as a
# workgroup keeps runs of (512) and one more
LONG = {"one": [3, 0, 600, 1, 17, 0, 2, 9, 1, 0, 0, 5, 0, 1, 0, 1], "first": [512] + [0] * 7, "last": [0] * 7 + [513],
        "two": [0] * 20 + [700] + [1] * 20 + [900] + [2] * 22, "512": [8, 700] * 4 + [3] * 504, "513": [8, 700] * 4 + [3] * 505}


@pytest.mark.parametrize("bits,gs,K", [(4, 64, 192), (8, 64, 320)])
@pytest.mark.parametrize("mt", [1, 2, 3, 8])
@pytest.mark.parametrize("name", sorted(LONG))
def test_sorted_gather_with_long_runs(monkeypatch, bits, gs, K, mt, name):
    # runs far above the average are dealt out over the workgroups
    setknob(monkeypatch, "MLXQ_STRIP", "2")
    setknob(monkeypatch, "MLXQ_STRIP_MT", str(mt))
    counts = LONG[name]
    E, N = len(counts), 68 if len(counts) > 64 else 200
    rng = np.random.default_rng(45500 + bits + mt)
    ids = np.repeat(np.arange(E), counts)
    announce("strip gather long runs", bits, mt, name)
    x, xv = _dev(rng.standard_normal((len(ids), 1, K)), "bfloat16")
    (wq, s, b), (wqn, sv, bv) = _weights(rng, (E, N), K, bits, gs, "bfloat16")
    want = np.concatenate([og.qmm(xv[ids == e, 0], wqn[e], sv[e], bv[e], True, gs, bits) for e in range(E) if counts[e]])
    for idx in (torch.int32, torch.int64):
        i = torch.from_numpy(ids).to(idx).cuda()
        y = mq.gather_qmm(x, wq, s, b, None, i, True, gs, bits, "affine", True)
        assert _rel(y[:, 0], want, "bfloat16") <= 1e-2
        assert torch.equal(y, mq.gather_qmm(x, wq, s, b, None, i, True, gs, bits, "affine", True))
    # indices past the experts belong to the last one
    i = torch.from_numpy(np.where(ids == E - 1, E + 5 + np.arange(len(ids)), ids)).to(torch.int32).cuda()
    assert torch.equal(y, mq.gather_qmm(x, wq, s, b, None, i, True, gs, bits, "affine", True))
