"""Calls whose default route must not be slower than another kernel of this
library takes for them: each was once given a kernel 1.4 to 8 times slower.
Both are timed here in turn (captured calls, medians); a quarter over is
allowed."""
import pytest
import torch

import mlxcel_amd as mq
from helpers import announce, graph_us, kernels_of, setknob

pytestmark = pytest.mark.gpu


def _matrix(shape, K, bits, gs):
    g = torch.Generator(device="cuda").manual_seed(7)
    w = torch.randint(-2 ** 31, 2 ** 31, (*shape, K * bits // 32), generator=g, device="cuda").to(torch.int32)
    s = torch.rand((*shape, K // gs), generator=g, device="cuda").to(torch.bfloat16) * 0.01
    return w.view(torch.uint32), s, -8 * s


def _timed(monkeypatch, call, other):
    """(us of the default route, us with the switches of `other` set)"""
    def switched():
        with monkeypatch.context() as m:
            for k, v in other.items():
                setknob(m, k, v)
            call()
        setknob(monkeypatch, "MLXQ_NONE", "")  # re-read the switches

    return graph_us([call, switched])


def _dense(M, N, K, bits, gs, dt):
    w, s, b = _matrix((N,), K, bits, gs)
    x, s, b = (t.to(dt) for t in (torch.randn(M, K, device="cuda"), s, b))
    return lambda: mq.quantized_matmul(x, w, s, b, True, gs, bits)


@pytest.mark.parametrize("bits,M,N,K,gs", [(4, 78, 151936, 256, 32), (4, 97, 151936, 576, 64), (4, 52, 151936, 256, 128),
                                           (8, 49, 151936, 1152, 128), (2, 831, 17072, 288, 32), (5, 739, 5645, 544, 32)])
def test_strip_kernel_and_the_ones_it_replaces(monkeypatch, bits, M, N, K, gs):
    # many rounds of strips with a short K, several passes over an odd width
    announce("route time, strip", bits, M, N, K)
    now, other = _timed(monkeypatch, _dense(M, N, K, bits, gs, torch.bfloat16), {"MLXQ_STRIP": "0"})
    assert now <= 1.25 * other, (now, other)


@pytest.mark.parametrize("bits,M,N,K,gs", [(3, 257, 155, 1024, 128), (6, 223, 142, 1152, 128), (3, 323, 146, 512, 64), (2, 488, 282, 512, 32)])
def test_odd_widths_of_small_matrices(monkeypatch, bits, M, N, K, gs):
    # the prefill tiles against the general kernel, which these switches leave the call to
    announce("route time, odd widths", bits, M, N, K)
    now, other = _timed(monkeypatch, _dense(M, N, K, bits, gs, torch.float16), {"MLXQ_QMM_MIN_ROWS": "100000", "MLXQ_STRIP": "0"})
    assert now <= 1.25 * other, (now, other)


@pytest.mark.parametrize("bits,M,N,K,gs", [(4, 469, 17388, 1152, 128), (4, 462, 18864, 1024, 128), (4, 442, 17336, 448, 64)])
def test_prefill_tiles_of_short_k(monkeypatch, bits, M, N, K, gs):
    # the planned tile and K split against each tile unsplit
    announce("route time, prefill tiles", bits, M, N, K)
    call = _dense(M, N, K, bits, gs, torch.bfloat16)
    for tile in ("4", "6", "8"):
        now, other = _timed(monkeypatch, call, {"MLXQ_QMM_TILE": tile, "MLXQ_QMM_KSPLIT": "1"})
        assert now <= 1.2 * other, (tile, now, other)


@pytest.mark.parametrize("E,N,K,B,bits", [(128, 2026, 640, 16328, 4), (60, 5641, 896, 3300, 8), (8, 5186, 1664, 928, 4), (64, 3282, 640, 3234, 8)])
def test_evenly_routed_sorted_gather(monkeypatch, E, N, K, B, bits):
    # many rounds of strips with a short K, against the grouped tiles
    announce("route time, even gather", E, N, K, B, bits)
    w, s, b = _matrix((E, N), K, bits, 128)
    x = torch.randn(B, 1, K, device="cuda").to(torch.bfloat16)
    ids = torch.randint(0, E, (B,), generator=torch.Generator().manual_seed(B)).sort().values.to(torch.int32).cuda()
    now, tiles = _timed(monkeypatch, lambda: mq.gather_qmm(x, w, s, b, None, ids, True, 128, bits, "affine", True), {"MLXQ_STRIP": "0"})
    assert now <= 1.2 * tiles, (now, tiles)


@pytest.mark.parametrize("E,N,K,B,hot", [(128, 768, 2048, 8192, 8), (128, 768, 2048, 1024, 8), (32, 2048, 1024, 2048, 2)])
def test_skewed_sorted_gather(monkeypatch, E, N, K, B, hot):
    # all entries on a few experts, against the grouped tiles
    announce("route time, skewed gather", E, N, K, B, hot)
    w, s, b = _matrix((E, N), K, 4, 64)
    x = torch.randn(B, 1, K, device="cuda").to(torch.bfloat16)
    ids = (torch.arange(hot, device="cuda").repeat_interleave(B // hot) * (E // hot)).to(torch.int32)

    def call():
        return mq.gather_qmm(x, w, s, b, None, ids, True, 64, 4, "affine", True)

    now, tiles = _timed(monkeypatch, call, {"MLXQ_STRIP": "0"})
    assert any("qmm_strip" in k for k in kernels_of(call))
    assert now <= 1.25 * tiles, (now, tiles)
