"""GPU parity of the prefill tile kernel on affine codes of 2, 3, 5 and 6 bits
(qmm_odd.hip), bfloat16 and float16, against the float64 numpy restatement of
MLX's CPU kernels (oracle/generic.py): more than 128 rows, both tiles, with
and without a K split, rows and columns at the edges of the tiles, K from one
64-wide step to an odd number of groups.  Tolerance: max|y - y_ref| /
max|y_ref| <= 1e-2, the bound of every 16-bit result here.
"""
import numpy as np
import pytest
import torch

import mlxcel_amd as mq
from oracle import generic as og
from helpers import announce, setknob
from test_gpu_strip import _dev, _rel, _weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [2, 3, 5, 6])
@pytest.mark.parametrize("dt", ["bfloat16", "float16"])
@pytest.mark.parametrize("M,N,K,gs,tile,ks", [(129, 257, 64, 32, 4, 1), (256, 256, 576, 64, 4, 3),
                                              (300, 1, 192, 32, 6, 1), (130, 129, 1088, 64, 6, 4),
                                              (257, 100, 640, 128, -1, 0), (1025, 33, 128, 64, -1, 0)])
def test_edges(monkeypatch, bits, dt, M, N, K, gs, tile, ks):
    if tile >= 0:
        setknob(monkeypatch, "MLXQ_QMM_TILE", str(tile))
        setknob(monkeypatch, "MLXQ_QMM_KSPLIT", str(ks))
    rng = np.random.default_rng(46000 + 100 * bits + M)
    announce("qmm odd", bits, dt, M, N, K, gs, tile, ks)
    x, xv = _dev(rng.standard_normal((M, K)), dt)
    (wq, s, b), (wqn, sv, bv) = _weights(rng, (N,), K, bits, gs, dt)
    y = mq.quantized_matmul(x, wq, s, b, True, gs, bits)
    assert _rel(y, og.qmm(xv, wqn, sv, bv, True, gs, bits), dt) <= 1e-2


@pytest.mark.parametrize("bits,dt", [(4, "bfloat16"), (8, "bfloat16"), (4, "float16")])
@pytest.mark.parametrize("M,N,K,gs", [(129, 1900, 1152, 64), (333, 770, 4096, 64), (768, 600, 2048, 128), (1024, 129, 576, 32)])
def test_splits_that_fill_a_round(bits, dt, M, N, K, gs):
    # 4- and 8-bit codes take the same tile and K-split choice at 129-1024 rows
    rng = np.random.default_rng(47000 + bits + M)
    announce("qmm mid plan", bits, dt, M, N, K, gs)
    x, xv = _dev(rng.standard_normal((M, K)), dt)
    (wq, s, b), (wqn, sv, bv) = _weights(rng, (N,), K, bits, gs, dt)
    y = mq.quantized_matmul(x, wq, s, b, True, gs, bits)
    assert _rel(y, og.qmm(xv, wqn, sv, bv, True, gs, bits), dt) <= 1e-2
