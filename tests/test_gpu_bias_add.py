"""The linear bias of quantized_linear in 16-bit types, bit for bit the matmul's
result plus the bias in fp32, rounded once: column counts that are and are not
multiples of the 8 elements a thread adds, a bias of the output's shape."""
import numpy as np
import pytest
import torch

import mlxcel_amd as mq
from helpers import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("M,N", [(1, 8), (3, 7), (5, 1001), (33, 264), (1, 1)])
@pytest.mark.parametrize("full", [False, True])
def test_bias_is_the_rounded_sum(dt, M, N, full):
    announce("bias add", dt, M, N, full)
    rng = np.random.default_rng(54000 + M + N)
    td = getattr(torch, dt)
    x = torch.from_numpy(rng.standard_normal((M, 64)).astype(np.float32)).to(td).cuda()
    codes = torch.from_numpy(rng.integers(0, 1 << 32, size=(N, 8), dtype=np.uint32)).cuda()
    s = torch.full((N, 1), 0.01, dtype=td, device="cuda")
    b = torch.full((N, 1), -0.05, dtype=td, device="cuda")
    bias = torch.from_numpy(rng.standard_normal((M, N) if full else (N,)).astype(np.float32)).to(td).cuda()
    y = mq.quantized_matmul(x, codes, s, b)
    got = mq.quantized_linear(x, codes, s, b, bias)
    assert torch.equal(got, (y.float() + bias.float()).to(td))
