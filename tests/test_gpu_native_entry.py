"""The entry points' native module (csrc/pyext.cpp) against the ctypes path it
stands in for: the same bytes for every wrapper, the same errors, the caller's
stream, and the argument forms it hands back (tensor subclasses, other Python
number types, torch-function modes, CPU tensors).  Whether the module took a
call is asserted each time."""
import sys
import threading

import numpy as np
import pytest
import torch

import mlxcel_amd as mq
from mlxcel_amd import ops
from torch.utils._python_dispatch import TorchDispatchMode
from test_gpu_strip import _weights

pytestmark = pytest.mark.gpu


class _Sub(torch.Tensor):
    pass


NAMES = ("quantized_matmul", "quantized_matmul_multi", "gather_qmm", "dequantize", "quantize", "fused_moe")


def _both(monkeypatch, f, handled=True):
    """f() through the native module and through ctypes; the native module
    must have taken the call (handled) or handed it back as None."""
    assert ops._native is not ops._ctypes_only
    native, results = ops._native, []
    with monkeypatch.context() as m:
        for name in NAMES:
            def record(*a, fn=getattr(native, name)):
                results.append(fn(*a))
                return results[-1]
            m.setattr(native, name, record)
        got = f()
        assert len(results) == 1 and (results[0] is not None) == handled
        for name in NAMES:
            m.setattr(native, name, lambda *a: None)
        return got, f()


def _flat(r):
    return list(r) if isinstance(r, (list, tuple)) else [r]


def test_same_results_as_the_ctypes_path(monkeypatch):
    rng = np.random.default_rng(48000)
    E, N, K = 4, 64, 128
    x = torch.from_numpy(rng.standard_normal((3, K)).astype(np.float32)).to(torch.bfloat16).cuda()
    (w, s, b), _ = _weights(rng, (N,), K, 4, 64, "bfloat16")
    (we, se, be), _ = _weights(rng, (E, N), K, 4, 64, "bfloat16")
    (wg, sg, bg), _ = _weights(rng, (E, N), K, 4, 64, "bfloat16")
    (wd, sd, bd), _ = _weights(rng, (E, K), N, 4, 64, "bfloat16")
    lin = torch.ones(N, dtype=torch.bfloat16, device="cuda")
    ids = torch.tensor([[2, 0], [1, 3], [0, 1]], device="cuda")
    score = torch.tensor([0.25, 0.75], device="cuda")
    side = torch.cuda.Stream()

    def on_side():
        # x is written on the side stream behind a wait of some 10 ms: a launch
        # on any other stream would read zeros
        late = torch.zeros_like(x)
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            torch.cuda._sleep(1 << 24)
            late.copy_(x)
            y = mq.quantized_matmul(late, w, s, b)
        side.synchronize()
        assert torch.equal(y, mq.quantized_matmul(x, w, s, b))
        return y

    def in_mode():
        with torch.device("cuda"):  # a torch-function mode
            return mq.quantized_matmul(x, w, s, b)

    # forms that the native module hands back
    for f in (lambda: mq.quantized_matmul(x, w, s, b, group_size=np.int64(64), bits=4), in_mode,
              lambda: mq.quantized_matmul(x.as_subclass(_Sub), w, s, b).as_subclass(torch.Tensor),
              lambda: mq.quantized_matmul(x, w, s, b, bits=np.int64(4))):
        got, want = _both(monkeypatch, f, handled=False)
        assert torch.equal(got, want)
    for f in (lambda: mq.quantized_matmul(x, w, s, b), lambda: mq.quantized_matmul(x[None], w, s, b, True, 64, 4, "affine"),
              lambda: mq.quantized_matmul(x, w, s, b, out=torch.empty(3, N, dtype=torch.bfloat16, device="cuda")),
              lambda: mq.quantized_linear(x, w, s, b, lin), lambda: mq.quantized_linear(x, w, s, b),
              lambda: mq.quantized_matmul_multi(x, [w, w], (s, s), [b, b]),
              lambda: mq.gather_qmm(x.view(3, 1, 1, K), we, se, be, None, ids),
              lambda: mq.dequantize(w, s, b), lambda: mq.quantize(lin.expand(4, N).contiguous()),
              lambda: mq.fused_moe_expert(x[0], ids[0], wg, sg, bg, we, se, be, wd, sd, bd, score, K, N, 2, 4, 4, 64)):
        got, want = _both(monkeypatch, f)
        assert type(got) is type(want)
        for g, h in zip(_flat(got), _flat(want)):
            assert g.shape == h.shape and g.dtype == h.dtype and torch.equal(g.view(torch.uint8), h.view(torch.uint8))
    on_side()


@pytest.mark.parametrize("change", ["w_dtype", "no_biases", "inner", "mode", "out_shape", "cpu", "bits"])
def test_same_errors_as_the_ctypes_path(monkeypatch, change):
    rng = np.random.default_rng(49000)
    x = torch.ones((2, 128), dtype=torch.bfloat16, device="cuda")
    (w, s, b), _ = _weights(rng, (8,), 128, 4, 64, "bfloat16")
    a = dict(x=x, w=w, scales=s, biases=b)
    if change == "w_dtype":
        a["w"] = w.view(torch.int32)
    elif change == "no_biases":
        a["biases"] = None
    elif change == "inner":
        a["x"] = x[:, :64].contiguous()
    elif change == "mode":
        a["mode"] = "nonsense"
    elif change == "out_shape":
        a["out"] = torch.empty((3, 8), dtype=torch.bfloat16, device="cuda")
    elif change == "cpu":
        a["x"] = x.cpu()
    else:
        a["bits"] = 7

    def message():
        with pytest.raises((ValueError, NotImplementedError, ops.QuantizedOpError)) as e:
            mq.quantized_matmul(**a)
        return type(e.value), str(e.value)

    # (a tensor off the GPU is handed back: the ctypes path has the message)
    got, want = _both(monkeypatch, message, handled=change != "cpu")
    assert got == want and got[1]


def test_multi_holds_the_outputs_of_a_list_that_changes():
    # another thread empties the list while the call runs without the GIL
    rng = np.random.default_rng(49500)
    x = torch.ones((2, 128), dtype=torch.bfloat16, device="cuda")
    (w, s, b), _ = _weights(rng, (8,), 128, 4, 64, "bfloat16")
    want = mq.quantized_matmul(x, w, s, b)
    lists, stop = [[]], threading.Event()

    def empty():
        while not stop.is_set():
            lists[0].clear()

    t = threading.Thread(target=empty)
    t.start()
    try:
        for i in range(300):
            outs = [torch.empty(2, 8, dtype=torch.bfloat16, device="cuda") for _ in range(3)]
            lists[0] = outs
            r = ops._native.quantized_matmul_multi(x, [w] * 3, [s] * 3, [b] * 3, None, None, "affine", outs)
            # None: emptied before the call looked at it
            assert r is None or all(torch.equal(y, want) for y in r)
    finally:
        stop.set()
        t.join()
    outs = [torch.empty(2, 8, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    held = [sys.getrefcount(o) for o in (w, s, b, *outs)]
    r = ops._native.quantized_matmul_multi(x, [w] * 2, (s,) * 2, [b] * 2, None, None, "affine", outs)
    assert all(y is o for y, o in zip(r, outs))
    del r
    assert [sys.getrefcount(o) for o in (w, s, b, *outs)] == held


def test_an_exception_of_a_dispatch_mode_reaches_the_caller():
    rng = np.random.default_rng(49600)
    x = torch.ones((2, 128), dtype=torch.bfloat16, device="cuda")
    (w, s, b), _ = _weights(rng, (8,), 128, 4, 64, "bfloat16")
    seen = []

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            if self.refuse:
                raise LookupError("no allocation here")
            return func(*args, **(kwargs or {}))

    with Mode() as mode:
        mode.refuse = False
        y = mq.quantized_matmul(x, w, s, b)
        assert seen  # the result was allocated through the mode
        mode.refuse = True
        with pytest.raises(LookupError, match="no allocation"):
            mq.quantized_matmul(x, w, s, b)
    assert torch.equal(y, mq.quantized_matmul(x, w, s, b))
