"""Argument handling of the operator calls in csrc/kh_pyops.c: what each accepts, what it raises, what it returns."""
import ctypes
import threading

import numpy as np
import pytest
import torch

from kuiperllama_amd import _ffi, ops

f = lambda *s: torch.zeros(*s)  # noqa: E731
CALLS = {"add": lambda t: ops.add(t, t, t), "swiglu": lambda t: ops.swiglu(t, t, t), "matmul": lambda t: ops.matmul(t, f(4, 4), t),
         "matmul_q8": lambda t: ops.matmul_q8(t, f(4, 4), t, 64, t), "rmsnorm": lambda t: ops.rmsnorm(t, t, t, 1e-5),
         "rope": lambda t: ops.rope(t, t, 0, t, t, 4, 0), "mha": lambda t: ops.mha(0, 1, 0, 1, 4, 1, 4, t, t, None, t, t)}


@pytest.mark.parametrize("name", sorted(CALLS))
def test_host_tensors_are_refused(name):
    with pytest.raises(ValueError, match="GPU"):
        CALLS[name](f(4))


def test_shapes_and_counts():
    with pytest.raises(ValueError):
        ops.matmul(f(4), f(4), f(4))  # a matrix has two dimensions
    with pytest.raises(TypeError):
        ops.add(f(4), f(4))
    with pytest.raises(AttributeError):
        ops.add([1.0], f(4), f(4))


def test_first_calls_of_several_threads():
    ops._n = ops._Unbound()
    seen = []

    def call():
        try:
            ops.add(f(4), f(4), f(4))
        except Exception as e:  # noqa: BLE001
            seen.append(type(e))

    ts = [threading.Thread(target=call) for _ in range(8)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert seen == [ValueError] * 8


@pytest.mark.gpu
def test_device_calls(gpu):
    d = lambda a: torch.as_tensor(a).to(gpu)  # noqa: E731
    x, y, out = d(np.arange(8, dtype=np.float32)), d(np.ones(8, np.float32)), torch.zeros(8, device=gpu)
    assert ops.add(in1=x, in2=y, out=out) is out and out.cpu().tolist() == list(range(1, 9))
    w = torch.eye(8, device=gpu)
    assert ops.matmul(x, w, out, scale=2) is out and out.cpu().tolist() == [2.0 * i for i in range(8)]
    with pytest.raises(TypeError, match="float32"):
        ops.add(x.int(), y, out)
    with pytest.raises(ValueError, match="contiguous"):
        ops.matmul(x, torch.zeros(8, 16, device=gpu)[:, ::2], out)
    with pytest.raises(ctypes.ArgumentError):
        ops.matmul_q8(x, torch.zeros(8, 64, dtype=torch.int8, device=gpu), y, 64.0, out)
    k, q = torch.randn(2, 64, device=gpu), torch.randn(64, device=gpu)
    one, two, score = torch.zeros(64, device=gpu), torch.zeros(64, device=gpu), torch.zeros(2, device=gpu)
    assert ops.mha(torch.tensor([0], dtype=torch.int32, device=gpu), 1, 0, 2, 64, 1, 64, one, q, score, k, k) is one
    assert ops.mha(np.int64(0), 1, 0, 2, 64, 1, 64, two, q, None, k, k) is two
    assert torch.equal(one, k[0]) and torch.equal(two, k[0]) and score.cpu().tolist() == [1.0, 0.0]
    with pytest.raises(_ffi.KhError):
        ops.mha(2, 1, 0, 2, 64, 1, 64, one, q, None, k, k)  # behind the cache
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        ops.add(x, y, out)
    side.synchronize()
    assert out.cpu().tolist() == list(range(1, 9))
