"""The ops library's workspaces: as many streams as its table of reduction
buffers has entries, each with products that split k as well, through a linear
layer's backward (products, bias gradient) against float64."""
import ctypes

import pytest

from gpt_amd import ops

pytestmark = pytest.mark.gpu

STREAMS = 64


def rel(x, r):
    return float((x.double() - r).norm() / r.norm())


@pytest.fixture
def streams():
    """64 raw streams of the default priority (torch's pool hands out 32)."""
    import torch

    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipStreamCreate.argtypes = [ctypes.POINTER(ctypes.c_void_p)]
    hip.hipStreamDestroy.argtypes = [ctypes.c_void_p]
    torch.cuda.synchronize()
    ops.release_workspaces()
    out = []
    for _ in range(STREAMS):
        s = ctypes.c_void_p()
        assert hip.hipStreamCreate(ctypes.byref(s)) == 0
        out.append(s.value)
    yield out
    torch.cuda.synchronize()
    ops.release_workspaces()
    for s in out:
        assert hip.hipStreamDestroy(s) == 0


def test_backward_on_64_streams(dev, streams):
    """grad_y w^T splits k at this size; streams past the 16 that hold a split
    workspace run it otherwise, to the same precision (2^-25 sqrt(K / 2) for K terms)."""
    import torch

    M, K, N = 77, 768, 3072
    g = torch.Generator(device=dev).manual_seed(1)
    x, w, gy = (torch.empty(s, device=dev).normal_(0.0, 1.0, generator=g) for s in ((M, K), (K, N), (M, N)))
    gx = [torch.empty((M, K), device=dev) for _ in streams]
    gw, gb = ([torch.zeros(s, device=dev) for _ in streams] for s in ((K, N), (N,)))
    torch.cuda.synchronize()
    for i, s in enumerate(streams):
        ops.device_linear_backward(gx[i], gw[i], gb[i], gy, x, w, 1, M, K, N, stream=s)
    torch.cuda.synchronize()
    rx, rw, rb = gy.double() @ w.double().t(), x.double().t() @ gy.double(), gy.double().sum(0)
    for i in range(STREAMS):
        assert rel(gx[i], rx) < 1.2e-6 and rel(gw[i], rw) < 3e-7 and rel(gb[i], rb) < 3e-7, i
