"""The ops library's workspaces: as many streams as its table of reduction
buffers has entries, each with products that split k as well, through a linear
layer's backward (products, bias gradient) against float64; captured products
that split k, which are the eager ones bit for bit, and more captures than hold a
split workspace."""
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


def captured(fn):
    import torch

    st, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(graph, stream=st):
        fn(st)
    return graph, st


@pytest.mark.parametrize("M,K,N", [(77, 768, 3072), (4096, 768, 768)])
def test_captured_split_products_are_the_eager_ones(dev, M, K, N):
    """grad_y w^T splits k at the first size, x^T grad_y at the second. The graph is
    replayed on a stream of its own while eager calls run on the one it was captured
    on; both give the eager bits each time."""
    import torch

    g = torch.Generator(device=dev).manual_seed(M)
    x, w, gy = (torch.empty(s, device=dev).normal_(0.0, 1.0, generator=g) for s in ((M, K), (K, N), (M, N)))
    out = [[torch.zeros(s, device=dev) for s in ((M, K), (K, N), (N,))] for _ in range(3)]

    def backward(o, st):
        ops.device_linear_backward(*o, gy, x, w, 1, M, K, N, stream=st)

    first = torch.cuda.Stream()
    first.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(first):
        backward(out[0], first)
        first.synchronize()
        graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=first):
        backward(out[1], first)
    other = torch.cuda.Stream()
    for _ in range(4):
        for o in out[1:]:
            o[1].zero_(), o[2].zero_(), o[0].fill_(float("nan"))
        torch.cuda.synchronize()
        with torch.cuda.stream(other):
            graph.replay()
        backward(out[2], first)
        torch.cuda.synchronize()
        # (grad_b's reduction shares its buffer with the capture's stream, and is not compared)
        for o in out[1:]:
            assert torch.equal(o[0], out[0][0]) and torch.equal(o[1], out[0][1])


def test_first_split_product_of_a_stream_beside_a_capture(dev):
    """An eager product that allocates its split workspace while another stream is
    being captured ends neither."""
    import torch

    M, K, N = 77, 3072, 768
    g = torch.Generator(device=dev).manual_seed(6)
    x, w = (torch.empty(s, device=dev).normal_(0.0, 1.0, generator=g) for s in ((M, K), (K, N)))
    b, y, z = torch.zeros(N, device=dev), torch.empty((M, N), device=dev), torch.zeros(4, device=dev)
    eager = torch.cuda.Stream()
    torch.cuda.synchronize()
    ops.release_workspaces()

    def both(st):
        z.add_(1.0)
        ops.device_linear_activation_fused_forward(y, None, x, w, b, False, 1, M, K, N, stream=eager)

    graph, _ = captured(both)
    graph.replay()
    torch.cuda.synchronize()
    assert z.tolist() == [1.0] * 4
    assert rel(y, x.double() @ w.double()) < 1.2e-6


def test_graphs_outlive_a_release_and_a_larger_call(dev):
    """A captured LayerNorm backward, linear backward and clipping call keep the
    buffer that they were captured with when the workspaces are released, and when a
    larger call on the stream needs more; memory allocated afterwards is not theirs."""
    import torch

    M, C = 512, 768
    g = torch.Generator(device=dev).manual_seed(9)

    def rnd(*s):
        return torch.empty(s, device=dev).normal_(0.0, 1.0, generator=g)

    x, w, gy, gamma = rnd(M, C), rnd(C, C), rnd(M, C), rnd(C)
    mean, var = x.mean(1), x.var(1, unbiased=False)
    big = rnd(4096, 4 * C), rnd(4096, C), rnd(C, 4 * C)
    big_out = torch.empty((4096, C), device=dev), torch.zeros((C, 4 * C), device=dev), torch.zeros(4 * C, device=dev)
    out = [torch.zeros(s, device=dev) for s in ((M, C), (C,), (C,), (M, C), (C, C), (C,))]
    clip = gy.clone()

    def calls(st):
        ops.device_layernorm_residual_fused_backward(*out[:3], gy, None, x, mean, var, gamma, 1, M, C, stream=st)
        ops.device_linear_backward(*out[3:], gy, x, w, 1, M, C, C, stream=st)
        ops.device_scale_and_clip_grad(clip, M * C, 1.0, 1, stream=st)

    def reset():
        for o in out:
            o.zero_()
        clip.copy_(gy)
        torch.cuda.synchronize()

    torch.cuda.synchronize()
    ops.release_workspaces()
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    calls(st)
    torch.cuda.synchronize()
    want = [t.clone() for t in out + [clip]]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        calls(st)
    for step in range(4):
        if step == 1:
            ops.release_workspaces()
        if step == 2:
            ops.device_linear_backward(*big_out, big[0], big[1], big[2], 1, 4096, C, 4 * C, stream=st)
            torch.cuda.synchronize()
        if step == 3:
            ops.release_workspaces()
        held = [torch.full((1 << 18,), 7.0, device=dev) for _ in range(64)]  # 64 MB of what might have been freed
        reset()
        graph.replay()
        torch.cuda.synchronize()
        for t, e in zip(out + [clip], want):
            assert torch.equal(t, e), step
        assert all(bool((h == 7.0).all()) for h in held), step
        del held


def test_more_captures_than_split_workspaces(dev):
    import torch

    M, K, N = 77, 3072, 768
    g = torch.Generator(device=dev).manual_seed(5)
    x, w = (torch.empty(s, device=dev).normal_(0.0, 1.0, generator=g) for s in ((M, K), (K, N)))
    b, r = torch.zeros(N, device=dev), x.double() @ w.double()
    made = []
    for _ in range(20):
        y = torch.full((M, N), float("nan"), device=dev)
        made.append((captured(lambda st: ops.device_linear_activation_fused_forward(y, None, x, w, b, False, 1, M, K, N,
                                                                                      stream=st)), y))
    for _ in range(2):
        for (graph, _), y in made:
            y.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert rel(y, r) < 1.2e-6
