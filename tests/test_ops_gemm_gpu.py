"""The ops library's own matrix products (gpt_amd/csrc/ops_gemm.hip) at the
sizes where they can go wrong, through the C ABI against float64: rows and
columns off every tile's edge, k with a remainder of 4 and of fewer than one
step, one row, every layout (x w, grad_y w^T, x^T grad_y), split and unsplit k,
the GELU epilogue, and infinities, NaN and values beyond bf16's largest.

Tolerance on the 2-norm: an fp32 accumulation of K random terms in order has a
relative error of about 2^-25 sqrt(K / 2) (K roundings of a sum that grows as
the square root), and no less than 3e-7 is asked, for the few roundings of a
short product and its epilogue. The BLAS libraries' fp32 products, which take
some of these sizes, come within 0.6 of that; the library's own kernels stay
below a third (the tiled one rounds its running sums once per 32 k, the few-row
one six times)."""
import numpy as np
import pytest

from gpt_amd import ops

pytestmark = pytest.mark.gpu


def tol(K):
    return max(3e-7, 2.0 ** -25 * (K / 2) ** 0.5)


def rel(x, r):
    return float((x.double() - r).norm() / r.norm())


def gelu64(s):
    import torch

    return 0.5 * s * (1 + torch.tanh(0.79788456 * (s + 0.044715 * s ** 3)))


SHAPES = [(1, 768, 2304), (33, 768, 768), (77, 100, 132), (77, 3072, 768), (127, 36, 3072), (300, 1600, 6400),
          (1025, 768, 3076), (4096, 768, 768), (3001, 2304, 772), (2050, 3072, 768),
          # tiles of 32 x 48 and 32 x 64 (few rows), with remainders of each
          (70, 768, 3072), (97, 100, 3084), (130, 36, 3076), (66, 1000, 4100), (50, 1600, 6400), (150, 768, 768)]


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_linear_products(dev, M, K, N):
    import torch

    g = torch.Generator(device=dev).manual_seed(M + K + N)

    def rnd(*s, std=1.0):
        return torch.empty(s, device=dev).normal_(0.0, std, generator=g)

    x, w, b, gy = rnd(M, K), rnd(K, N, std=K ** -0.5), rnd(N), rnd(M, N)
    y, act = torch.full((M, N), np.nan, device=dev), torch.full((M, N), np.nan, device=dev)
    gw0, gb = rnd(K, N), torch.zeros(N, device=dev)
    gx, gw = torch.full((M, K), np.nan, device=dev), gw0.clone()
    ops.device_linear_activation_fused_forward(y, act, x, w, b, True, 1, M, K, N)
    ops.device_linear_backward(gx, gw, gb, gy, x, w, 1, M, K, N)
    y64 = x.double() @ w.double() + b.double()
    assert rel(y, y64) < tol(K)
    assert rel(act, gelu64(y64)) < tol(K)
    assert rel(gx, gy.double() @ w.double().t()) < tol(N)
    assert rel(gw - gw0, x.double().t() @ gy.double()) < tol(M) + 2.0 ** -23 * float(gw.norm() / (gw - gw0).norm())
    y2 = torch.empty_like(y)
    ops.device_linear_activation_fused_forward(y2, None, x, w, b, False, 1, M, K, N)
    assert torch.equal(y2, y)


@pytest.mark.parametrize("M,C,V", [(5, 768, 50304), (1000, 768, 8192), (2500, 128, 50304)])
def test_unembedding_products(dev, M, C, V):
    import torch

    g = torch.Generator(device=dev).manual_seed(M)
    x, wte = (torch.empty(s, device=dev).normal_(0.0, std, generator=g) for s, std in (((M, C), 1.0), ((V, C), 0.02)))
    gl = torch.empty((M, V), device=dev).normal_(0.0, 1e-6, generator=g)
    logits, gx, gw = torch.empty((M, V), device=dev), torch.empty((M, C), device=dev), torch.zeros((V, C), device=dev)
    ops.device_unembedding_forward(logits, x, wte, 1, M, C, V)
    ops.device_unembedding_backward(gx, gw, gl, x, wte, 1, M, C, V)
    assert rel(logits, x.double() @ wte.double().t()) < tol(C)
    assert rel(gx, gl.double() @ wte.double()) < tol(V)
    assert rel(gw, gl.double().t() @ x.double()) < tol(M)


@pytest.mark.parametrize("M,K,N", [(64, 768, 768), (4096, 768, 2304)])
def test_non_finite_operands(dev, M, K, N):
    """Where the fp32 product of some row and column is infinite or NaN, so is
    the library's, with its sign; a value beyond bf16's largest finite one is
    no infinity; every other entry is untouched."""
    import torch

    g = torch.Generator(device=dev).manual_seed(7)
    x, w = (torch.empty(s, device=dev).normal_(0.0, 1.0, generator=g) for s in ((M, K), (K, N)))
    b, y = torch.zeros(N, device=dev), torch.empty((M, N), device=dev)
    x[3, 5], x[40, 7], x[50, 1], w[9, 100] = np.inf, -np.inf, 3.4e38, np.nan
    w[1] *= 1e-3
    ops.device_linear_activation_fused_forward(y, None, x, w, b, False, 1, M, K, N)
    r = (x.double() @ w.double()).float()
    assert torch.equal(torch.isnan(y), torch.isnan(r))
    assert torch.equal(torch.isinf(y), torch.isinf(r))
    assert torch.equal(y[torch.isinf(r)], r[torch.isinf(r)])
    for rows in (torch.tensor([50]), torch.tensor([m for m in range(M) if m not in (3, 40, 50)])):
        a, e = y[rows.to(dev)], (x[rows.to(dev)].double() @ w.double())
        ok = torch.isfinite(e)
        assert rel(a[ok], e[ok]) < tol(K)


@pytest.mark.parametrize("row,col", [(None, 0), (None, 31), (None, 45), (0, None), (17, None), (63, None)])
def test_second_pass_where_few_lanes_overflow(dev, row, col):
    """A value beyond bf16's largest in one row or one column only, so that most
    lanes of a wave (the first among them, or not) have finite sums."""
    import torch

    M, K, N = 64, 768, 768
    g = torch.Generator(device=dev).manual_seed(11)
    x, w = (torch.empty(s, device=dev).normal_(0.0, 1.0, generator=g) for s in ((M, K), (K, N)))
    b, y = torch.zeros(N, device=dev), torch.empty((M, N), device=dev)
    if col is None:
        x[row, 300], w[300] = 3.4e38, w[300] * 1e-37
    else:
        w[300, col], x[:, 300] = -3.4e38, x[:, 300] * 1e-37
    ops.device_linear_activation_fused_forward(y, None, x, w, b, False, 1, M, K, N)
    r = x.double() @ w.double()
    assert torch.isfinite(y).all()
    part = (slice(None), col) if row is None else row
    assert rel(y, r) < tol(K) and rel(y[part], r[part]) < tol(K)


@pytest.mark.parametrize("M,K,N", [(90, 768, 1540), (2048, 772, 2308)])
def test_non_finite_operands_of_the_transposed_forms(dev, M, K, N):
    """The same for grad_y w^T (few rows, and tiles of split k) and x^T grad_y, all on
    the library's own kernels at these sizes."""
    import torch

    g = torch.Generator(device=dev).manual_seed(8)
    x, w, gy = (torch.empty(s, device=dev).normal_(0.0, 1.0, generator=g) for s in ((M, K), (K, N), (M, N)))
    x[3, 5], gy[40, 7], gy[50, 1], w[100, 9] = np.inf, -np.inf, 3.4e38, np.nan
    w[:, 1] *= 1e-3
    x[50] *= 1e-3
    gx, gw, gb = torch.empty((M, K), device=dev), torch.zeros((K, N), device=dev), torch.zeros(N, device=dev)
    before = ops.gemm_info()["tuned"]
    ops.device_linear_backward(gx, gw, gb, gy, x, w, 1, M, K, N)
    assert ops.gemm_info()["tuned"] == before + 2
    for y, r, k in ((gx, gy.double() @ w.double().t(), N), (gw, x.double().t() @ gy.double(), M)):
        f = r.float()
        assert torch.equal(torch.isnan(y), torch.isnan(f))
        assert torch.equal(torch.isinf(y), torch.isinf(f))
        assert torch.equal(y[torch.isinf(f)], f[torch.isinf(f)])
        big = r.abs() > 1e30
        for part in (torch.isfinite(f) & big, torch.isfinite(f) & ~big):
            assert rel(y[part], r[part]) < tol(k)


def test_captured_products_replay(dev):
    """A captured linear layer replayed between eager calls gives the eager
    results' values, and the same bits on every replay."""
    import torch

    M, K, N = 4096, 3072, 768
    g = torch.Generator(device=dev).manual_seed(3)
    x, w = (torch.empty(s, device=dev).normal_(0.0, 1.0, generator=g) for s in ((M, K), (K, N)))
    b, y, e = torch.zeros(N, device=dev), torch.empty((M, N), device=dev), torch.empty((M, N), device=dev)
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        ops.device_linear_activation_fused_forward(y, None, x, w, b, False, 1, M, K, N, stream=st)
    first = None
    for _ in range(3):
        y.fill_(np.nan)
        graph.replay()
        ops.device_linear_activation_fused_forward(e, None, x, w, b, False, 1, M, K, N)
        torch.cuda.synchronize()
        first = y.clone() if first is None else first
        assert torch.equal(y, first)
        assert rel(y, e.double()) < tol(K)
    ops.release_workspaces()
    ops.device_linear_activation_fused_forward(e, None, x, w, b, False, 1, M, K, N)
    assert rel(e, x.double() @ w.double()) < tol(K)


@pytest.mark.parametrize("M,K,N", [(77, 768, 768), (2050, 768, 2304)])
@pytest.mark.parametrize("e", [94, 112, 118, 124])
def test_tiny_operands(dev, M, K, N, e):
    """Operands of 2^-e, where bf16 terms are subnormal: all of them, and one
    row or column among ordinary ones, keep the precision of an fp32 product."""
    import torch

    g = torch.Generator(device=dev).manual_seed(e)

    def rnd(*s, std=1.0):
        return torch.empty(s, device=dev).normal_(0.0, std, generator=g)

    x, w, gy, b, y = rnd(M, K), rnd(K, N), rnd(M, N), torch.zeros(N, device=dev), torch.empty((M, N), device=dev)
    small = 2.0 ** -e
    xt, wt, gt = x.clone(), w.clone(), gy * small
    xt[M // 2] *= small
    wt[:, N // 3] *= small
    xz, wz = xt.clone(), wt.clone()  # the first k zeros
    xz[:, :40] = 0
    wz[:40] = 0
    for a, c in ((x * small, w), (x, w * small), (xt, w), (x, wt), (xz, w), (x, wz)):
        ops.device_linear_activation_fused_forward(y, None, a, c, b, False, 1, M, K, N)
        r = a.double() @ c.double()
        assert rel(y, r) < tol(K)
        assert rel(y[M // 2], r[M // 2]) < tol(K)
        assert rel(y[:, N // 3], r[:, N // 3]) < tol(K)
    gx, gw, gb = torch.empty((M, K), device=dev), torch.zeros((K, N), device=dev), torch.zeros(N, device=dev)
    ops.device_linear_backward(gx, gw, gb, gt, x, w, 1, M, K, N)
    assert rel(gx, gt.double() @ w.double().t()) < tol(N)
    assert rel(gw, x.double().t() @ gt.double()) < tol(M)


@pytest.mark.parametrize("M,K,N", [(77, 768, 768), (2050, 768, 2304), (4096, 3072, 768)])
@pytest.mark.parametrize("at", [33, 300, 700])
def test_tiny_rows_after_zeros(dev, M, K, N, at):
    """Rows and columns that are zero up to k = at, then tiny, then ordinary or zero, among
    rows of zeros: the look at their further steps."""
    import torch

    g = torch.Generator(device=dev).manual_seed(at)
    x, w = (torch.empty(s, device=dev).normal_(0.0, 1.0, generator=g) for s in ((M, K), (K, N)))
    b, y = torch.zeros(N, device=dev), torch.empty((M, N), device=dev)
    x[M // 3] = 0
    x[[M // 2, M // 4], :at] = 0
    x[M // 2] *= 2.0 ** -118
    w[:, N // 3] = 0
    w[:at, [N // 2, N // 4]] = 0
    w[:, N // 4] *= 2.0 ** -118
    ops.device_linear_activation_fused_forward(y, None, x, w, b, False, 1, M, K, N)
    r = x.double() @ w.double()
    assert not y[M // 3].any() and not y[:, N // 3].any()
    rest = [n for n in range(N) if n != N // 4]
    assert rel(y[:, rest], r[:, rest]) < tol(K)
    assert rel(y[M // 2][rest], r[M // 2][rest]) < tol(K)
    assert rel(y[M // 4][rest], r[M // 4][rest]) < tol(K)
    rows = [m for m in range(M) if m != M // 2]
    assert rel(y[rows, N // 4], r[rows, N // 4]) < tol(K)


@pytest.mark.parametrize("form", ["nn", "nt"])
@pytest.mark.parametrize("M,K,N", [(77, 3072, 768), (512, 768, 768), (128, 768, 2304), (4096, 768, 2304)])
def test_errors_do_not_add_up_over_rows(dev, M, K, N, form):
    """Sums of the errors over C's rows, as a bias gradient forms them, are as large
    as sums of independent errors (a factor of 1.3 for the 13 of 77 rows that have no
    counterpart of the other sign): the matrix cores round towards minus infinity,
    which adds up to 2 to 4 times that where every error has one sign."""
    import torch

    g = torch.Generator(device=dev).manual_seed(M + K)
    x, w = (torch.empty(s, device=dev).normal_(0.0, 1.0, generator=g) for s in ((M, K), (K, N)))
    y, b = torch.empty((M, N), device=dev), torch.zeros(N, device=dev)
    if form == "nn":
        ops.device_linear_activation_fused_forward(y, None, x, w, b, False, 1, M, K, N)
    else:
        ops.device_unembedding_forward(y, x, w.t().contiguous(), 1, M, K, N)
    e = y.double() - x.double() @ w.double()
    alone = float(e.pow(2).mean().sqrt()) * M ** 0.5
    assert float(e.sum(0).pow(2).mean().sqrt()) < 1.3 * alone


# (form, M, N, K, products on the library's own kernels). Per form a size for each tile
# of ops_gemm.hip (128 x 128 .. 32 x 64, in its order), unsplit and with k split where
# the rule does that, and one that the BLAS libraries take. "ta" is a whole linear
# backward over K rows: grad_x and grad_w.
ROUTES = [("nn", 2195, 2168, 40, 1), ("nn", 730, 2948, 656, 1), ("nn", 1637, 1180, 956, 1), ("nn", 568, 2872, 40, 1),
          ("nn", 191, 2820, 352, 1), ("nn", 1059, 48, 60, 1), ("nn", 112, 2128, 1060, 1), ("nn", 577, 3252, 56, 1),
          ("nn", 92, 3020, 1284, 1), ("nn", 3, 216, 88, 1), ("nn", 4, 40, 1032, 1), ("nn", 98, 2724, 40, 1),
          ("nn", 79, 3172, 40, 1), ("nn", 700, 300, 1500, 0), ("nn", 77, 771, 768, 0),
          ("nt", 2610, 1896, 36, 1), ("nt", 1584, 1524, 768, 1), ("nt", 624, 3204, 1420, 1), ("nt", 610, 2476, 36, 1),
          ("nt", 126, 3488, 1680, 1), ("nt", 1221, 88, 48, 1), ("nt", 2314, 1708, 40, 1), ("nt", 4, 52, 100, 1),
          ("nt", 1, 36, 700, 1), ("nt", 322, 864, 44, 1), ("nt", 147, 1664, 36, 1), ("nt", 700, 308, 1500, 0),
          ("ta", 2164, 1252, 804, 2), ("ta", 636, 3264, 1875, 2), ("ta", 1504, 1048, 68, 2), ("ta", 1152, 1780, 748, 1),
          ("ta", 52, 472, 60, 2), ("ta", 2708, 644, 116, 2), ("ta", 302, 406, 1000, 0)]


@pytest.mark.parametrize("form,M,N,K,own", ROUTES)
def test_which_products_the_own_kernels_take(dev, form, M, N, K, own):
    """Sizes that no other test of the process calls, so that the count of shapes on the
    own kernels tells where each product ran."""
    import torch

    g = torch.Generator(device=dev).manual_seed(M + N + K)

    def rnd(*s):
        return torch.empty(s, device=dev).normal_(0.0, 1.0, generator=g)

    before = ops.gemm_info()
    if form == "ta":
        x, w, gy = rnd(K, M), rnd(M, N), rnd(K, N)
        gx, gw, gb = torch.empty((K, M), device=dev), torch.zeros((M, N), device=dev), torch.zeros(N, device=dev)
        ops.device_linear_backward(gx, gw, gb, gy, x, w, 1, K, M, N)
        assert rel(gx, gy.double() @ w.double().t()) < tol(N)
        assert rel(gw, x.double().t() @ gy.double()) < tol(K)
    else:
        x, w, b, y = rnd(M, K), rnd(K, N), torch.zeros(N, device=dev), torch.empty((M, N), device=dev)
        if form == "nn":
            ops.device_linear_activation_fused_forward(y, None, x, w, b, False, 1, M, K, N)
        else:
            ops.device_unembedding_forward(y, x, w.t().contiguous(), 1, M, K, N)
        assert rel(y, x.double() @ w.double()) < tol(K)
    after = ops.gemm_info()
    assert after["tuned"] - before["tuned"] == own
    assert after["plans"] - before["plans"] >= own


def test_gelu_keeps_32_bits(dev):
    """The GELU of the products' epilogue and its derivative over N(0, 3), against float64.
    One rounding of a result is 2.4e-8 in the 2-norm (0.41 of 2^-24): the GELU may be two
    of them off and the derivative, a sum of two terms, three. (exp and 1 - g with their
    full rounding came to 3.6e-7 in the derivative.) Then the ends of the range: GELU is x
    or nothing there, infinity included, its derivative 1 or 0."""
    import torch

    g = torch.Generator(device=dev).manual_seed(3)
    M, N = 16384, 4
    x = torch.empty((M, N), device=dev).normal_(0.0, 3.0, generator=g)
    ends = torch.tensor([0.0, 14.0, 1e15, 1e30, float("inf"), -14.0, -1e15, -1e30], device=dev)
    x[:2] = ends.view(2, 4)
    y, act, gx = (torch.empty((M, N), device=dev) for _ in range(3))
    ops.device_activation_backward(gx, torch.ones_like(x), x, 1, M, N)
    a = x[2:].double().requires_grad_(True)
    r = gelu64(a)
    d, = torch.autograd.grad(r.sum(), a)
    assert rel(gx[2:], d) < 7.3e-8
    assert gx[:2].view(-1)[[0, 1, 2, 5, 6]].tolist() == [0.5, 1.0, 1.0, 0.0, 0.0]
    w, b, zero = torch.eye(4, device=dev), torch.zeros(4, device=dev), torch.zeros((4, 4), device=dev)
    for v in ends.tolist():
        b[1] = v
        ops.device_linear_activation_fused_forward(y[:4], act[:4], zero, w, b, True, 1, 4, 4, 4)
        assert torch.equal(act[:4, 1], torch.clamp(y[:4, 1], min=0.0)) and torch.equal(y[:4, 1], b[1].expand(4))
    x = torch.empty((M, N), device=dev).normal_(0.0, 3.0, generator=g)
    ops.device_linear_activation_fused_forward(y, act, x, torch.eye(4, device=dev), torch.zeros(4, device=dev), True,
                                               1, M, 4, N)
    assert torch.equal(y, x)
    assert rel(act, gelu64(x.double())) < 4.9e-8
