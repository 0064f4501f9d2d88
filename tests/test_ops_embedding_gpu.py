"""Embedding gradients where a token's rows are many or far apart, against the
CPU oracle bit for bit: one id on every row, more rows than one list holds
(2048), a row count off every unrolled group, and a width of more than one
column range."""
import numpy as np
import pytest

from gpt_amd import ops
from oracle import pyops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,C,V,ids", [(1, 768, 10, 1), (37, 768, 40, 2), (2048, 12, 9, 1), (2049, 8, 70, 3),
                                          (5003, 36, 50, 7), (600, 1540, 20, 4), (300, 30, 11, 2)])
def test_embedding_backward_many_rows_per_token(dev, rows, C, V, ids):
    import torch

    r = np.random.default_rng(rows)
    tok = r.integers(0, ids, size=rows).astype(np.int32)
    gy, w0 = (r.standard_normal(s, dtype=np.float32) for s in ((rows, C), (V, C)))
    p0 = r.standard_normal((rows, C), dtype=np.float32)
    w, p = w0.copy(), p0.copy()
    pyops.embedding_backward(w, p, gy, tok, 1, rows, C)
    dw, dp, dg, dt = (torch.from_numpy(a).to(dev) for a in (w0, p0, gy, tok))
    ops.device_embedding_backward(dw, dp, dg, dt, 1, rows, C, vocab_rows=V)
    assert np.array_equal(dw.cpu().numpy().view(np.uint32), w.view(np.uint32))
    assert np.array_equal(dp.cpu().numpy().view(np.uint32), p.view(np.uint32))


@pytest.mark.parametrize("C", [36, 768, 1540, 30])
def test_embedding_backward_lists_between_empty_ones(dev, C):
    """Ids that hardly repeat: of an id's lists of 2048 rows the first, the last or some
    between are empty, and full groups of loads (12, then 4) end at, before and after
    a list's end."""
    import torch

    rows = 5 * 2048 + 77
    tok = np.arange(rows, dtype=np.int32)
    for id, at in enumerate(([0, 4096, 10316], [1, 2047, 2048, 8191], list(range(7, 7 + 2 * 11, 2)),
                             list(range(100, 112)), list(range(2040, 2053)), list(range(2 * 2048, 3 * 2048, 73)),
                             [9000] + list(range(9001, 9029)))):
        tok[at] = rows + id
    V = rows + 7
    r = np.random.default_rng(C)
    gy, w0 = (r.standard_normal(s, dtype=np.float32) for s in ((rows, C), (V, C)))
    p0 = np.zeros((rows, C), np.float32)
    w, p = w0.copy(), p0.copy()
    pyops.embedding_backward(w, p, gy, tok, 1, rows, C)
    dw, dp, dg, dt = (torch.from_numpy(a).to(dev) for a in (w0, p0, gy, tok))
    ops.device_embedding_backward(dw, dp, dg, dt, 1, rows, C, vocab_rows=V)
    assert np.array_equal(dw.cpu().numpy().view(np.uint32), w.view(np.uint32))
    assert np.array_equal(dp.cpu().numpy().view(np.uint32), p.view(np.uint32))


def test_embedding_backward_more_rows_than_one_grid_dimension(dev):
    """2^23 + 5 rows, a launch of two dimensions. All ids but the last are out of
    range, which adds nothing to grad_wte (and leaves one search of the rows)."""
    import torch

    rows, C = (1 << 23) + 5, 4
    gy = torch.empty((rows, C), device=dev).normal_(generator=torch.Generator(device=dev).manual_seed(5))
    tok = torch.full((rows,), 7, dtype=torch.int32, device=dev)
    tok[-1] = 1
    gw, gp = torch.ones((3, C), device=dev), torch.ones((rows, C), device=dev)
    ops.device_embedding_backward(gw, gp, gy, tok, 1, rows, C, vocab_rows=3)
    want = torch.ones((3, C), device=dev)
    want[1] += gy[-1]
    assert torch.equal(gw, want)
    assert torch.equal(gp, gy + 1)
