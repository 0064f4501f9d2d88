"""Attention for head sizes other than 64 (gpt_amd/csrc/attn_general.hip) at
the edges of its blocks, against dense float64: every padded head size and its
neighbours, lengths around multiples of 16 and of the 64 keys that four waves
take in a turn, one row, head sizes and pointers that only allow 4-byte loads,
and guard bands around every output.

Tolerance 2e-6 of the largest value (the interface asks 1e-5 forward and 1e-4
backward): sums of at most 400 terms of size one in fp32, whose error in any
order is below 400 x 2^-24 / 10 relative to the row's largest."""
import numpy as np
import pytest

import gpt_amd

pytestmark = pytest.mark.gpu

TOL = 2e-6


def run(dev, B, T, H, d, off=0, pad=64):
    import torch

    C = H * d
    g = torch.Generator(device=dev).manual_seed(B * 1000 + T + d)

    def buf(n, fill):
        t = torch.full((n + 2 * pad + off,), fill, device=dev)
        return t, t[pad + off:pad + off + n]

    _, x = buf(B * T * 3 * C, 0.0)
    x.normal_(generator=g)
    _, gy = buf(B * T * C, 0.0)
    gy.normal_(generator=g)
    outs = {k: buf(n, 777.0) for k, n in (("y", B * T * C), ("lse", B * T * H), ("gx", 3 * B * T * C), ("D", B * T * H))}
    v = {k: t[1] for k, t in outs.items()}
    gpt_amd.device_flash_attention_forward(v["y"], v["lse"], x, B, T, C, H)
    gpt_amd.device_flash_attention_backward(v["gx"], v["D"], v["lse"], gy, v["y"], x, B, T, C, H)
    first = v["gx"].clone()
    gpt_amd.device_flash_attention_backward(v["gx"], v["D"], v["lse"], gy, v["y"], x, B, T, C, H)
    torch.cuda.synchronize()
    assert torch.equal(first, v["gx"])
    for whole, part in outs.values():
        n = part.numel()
        assert torch.all(whole[:pad + off] == 777.0) and torch.all(whole[pad + off + n:] == 777.0)

    q, k, w = (t.double().reshape(B, T, H, d).transpose(1, 2) for t in x.reshape(B, T, 3, C).unbind(2))
    go = gy.double().reshape(B, T, H, d).transpose(1, 2)
    s = (q @ k.transpose(2, 3).contiguous()) / np.sqrt(d)
    s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=dev).triu(1), -np.inf)
    lse = torch.logsumexp(s, -1)
    p = torch.exp(s - lse[..., None])
    o = p @ w
    D = (go * o).sum(-1)
    ds = p * (go @ w.transpose(2, 3).contiguous() - D[..., None]) / np.sqrt(d)
    gx = torch.stack([ds @ k, ds.transpose(2, 3).contiguous() @ q, p.transpose(2, 3).contiguous() @ go])
    ref = {"y": o.transpose(1, 2), "lse": lse.transpose(1, 2), "D": D.transpose(1, 2), "gx": gx.permute(1, 3, 0, 2, 4)}
    for name, r in ref.items():
        r = r.reshape(-1)
        e = float((v[name].double() - r).abs().max() / max(float(r.abs().max()), 1e-3))
        assert e < TOL, (name, e)


@pytest.mark.parametrize("d", [1, 4, 8, 15, 16, 20, 32, 36, 48, 60, 65, 80, 96, 100, 128, 160, 192, 250, 256])
@pytest.mark.parametrize("T", [33, 130])
def test_head_sizes(dev, d, T):
    run(dev, 2, T, 3, d)


@pytest.mark.parametrize("T", [1, 15, 16, 17, 63, 64, 65, 256, 400])
@pytest.mark.parametrize("d", [32, 128])
def test_lengths(dev, T, d):
    run(dev, 1, T, 5, d)


@pytest.mark.parametrize("d", [64, 128])
def test_misaligned_pointers(dev, d):
    run(dev, 2, 70, 2, d, off=1)


def pairs64(x, gy, T, d):
    """y, dq, dk, dv and lse of one head in float64, every query over its own keys
    alone, so that no value meets a masked one."""
    q, k, v = x.double().unbind(1)
    g, sc = gy.double(), d ** -0.5
    y, dq, dk, dv = (np.zeros((T, d)) for _ in range(4))
    lse = np.zeros(T)
    q, k, v, g = (t.cpu().numpy() for t in (q, k, v, g))
    with np.errstate(all="ignore"):
        for i in range(T):
            s = (k[:i + 1] * q[i]).sum(1) * sc
            m = np.nanmax(s) if np.isfinite(s).any() else 0.0
            e = np.exp(s - m)
            p = e / e.sum()
            lse[i] = m + np.log(e.sum())
            y[i] = (p[:, None] * v[:i + 1]).sum(0)
            ds = p * ((v[:i + 1] * g[i]).sum(1) - (y[i] * g[i]).sum()) * sc
            dq[i] = (ds[:, None] * k[:i + 1]).sum(0)
            dk[:i + 1] += ds[:, None] * q[i]
            dv[:i + 1] += p[:, None] * g[i]
    return {"y": y, "lse": lse, "dq": dq, "dk": dk, "dv": dv}


@pytest.mark.parametrize("d", [16, 20, 33, 128, 250])
@pytest.mark.parametrize("what", ["k", "v", "q", "g", "low"])
@pytest.mark.parametrize("row", [5, 20, 37])
def test_non_finite_values_stay_with_their_pairs(dev, d, what, row):
    """An infinity or NaN reaches the rows that causality gives it and no others of
    their 16-row blocks; scores of -infinity (low) weigh nothing."""
    import torch

    T, H = 40, 2
    C = H * d
    g = torch.Generator(device=dev).manual_seed(d + row)
    x = torch.empty((1, T, 3, H, d), device=dev).normal_(generator=g)
    gy = torch.empty((1, T, H, d), device=dev).normal_(generator=g)
    if what == "g":
        gy[0, row, 1, 1] = np.nan
    elif what == "low":
        x[0, :, 0, 1, 0], x[0, :, 1, 1, 0] = 1e25, 0.0
        x[0, 16:32, 1, 1, 0] = x[0, row + 1, 1, 1, 0] = -1e25
    else:
        x[0, row, "qkv".index(what), 1, 1] = np.inf if what == "v" else np.nan
    y, lse, gx, D = (torch.empty(s, device=dev) for s in ((1, T, C), (1, T, H), (1, T, 3 * C), (1, T, H)))
    gpt_amd.device_flash_attention_forward(y, lse, x, 1, T, C, H)
    gpt_amd.device_flash_attention_backward(gx, D, lse, gy, y, x, 1, T, C, H)
    for h in range(H):
        r = pairs64(x[0, :, :, h], gy[0, :, h], T, d)
        o = gx.view(T, 3, H, d)[:, :, h]
        a = {"y": y.view(T, H, d)[:, h], "lse": lse.view(T, H)[:, h], "dq": o[:, 0], "dk": o[:, 1], "dv": o[:, 2]}
        for name, t in a.items():
            t, e = t.double().cpu().numpy(), r[name]
            ok = np.isfinite(e)
            assert np.array_equal(np.isfinite(t), ok), (name, h)
            if ok.any():
                assert np.abs(t[ok] - e[ok]).max() <= TOL * max(np.abs(e[ok]).max(), 1e-3), (name, h)


def test_rows_beyond_buffer_offsets_and_one_grid_dimension(dev):
    """16 rows of 400 MB each are past a buffer range's 31-bit offsets, and one
    workgroup per head is more than a launch dimension takes."""
    run(dev, 1, 2, (1 << 23) + 3, 4)
