"""AdamW and gradient clipping at the sizes where their launches change: the
last partial workgroup, lengths that only allow 4-byte accesses, the size from
which the streams take the non-temporal hint (8 Mi elements), and clipping that
leaves the gradient alone (accum 1, norm below the limit), against the CPU oracle
and float64."""
import numpy as np
import pytest

from gpt_amd import ops
from oracle import pyops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 4, 1023, 1024, 4100, (8 << 20) - 4, 8 << 20, (8 << 20) + 1, 10000004])
def test_adamw_sizes(dev, n):
    """Bit for bit against the CPU oracle; nothing past n is touched."""
    import torch

    r = np.random.default_rng(n)
    p, g, m, v = (r.standard_normal(n, dtype=np.float32) * np.float32(s) for s in (0.02, 1e-3, 1e-4, 1e-3))
    v *= v
    d = [torch.from_numpy(np.concatenate([a, np.full(8, 7, np.float32)])).to(dev) for a in (p, g, m, v)]
    ops.device_adamw_step(*d, n, 3e-4, 0.9, 0.999, 1e-8, 0.1, 3)
    pyops.adamw(p, g, m, v, n, 3e-4, 0.9, 0.999, 1e-8, 0.1, 3)
    for t, a in zip(d, (p, g, m, v)):
        t = t.cpu().numpy()
        assert np.array_equal(t[:n].view(np.uint32), a.view(np.uint32))
        assert np.all(t[n:] == 7)


@pytest.mark.parametrize("n", [3, 4096, 1024 * 1024 + 4, 9000001, (1 << 24) + 1])
@pytest.mark.parametrize("max_norm,accum", [(1e9, 1), (0.5, 1), (1e9, 3), (0.5, 3)])
def test_clip(dev, n, max_norm, accum):
    import torch

    g = torch.Generator(device=dev).manual_seed(n)
    x = torch.empty(n + 4, device=dev).normal_(0, 1, generator=g)
    before = x.clone()
    ops.device_scale_and_clip_grad(x, n, max_norm, accum)
    e = before[:n].double() / accum
    norm = float(e.norm())
    if norm > max_norm:
        e = e * (max_norm / (norm + 1e-6))
    elif accum == 1:
        assert torch.equal(x, before)
    # division, the norm's sum (1e-7), the factor and the product
    assert float(((x[:n].double() - e).abs() / e.abs().clamp_min(1e-30)).max()) < 6e-7
    assert torch.equal(x[n:], before[n:])
