"""Prompt attention over shared K / V blocks at scores that are not the usual ones: a scale of 0 (every visible key weighs the
same) or next to it, a negative one."""
import math

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _ref(q, k, v, see, scale):
    """In 64 bits, from the f16 q."""
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    g = q.shape[1] // k.shape[0]
    for h in range(q.shape[1]):
        s = (q[:, h].half().double() @ k[h // g].double().T * scale).masked_fill(~see, -math.inf)
        out[:, h] = s.softmax(-1) @ v[h // g].double()
    return out


def _rel(y, r):
    return ((y - r).norm() / r.norm()).item()


@pytest.mark.parametrize("scale", [0.0, -0.0, 1e-45, -0.07])
@pytest.mark.parametrize("n,keys,kind", [(800, 800, "causal"), (800, 817, "open"), (520, 530, "mask")])
def test_scale_zero_and_below(scale, n, keys, kind):
    from ameva_compute_amd import ops
    print(scale, n, keys, kind, flush=True)
    torch.manual_seed(n)
    q = torch.randn(n, 32, 128, device="cuda")
    k, v = (torch.randn(8, keys, 128, device="cuda").half() for _ in "kv")
    limit = torch.arange(n, device="cuda")[:, None] + (0 if kind == "causal" else 9)
    see = torch.arange(keys, device="cuda")[None, :] <= limit
    if kind == "open":
        see = torch.ones_like(see)
    mask = torch.zeros(n, keys, dtype=torch.float16, device="cuda").masked_fill_(~see, -math.inf) if kind == "mask" else None
    y = ops.flash_attn_prefill(q, k, v, scale, n_kv=keys, mask=mask, causal_pos0=0 if kind == "causal" else -1)
    assert _rel(y, _ref(q, k, v, see, scale)) < 2.0 ** -11  # weights rounded to f16
