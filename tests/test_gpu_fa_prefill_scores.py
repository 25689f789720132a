"""Prompt attention over shared K / V blocks at scores that are not the usual ones: a scale of 0 (every visible key weighs the
same) or next to it, a negative one; one key that outweighs all others; scores so far apart that f32 rounds them to whole
numbers."""
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


@pytest.mark.parametrize("above,sinks", [(8, 1), (11, 16), (14, 1)])
@pytest.mark.parametrize("kind", ["causal", "mask"])
def test_dominating_first_keys(above, sinks, kind):
    """Keys that draw most of every query's weight and hold no value: what is left of the others' weights is the result."""
    from ameva_compute_amd import ops
    n = 1024
    torch.manual_seed(above)
    q, k = torch.randn(n, 32, 128, device="cuda"), torch.randn(8, n, 128, device="cuda")
    v = torch.randn(8, n, 128, device="cuda").half()
    q[..., 0], k[..., 0], k[:, :sinks], v[:, :sinks] = 4.0, 0.0, 0.0, 0.0
    k[:, :sinks, 0] = above * 128 ** 0.5 / 4
    k = k.half()
    see = torch.tril(torch.ones(n, n, dtype=torch.bool, device="cuda"))
    mask = torch.zeros(n, n, dtype=torch.float16, device="cuda").masked_fill_(~see, -math.inf) if kind == "mask" else None
    y = ops.flash_attn_prefill(q, k, v, 128 ** -0.5, n_kv=n, mask=mask, causal_pos0=0 if kind == "causal" else -1)
    r = _ref(q, k, v, see, 128 ** -0.5)
    # the others' weights, 2^(-1.44 (above + 4)) and more of the largest, rounded to f16 in full: 2^-11 at most each
    assert _rel(y[sinks:], r[sinks:]) < 2.0 ** -11


@pytest.mark.parametrize("size", [3000.0, 20000.0])
@pytest.mark.parametrize("kind", ["causal", "mask"])
def test_huge_scores(size, kind):
    """q and k near the end of f16's range: scores of 2^24 to 2^30, where the nearest f32 numbers are up to 64 apart and all
    of a query's weight is on one key."""
    from ameva_compute_amd import ops
    n = 900
    torch.manual_seed(int(size))
    q, k = ((torch.randn(s, device="cuda") * size).clamp(-65000, 65000) for s in ((n, 32, 128), (8, n, 128)))
    k, v = k.half(), torch.randn(8, n, 128, device="cuda").half()
    see = torch.tril(torch.ones(n, n, dtype=torch.bool, device="cuda"))
    mask = torch.zeros(n, n, dtype=torch.float16, device="cuda").masked_fill_(~see, -math.inf) if kind == "mask" else None
    y = ops.flash_attn_prefill(q, k, v, 128 ** -0.5, n_kv=n, mask=mask, causal_pos0=0 if kind == "causal" else -1)
    r = _ref(q, k, v, see, 128 ** -0.5)
    assert bool(y.isfinite().all())
    # two keys whose scores f32 cannot tell apart (about one query in a thousand at the larger size) share the weight
    near = ((y - r).norm(dim=-1) < 2.0 ** -10 * r.norm(dim=-1)).float().mean().item()
    assert near > 0.99
