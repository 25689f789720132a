"""Prompt attention over shared K / V blocks (k_fa_prefill_sh, launches of many tiles) against float64: head groups that do and
do not fill its four units, ragged last tiles, chunks after a past, no position limit, ggml masks (aligned or not, rows that
see nothing), fewer keys than the cache holds."""
import math

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _ref(q, k, v, see):
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    g = q.shape[1] // k.shape[0]
    for h in range(q.shape[1]):
        s = (q[:, h].half().double() @ k[h // g].double().T / 128 ** 0.5).masked_fill(~see, -math.inf)
        out[:, h] = torch.nan_to_num(s.softmax(-1)) @ v[h // g].double()
    return out


@pytest.mark.parametrize("heads,kv,n,pos0,kind", [
    (32, 8, 777, 0, "causal"), (64, 64, 380, 33, "causal"), (40, 8, 600, 1, "causal"), (16, 8, 1536, 7, "causal"),
    (32, 8, 800, 0, "open"), (32, 8, 500, 40, "mask"), (32, 8, 500, 41, "mask"), (32, 8, 513, 0, "holes")])
def test_shared_blocks(heads, kv, n, pos0, kind):
    from ameva_compute_amd import ops
    print(heads, kv, n, pos0, kind, flush=True)
    torch.manual_seed(n + pos0)
    keys = pos0 + n
    q = torch.randn(n, heads, 128, device="cuda")
    kc, vc = (torch.randn(keys + 5, kv, 128, device="cuda").half() for _ in "kv")
    k, v = kc.permute(1, 0, 2), vc.permute(1, 0, 2)
    at = torch.arange(n, device="cuda")[:, None] + pos0
    see = torch.arange(keys, device="cuda")[None, :] <= at if kind != "open" else torch.ones(n, keys, dtype=torch.bool, device="cuda")
    mask = None
    if kind in ("mask", "holes"):
        if kind == "holes":  # a query that sees nothing, blocks that a whole tile does not see
            see = see & (torch.rand(n, keys, device="cuda") < 0.5)
            see[3] = False
            see[64:96, :64] = False
        mask = torch.zeros(n, keys, dtype=torch.float16, device="cuda").masked_fill_(~see, -math.inf)
    y = ops.flash_attn_prefill(q, k, v, 128 ** -0.5, n_kv=keys, mask=mask, causal_pos0=pos0 if kind == "causal" else -1)
    r = _ref(q, k[:, :keys], v[:, :keys], see)
    # weights rounded to f16 (2^-11 at most each): the sum's relative error stays below that
    assert ((y - r).norm() / r.norm()).item() < 2.0 ** -11
    if kind == "holes":
        assert not y[3].any()
