"""Batched products whose operands are followed by 0xFF bytes (NaN scales, digits of -1): what lies behind an activation or a
weight never reaches a product, where the last step has fewer blocks than the four a step holds and where wave groups sharing k have no
blocks at all."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _framed(t):
    """t's bytes in a buffer that goes on with 64 KB of 0xFF."""
    b = torch.full((t.numel() + (1 << 16),), 0xFF, dtype=torch.uint8, device="cuda")
    b[:t.numel()] = t
    return b[:t.numel()]


def _weight(ops, wtype, n, k):
    w = torch.randn((n, k), device="cuda") * 0.02
    return ops.QWeight.from_ggml(wtype, ops.quantize_q4_0(w) if wtype == ops.Q4_0
                                 else ops.quantize_act(w, ops.Q8_0, ggml=True)[1], n, k)


@pytest.mark.parametrize("wtype", ["Q4_0", "Q8_0"])
@pytest.mark.parametrize("n,k,m", [(1, 32, 33), (1, 96, 65), (3, 160, 40), (65, 416, 129), (8200, 32, 100),
                                   (12415, 224, 500)])
def test_int8(wtype, n, k, m):
    from ameva_compute_amd import ops
    print(wtype, n, k, m, flush=True)
    torch.manual_seed(n + k + m)
    w = _weight(ops, getattr(ops, wtype), n, k)
    act = ops.quantize_act(torch.randn((m, k), device="cuda"), ops.Q8_0)[0]
    want = ops.mul_mat_q(w, act, m, act_t=ops.Q8_0)
    assert bool(want.isfinite().all())
    w.data = _framed(w.data)
    assert torch.equal(ops.mul_mat_q(w, _framed(act), m, act_t=ops.Q8_0), want)
