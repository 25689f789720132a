"""MUL_MAT of 3 to 7 tokens where the rows are long: a GEMV per token while that is faster than one launch's chain along k, bit
for bit each token by itself, and one launch elsewhere; every output against float64 over the same quantized operands (the
reference's per-output gate) on both sides of the line."""
import pytest

torch = pytest.importorskip("torch")
from parity import act_type_of, dequant_act, per_output_gate

pytestmark = pytest.mark.gpu
Q4_0, Q8_0, Q4_K, Q6_K = 2, 8, 12, 14


# per_token: the counts of tokens that take a GEMV each
@pytest.mark.parametrize("t,n,k,per_token", [
    (Q4_0, 64, 14336, (3, 4)), (Q8_0, 64, 14336, range(3, 8)), (Q4_K, 64, 14336, range(3, 6)), (Q6_K, 64, 14336, (3, 4, 5)),
    (Q4_0, 17, 8224, range(3, 7)), (Q8_0, 16, 8224, range(3, 7)), (Q8_0, 2048, 4096, ()), (Q4_K, 1024, 4096, ()),
    (Q6_K, 2048, 8192, ()), (Q4_0, 1024, 8192, ())])
def test_long_rows(orc, t, n, k, per_token):
    from ameva_compute_amd import ops
    print(t, n, k, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + k + t)
    x = torch.randn((n, k), generator=g, device="cuda")
    wb = (ops.quantize_q4_0(x) if t == Q4_0 else ops.quantize_act(x, Q8_0, ggml=True)[1] if t == Q8_0
          else ops.quantize_k(x, t))
    w = ops.QWeight.from_ggml(t, wb, n, k)
    w_deq = orc.dequantize(t, wb.cpu().numpy().reshape(n, -1), k)
    for m in range(3, 8):
        a = torch.randn((m, k), generator=g, device="cuda")
        y = ops.mul_mat(w, a)
        blocks = ops.quantize_act(a, act_type_of(t), ggml=True)[1].cpu().numpy()
        per_output_gate(y.cpu().numpy(), w_deq, dequant_act(blocks, act_type_of(t), k), what=f"type {t} {n} x {k} m={m}")
        if m in per_token:
            assert torch.equal(y, torch.cat([ops.mul_mat(w, a[i:i + 1]) for i in range(m)])), m
