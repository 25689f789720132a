"""MUL_MAT of 2 to 8 tokens, where calls pass from a GEMV per token to one batched launch: every output against float64 over
the same quantized operands (the reference's per-output gate), with odd row counts, k in odd numbers of blocks and rows past
a 16-row tile."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
from parity import act_type_of, dequant_act, per_output_gate

pytestmark = pytest.mark.gpu
Q4_0, Q8_0, Q4_K, Q6_K = 2, 8, 12, 14


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ameva_compute_amd import ops
    return ops


@pytest.mark.parametrize("t", [Q4_0, Q8_0, Q4_K, Q6_K])
@pytest.mark.parametrize("n,k", [(2, 256), (34, 1024), (257, 512), (8208, 256), (48, 4352), (130, 288)])
def test_few_tokens(ops, orc, t, n, k):
    if t in (Q4_K, Q6_K) and k % 256:
        k = 512
    g = torch.Generator(device="cuda").manual_seed(n + k + t)
    x = torch.randn((n, k), generator=g, device="cuda")
    wb = (ops.quantize_q4_0(x) if t == Q4_0 else ops.quantize_act(x, Q8_0, ggml=True)[1] if t == Q8_0
          else ops.quantize_k(x, t))
    w = ops.QWeight.from_ggml(t, wb, n, k)
    w_deq = orc.dequantize(t, wb.cpu().numpy().reshape(n, -1), k)
    for m in range(2, 9):
        a = torch.randn((m, k), generator=g, device="cuda")
        blocks = ops.quantize_act(a, act_type_of(t), ggml=True)[1].cpu().numpy()
        per_output_gate(ops.mul_mat(w, a).cpu().numpy(), w_deq, dequant_act(blocks, act_type_of(t), k),
                        what=f"type {t} {n} x {k} m={m}")
