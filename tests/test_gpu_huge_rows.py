"""MUL_MAT of 33 to 64 tokens with rows of 2^25 elements, where a tile's bytes pass 32-bit offsets: the product of short rows
repeated is that of the short rows times the repetitions."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,n,m", [("Q8_0", 130, 33), ("Q4_0", 2, 64), ("Q4_K", 3, 40)])
def test_huge_rows(orc, t, n, m):
    from ameva_compute_amd import ops
    from parity import act_type_of, dequant_act
    print(t, n, m, flush=True)
    t, k0, rep = getattr(ops, t), 4096, 8192
    k = k0 * rep
    torch.manual_seed(t)
    w0, x0 = torch.randn((n, k0), device="cuda"), torch.randn((m, k0), device="cuda")
    wb = (ops.quantize_q4_0(w0) if t == ops.Q4_0 else ops.quantize_act(w0, ops.Q8_0, ggml=True)[1] if t == ops.Q8_0
          else ops.quantize_k(w0, t)).reshape(n, -1)
    w = ops.QWeight.from_ggml(t, wb.repeat(1, rep), n, k)
    at = ops.Q8_K_MMA if t == ops.Q4_K else ops.Q8_0
    act = ops.quantize_act(x0.repeat(1, rep), at)[0]
    y = ops.mul_mat_q(w, act, m, act_t=at)
    e = torch.randn_like(y)
    assert torch.equal(ops.mul_mat_q_add(w, act, m, e, act_t=at), y + e)
    del act
    wd = torch.from_numpy(orc.dequantize(t, wb.cpu().numpy(), k0).reshape(n, k0)).double()
    blocks = ops.quantize_act(x0, act_type_of(t), ggml=True)[1].cpu().numpy()
    ad = torch.from_numpy(dequant_act(blocks, act_type_of(t), k0).reshape(m, k0)).double()
    # the reference's per-output gate: 1e-5 of the sum of magnitudes
    assert bool(((y.cpu().double() - rep * (ad @ wd.T)).abs() <= 1e-5 * rep * (ad.abs() @ wd.abs().T)).all())
    torch.cuda.empty_cache()
