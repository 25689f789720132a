"""The tiled int8 MUL_MAT above 32 tokens with k of one to four steps, where fewer groups of waves share it: block integers
against the oracle bit for bit, every output within the reference's per-output gate."""
import numpy as np
import pytest

from parity import dequant_act, per_output_gate

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(65, 40), (8200, 100), (16500, 129)])  # 64 x 64 tiles, 64 x 128, 64 x 128 with more of them
@pytest.mark.parametrize("wtype,k", [(2, 64), (2, 128), (2, 256), (2, 288), (8, 32), (8, 160), (8, 256), (8, 384), (12, 256),
                                     (12, 512), (12, 768)])
def test_short_k(orc, n, m, wtype, k):
    from ameva_compute_amd import ops
    print(wtype, n, k, m, flush=True)
    rng = np.random.default_rng(n + m + k + wtype)
    wf = torch.from_numpy((rng.standard_normal((n, k)) * 0.02).astype(np.float32)).cuda()
    wg = (ops.quantize_q4_0(wf) if wtype == 2 else ops.quantize_act(wf, ops.Q8_0, ggml=True)[1] if wtype == 8
          else ops.quantize_k(wf, wtype))
    at = ops.Q8_K if wtype == 12 else ops.Q8_0
    act, ag = ops.quantize_act(torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).cuda(), at, ggml=True)
    w = ops.QWeight.from_ggml(wtype, wg, n, k)
    wg, ag = wg.cpu().numpy(), ag.cpu().numpy()
    _, ref = orc.mul_mat(wtype, wg, n, k, ag, m, with_blocks=True)
    assert np.array_equal(ops.block_sums(w, act, m, kernel="mmq").cpu().numpy().reshape(ref.shape), ref)
    y = ops.mul_mat_q(w, act, m, act_t=at)
    per_output_gate(y.cpu().numpy(), orc.dequantize(wtype, wg, k).reshape(n, k), dequant_act(ag, at, k),
                    what=f"{wtype} {n} {k} {m}")
    e = torch.randn((m, n), device="cuda")
    assert torch.equal(ops.mul_mat_q_add(w, act, m, e, act_t=at), y + e)
