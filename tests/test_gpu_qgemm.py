"""The tiled int8 MUL_MAT (amv_qgemm.hip) above 32 tokens at the edges of its choices: 64 x 64, 64 x 128 and 128 x 128 tiles with
one, two or four groups of waves sharing k (some of them without blocks of their own), ragged rows and tokens, a last step of
one to three blocks: block integers against the oracle bit for bit, every output within the reference's per-output gate."""
import numpy as np
import pytest

from parity import dequant_act, per_output_gate

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# (rows, tokens): 64 x 64 four groups; 64 x 128 four (Q8_0: two); 64 x 128 two (Q4_K, Q4_0); 64 x 128 one (Q4_K); 128 x 128
TILES = [(1, 33), (63, 64), (65, 65), (129, 40), (8200, 100), (16500, 129), (14300, 270), (16500, 300)]


@pytest.mark.parametrize("n,m", TILES)
@pytest.mark.parametrize("wtype,k", [(2, 32), (2, 352), (8, 96), (8, 544), (12, 256), (12, 1280)])
def test_tiles(orc, n, m, wtype, k):
    from ameva_compute_amd import ops
    if n > 1000 and k > 600:
        k = 512 if wtype == 12 else k
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
    wd, ad = orc.dequantize(wtype, wg, k).reshape(n, k), dequant_act(ag, at, k)
    per_output_gate(y.cpu().numpy(), wd, ad, what=f"{wtype} {n} {k} {m}")
    e = torch.randn((m, n), device="cuda")
    assert torch.equal(ops.mul_mat_q_add(w, act, m, e, act_t=at), y + e)
