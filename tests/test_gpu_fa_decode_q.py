"""Decode attention over Q8_0 / Q4_0 caches at the edges of its key tiles (a wave owns 16 or 32 keys, a workgroup 4
waves): one key, one past a chunk, a wave and a split, and the 32-key form that n_kv * n_head_kv > 65536 selects; every
GQA group; a key count below the launch's n_kv_max, with rows past it that hold NaN scales.

Reference: float64 softmax over q quantized to Q8_0 by the oracle and dequantized K and V. The block integers are exact on
both sides; a score is 4 products and 3 sums in f32, a relative error of at most 8 * 2^-24 of sum |t_b| < 64 here (scale
1 / sqrt(128), |q k| blocks of normal data), so a probability is off by at most 3.1e-5 relative at worst and about 1e-6 in
the mean; the P V sums add f32 rounding of the same order: 1e-5 relative L2."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

Q8_0, Q4_0 = 8, 2


@pytest.mark.parametrize("t", [Q8_0, Q4_0])
@pytest.mark.parametrize("G,n_head_kv,n_kv,n_max", [
    (1, 3, 1, 1), (2, 1, 17, 40), (4, 2, 65, 65), (8, 2, 64, 300), (4, 8, 129, 129), (1, 2, 1000, 1003),
    (4, 8, 8221, 8221), (8, 8, 8193, 9000), (2, 16, 4127, 4130), (1, 33, 2047, 2047)])
def test_decode_quantized_key_tiles(orc, t, G, n_head_kv, n_kv, n_max):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ameva_compute_amd import ops
    dev, D = torch.device("cuda:0"), 128
    rng = np.random.default_rng(n_kv + G)
    quant = (lambda x: orc.quantize_q8_0(x, 0)) if t == Q8_0 else orc.quantize_q4_0
    n_head = n_head_kv * G
    cache, deq = [], []
    for _ in range(2):
        b = quant(rng.standard_normal((n_max * n_head_kv, D)).astype(np.float32))
        deq.append(orc.dequantize(t, b, D).reshape(n_max, n_head_kv, D).astype(np.float64)[:n_kv])
        b = b.reshape(n_max, n_head_kv, -1).copy()
        b[n_kv:] = 0xFF  # f16 NaN scales
        cache.append(torch.from_numpy(b).to(dev).permute(1, 0, 2))
    q = rng.standard_normal((n_head, D)).astype(np.float32)
    q64 = orc.dequantize(Q8_0, orc.quantize_q8_0(q, 0), D).reshape(n_head_kv, G, D).astype(np.float64)
    s = np.einsum("hgd,khd->hgk", q64, deq[0]) / D ** 0.5
    p = np.exp(s - s.max(-1, keepdims=True))
    want = (np.einsum("hgk,khd->hgd", p, deq[1]) / p.sum(-1, keepdims=True)).reshape(n_head, D)
    nkv = torch.tensor([n_kv], dtype=torch.int32, device=dev)
    for one in (False, True):
        got = ops.flash_attn_decode_kv(torch.from_numpy(q).to(dev), cache[0], cache[1], t, 1 / D ** 0.5, n_kv_max=n_max,
                                       n_kv_dev=nkv, one_launch=one).cpu().numpy().astype(np.float64).reshape(n_head, D)
        assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)
