"""I2_S of 3 to 8 tokens with few long rows (a GEMV per token or one batched launch, by rows, k and tokens), and the activation
quantizer's shortest rows (up to 1024 elements in one load, just past it), bit for bit against the oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
from test_gpu_ops import pack_i2s

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(320, 17024), (64, 6912), (2560, 1024), (65, 128), (40, 640), (33, 1152)])
def test_i2s_long_rows(orc, n, k):
    from ameva_compute_amd import ops
    print(n, k, flush=True)
    rng = np.random.default_rng(n + k)
    w = pack_i2s(rng.integers(0, 3, (n, k)))
    wd = torch.from_numpy(w.reshape(-1).copy()).cuda()
    for m in range(3, 9):
        x = rng.standard_normal((m, k)).astype(np.float32)
        q_ref, deq_ref = orc.i2s_quantize_act(x)
        out_ref, _ = orc.i2s_gemv(w, n, k, q_ref, deq_ref, 0.7)
        act = ops.i2s_quantize_act(torch.from_numpy(x).cuda())
        a = act.cpu().numpy()
        meta = a[m * k:].view(np.int32).reshape(m, 2)
        assert np.array_equal(a[:m * k].view(np.int8).reshape(m, k), q_ref)
        assert np.array_equal(meta[:, 0].view(np.float32), deq_ref)
        assert np.array_equal(ops.i2s_gemv(wd, n, k, act, m, 0.7).cpu().numpy(), out_ref.reshape(m, n))
