"""I2_S of 3 to 8 tokens, where calls pass from a GEMV per token to the batched kernel, and the activation quantizer's row
lengths (rows held in registers, the rest of a longer row, rows that are not 16-byte aligned), bit for bit against the
oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
from test_gpu_ops import pack_i2s

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,off", [(130, 2560, 0), (67, 128, 1), (5, 3072, 0), (64, 3200, 2), (33, 8192, 0),
                                     (40, 8320, 0), (16, 17024, 3)])
def test_i2s_few_tokens(orc, n, k, off):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ameva_compute_amd import ops
    rng = np.random.default_rng(n + k)
    w = pack_i2s(rng.integers(0, 3, (n, k)))
    wd = torch.from_numpy(w.reshape(-1).copy()).cuda()
    for m in range(3, 9):
        x = rng.standard_normal((m, k)).astype(np.float32)
        q_ref, deq_ref = orc.i2s_quantize_act(x)
        out_ref, _ = orc.i2s_gemv(w, n, k, q_ref, deq_ref, 1.37)
        buf = torch.zeros(m * k + off, device="cuda")
        buf[off:] = torch.from_numpy(x.reshape(-1)).cuda()
        act = ops.i2s_quantize_act(buf[off:].view(m, k))
        a = act.cpu().numpy()
        meta = a[m * k:].view(np.int32).reshape(m, 2)
        assert np.array_equal(a[:m * k].view(np.int8).reshape(m, k), q_ref)
        assert np.array_equal(meta[:, 0].view(np.float32), deq_ref)
        assert np.array_equal(meta[:, 1], q_ref.astype(np.int32).sum(axis=1))
        assert np.array_equal(ops.i2s_gemv(wd, n, k, act, m, 1.37).cpu().numpy(), out_ref.reshape(m, n))
