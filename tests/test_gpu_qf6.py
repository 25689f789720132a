"""The activation type AMV_ACT_Q8_0_F6 is accepted as the plain Q8_0 layout: the same bytes, block integers (against the oracle,
bit for bit) and outputs, at the edges of the tiled kernels' tiles and where k is split."""
import numpy as np
import pytest
import torch

import oracle
from ameva_compute_amd import ops
from ameva_compute_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def _case(n, k, m, seed):
    rng = np.random.default_rng(seed)
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    x = (rng.standard_normal((m, k)) * rng.uniform(0.01, 30, (m, 1))).astype(np.float32)
    wg = ops.quantize_q4_0(torch.from_numpy(w).cuda())
    return ops.QWeight.from_ggml(ops.Q4_0, wg, n, k), wg, torch.from_numpy(x).cuda()


# (rows, k, tokens, exact): exact where all of k is summed in one order
@pytest.mark.parametrize("n,k,m,exact", [
    (128, 32, 65, True), (1025, 512, 257, True), (12416, 256, 512, True), (12415, 224, 500, True), (12290, 32, 511, True),
    (49100, 96, 65, True), (3072, 7200, 500, False)])
def test_f6_against_int8(n, k, m, exact):
    w, _, x = _case(n, k, m, n + k + m)
    print(n, k, m, flush=True)
    a0, _ = ops.quantize_act(x, ops.Q8_0)
    a1, _ = ops.quantize_act(x, ops.Q8_0_F6)
    assert torch.equal(a1[:a0.numel()], a0)
    y0, y1 = (ops.mul_mat_q(w, a, m, act_t=t) for a, t in ((a0, ops.Q8_0), (a1, ops.Q8_0_F6)))
    e = torch.randn(m, n, device="cuda")
    z1 = ops.mul_mat_q_add(w, a1, m, e, act_t=ops.Q8_0_F6)
    assert torch.equal(z1, y1 + e)
    if exact:
        assert torch.equal(y0, y1)
    else:  # sum |w a| is below |row| |column|
        bound = 2 * (k / 32) * 2.0 ** -24 * torch.outer(x.norm(dim=1), torch.full((n,), 0.03 * k ** 0.5, device="cuda"))
        assert bool(((y0 - y1).abs() <= bound).all())


@pytest.mark.parametrize("n,k,m", [(131, 96, 70), (12300, 96, 490)])
def test_f6_block_sums(n, k, m):
    w, wg, x = _case(n, k, m, n * 3 + m)
    x[0, :32] = 127.0  # the largest digits
    x[1, :32] = -127.0
    act, ag = ops.quantize_act(x, ops.Q8_0_F6, ggml=True)
    out = torch.empty((m, n, k // 32), dtype=torch.int32, device="cuda")
    check(lib().amv_mul_mat_q_act_block_sums(ops.Q4_0, w.data.data_ptr(), n, k, act.data_ptr(), ops.Q8_0_F6, m,
                                             out.data_ptr(), torch.cuda.current_stream().cuda_stream), "block sums")
    _, ref = oracle.mul_mat(oracle.Q4_0, wg.cpu().numpy(), n, k, ag.cpu().numpy(), m, with_blocks=True)
    assert np.array_equal(out.cpu().numpy(), ref)


def test_f6_is_plain_elsewhere():
    """Up to 64 tokens, and for Q8_0 weights."""
    w, _, x = _case(256, 512, 40, 5)
    a0, a1 = (ops.quantize_act(x, t)[0] for t in (ops.Q8_0, ops.Q8_0_F6))
    assert torch.equal(ops.mul_mat_q(w, a0, 40, act_t=ops.Q8_0), ops.mul_mat_q(w, a1, 40, act_t=ops.Q8_0_F6))
    w8 = ops.QWeight.from_ggml(ops.Q8_0, ops.quantize_act(torch.randn(64, 512, device="cuda"), ops.Q8_0, ggml=True)[1],
                               64, 512)
    x = torch.randn(80, 512, device="cuda")
    a0, a1 = (ops.quantize_act(x, t)[0] for t in (ops.Q8_0, ops.Q8_0_F6))
    assert torch.equal(ops.mul_mat_q(w8, a0, 80, act_t=ops.Q8_0), ops.mul_mat_q(w8, a1, 80, act_t=ops.Q8_0_F6))
