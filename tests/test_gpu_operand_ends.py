"""Batched products whose operands are followed by 0xFF bytes (NaN scales, digits of -1): what lies behind an activation or a
weight never reaches a product, where the last step has fewer blocks than a step holds (an odd number of 32-blocks for the
6-bit kernel, a number that 4 does not divide for the int8 one) and where wave groups sharing k have no blocks at all."""
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


# at least 384 tiles of 128 x 128, so that the 6-bit kernel takes them; 1, 3 and 7 blocks of k, tokens past one token tile
@pytest.mark.parametrize("n,k,m", [(24500, 32, 200), (12290, 96, 490), (12415, 224, 500)])
def test_f6(n, k, m):
    from ameva_compute_amd import ops
    from ameva_compute_amd._lib import check, lib
    print(n, k, m, flush=True)
    torch.manual_seed(k)
    w = _weight(ops, ops.Q4_0, n, k)
    x = torch.randn((m, k), device="cuda")
    want = ops.mul_mat_q(w, ops.quantize_act(x, ops.Q8_0)[0], m, act_t=ops.Q8_0)
    act = _framed(ops.quantize_act(x, ops.Q8_0_F6)[0])
    w.data = _framed(w.data)
    assert torch.equal(ops.mul_mat_q(w, act, m, act_t=ops.Q8_0_F6), want)
    sums = [torch.empty((m, n, k // 32), dtype=torch.int32, device="cuda") for _ in "ab"]
    for s, at in zip(sums, (ops.Q8_0, ops.Q8_0_F6)):
        check(lib().amv_mul_mat_q_act_block_sums(ops.Q4_0, w.data.data_ptr(), n, k, act.data_ptr(), at, m, s.data_ptr(),
                                                 torch.cuda.current_stream().cuda_stream), "block sums")
    assert torch.equal(*sums)


@pytest.mark.parametrize("wtype", ["Q4_0", "Q8_0"])
@pytest.mark.parametrize("n,k,m", [(1, 32, 33), (1, 96, 65), (3, 160, 40), (65, 416, 129), (8200, 32, 100)])
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
