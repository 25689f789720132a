"""A captured prefill keeps its buffers: prompts of another length, with another activation layout, use a set of their own."""
import types

import pytest

torch = pytest.importorskip("torch")
from ameva_compute_amd import llama, ops


@pytest.mark.parametrize("wtype", [ops.Q4_0, ops.Q4_K])
def test_prefill_buffers_kept_per_layout(wtype):
    lay = types.SimpleNamespace(H=256, FF=512, attn_norm=torch.empty(1), wqkv=types.SimpleNamespace(type=wtype, n_rows=384),
                                wgu=types.SimpleNamespace(n_rows=1024))
    first = {n: llama.LlamaLayer._prefill_buffers(lay, n) for n in (512, 32, 5)}
    for n, b in first.items():
        at = ops.gemm_act_type(wtype, n)
        assert b["at"] == at and b["n"] >= n
        assert b["act_h"].numel() >= ops.lib().amv_act_bytes(at, n, lay.H)
        assert llama.LlamaLayer._prefill_buffers(lay, n) is b
