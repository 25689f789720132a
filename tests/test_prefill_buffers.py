"""A captured prefill keeps its buffers: prompts of another length, with another activation layout, use a set of their own.
In a model, layers whose weight types take other layouts have sets of their own, all with the prompt's positions."""
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


@pytest.mark.parametrize("wtype", [ops.Q4_0, ops.Q8_0, ops.Q4_K, ops.Q6_K])
def test_short_prompt_keeps_its_buffers_through_a_long_one(wtype):
    lay = types.SimpleNamespace(H=256, FF=512, attn_norm=torch.empty(1), wqkv=types.SimpleNamespace(type=wtype, n_rows=384),
                                wgu=types.SimpleNamespace(n_rows=1024))
    short = llama.LlamaLayer._prefill_buffers(lay, 20)
    long = llama.LlamaLayer._prefill_buffers(lay, 300)
    assert llama.LlamaLayer._prefill_buffers(lay, 20) is short and llama.LlamaLayer._prefill_buffers(lay, 300) is long


@pytest.mark.parametrize("wtypes,n", [((ops.Q4_0, ops.Q8_0), 100), ((ops.Q4_K, ops.Q6_K), 5), ((ops.Q4_K, ops.Q6_K), 20),
                                     ((ops.Q4_K, ops.Q6_K, ops.Q4_K), 40), ((ops.Q8_0, ops.Q4_0, ops.Q8_0), 3)])
def test_model_positions_reach_every_layer(wtypes, n):
    """Layers of other weight types may take other activation layouts: each has the prompt's positions, layers of one layout
    share a set, and an older prompt's positions are replaced."""
    from ameva_compute_amd.model import LlamaModel

    class Layer(llama.LlamaLayer):
        def __init__(self, t):
            self.H, self.FF, self.attn_norm = 256, 512, torch.empty(1)
            self.wqkv, self.wgu = types.SimpleNamespace(type=t, n_rows=384), types.SimpleNamespace(n_rows=1024)

    model = LlamaModel.__new__(LlamaModel)
    model.layers = [Layer(t) for t in wtypes]
    for lay in model.layers:
        lay.set_prefill_position(50, n)
    for m in (n, 200, n):
        model._prompt_buffers(m)
        for lay in model.layers:
            b = lay._prefill_buffers(lay.pf_n)  # what the layer's prefill takes
            assert (lay.pf_pos0, lay.pf_n) == (0, m) and b["at"] == ops.gemm_act_type(lay.wqkv.type, m)
            assert torch.equal(b["pos"][:m], torch.arange(m, dtype=torch.int32))
            assert torch.equal(b["idx"][:m], torch.arange(m))
        for a in model.layers:
            for b in model.layers:
                same = ops.gemm_act_type(a.wqkv.type, m) == ops.gemm_act_type(b.wqkv.type, m)
                assert (a._pf is b._pf) == same
