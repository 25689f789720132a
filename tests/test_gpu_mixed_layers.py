"""A model whose layers hold weights of different types, so that a prompt's layers take different activation layouts: cache rows
and logits of prompts of several lengths equal, bit for bit, those of the same layers run one by one at positions of their
own."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pair,lengths", [(("Q4_0", "Q8_0"), (100, 5, 70)), (("Q4_K", "Q6_K"), (5, 20, 40, 100)),
                                          (("Q8_0", "Q4_0"), (130, 3))])
def test_mixed_layers(pair, lengths):
    from ameva_compute_amd import llama, model, ops
    dev = torch.device("cuda:0")
    dims = dict(H=256, n_head=2, n_head_kv=1, D=128, FF=512, ctx=256)

    def layers():
        out = []
        for i, t in enumerate((*pair, pair[0])):
            t = getattr(ops, t)
            if t == ops.Q8_0:  # random_layer makes the other types
                lay = llama.random_layer(dev, seed=i, wtype=ops.Q4_0, **dims)
                g = torch.Generator(device=dev).manual_seed(i)
                for name in ("wqkv", "wo", "wgu", "wdown"):
                    w = getattr(lay, name)
                    x = torch.randn((w.n_rows, w.k), generator=g, device=dev) * 0.02
                    b = ops.quantize_act(x, ops.Q8_0, ggml=True)[1]
                    setattr(lay, name, ops.QWeight.from_ggml(t, b, w.n_rows, w.k))
                lay = llama.LlamaLayer(lay.wqkv, lay.wo, lay.wgu, lay.wdown, lay.attn_norm, lay.ffn_norm, 2, 1, 128, 256)
            else:
                lay = llama.random_layer(dev, seed=i, wtype=t, **dims)
            out.append(lay)
        return out

    g = torch.Generator(device=dev).manual_seed(7)
    emb = ops.quantize_q4_0(torch.randn((500, 256), generator=g, device=dev)).reshape(500, -1)
    head = ops.QWeight.from_ggml(ops.Q4_0, ops.quantize_q4_0(torch.randn((500, 256), generator=g, device=dev)), 500, 256)
    norm = 1 + 0.1 * torch.randn(256, generator=g, device=dev)
    m = model.LlamaModel(emb, ops.Q4_0, layers(), norm, head)
    for n in lengths:
        tokens = torch.randint(500, (n,), generator=g, device=dev, dtype=torch.int32)
        m.prefill(tokens)
        ref = layers()
        x, y = (torch.empty((n, 256), device=dev) for _ in "xy")
        m._embed(tokens, x, n, torch.cuda.current_stream().cuda_stream)
        for lay, got in zip(ref, m.layers):
            lay.set_prefill_position(0, n)
            lay.prefill(x, y)
            x, y = y, x
            assert torch.equal(got.k_cache[:n], lay.k_cache[:n]) and torch.equal(got.v_cache[:n], lay.v_cache[:n])
        single = model.LlamaModel(emb, ops.Q4_0, ref, norm, head)
        single._head(x[n - 1], torch.cuda.current_stream().cuda_stream)
        assert torch.equal(m.logits, single.logits), n
