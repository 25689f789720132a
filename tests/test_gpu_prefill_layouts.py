"""Prompts of different lengths on one model: the activation layout of the MUL_MATs changes with the token count, and every
layer has to see the positions and buffers of the prompt at hand. Each prompt's logits equal those of a model that has run
nothing else, bit for bit (the same launches on the same inputs); a captured prompt replays the same after shorter ones."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wtype", [2, 12])
def test_prompts_of_other_lengths(wtype):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ameva_compute_amd.model import random_model
    dev = torch.device("cuda:0")

    def make():
        return random_model(dev, n_layers=2, H=256, n_head=2, n_head_kv=1, D=128, FF=512, vocab=1000, ctx=256, seed=3,
                            wtype=wtype, max_new=8)

    g = torch.Generator(device=dev).manual_seed(1)
    prompts = [torch.randint(1000, (n,), generator=g, device=dev, dtype=torch.int32) for n in (200, 20, 5, 40, 2, 100, 30)]
    m = make()
    for p in prompts:
        m.prefill(p)
        ref = make()
        ref.prefill(p)
        assert torch.equal(m.logits, ref.logits), p.numel()

    lay = m.layers[0]
    x = torch.randn((200, lay.H), generator=g, device=dev)
    out = torch.empty_like(x)
    lay.set_prefill_position(0, 200)
    lay.prefill(x, out)
    want = out.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        lay.prefill(x, out)
    for n in (5, 30, 2):
        lay.set_prefill_position(0, n)
        lay.prefill(x[:n].contiguous(), torch.empty((n, lay.H), device=dev))
        trash = [torch.full((1 << 18,), 7.0, device=dev) for _ in range(16)]  # freed buffers would be handed out again
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), n
        del trash
