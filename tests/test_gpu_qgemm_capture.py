"""Batched products with at least 1024 tiles of 64 x 64 and fewer than 384 of 128 x 128 keep k whole: they run without the
split's workspace, so such a product may be a process's first under capture (in a child process: the workspace, once
allocated, stays)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = """
import sys, torch
from ameva_compute_amd import ops
n, k, m = map(int, sys.argv[1:])
for wtype, at in ((ops.Q4_0, ops.Q8_0), (ops.Q4_0, ops.Q8_0_F6), (ops.Q8_0, ops.Q8_0), (ops.Q4_K, ops.Q8_K)):
    print(wtype, at, flush=True)
    w = torch.randn((n, k), device="cuda") * 0.02
    wg = (ops.quantize_q4_0(w) if wtype == ops.Q4_0 else ops.quantize_act(w, ops.Q8_0, ggml=True)[1]
          if wtype == ops.Q8_0 else ops.quantize_k(w, wtype))
    w = ops.QWeight.from_ggml(wtype, wg, n, k)
    act = ops.quantize_act(torch.randn((m, k), device="cuda"), at)[0]
    out = torch.zeros((m, n), device="cuda")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ops.mul_mat_q(w, act, m, out=out, act_t=at)
    ref = ops.mul_mat_q(w, act, m, act_t=at)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
print("captured")
"""


@pytest.mark.parametrize("n,m", [(11000, 331), (16400, 200)])  # 1032 and 1028 tiles of 64 x 64, 258 of 128 x 128
def test_first_product_under_capture(n, m):
    r = subprocess.run([sys.executable, "-c", CHILD, str(n), "6144", str(m)], cwd=ROOT, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0 and "captured" in r.stdout, r.stdout + r.stderr[-2000:]
