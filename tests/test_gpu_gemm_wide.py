"""256 x 256 tiles (two 64-deep slab buffers filled by units): K of one slab,
of even and odd slab counts, ragged rows and columns, every epilogue, and
q|k|v heads two to a tile against launches on other tiles, bit for bit."""

import pytest
import torch
import torch.nn.functional as F

from layer_streaming import _hip
from oracle import cases
from oracle import llama_oracle as ref
from test_gpu_prefill import linear_bound_report

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.mark.parametrize("m,n,k", [(4000, 4096, 64), (4096, 4096, 128), (4001, 4090, 192),
                                   (3900, 4040, 320)])
def test_wide_tiles(gpu_device, m, n, k):
    # 16 x 16 tiles of 256 x 256: one round, against two of 256 x 128
    print("wide m={} n={} k={}".format(m, n, k), flush=True)
    dev = gpu_device
    x, w = cases.normal_bf16((m, k), 601), cases.normal_bf16((n, k), 602, 0.05)
    res = cases.normal_bf16((m, n), 603).to(dev)
    xd, wd = x.to(dev), w.to(dev)
    y = torch.empty((m, n), dtype=BF16, device=dev)
    _hip.gemm(xd, wd, y)
    assert linear_bound_report(y, x, w) <= 1.0
    # a few of the rows on another tile shape: the same sums
    few = torch.empty((300, n), dtype=BF16, device=dev)
    _hip.gemm(xd[m - 300:], wd, few)
    assert torch.equal(few, y[m - 300:])
    out = torch.empty_like(y)
    _hip.gemm_residual(xd, wd, res, out)
    assert torch.equal(out, res + y)
    yf = torch.empty((m, n), dtype=torch.float32, device=dev)
    _hip.gemm_f32out(xd, wd, yf)
    assert torch.equal(yf.to(BF16), y)
    gate, prod = torch.empty_like(y), torch.empty_like(y)
    _hip.gate_silu_gemm(xd, wd, gate)
    _hip.up_mul_gemm(xd, wd, gate, prod)
    assert cases.compare(gate.cpu(), F.silu(y.cpu()))["ok"]
    assert torch.equal(prod, gate * y)


@pytest.mark.parametrize("m", [4096, 3990])
@pytest.mark.parametrize("k", [64, 192, 256])
def test_wide_qkv_equals_split(gpu_device, m, k):
    dev = gpu_device
    cap = m + 9
    x = cases.normal_bf16((m, k), 611).to(dev)
    w = [cases.normal_bf16((rows, k), 612 + i, 0.05).to(dev)
         for i, rows in enumerate((4096, 1024, 1024))]
    c, s = ref.rope_cos_sin(ref.llama3_inv_freq(128), list(range(cap)))
    c, s = c[:, :64].contiguous().to(dev), s[:, :64].contiguous().to(dev)
    outs = []
    for groups in ([w], [[w[0][:2048], None, None], [None, w[1], None], [None, None, w[2]]]):
        q = torch.zeros((m, groups[0][0].shape[0]), dtype=BF16, device=dev)
        kc = torch.zeros((8, cap, 128), dtype=BF16, device=dev)
        vc = torch.zeros_like(kc)
        for wq, wk, wv in groups:
            _hip.qkv_rope_gemm(x, wq, wk, wv, c, s, 4, q, kc.view(-1), vc.view(-1),
                               cap * 128, 5)
        outs.append((q[:, :2048], kc, vc))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
