"""Streaming GEMM of short prompts (gemm_stream.hip) at the edges of its
shapes: token counts at both sides of each fragment and plan boundary, weight
rows that do not fill the last workgroup, odd pitches (element-wise stores),
K below, at and past whole slabs.  Bound of a bf16 product as in
test_gpu_prefill.py: one bf16 ulp plus 2^-22 sum |x w| of fp32 accumulation.
"""

import pytest
import torch
import torch.nn.functional as F

from layer_streaming import _hip
from oracle import cases
from oracle import llama_oracle as ref
from test_gpu_prefill import linear_bound_report

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.mark.parametrize("m,n,k", [
    (1, 4096, 64), (15, 16, 128), (16, 4097, 192), (17, 6144, 320),
    (48, 1024, 1088), (49, 1003, 256), (64, 28672, 64), (65, 4096, 576),
    (112, 4100, 192), (113, 4096, 448), (159, 8191, 128), (160, 30000, 64),
    (161, 4096, 320), (256, 6100, 192), (129, 7000, 64)])
def test_stream_gemm_edges(gpu_device, m, n, k):
    print("stream gemm m={} n={} k={}".format(m, n, k), flush=True)
    dev = gpu_device
    x, w = cases.normal_bf16((m, k), 301), cases.normal_bf16((n, k), 302, 0.05)
    res = cases.normal_bf16((m, n), 303)
    xd, wd = x.to(dev), w.to(dev)
    # rows around the output stay as they were
    guard = torch.full((m + 2, n), 7.0, dtype=BF16, device=dev)
    y = torch.empty((m, n), dtype=BF16, device=dev)
    _hip.gemm(xd, wd, y)
    assert linear_bound_report(y, x, w) <= 1.0
    if (n * 2) % 16 == 0:
        inner = guard[1:m + 1]
        _hip.gemm_residual(xd, wd, res.to(dev), inner)
        assert torch.equal(inner, res.to(dev) + y)
        assert bool((guard[0] == 7.0).all()) and bool((guard[m + 1] == 7.0).all())
    yf = torch.empty((m, n), dtype=torch.float32, device=dev)
    _hip.gemm_f32out(xd, wd, yf)
    if m <= 128:
        assert torch.equal(yf.to(BF16), y)
    else:  # logits of more rows run on tiles, whose sums add in another order
        assert linear_bound_report(yf.to(BF16), x, w) <= 1.0


@pytest.mark.parametrize("m,n,k", [(16, 64, 64), (33, 2048, 320), (81, 2112, 576),
                                   (160, 14336, 256), (97, 14400, 192)])
def test_stream_swiglu_edges(gpu_device, m, n, k):
    print("stream swiglu m={} n={} k={}".format(m, n, k), flush=True)
    dev = gpu_device
    x = cases.normal_bf16((m, k), 311)
    wg, wu = (cases.normal_bf16((n, k), s, 0.05) for s in (312, 313))
    xd, wgd, wud = x.to(dev), wg.to(dev), wu.to(dev)
    fused, gate, split = (torch.empty((m, n), dtype=BF16, device=dev) for _ in range(3))
    _hip.gate_up_swiglu_gemm(xd, wgd, wud, fused)
    _hip.gate_silu_gemm(xd, wgd, gate)
    _hip.up_mul_gemm(xd, wud, gate, split)
    assert torch.equal(fused, split)
    r = cases.compare(fused, F.silu(ref.linear(x, wg)) * ref.linear(x, wu))
    assert r["ok"], r


@pytest.mark.parametrize("m", [1, 17, 49, 160, 161, 256])
def test_stream_qkv_split_equals_fused(gpu_device, m):
    # q, k and v as three launches (other weight rows per workgroup) add in
    # the same order; the last workgroup of the fused launch crosses from k
    # to v heads when 24 or 48 rows do not divide a matrix
    dev = gpu_device
    k, cap = 192, m + 3
    x = cases.normal_bf16((m, k), 321).to(dev)
    w = [cases.normal_bf16((rows, k), 322 + i, 0.05).to(dev)
         for i, rows in enumerate((4096, 1024, 1024))]
    inv = ref.llama3_inv_freq(128)
    c, s = ref.rope_cos_sin(inv, list(range(cap)))
    c, s = c[:, :64].contiguous().to(dev), s[:, :64].contiguous().to(dev)
    outs = []
    for groups in ([w], [[w[0], None, None], [None, w[1], None], [None, None, w[2]]]):
        q = torch.zeros((m, 4096), dtype=BF16, device=dev)
        kc = torch.zeros((8, cap, 128), dtype=BF16, device=dev)
        vc = torch.zeros_like(kc)
        for wq, wk, wv in groups:
            _hip.qkv_rope_gemm(x, wq, wk, wv, c, s, 2, q, kc.view(-1), vc.view(-1),
                               cap * 128, 1)
        outs.append((q, kc, vc))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    v = ref.linear(x.cpu(), w[2].cpu()).view(m, 8, 128).transpose(0, 1)
    assert cases.compare(outs[0][2][:, 1:m + 1].cpu(), v)["ok"]
    assert int(outs[0][2][:, 0].abs().sum()) == 0


@pytest.mark.parametrize("m,n", [(6, 8192), (64, 8192), (128, 8192), (6, 66048)])
def test_stream_sums_are_quarters_of_k(gpu_device, m, n):
    # rounding errors of a chain of fp32 additions grow as the root of its
    # length: four chains leave half the error of one (tiles of more rows),
    # two would leave 0.71 of it
    dev, k = gpu_device, 4096
    x = cases.normal_bf16((192, k), 331).to(dev)
    w = cases.normal_bf16((n, k), 332, 0.02).to(dev)
    exact = x[:m].double() @ w.double().t()
    errors = []
    for rows in (m, 192):
        y = torch.empty((rows, n), dtype=torch.float32, device=dev)
        _hip.gemm_f32out(x[:rows], w, y)
        errors.append(float((y[:m].double() - exact).norm()))
    assert errors[0] <= 0.6 * errors[1], errors


@pytest.mark.parametrize("m,n,k", [(2, 65544, 256), (33, 65700, 640), (64, 128256, 896),
                                   (128, 70000, 1024), (17, 66048, 576)])
def test_stream_rotated_logits(gpu_device, m, n, k):
    # more than 65536 columns: each tile starts at another 256 columns of K
    # (640, 896: the last slab of 256 or 128 is short; 576: an odd number of
    # 64-deep slabs, not rotated).  Bound of fp32 accumulation as above.
    print("rotated logits m={} n={} k={}".format(m, n, k), flush=True)
    dev = gpu_device
    x = cases.normal_bf16((m, k), 341).to(dev)
    w = cases.normal_bf16((n, k), 342, 0.05).to(dev)
    y = torch.full((m, n), float("nan"), dtype=torch.float32, device=dev)
    _hip.gemm_f32out(x, w, y)
    exact = x.double() @ w.double().t()
    bound = 2.0 ** -22 * (x.double().abs() @ w.double().abs().t())
    assert bool(((y.double() - exact).abs() <= bound).all())


@pytest.mark.parametrize("m,n,k", [(16, 14336, 640), (33, 7168, 896), (100, 14336, 640),
                                   (160, 14336, 768), (49, 6208, 1152), (16, 6144, 640)])
def test_stream_rotated_swiglu_equals_its_halves(gpu_device, m, n, k):
    # the fused launch and its halves walk K in slabs of other depths from the
    # same starts, and add in the same order
    dev = gpu_device
    x = cases.normal_bf16((m, k), 351).to(dev)
    wg, wu = (cases.normal_bf16((n, k), s, 0.05).to(dev) for s in (352, 353))
    fused, gate, split = (torch.empty((m, n), dtype=BF16, device=dev) for _ in range(3))
    _hip.gate_up_swiglu_gemm(x, wg, wu, fused)
    _hip.gate_silu_gemm(x, wg, gate)
    _hip.up_mul_gemm(x, wu, gate, split)
    assert torch.equal(fused, split)
    exact = F.silu(x.double() @ wg.double().t())
    assert cases.compare(gate, exact.to(BF16).cpu())["ok"]


@pytest.mark.parametrize("m,n,k", [(1, 40, 512), (16, 1000, 576), (7, 520, 1088), (9, 4096, 1984),
                                   (16, 2056, 4160), (3, 8, 64)])
def test_stream_deep_slabs(gpu_device, m, n, k):
    # up to 16 rows and 16 columns a workgroup: 512-deep slabs, K below, at and
    # past whole ones, with and without the nontemporal hint (K >= 4096)
    print("deep slabs m={} n={} k={}".format(m, n, k), flush=True)
    dev = gpu_device
    x, w = cases.normal_bf16((m, k), 361), cases.normal_bf16((n, k), 362, 0.05)
    res = cases.normal_bf16((m, n), 363).to(dev)
    xd, wd = x.to(dev), w.to(dev)
    y, out, gate, prod = (torch.empty((m, n), dtype=BF16, device=dev) for _ in range(4))
    _hip.gemm(xd, wd, y)
    assert linear_bound_report(y, x, w) <= 1.0
    _hip.gemm_residual(xd, wd, res, out)
    assert torch.equal(out, res + y)
    yf = torch.empty((m, n), dtype=torch.float32, device=dev)
    _hip.gemm_f32out(xd, wd, yf)
    assert torch.equal(yf.to(BF16), y)
    _hip.gate_silu_gemm(xd, wd, gate)
    assert cases.compare(gate.cpu(), F.silu(y.cpu()))["ok"]
    _hip.up_mul_gemm(xd, wd, gate, prod)
    assert torch.equal(prod, gate * y)


@pytest.mark.parametrize("n", [3584, 4096, 5120, 7168])
@pytest.mark.parametrize("m", [5, 16, 33, 100, 129, 160])
def test_stream_widths(gpu_device, m, n):
    # 32 and 64 gate and up rows a workgroup (16 and 32 in the halves), token
    # tiles that share an XCD (tile counts that are no multiple of 8), 32 and
    # 112 rows for logits; past 128 rows 5120 and 7168 gate rows run tiles
    dev, k = gpu_device, 768
    print("stream widths m={} n={}".format(m, n), flush=True)
    x = cases.normal_bf16((m, k), 371).to(dev)
    wg, wu = (cases.normal_bf16((n, k), s, 0.05).to(dev) for s in (372, 373))
    fused, gate, split = (torch.empty((m, n), dtype=BF16, device=dev) for _ in range(3))
    _hip.gate_up_swiglu_gemm(x, wg, wu, fused)
    _hip.gate_silu_gemm(x, wg, gate)
    _hip.up_mul_gemm(x, wu, gate, split)
    assert torch.equal(fused, split)
    product = x.double() @ wg.double().t()
    assert cases.compare(gate.cpu(), F.silu(product).to(BF16).cpu())["ok"]
    # all rows of both matrices in one product
    both = torch.cat((wg, wu))
    wide = torch.empty((m, 2 * n), dtype=torch.float32, device=dev)
    y = torch.empty((m, 2 * n), dtype=BF16, device=dev)
    _hip.gemm_f32out(x, both, wide)
    _hip.gemm(x, both, y)
    bound = 2.0 ** -22 * (x.double().abs() @ both.double().abs().t())
    assert bool(((wide.double() - x.double() @ both.double().t()).abs() <= bound).all())
    if m <= 128:
        assert torch.equal(wide.to(BF16), y)
    assert linear_bound_report(y, x.cpu(), both.cpu()) <= 1.0
