"""160 x 256 tiles (waves 4 .. 7 load one X instruction fewer than waves
0 .. 3): one slab of K, even and odd slab counts, ragged rows and columns,
every epilogue, and the partials of split K."""

import pytest
import torch
import torch.nn.functional as F

from layer_streaming import _hip
from oracle import cases
from oracle import llama_oracle as ref
from test_gpu_prefill import linear_bound_report

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.mark.parametrize("m,n,k", [(257, 28672, 64), (320, 28672, 128), (301, 28600, 192)])
def test_low_tiles(gpu_device, m, n, k):
    # two rows of 112 tiles, one round; 13 000 columns run 128-row tiles
    print("low m={} n={} k={}".format(m, n, k), flush=True)
    dev = gpu_device
    x, w = cases.normal_bf16((m, k), 701), cases.normal_bf16((n, k), 702, 0.05)
    res = cases.normal_bf16((m, n), 703).to(dev)
    xd, wd = x.to(dev), w.to(dev)
    y = torch.empty((m, n), dtype=BF16, device=dev)
    _hip.gemm(xd, wd, y)
    assert linear_bound_report(y, x, w) <= 1.0
    few = torch.empty((m, 13000), dtype=BF16, device=dev)
    _hip.gemm(xd, wd[n - 13000:], few)
    assert torch.equal(few, y[:, n - 13000:])
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
    half = 14336
    fused = torch.empty((m, half), dtype=BF16, device=dev)
    up = wd[-half:].contiguous()
    _hip.gate_up_swiglu_gemm(xd, wd[:half], up, fused)
    assert torch.equal(fused, gate[:, :half] * y[:, -half:])


@pytest.mark.parametrize("m", [257, 309])
def test_low_qkv_equals_split(gpu_device, m):
    dev, k, cap = gpu_device, 192, m + 9
    x = cases.normal_bf16((m, k), 711).to(dev)
    w = [cases.normal_bf16((rows, k), 712 + i, 0.05).to(dev)
         for i, rows in enumerate((26624, 1024, 1024))]
    c, s = ref.rope_cos_sin(ref.llama3_inv_freq(128), list(range(cap)))
    c, s = c[:, :64].contiguous().to(dev), s[:, :64].contiguous().to(dev)
    kc = torch.zeros((2, 8, cap, 128), dtype=BF16, device=dev)
    vc = torch.zeros_like(kc)
    q = torch.zeros((m, 26624), dtype=BF16, device=dev)
    part = torch.zeros((2, m, 13312), dtype=BF16, device=dev)

    def launch(wq, wk, wv, out, at):
        _hip.qkv_rope_gemm(x, wq, wk, wv, c, s, 4, out, kc[at].view(-1), vc[at].view(-1),
                           cap * 128, 5)

    launch(w[0], w[1], w[2], q, 0)
    launch(w[0][:13312], None, None, part[0], 1)
    launch(w[0][13312:], None, None, part[1], 1)
    launch(None, w[1], None, part[0], 1)
    launch(None, None, w[2], part[0], 1)
    assert torch.equal(q, torch.cat((part[0], part[1]), 1))
    assert torch.equal(kc[0], kc[1]) and torch.equal(vc[0], vc[1])


@pytest.mark.parametrize("m,n,k,splits,refused", [
    (257, 4096, 14336, 8, True), (320, 4096, 14400, 8, True), (613, 4088, 8192, 4, True),
    (641, 4096, 8192, 3, True), (1100, 4096, 8192, 2, False)])
def test_low_split(gpu_device, m, n, k, splits, refused):
    # 28 slabs of K a split at least, so eight of them need K >= 14336
    print("low split m={} n={} k={}".format(m, n, k), flush=True)
    dev = gpu_device
    x, w = cases.normal_bf16((m, k), 721), cases.normal_bf16((n, k), 722, 0.02)
    res = cases.normal_bf16((m, n), 723).to(dev)
    xd, wd = x.to(dev), w.to(dev)
    need = _hip.gemm_workspace_bytes(m, n, k)
    assert need == splits * m * n * 4
    ws = torch.full((need,), 255, dtype=torch.uint8, device=dev)  # NaN where unwritten
    y, out = (torch.empty((m, n), dtype=BF16, device=dev) for _ in range(2))
    _hip.gemm(xd, wd, y, workspace=ws)
    assert linear_bound_report(y, x, w) <= 1.0
    _hip.gemm_residual(xd, wd, res, out, workspace=ws)
    assert torch.equal(out, res + y)
    # a short workspace is refused, or where the other tiles run one pass,
    # left alone
    if refused:
        with pytest.raises(_hip.HipCallError):
            _hip.gemm(xd, wd, y, workspace=ws[:-16])
    else:
        _hip.gemm(xd, wd, y, workspace=ws[:16])
        _hip.gemm(xd, wd, out)
        assert torch.equal(out, y)


def test_low_split_takes_what_the_one_pass_takes(gpu_device):
    # where only these tiles split, an unaligned workspace is left alone and
    # an unaligned residual is read element by element, as by the one pass
    dev, (m, n, k) = gpu_device, (1100, 4096, 8192)
    x, w = cases.normal_bf16((m, k), 731).to(dev), cases.normal_bf16((n, k), 732, 0.02).to(dev)
    need = _hip.gemm_workspace_bytes(m, n, k)
    ws = torch.empty(need + 16, dtype=torch.uint8, device=dev)
    shifted = cases.normal_bf16((m * n + 1,), 733).to(dev)[1:].view(m, n)
    one, y, out = (torch.empty((m, n), dtype=BF16, device=dev) for _ in range(3))
    _hip.gemm(x, w, one)
    _hip.gemm(x, w, y, workspace=ws[4:])
    assert torch.equal(y, one)
    _hip.gemm_residual(x, w, shifted, out, workspace=ws)
    assert torch.equal(out, shifted + one)
