"""RMSNorm rows around the widths that are kept in registers (2048, 4096,
8192 columns) and beside them, in place too: within one bf16 ulp of the
oracle (the mean of squares may add in another order)."""

import pytest
import torch

from layer_streaming import _hip
from oracle import cases
from oracle import llama_oracle as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 3, 300])
@pytest.mark.parametrize("n", [8, 2040, 2048, 2056, 4096, 4104, 8192, 16384])
def test_rmsnorm_widths(gpu_device, rows, n):
    print("rmsnorm rows={} n={}".format(rows, n), flush=True)
    x = cases.normal_bf16((rows, n), 401)
    w = cases.normal_bf16((n,), 402)
    expected = ref.rms_norm(x, w, 1e-5).float()
    xd, wd = x.to(gpu_device), w.to(gpu_device)
    out = torch.empty_like(xd)
    _hip.rmsnorm(xd, wd, out, 1e-5)
    _hip.rmsnorm(xd, wd, xd, 1e-5)
    assert torch.equal(out, xd)
    ulp = torch.exp2(torch.floor(torch.log2(expected.abs().clamp_min(1e-30))) - 7)
    # the normalised value may round the other way (half an ulp), and so may
    # its product with the weight
    assert bool(((out.cpu().float() - expected).abs() <= 2 * ulp).all())
