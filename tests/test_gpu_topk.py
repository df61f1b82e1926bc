"""Exact top-k at the edges of its two selections: passes of a maximum for up
to 5 keys, sorted 64-key lists from 6; row counts around the 64-lane chunks,
the 1024-logit spans and several spans; ties, signed zeros, NaN and -inf."""

import pytest
import torch

from layer_streaming import _hip

pytestmark = pytest.mark.gpu


def _expected(values, k):
    # value descending, index ascending; NaN above everything, -0.0 == +0.0
    def order(i):
        v = values[i]
        return (0, 0.0, i) if v != v else (1, -v, i)

    return sorted(range(len(values)), key=order)[:k]


@pytest.mark.parametrize("top_k", [1, 4, 5, 6, 33, 63, 64])
@pytest.mark.parametrize("rows", [1, 63, 65, 1023, 1025, 4097, 20000])
def test_topk_edges(gpu_device, rows, top_k):
    print("topk rows={} k={}".format(rows, top_k), flush=True)
    g = torch.Generator().manual_seed(rows * 100 + top_k)
    # few distinct values: ties across lanes, waves and spans
    values = (torch.randn(rows, generator=g) * 8).round() / 4
    values[values == 0.25] = -0.0
    if rows > 60:
        values[rows // 2] = float("nan")
        values[rows - 1] = float("nan")
        values[3] = float("-inf")
        values[7] = float("inf")
    dev = gpu_device
    ws = torch.full((_hip.lm_head_workspace_bytes(rows, top_k),), 0xAB, dtype=torch.uint8,
                    device=dev)
    out = torch.empty(top_k, dtype=torch.float32, device=dev)
    ids = torch.empty(top_k, dtype=torch.int64, device=dev)
    _hip.topk_f32(values.to(dev), top_k, ws, out, ids)
    n = min(rows, top_k)
    expected = _expected(values.tolist(), n)
    assert ids[:n].tolist() == expected
    picked = values[expected]
    got = out[:n].cpu()
    assert bool(((got == picked) | ((got != got) & (picked != picked))).all())
    assert ids[n:].tolist() == [-1] * (top_k - n)
