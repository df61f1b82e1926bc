"""Causal attention of short prompts (one workgroup per 8 tokens and KV head)
at the edges of its tiles and of its range: token counts around 8 and around
the 704-token switch to the lockstep kernel, cached positions around a
32-position block, few KV heads, many (16 switch at 352 tokens, 32 at 176), rows past the end poisoned with NaN.

P enters the products rounded to bf16 (relative 2^-9 each, averaging), the
result is rounded once more: 1e-2 + 1e-2 |b| as in test_gpu_prefill.py."""

import pytest
import torch

from layer_streaming import _hip
from oracle import cases

pytestmark = pytest.mark.gpu
DIM = 128


@pytest.mark.parametrize("past,tokens,kv", [
    (0, 1, 8), (0, 7, 8), (0, 8, 1), (0, 9, 8), (5, 33, 3), (31, 1, 8), (32, 64, 2),
    (300, 17, 8), (1000, 40, 8), (0, 703, 2), (0, 704, 8), (0, 705, 2), (37, 704, 1),
    (0, 352, 16), (9, 353, 16), (40, 176, 32), (0, 177, 32)])
def test_short_prompt_attention(gpu_device, past, tokens, kv):
    print("short attention past={} tokens={} kv={}".format(past, tokens, kv), flush=True)
    heads, total, cap = 4 * kv, past + tokens, past + tokens + 9
    q = cases.normal_bf16((tokens, heads * DIM), 501)
    k = cases.normal_bf16((kv, cap, DIM), 502)
    v = cases.normal_bf16((kv, cap, DIM), 503)
    k[:, total:] = float("nan")
    v[:, total:] = float("nan")
    kd, vd = k.to(gpu_device), v.to(gpu_device)
    out = torch.full((tokens + 1, heads * DIM), 5.0, dtype=torch.bfloat16,
                     device=gpu_device)
    _hip.prefill_attention(q.to(gpu_device), kd.view(-1), vd.view(-1), cap * DIM, past,
                           tokens, out[:tokens], DIM ** -0.5, heads, kv)
    assert bool((out[tokens] == 5.0).all())
    limit = torch.arange(past, total)
    column = torch.arange(total)
    for h in range(heads):
        qh = q[:, h * DIM:(h + 1) * DIM].double()
        s = qh @ k[h // 4, :total].double().t() * DIM ** -0.5
        s.masked_fill_(column[None, :] > limit[:, None], float("-inf"))
        expected = torch.softmax(s, -1) @ v[h // 4, :total].double()
        got = out[:tokens, h * DIM:(h + 1) * DIM].cpu().double()
        assert bool(((got - expected).abs() <= 1e-2 + 1e-2 * expected.abs()).all()), h
