"""GPU: B*H that is no multiple of the queue count: the left-over heads' tiles are dealt to all queues."""

from __future__ import annotations

import pytest
import torch

from tests.gpu_reference import attention_fp64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads", [9, 12, 15, 20])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("splits", ["1", "3"])
def test_left_over_heads(monkeypatch, heads, causal, splits):
    from flash_attn_npu_amd import flash_attention_forward as fa

    monkeypatch.setenv("KV_SPLITS", splits)
    g = torch.Generator().manual_seed(heads)
    q, k, v = (torch.randn((1, heads, 700, 64), generator=g).half().cuda() for _ in range(3))
    for programs in (None, "11"):  # one unit per workgroup; 11 workgroups over 8 queues
        if programs:
            monkeypatch.setenv("PERSISTENT_PROGRAMS", programs)
        out, lse = fa.attention(q, k, v, causal, 0.125, return_lse=True)
        o64, l64 = attention_fp64(q, k, v, causal, 0.125)
        # fp16 rounding of P and O: the bounds of the parity tests.
        assert (out.float() - o64.half().float()).abs().max().item() <= 5e-3
        assert (lse.double() - l64).abs().max().item() <= 1e-3
