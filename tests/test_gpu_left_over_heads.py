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


def _close(out, lse, q, k, v, causal, scale, o_tol):
    o64, l64 = attention_fp64(q, k, v, causal, scale)
    assert (out.float() - o64.to(q.dtype).float()).abs().max().item() <= o_tol
    assert (lse.double() - l64).abs().max().item() <= 1e-3


# (B, H, S, D, tile, bshd): each kernel family, a grid of several rounds, heads in more
# than one group of 8 per queue, a projection's layout.
@pytest.mark.parametrize("case", [(1, 9, 300, 256, None, False), (3, 5, 513, 128, (256, 64), False),
                                  (3, 3, 129, 64, (256, 64), True), (1, 73, 390, 16, None, False),
                                  (5, 26, 200, 128, None, True), (1, 15, 1100, 32, None, True)])
@pytest.mark.parametrize("causal", [False, True])
def test_left_over_heads_by_kernel(case, causal):
    from flash_attn_npu_amd import flash_attention_forward as fa

    B, H, S, D, tile, bshd = case
    g = torch.Generator().manual_seed(S)
    shape = (B, S, H, D) if bshd else (B, H, S, D)
    q, k, v = (torch.randn(shape, generator=g).bfloat16().cuda() for _ in range(3))
    if bshd:
        q, k, v = (t.permute(0, 2, 1, 3) for t in (q, k, v))
    bm, bn = tile or (None, None)
    out, lse = fa.attention(q, k, v, causal, D ** -0.5, BM=bm, BN=bn, return_lse=True)
    _close(out, lse, q, k, v, causal, D ** -0.5, 2e-2)  # bf16: the bound of the parity tests


@pytest.mark.parametrize("shape", [(1, 12, 700, 64), (3, 3, 300, 256), (1, 41, 260, 128)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("splits", ["1", "3"])
def test_left_over_heads_captured(monkeypatch, shape, causal, splits):
    """A captured launch walks the same order with no counters: replays equal the eager result."""
    from flash_attn_npu_amd import flash_attention_forward as fa

    monkeypatch.setenv("KV_SPLITS", splits)
    g = torch.Generator().manual_seed(shape[2])
    q, k, v = (torch.randn(shape, generator=g).half().cuda() for _ in range(3))
    want_o, want_l = fa.attention(q, k, v, causal, 0.1, return_lse=True)
    _close(want_o, want_l, q, k, v, causal, 0.1, 5e-3)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fa.attention(q, k, v, causal, 0.1, return_lse=True)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, lse = fa.attention(q, k, v, causal, 0.1, return_lse=True)
    for rep in range(3):
        out.zero_()
        lse.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want_o) and torch.equal(lse, want_l), rep
        assert torch.equal(fa.attention(q, k, v, causal, 0.1), want_o)
