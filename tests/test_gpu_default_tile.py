"""GPU: non-causal D = 128 on both sides of the sizes where the default tile changes."""

from __future__ import annotations

import pytest
import torch

from tests.gpu_reference import attention_fp64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,n_ctx", [(2, 1), (3, 48), (3, 49), (512, 96), (513, 96), (513, 97)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_default_tile_of_short_sequences(fa, heads, n_ctx, dtype):
    g = torch.Generator().manual_seed(heads + n_ctx)
    q, k, v = (torch.randn((1, heads, n_ctx, 128), generator=g).to(dtype).cuda() for _ in range(3))
    out, lse = fa.attention(q, k, v, False, 0.09, return_lse=True)
    o64, l64 = attention_fp64(q, k, v, False, 0.09)
    # 16-bit rounding of P and O: the bounds of the parity tests.
    assert (out.float() - o64.to(dtype).float()).abs().max().item() <= (2e-2 if dtype == torch.bfloat16 else 5e-3)
    assert (lse.double() - l64).abs().max().item() <= 1e-3
