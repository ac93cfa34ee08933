"""CPU: the planner's size rules (default tile, split-KV choice) at the sizes where they change."""

from __future__ import annotations

import pytest
import torch

from flash_attn_npu_amd import flash_attention_forward as fa


@pytest.mark.parametrize("head_dim,block_n", [(16, 128), (32, 64), (64, 64), (128, 64), (256, 32)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_default_tile_follows_head_dim(head_dim, block_n, causal, dtype):
    for n_ctx in (1, 64, 333, 1777, 8192):
        rt = fa._describe_runtime(3, 5, n_ctx, head_dim, causal, dtype=dtype)
        assert rt["tiling_source"] == "fallback"
        assert rt["selected_config"] == {"BLOCK_M": 128, "BLOCK_N": block_n}
