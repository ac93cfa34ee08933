"""CPU: the planner's size rules (default tile, split-KV choice) at the sizes where they change."""

from __future__ import annotations

import ctypes

import pytest
import torch

from flash_attn_npu_amd import flash_attention_forward as fa


@pytest.mark.parametrize("head_dim,block_n", [(16, 128), (32, 64), (64, 64), (128, 64), (256, 32)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_default_tile_follows_head_dim(head_dim, block_n, causal, dtype):
    for n_ctx in (49, 64, 333, 1777, 8192):
        rt = fa._describe_runtime(3, 5, n_ctx, head_dim, causal, dtype=dtype)
        assert rt["tiling_source"] == "fallback"
        assert rt["selected_config"] == {"BLOCK_M": 128, "BLOCK_N": block_n}


@pytest.mark.parametrize("heads,n_ctx,block_n", [
    (3, 1, 32), (3, 48, 32), (3, 49, 64), (2000, 48, 32),    # half a 64-key tile would be padding
    (512, 96, 64), (513, 96, 32), (513, 49, 32), (513, 97, 64), (257, 129, 64), (4095, 96, 32),
    (4096, 96, 64), (4096, 48, 32), (64, 16384, 64)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_non_causal_d128_tile_at_its_limits(heads, n_ctx, block_n, dtype):
    assert fa._query_config(1, heads, n_ctx, 128, False, dtype=dtype)[1] == block_n
    assert fa._query_config(1, heads, n_ctx, 128, True, dtype=dtype)[1] == 64


def _splits(z, h, n_ctx, head_dim, causal):
    return fa._describe_runtime(z, h, n_ctx, head_dim, causal)["kv_splits"]


def test_split_choice_at_its_limits():
    # 128 tiles of 1024 keys: the merge would cost more than the halved runs save.
    assert _splits(1, 16, 1024, 128, False) == 1
    assert _splits(1, 16, 1024, 256, True) == 1
    # 128 tiles of 4096 and 2048 keys: two runs fill the CUs.
    assert _splits(1, 4, 4096, 128, False) == 2
    assert _splits(1, 8, 2048, 16, False) == 2
    # One tile per CU and more: none.
    assert _splits(1, 8, 4096, 64, False) == 1
    assert _splits(1, 8, 4096, 64, True) == 1
    assert _splits(1, 9, 4096, 64, False) == 1
    # 192 tiles: causal runs may share CUs when they are long, others not.
    assert _splits(1, 3, 8192, 64, True) == 2
    assert _splits(1, 3, 8192, 64, False) == 1
    # Short runs are never made.
    assert _splits(1, 1, 128, 256, False) == 1
    for n_ctx in (129, 300, 1000, 4097, 100000):
        s = _splits(1, 1, n_ctx, 128, False)
        assert s == 1 or (n_ctx // s >= 128 and s * -(-n_ctx // 128) <= 256)


@pytest.mark.parametrize("head_dim", [32, 64, 128, 256])
def test_splits_fill_the_cus_between_powers_of_two(head_dim):
    # 80 tiles: 3 runs make 240 workgroups, 2 only 160; 40 and 48 tiles: 6 and 5.
    assert _splits(1, 1, 10240, head_dim, False) == 3
    assert _splits(1, 1, 5120, head_dim, False) in (4, 6)
    assert _splits(1, 1, 6144, head_dim, False) in (4, 5)
    # Causal, 96 tiles: 288 workgroups.
    assert _splits(1, 2, 6144, head_dim, True) in (3, 4)


def _choices(z, h, s_q, s_k, head_dim, causal, programs=0):
    lib = fa._load_library()
    p = fa._shape_params(z, h, s_q, head_dim, causal, programs=programs)
    p.Sk = s_k
    splits = [f(ctypes.byref(p)) for f in (lib.fa_default_kv_splits, lib.fa_workspace_kv_splits)]
    return splits, [lib.fa_split_workspace_bytes(ctypes.byref(p), s) for s in splits]


def test_default_choice_fits_the_static_buffer():
    """What fa_default_kv_splits returns can be passed to fa_fwd_split_static, but for long
    runs on grids of at most one tile per two CUs."""
    larger = 0
    for head_dim in (16, 64, 128, 256):
        for heads in range(1, 14):
            for n_ctx in (1024, 1500, 2048, 3000, 4096, 5000, 8192, 16384):
                for causal in (False, True):
                    tiles = heads * -(-n_ctx // 128)
                    (default, any_ws), (nbytes, _) = _choices(1, heads, n_ctx, n_ctx, head_dim, causal)
                    assert default <= 1 or nbytes <= 32 << 20 or (
                        tiles <= 128 and default * 65536 <= n_ctx * head_dim), (head_dim, heads, n_ctx, causal)
                    larger += any_ws != default
    assert larger > 0
    # 160 tiles, 40 MiB of partial results: only where a workspace can be had.
    assert _choices(1, 5, 4096, 4096, 256, True)[0] == [1, 2]
    assert _splits(1, 5, 4096, 256, True) == 2


def test_no_split_leaves_empty_runs():
    for head_dim, bn in ((16, 128), (64, 64), (128, 64), (256, 32)):
        for n_ctx in (1000, 1500, 2177, 3000, 4097, 5000, 8193, 8200, 10000):
            for heads in (1, 2, 3):
                s = _splits(1, heads, n_ctx, head_dim, False)
                kv_tiles = -(-n_ctx // bn)
                assert -(-kv_tiles // -(-kv_tiles // s)) == s, (head_dim, n_ctx, heads, s)


def test_splits_count_visible_keys_and_programs():
    # Causal with more keys than queries: only Sq keys are ever visible.
    for heads in (8, 100, 192):
        assert _choices(1, heads, 128, 8192, 64, True)[0] == [1, 1]
    # Fewer programs than tiles: splitting them shortens nothing.
    assert _choices(1, 3, 8192, 8192, 64, True)[0] == [2, 2]
    assert _choices(1, 3, 8192, 8192, 64, True, programs=64)[0] == [1, 1]
    assert _choices(1, 1, 4096, 4096, 128, False, programs=16)[0] == [1, 1]
    assert _choices(1, 1, 4096, 4096, 128, False, programs=256)[0] == [8, 8]
