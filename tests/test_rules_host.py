"""Dispatch rules that are decided on the host, without a GPU: where the fp32 state fork takes prepared tiles, and
where a decoding step's keys are split."""

import pytest
import torch

from dllm_qwen38_amd import _lib, attention


@pytest.mark.parametrize("args,taken", [
    ((1, 256, 16, 48, 128, 128, 32, 1), True),
    ((1, 32, 16, 48, 128, 128, 32, 0), True),      # one tile
    ((1, 8, 1, 1, 64, 64, 1, 1), True),            # one row per tile
    ((32, 256, 4, 4, 64, 64, 32, 1), True),        # 128 heads of 64
    ((33, 256, 4, 4, 64, 64, 32, 1), False),       # 132
    ((33, 256, 16, 48, 128, 128, 32, 1), True),    # heads of 128: any number
    ((64, 256, 16, 48, 128, 128, 32, 1), False),   # but a tile of them past the bound
    ((1, 256, 16, 48, 128, 64, 32, 1), False),
    ((1, 256, 4, 4, 32, 32, 32, 1), False),
    ((1, 256, 16, 48, 128, 128, 64, 1), False),
    ((1, 240, 16, 48, 128, 128, 32, 1), False),
    ((1, 256, 5, 48, 128, 128, 32, 1), False),
    ((0, 256, 16, 48, 128, 128, 32, 1), False),
])
def test_fp32_fork_workspace(args, taken):
    n = _lib.lib().dllm_gdn_fork_f32_workspace_bytes(*args)
    B, Hv, D = args[0], args[3], args[4]
    # 128 MB of operands (and states not kept), and the two states carried between ranges
    assert (0 < n <= (128 << 20) + 2 * B * Hv * D * D * 4) if taken else n == 0


@pytest.mark.parametrize("B,Hq,Hkv,d,last", [
    (1, 24, 4, 256, 8), (4, 24, 4, 256, 13), (16, 24, 4, 256, 31), (1, 16, 4, 128, 12), (4, 16, 4, 128, 14), (1, 8, 2, 64, 14),
])
def test_key_splits_begin_where_the_merge_pays(B, Hq, Hkv, d, last):
    q = torch.empty(B, 32, Hq, d, dtype=torch.bfloat16)
    assert attention._key_splits(q, 32, 32 * last, Hkv, d) == 1
    assert attention._key_splits(q, 32, 32 * last + 1, Hkv, d) > 1
    assert attention._key_splits(q, 65, 32 * last + 1, Hkv, d) == 1
    assert attention._key_splits(q.float(), 32, 32 * last + 1, Hkv, d) == 1
