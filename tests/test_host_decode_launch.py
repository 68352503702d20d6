"""Host checks of how decode launches are sized (no GPU: the library answers for 256 CUs)."""

import pytest
import torch

from falcon_perception_amd import ops
from falcon_perception_amd.paged_attention import PagedKVCache

HEADS = [(16, 8), (64, 8), (16, 16), (8, 4), (4, 1), (32, 32)]  # query heads, workgroup heads


@pytest.mark.parametrize("limit", [256, 512, 1024, 2048, 8192])
@pytest.mark.parametrize("table", [1, 3])
@pytest.mark.parametrize("max_batch", [9, 10, 12, 17, 24, 41, 65, 125])
def test_the_caches_workspace_holds_every_batch(native_lib, max_batch, limit, table):
    """A page table exactly as wide as the limit (`table` 1) leaves no slack: the one buffer of the cache has to hold the launch of
    every batch up to the largest, whose split may be finer than that of batch 1 and of the largest."""
    P, D = 128, 128
    for Hq, Hc in HEADS:
        cache = PagedKVCache(table * limit // P, P, max_batch, 1, 8, 1, torch.bfloat16, device="cpu")
        address = None
        for B in [8, *range(1, max_batch + 1)]:
            workspace, split = cache.decode_launch(B, Hq, D, limit, Hc)
            assert split == ops.decode_split_tokens(B, Hc, limit, P)
            need = ops.decode_workspace_bytes(B, Hq, D, limit, split)
            assert need <= (0 if workspace is None else workspace.numel()), (Hq, Hc, B, split)
            if workspace is not None:  # captured graphs of other batches keep writing to it
                address = address or workspace.data_ptr()
                assert workspace.data_ptr() == address, (Hq, Hc, B)
