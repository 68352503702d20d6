"""Host checks of how decode launches are sized (no GPU: the library answers for 256 CUs)."""

import pytest
import torch

from falcon_perception_amd import _native, ops
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


def plain_split(B, Hc, limit):
    """The split of a launch that goes split by split: the largest power of two up to 2048 that gives the workgroups wanted."""
    target = min(max(4 * B * Hc, 512), 2048)
    split = 2048
    while split > 128 and B * Hc * -(-limit // split) < target:
        split //= 2
    return split


@pytest.mark.parametrize("Hc", [1, 2, 4, 8, 16, 32])
def test_a_finer_split_only_where_the_even_cut_uses_it(native_lib, Hc):
    """The finer split that leaves workspace rows for the even cut: never where one split covers every context, not with more
    sequences than the cut takes, not with short splits, and without outgrowing the array of the entry point that cannot
    allocate."""
    finer = 0
    for B in [*range(1, 70), 96, 128, 255, 256, 257, 512, 1024, 1025, 2048, 4096]:
        for limit in (64, 128, 256, 512, 1024, 2048, 4096, 8192, 16384):
            split, plain = ops.decode_split_tokens(B, Hc, limit, 128), plain_split(B, Hc, limit)
            if split != plain:
                finer += 1
                assert split < plain < limit and B <= 1024 and 8 * B >= 512 // Hc
                assert plain >= 1024 or (plain == 512 and limit > 7 * 512)
                assert B * (-(-limit // split) - 1) >= 512 // Hc > B * (-(-limit // (2 * split)) - 1)
            need, before = (ops.decode_workspace_bytes(B, 8 * Hc, 128, limit, s) for s in (split, plain))
            room = _native.NOALLOC_SCRATCH_BYTES
            assert need <= room or before > room, (B, limit)
    assert finer > 0 or Hc > 16


@pytest.mark.parametrize("B,Hq,Hc", [(512, 128, 16), (1024, 64, 8), (2048, 32, 8)])
def test_large_batches_under_a_short_limit_need_no_scratch_array(native_lib, B, Hq, Hc):
    """One split covers a limit of 1024 tokens: the call gets past the size of the array to its null pointers."""
    rc = native_lib.fp_paged_decode_noalloc(None, 0, 0, None, None, None, 0, None, None, 0, None, 0, 0, None, None, B, Hq, Hc, 1,
                                            128, 128, 8, B, 8192, 1024, 0, 1.0, 1, None)
    assert rc == -1 and b"null pointer" in native_lib.fp_last_error()
    assert ops.decode_workspace_bytes(B, Hq, 128, 1024, ops.decode_split_tokens(B, Hc, 1024, 128)) == 0


@pytest.mark.parametrize("Hq,Hc,kv_rep,split", [(1, 1, 2, 128), (4, 4, 8, 128), (6, 6, 4, 128), (8, 4, 2, 128), (9, 4, 1, 128), (8, 4, 1, 100)])
def test_pieces_of_a_launch_that_cannot_be(native_lib, Hq, Hc, kv_rep, split):
    """More copies than heads would leave no workgroup heads to divide by."""
    with pytest.raises(RuntimeError, match="is no launch"):
        ops.decode_step_pieces(4, Hq, Hc, kv_rep, 64, 8192, 64, split)
