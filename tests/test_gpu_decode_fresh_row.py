"""GPU parity: a step's fresh row in a split of its own, the first and the last of a split's rows, for every number of lane groups a
wavefront's state is spread over (a row of 8, 16 or 32 lanes) and head count: split by split, in one launch and in two passes, in one split
that stores its result itself, piece by piece and cut evenly; against float64 over the pool the launch leaves, where the rows have to be."""

import re

import pytest
import torch

from falcon_perception_amd import ops
from tests.gpu_cases import DEV, kernels
from tests.test_gpu_decode_plan import decode, flat_state
from tests.test_gpu_decode_step import holds, inputs

pytestmark = pytest.mark.gpu

LENS = [0, 1, 31, 63, 64, 65, 127, 128, 129, 511, 512, 1000]


def ways(names):
    """(direct, cut evenly, piece by piece) of the split-K kernel among `names`, and whether a merge pass follows it."""
    main = [n for n in names if "paged_decode_kernel<" in n]
    assert len(main) == 1, names
    flags = re.search(r"<\w+, \d+, \d+, (\w+), \w+, \w+, (\w+), (\w+)>", main[0]).groups()
    return tuple(f == "true" for f in flags), any("merge" in n for n in names)


@pytest.mark.parametrize("way", ["one-launch", "two-passes", "direct", "pieces", "even"])
@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 64), (torch.float16, 128), (torch.float32, 64), (torch.float32, 128)], ids=str)
@pytest.mark.parametrize("G,rep,P", [(1, 1, 64), (2, 1, 48), (2, 2, 128), (4, 4, 64), (8, 1, 32)])
def test_the_fresh_row_at_the_edges_of_a_split(way, dtype, D, G, rep, P):
    """Split by split go launches of few sequences: two of the lengths at a time."""
    Hc, ctx = 8, 2048
    lens = LENS * 8 if way == "even" else LENS
    launches = [[i, len(lens) - 1 - i] for i in range(len(lens) // 2)] if way in ("one-launch", "two-passes") else [list(range(len(lens)))]
    B = len(launches[0])
    split = ops.decode_split_tokens(B, Hc, ctx, P) if way == "pieces" else ctx if way == "direct" else 64
    merged = G * D <= 256  # in the launch itself, with counters
    matrix = G >= 4 and dtype != torch.float32 and rep == 1
    if way == "pieces" and merged:
        assert ops.decode_step_pieces(B, Hc * G, Hc * rep, rep, D, ctx, P, split) > 0
    elif len(launches) > 1:
        chunks = 2 * torch.cuda.get_device_properties(0).multi_processor_count // Hc
        assert ops.decode_step_pieces(B, Hc * G, Hc * rep, rep, D, ctx, P, split) == 0 and B * (ctx // split - 1) < chunks
    st = flat_state(7 + D + G, len(lens), Hc, D, P, ctx, dtype, rep, lens)
    arrivals = torch.zeros(B * Hc, dtype=torch.int32, device=DEV)
    for which in launches:
        q, k_new, v_new = inputs(st, B, Hc, G, D, dtype, rep)
        pos = torch.tensor([lens[i] for i in which], dtype=torch.int32, device=DEV)
        bidx = torch.tensor([st.slots[i] for i in which], dtype=torch.int64, device=DEV)
        expected = st.cache.kv_cache.clone()
        kw = dict(max_context=ctx, split_tokens=split, kv_rep=rep, bidx=bidx, k_new=k_new, v_new=v_new)
        if way in ("one-launch", "pieces"):
            kw["arrivals"] = arrivals
        got = decode(st, q, pos, **kw)
        at = st.cache.page_table[bidx, pos // P] * P + pos % P
        expected[0, 0, 0][:, at], expected[0, 1, 0][:, at] = k_new[:, :, 0].transpose(0, 1), v_new[:, :, 0].transpose(0, 1)
        assert torch.equal(st.cache.kv_cache, expected) and not arrivals.any()
        holds(got, st, q, pos, bidx, ctx, dtype, matrix)
    if not matrix:
        flags, merge = ways(kernels(lambda: decode(st, q, pos, **kw)))
        if way != "pieces" or merged:
            assert flags == (way == "direct", way == "even", way == "pieces")
            assert merge == (way in ("two-passes", "even") or (way == "one-launch" and not merged))
