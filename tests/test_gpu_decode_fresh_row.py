"""GPU parity: a step's fresh row in a split of its own, the first and the last of a split's rows, for every number of lane groups a
wavefront's state is spread over (a row of 8, 16 or 32 lanes) and head count, split by split in one launch and in two passes, piece by piece and
cut evenly; against float64 over the pool the launch leaves, where the rows have to be."""

import pytest
import torch

from falcon_perception_amd import ops
from tests.gpu_cases import DEV
from tests.test_gpu_decode_plan import decode, flat_state
from tests.test_gpu_decode_step import holds, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("way", ["one-launch", "two-passes", "pieces", "even"])
@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 64), (torch.float16, 128), (torch.float32, 64), (torch.float32, 128)], ids=str)
@pytest.mark.parametrize("G,rep,P", [(1, 1, 64), (2, 1, 48), (2, 2, 128), (4, 4, 64), (8, 1, 32)])
def test_the_fresh_row_at_the_edges_of_a_split(way, dtype, D, G, rep, P):
    lens = [0, 1, 31, 63, 64, 65, 127, 128, 129, 511, 512, 1000]
    Hc, ctx = 8, 2048
    if way == "even":
        lens = lens * 8
    B = len(lens)
    split = ops.decode_split_tokens(B, Hc, ctx, P) if way == "pieces" else 64
    if way == "pieces" and G * D <= 256:
        assert ops.decode_step_pieces(B, Hc * G, Hc * rep, rep, D, ctx, P, split) > 0
    st = flat_state(7 + D + G, B, Hc, D, P, ctx, dtype, rep, lens)
    q, k_new, v_new = inputs(st, B, Hc, G, D, dtype, rep)
    pos = torch.tensor(lens, dtype=torch.int32, device=DEV)
    bidx = torch.tensor(st.slots, dtype=torch.int64, device=DEV)
    expected = st.cache.kv_cache.clone()
    arrivals = torch.zeros(B * Hc, dtype=torch.int32, device=DEV)
    kw = dict(max_context=ctx, split_tokens=split, kv_rep=rep, bidx=bidx)
    if way in ("one-launch", "pieces"):
        kw["arrivals"] = arrivals
    got = decode(st, q, pos, k_new=k_new, v_new=v_new, **kw)
    at = st.cache.page_table[bidx, pos // P] * P + pos % P
    expected[0, 0, 0][:, at], expected[0, 1, 0][:, at] = k_new[:, :, 0].transpose(0, 1), v_new[:, :, 0].transpose(0, 1)
    assert torch.equal(st.cache.kv_cache, expected) and not arrivals.any()
    holds(got, st, q, pos, bidx, ctx, dtype, G >= 4 and dtype == torch.bfloat16 and rep == 1)
