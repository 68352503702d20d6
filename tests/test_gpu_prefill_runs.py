"""GPU: query tiles that hold rows of several sequences and of padding, with their boundaries at the edges of the lanes that look
for them (64 rows to a lane register, up to four of them), against the oracle; whole workgroups, workgroups whose halves take the
key tiles in turn, and key shares."""

import pytest
import torch

from falcon_perception_amd import ops
from tests.gpu_cases import DEV
from tests.test_gpu_prefill_few_rows import check
from tests.test_gpu_prefill_key_shares import make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,bound", [(torch.bfloat16, 0.0), (torch.bfloat16, 39.0), (torch.float16, 0.0)], ids=str)
@pytest.mark.parametrize("D,G,P", [(128, 1, 64), (64, 1, 128), (128, 2, 32), (128, 4, 64), (64, 8, 64)])
@pytest.mark.parametrize("lens,pads", [
    ([1, 62, 1, 64, 63, 1], [0, 0, 0, 0, 0, 0]),   # boundaries at rows 1, 63, 64, 128, 191, 192
    ([31, 33, 65, 127], [1, 0, 0, 1]),             # 31, 32, 65, 130, 257 with single padding rows between
    ([5], [251]),                                  # one short run, the rest of a tile of 256 rows is padding
    ([256, 1], [0, 254]),                          # a run as long as the largest tile, then one row
], ids=str)
@pytest.mark.parametrize("shares", [False, True], ids=["uncut", "key-shares"])
def test_runs_inside_a_tile(dtype, bound, D, G, P, lens, pads, shares):
    st, q, bidx, lim = make_case(dtype, D, G, P, lens=lens, pads=pads)
    if bound:
        q = q / 3  # N(0, 1) rows: |q.k| / sqrt(D) stays far below the bound
    need = ops.prefill_workspace_bytes(q.shape[2], q.shape[1], 2, D, dtype)
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device=DEV) if shares and need else False
    check(st, q, bidx, lim, P, dtype, workspace=ws, score_bound=bound)


@pytest.mark.parametrize("lens,pads", [([1], [0]), ([63, 64], [1, 0]), ([65], [62]), ([128, 129], [0, 63]), ([1000, 20], [0, 4]), ([1900, 1], [12, 0])],
                         ids=str)
@pytest.mark.parametrize("P", [64, 256])
@pytest.mark.parametrize("Hc_more", [1, 8], ids=["64-row-tiles", "past-their-line"])
def test_bounded_prompts_of_one_head_to_a_cache_head(lens, pads, P, Hc_more):
    """Tiles of 64 rows by four wavefronts, and (16 heads of 1913 rows: 480 of these tiles) the launches that do not take them: tiles of 128,
    whose halves take the key tiles in the same turns, so that the bits are the same."""
    dtype, D = torch.bfloat16, 128
    st, q, bidx, lim = make_case(dtype, D, 1, P, lens=lens, pads=pads)
    q = q / 3
    out, lse = check(st, q, bidx, lim, P, dtype, workspace=False, score_bound=39.0)
    pk, pv = (x.repeat(Hc_more, 1, 1) for x in st.pool_planes())
    more, more_lse = ops.paged_prefill(q.repeat(1, Hc_more, 1, 1).to(DEV), pk, pv, st.cache.page_table, bidx, lim, P, workspace=False, score_bound=39.0)
    assert torch.equal(more, out.repeat(1, Hc_more, 1, 1)) and torch.equal(more_lse.view(Hc_more, 2, -1), lse.view(1, 2, -1).expand(Hc_more, -1, -1))
