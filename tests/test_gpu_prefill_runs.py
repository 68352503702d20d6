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
