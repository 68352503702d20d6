"""GPU: heads and rows whose vectors per token are and are not a power of two (shifts and divisions in the append kernel), both memory orders
of the source, against an index assignment.  Byte-exact."""

import pytest
import torch

from falcon_perception_amd import ops
from tests.gpu_cases import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [1, 2, 3, 16, 24])
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (80, torch.float16), (128, torch.float32), (6, torch.bfloat16), (1, torch.float32)], ids=str)
@pytest.mark.parametrize("order", ["tokens-outside", "heads-outside"])
def test_vectors_per_token(H, D, dtype, order):
    T, P, n_pages = 77, 8, 12
    gen = torch.Generator().manual_seed(H * 100 + D)
    shape = (T, H, D) if order == "tokens-outside" else (H, T, D)
    k, v = (torch.randn(shape, generator=gen).to(dtype).to(DEV) for _ in range(2))
    if order == "heads-outside":
        k, v = k.transpose(0, 1), v.transpose(0, 1)
    table = (torch.randperm(n_pages - 1, generator=gen) + 1)[None].repeat(2, 1).to(DEV)
    bidx = torch.ones(1, T, dtype=torch.int64, device=DEV)
    pos = torch.randperm(table.shape[1] * P, generator=gen)[:T][None].to(DEV)
    pools = [torch.zeros(H, n_pages * P, D, dtype=dtype, device=DEV) for _ in range(2)]
    expected = [p.clone() for p in pools]
    packed = [x.transpose(0, 1)[None] for x in (k, v)]  # [1, H, T, D]
    ops.kv_append(*pools, *packed, table, bidx, pos, P, clamp_negative=False, packed=True)
    slot = table[1, pos[0] // P] * P + pos[0] % P
    for e, x, p in zip(expected, packed, pools):
        e[:, slot] = x[0]
        assert torch.equal(e, p)
