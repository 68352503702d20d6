"""GPU: the cut of a decode launch whose sequences are much shorter than the limit the launch is sized for, as an
engine's are (its mask is as long as the longest sequence it may ever hold)."""

import numpy as np
import pytest
import torch

from falcon_perception_amd import ops
from oracle import paged_kv_oracle as O
from tests.gpu_cases import DEV, PagedState, f64, randn

pytestmark = pytest.mark.gpu

ATOL, RTOL = 2e-2, 1e-2


# chunks per cache head: 2 * 256 CUs / 8 heads = 64.  8 and 13 sequences (8 chunks each, eight splits of 512 tokens) are cut
# evenly, 7 and 64 because their workgroups do not fit the GPU at once, one goes split by split
@pytest.mark.parametrize("B", [1, 7, 8, 13, 64])
@pytest.mark.parametrize("P", [32, 24], ids=["pages-of-32", "pages-of-24"])
def test_short_sequences_under_a_long_limit(B, P):
    dtype, Hc, G, D, limit = torch.bfloat16, 8, 2, 128, 4096
    lens = [1, 63, 64, 65, 700, 320, 127, 511][:B] + [33 + 7 * i for i in range(max(0, B - 8))]
    st = PagedState(210 + B, n_pages=limit // P + 1 + sum(-(-L // P) for L in lens), page_size=P, max_batch=B + 2, Hc=Hc,
                    D=D, dtype=dtype)
    for L in lens:
        st.add_sequence(L)
    st.prefill_random()
    q = randn(st.gen, (B, Hc * G, 1, D), dtype).to(DEV)
    pos = torch.tensor(lens, dtype=torch.int32, device=DEV) - 1
    bidx = torch.tensor(st.slots, dtype=torch.int64, device=DEV)
    pk, pv = st.pool_planes()
    args = (q, pk, pv, st.cache.page_table, bidx, pos, P, limit // P * P)
    out, lse = ops.paged_decode(*args)
    plan = torch.zeros(ops.decode_plan_bytes(), dtype=torch.uint8, device=DEV)
    ops.paged_decode(*args, phase="plan", plan=plan)
    planned_batch = int(plan.view(torch.int32)[1])  # the even cut writes a plan, a launch split by split does not
    assert planned_batch == (B if B >= 7 else 0)
    planned = ops.paged_decode(*args, plan=plan)
    assert torch.equal(planned[0], out) and torch.equal(planned[1], lse)
    eo, el = O.decode_attention(f64(q), f64(pk), f64(pv), st.mirror.page_table, st.slots, np.array(lens) - 1, P)
    np.testing.assert_allclose(f64(out), eo, atol=ATOL, rtol=RTOL)
    np.testing.assert_allclose(f64(lse), el, atol=ATOL * 0.1, rtol=RTOL)
