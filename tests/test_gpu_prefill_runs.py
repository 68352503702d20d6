"""GPU: query tiles that hold rows of several sequences and of padding, with their boundaries at the edges of the lanes that look
for them (64 rows to a lane register, up to four of them), against the oracle; whole workgroups, workgroups whose halves take the
key tiles in turn, and key shares.  Workgroups of 64 rows, which stage a key tile with two wavefronts: against the oracle and against
those of 128 rows, whose halves take the key tiles in the same turns, bit for bit."""

import numpy as np
import pytest
import torch

from falcon_perception_amd import ops
from oracle import paged_kv_oracle as O
from tests.gpu_cases import DEV, f64, kernels
from tests.test_gpu_prefill_few_rows import EIGHT, FOUR, check
from tests.test_gpu_prefill_key_shares import TOL, make_case
from tests.test_gpu_sink_gate import check_gated

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,bound", [(torch.bfloat16, 0.0), (torch.bfloat16, 39.0), (torch.float16, 0.0)], ids=str)
@pytest.mark.parametrize("D,G,P", [(128, 1, 64), (64, 1, 128), (128, 2, 32), (128, 4, 64), (64, 8, 64)])
@pytest.mark.parametrize("lens,pads", [
    ([1, 62, 1, 64, 63, 1], [0, 0, 0, 0, 0, 0]),   # boundaries at rows 1, 63, 64, 128, 191, 192
    ([31, 33, 65, 127], [1, 0, 0, 1]),             # 31, 32, 65, 130, 257 with single padding rows between
    ([5], [251]),                                  # one short run, the rest of a tile of 256 rows is padding
    ([256, 1], [0, 254]),                          # a run as long as the largest tile, then one row
    ([1000, 31, 1, 200], [0, 1, 0, 0]),            # with a workspace the first is cut along the keys, beside runs that are not
], ids=str)
@pytest.mark.parametrize("shares", [False, True], ids=["uncut", "key-shares"])
def test_runs_inside_a_tile(dtype, bound, D, G, P, lens, pads, shares):
    st, q, bidx, lim = make_case(dtype, D, G, P, lens=lens, pads=pads)
    if bound:
        q = q / 3  # N(0, 1) rows: |q.k| / sqrt(D) stays far below the bound
    need = ops.prefill_workspace_bytes(q.shape[2], q.shape[1], 2, D, dtype)
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device=DEV) if shares else False
    if shares:
        assert need > 0 and (ops.prefill_uncut_keys(q.shape[2], q.shape[1], 2, D, P, dtype) < max(lens)) == (max(lens) == 1000)
    check(st, q, bidx, lim, P, dtype, workspace=ws, score_bound=bound)


class Sixteen:
    """A bounded launch of one query head to a cache head on 16 heads, copies of the two of `make_case`: with the columns of the page table
    that its longest sequence needs, and with a wide table."""

    P: int

    def __init__(self, lens, pads, P):
        self.st, q, self.bidx, self.lim = make_case(torch.bfloat16, 128, 1, P, lens=lens, pads=pads)
        self.P, self.q2 = P, q / 3
        self.q = self.q2.repeat(1, 8, 1, 1).to(DEV)
        self.pk, self.pv = (x.repeat(8, 1, 1) for x in self.st.pool_planes())
        self.table = self.st.cache.page_table
        self.pages = -(-max(lens) // P)

    def run(self, wide=False, **kw):
        table = torch.cat([self.table, torch.full((self.table.shape[0], 64), -1, device=DEV)], 1) if wide else self.table[:, :self.pages]
        return ops.paged_prefill(self.q, self.pk, self.pv, table, self.bidx, self.lim, self.P, workspace=False, score_bound=39.0, **kw)

    def same(self, four=True, **kw):
        """The results, bit for bit those of the wide table."""
        got, wide = self.run(**kw), self.run(wide=True, **kw)
        names = [kernels(lambda: self.run(w, **kw)) for w in (False, True)]
        assert [len(n) for n in names] == [1, 1] and (FOUR if four else EIGHT) in names[0][0] and EIGHT in names[1][0]
        for a, b in zip(got, wide):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
        return got

    def holds(self, out, lse):
        """Every pair of heads against the oracle over the pool and the table as they are."""
        pk, pv = (f64(x[:2]) for x in (self.pk, self.pv))
        eo, el = O.prefill_attention_paged(f64(self.q2), pk, pv, self.table.cpu().numpy(), self.bidx.cpu().numpy(), None,
                                           self.lim.cpu().numpy(), self.P)
        atol, rtol = TOL[torch.bfloat16]
        for h in range(0, 16, 2):
            np.testing.assert_allclose(f64(out[:, h:h + 2]), eo, atol=atol, rtol=rtol)
            np.testing.assert_allclose(f64(lse[:, h:h + 2]), el, atol=max(atol * 0.1, 1e-4), rtol=rtol)


# `four`: goes out as workgroups of 64 rows in pages of 64 tokens; in pages of 256 the table ends up to three key tiles later
@pytest.mark.parametrize("lens,pads,four", [
    ([1], [0], True), ([63, 64], [1, 0], True), ([65], [62], True), ([128, 129], [0, 63], True), ([512], [0], True), ([704, 20], [0, 0], True),
    ([832], [0], True), ([833], [0], False), ([1000, 20], [0, 4], False), ([1900, 1], [12, 0], False)], ids=str)
@pytest.mark.parametrize("P", [64, 256])
def test_bounded_prompts_of_one_head_to_a_cache_head(lens, pads, four, P):
    case = Sixteen(lens, pads, P)
    rows = sum(lens) + sum(pads)
    short = case.pages * P <= 64 * min(5 + rows * 16 // 1500, 13)
    assert short == four or P == 256
    case.holds(*case.same(four=short))


@pytest.mark.parametrize("lens,pads", [([63, 64], [1, 0]), ([613], [27]), ([100, 300, 40], [28, 0, 3])], ids=str)
def test_the_sink_gate_of_64_row_workgroups(lens, pads):
    case = Sixteen(lens, pads, 64)
    plain, lse = case.same()
    sinks = torch.linspace(-2, 3, 16, device=DEV)
    gated, lse2 = case.same(sinks=sinks)
    assert torch.equal(lse, lse2)
    check_gated(gated, plain, lse, sinks, torch.bfloat16)


@pytest.mark.parametrize("value", [float("nan"), float("inf")], ids=str)
@pytest.mark.parametrize("lens,pads", [([1], [0]), ([63, 64, 65], [1, 0, 2]), ([613], [27]), ([127, 129], [1, 0])], ids=str)
@pytest.mark.parametrize("P", [64, 128])
def test_64_row_workgroups_leave_out_what_is_behind_the_last_key(lens, pads, P, value):
    case = Sixteen(lens, pads, P)
    clean = case.same()
    for slot, n in zip(case.st.slots, lens):
        for at in range(n, -(-n // P) * P):
            row = int(case.table[slot, at // P]) * P + at % P
            case.pk[:, row], case.pv[:, row] = value, value
    for a, b in zip(case.same(), clean):
        assert torch.equal(a, b)


@pytest.mark.parametrize("value", [float("nan"), float("inf")], ids=str)
@pytest.mark.parametrize("L", [1, 63, 64, 100, 576])
def test_the_last_key_of_64_row_workgroups(L, value):
    """An element of the last key's V in rows that all see it: there and nowhere else."""
    case = Sixteen([L], [0], 64)
    case.lim = torch.full_like(case.lim, L)
    out, lse = case.same()
    last = int(case.table[case.st.slots[0], (L - 1) // 64]) * 64 + (L - 1) % 64
    case.pv[:, last, 5] = value
    got, lse2 = case.same()
    keep = [d for d in range(128) if d != 5]
    assert (got[..., 5].isnan() if value != value else got[..., 5] == value).all()
    assert torch.equal(got[..., keep], out[..., keep]) and torch.equal(lse2, lse)


@pytest.mark.parametrize("lens,pads,hole", [([613], [27], 0), ([613], [27], 1), ([200, 128], [0, 0], 1), ([63, 300], [1, 0], 4)], ids=str)
@pytest.mark.parametrize("P", [64, 128])
def test_64_row_workgroups_over_a_page_that_is_not_there(lens, pads, hole, P):
    """A page without an entry is staged row by row, every row of it slot 0: what a page full of copies of that row gives."""
    case = Sixteen(lens, pads, P)
    slot = case.st.slots[lens.index(max(lens))]
    hole = min(hole, case.pages - 1)
    spare = min(set(range(1, case.pk.shape[1] // P)) - set(case.table.flatten().tolist()))
    for x in (case.pk, case.pv):
        x[:, spare * P:(spare + 1) * P] = x[:, :1]
    case.table[slot, hole] = spare
    mapped = case.same()
    case.holds(*mapped)
    case.table[slot, hole] = -1
    for a, b in zip(case.same(), mapped):
        assert torch.equal(a, b)
