"""GPU: prefill launches of few rows, whose workgroups split the key tiles between their two halves, and the tail tile of a
run, against the oracle.  The tolerances are those of the other prefill tests: the rounding of the results and of the
probabilities to the dtype."""

import numpy as np
import pytest
import torch
from torch.nn.attention.flex_attention import AuxRequest

from falcon_perception_amd import attention as A
from falcon_perception_amd import ops
from oracle import paged_kv_oracle as O
from tests.gpu_cases import DEV, PagedState, f64, kernels, randn
from tests.test_gpu_prefill_key_shares import TOL, make_case

pytestmark = pytest.mark.gpu


def check(st, q, bidx, lim, P, dtype, **kw):
    pk, pv = st.pool_planes()
    out, lse = ops.paged_prefill(q.to(DEV), pk, pv, st.cache.page_table, bidx, lim, P, **kw)
    eo, el = O.prefill_attention_paged(f64(q), f64(pk), f64(pv), st.mirror.page_table, bidx.cpu().numpy(), None,
                                       lim.cpu().numpy(), P)
    atol, rtol = TOL[dtype]
    np.testing.assert_allclose(f64(out), eo, atol=atol, rtol=rtol)
    np.testing.assert_allclose(f64(lse), el, atol=max(atol * 0.1, 1e-4), rtol=rtol)
    return out, lse


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("D,G,P", [(128, 1, 128), (64, 2, 64), (128, 4, 16), (64, 1, 24), (128, 2, 256), (64, 4, 128)])
@pytest.mark.parametrize("lens,pads", [([1], [0]), ([63, 64, 65], [1, 0, 2]), ([127], [1]), ([129, 3], [0, 60]), ([192, 1], [0, 0])], ids=str)
def test_sizes_around_the_tiles(dtype, D, G, P, lens, pads):
    """One key tile (the second half of the workgroup has none), odd and even numbers of them, tails of one key."""
    st, q, bidx, lim = make_case(dtype, D, G, P, lens=lens, pads=pads)
    check(st, q, bidx, lim, P, dtype, workspace=False)


@pytest.mark.parametrize("lens", [[256], [320], [321, 40], [385, 20], [960], [961, 40], [1025, 20]], ids=str)
@pytest.mark.parametrize("D,G", [(128, 1), (64, 4), (128, 8)])
def test_ranges_around_the_first_second_share(lens, D, G):
    """4 to 7 and 15 to 17 key tiles: the launch has key shares, a run of up to about five tiles is not cut, and a launch
    holds cut and uncut runs side by side.  The workspace starts as NaN: nothing that no share wrote may come through."""
    dtype, P = torch.bfloat16, 64
    st, q, bidx, lim = make_case(dtype, D, G, P, lens=lens, pads=[5] + [0] * (len(lens) - 1))
    need = ops.prefill_workspace_bytes(q.shape[2], q.shape[1], 2, D, dtype)
    assert need > 0
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device=DEV)
    check(st, q, bidx, lim, P, dtype, workspace=ws)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("rows", [100, 2 * 128 * 140])
def test_rows_behind_the_last_key_stay_out(dtype, rows):
    """The page rows behind a sequence's last key hold NaN: launches of few rows and of many (one sequence repeated
    as rows over the same keys)."""
    D, G, P = 128, 1, 128
    st, q, bidx, lim = make_case(dtype, D, G, P, lens=[100], pads=[0])
    pk, pv = st.pool_planes()
    page = int(st.cache.page_table[st.slots[0], 0])
    pk[:, page * P + 100:(page + 1) * P] = float("nan")
    pv[:, page * P + 100:(page + 1) * P] = float("nan")
    n = -(-rows // 100)
    out, lse = ops.paged_prefill(q.repeat(1, 1, n, 1).to(DEV), pk, pv, st.cache.page_table, bidx.repeat(n), lim.repeat(n), P,
                                 workspace=False)
    assert torch.isfinite(out).all() and torch.isfinite(lse).all()
    for part in (pk, pv):
        part[:, page * P + 100:(page + 1) * P] = 0.0
    ref, _ = check(st, q, bidx, lim, P, dtype, workspace=False)
    atol, rtol = TOL[dtype]
    np.testing.assert_allclose(f64(out[:, :, -100:]), f64(ref), atol=atol, rtol=rtol)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("D,G", [(128, 1), (64, 4), (128, 8)])
@pytest.mark.parametrize("L", [1, 63, 100, 700])
@pytest.mark.parametrize("repeat", [1, 60])
@pytest.mark.parametrize("cut", [False, True], ids=["uncut", "key-shares"])
def test_an_infinite_value_in_the_last_key(dtype, D, G, L, repeat, cut):
    """The rows of the last tile behind the last key have no weight, and none of its infinity either: every row sees every key,
    so the element is infinite in every row and the others keep their bits (launches of few rows and of many)."""
    P = 128
    st, q, bidx, lim = make_case(dtype, D, G, P, lens=[L], pads=[0])
    q, bidx, lim = (0.1 * q).repeat(1, 1, repeat, 1).to(DEV), bidx.repeat(repeat), torch.full_like(lim, L).repeat(repeat)
    pk, pv = st.pool_planes()
    last = int(st.cache.page_table[st.slots[0], (L - 1) // P]) * P + (L - 1) % P
    args = (q, pk, pv, st.cache.page_table, bidx, lim, P)
    out, lse = ops.paged_prefill(*args, workspace=None if cut else False)
    pv[:, last, 5] = float("inf")
    got, lse2 = ops.paged_prefill(*args, workspace=None if cut else False)
    keep = [d for d in range(D) if d != 5]
    assert (got[..., 5] == float("inf")).all() and torch.equal(got[..., keep], out[..., keep]) and torch.equal(lse2, lse)


@pytest.mark.parametrize("P", [64, 32, 24])
@pytest.mark.parametrize("D,G,rows", [(128, 1, 64), (64, 2, 250), (128, 8, 100), (128, 4, 200)])
def test_a_launch_without_key_shares_needs_no_workspace(D, G, rows, P):
    """Up to `prefill_uncut_keys` the bits are those of the launch without a workspace; four tiles on it is cut."""
    dtype, Hc = torch.bfloat16, 2
    uncut = ops.prefill_uncut_keys(rows, Hc * G, Hc, D, P, dtype)
    assert uncut % 64 == 0 and uncut >= rows and ops.prefill_workspace_bytes(rows, Hc * G, Hc, D, dtype) > 0
    for keys, same in ((uncut, True), (uncut + 256, False)):
        st, q, bidx, lim = make_case(dtype, D, G, P, lens=[keys], pads=[0])
        q, bidx, lim = q[:, :, -rows:].to(DEV), bidx[-rows:].contiguous(), lim[-rows:].contiguous()
        pk, pv = st.pool_planes()
        args = (q, pk, pv, st.cache.page_table, bidx, lim, P)
        out, lse = ops.paged_prefill(*args)
        plain = ops.paged_prefill(*args, workspace=False)
        assert (torch.equal(out, plain[0]) and torch.equal(lse, plain[1])) == same


@pytest.mark.parametrize("rows", [100, 613])
def test_a_prompt_does_not_depend_on_who_else_is_cached(rows):
    """The drop-in leaves the workspace out where no cached sequence is long enough for key shares: a long sequence that
    is not in the step brings the workspace back and changes no bit."""
    dtype, Hc, D, P = torch.bfloat16, 16, 128, 128
    results, used = [], []
    for resident in (0, 6000):
        st = PagedState(19, n_pages=64, page_size=P, max_batch=4, Hc=Hc, D=D, dtype=dtype)
        cache = st.cache
        slot = st.add_sequence(rows)
        if resident:
            st.add_sequence(resident)
        L = -(-rows // 128) * 128
        gen = torch.Generator().manual_seed(5)
        q, k, v = (randn(gen, (1, Hc, L, D), dtype).to(DEV) for _ in range(3))
        live = torch.arange(L, device=DEV)[None] < rows
        bidx = torch.where(live, slot, 0)
        pos = torch.where(live, torch.arange(L, device=DEV)[None], 0)
        mask = cache.create_prefill_blockmask(bidx, torch.full_like(bidx, 9), 1, 2)
        K, V = cache.insert_kv(0, k, v, input_pos=pos, batch_idx=bidx)
        out, aux = A.compiled_flex_attn_prefill(q, K, V, block_mask=mask, return_aux=AuxRequest(lse=True))
        results.append((out, aux.lse))
        used.append(cache.prefill_workspace(L, Hc, D, Hc, dtype, mask.most_keys) is not False)
    assert used == [False, True]
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])


FOUR, EIGHT = ("paged_prefill_kernel<BF16, 128, 1, true, %d, true, 2>" % w for w in (4, 8))


@pytest.mark.parametrize("lens,pages,rows", [
    ([320], 5, 64), ([320], 6, 64), ([1464], 23, 64), ([613], 11, 613), ([613], 12, 613), ([704], 11, 613), ([1400], 22, 613),
    ([832], 13, 832), ([832], 14, 832), ([500, 500], 13, 1000), ([500, 500], 14, 1000), ([1000], 16, 1000)], ids=str)
def test_workgroups_of_64_rows_are_for_short_ranges(lens, pages, rows):
    """What a launch knows of the rows' key ranges is the width of the page table.  Over long ranges workgroups of 64 rows are the
    slower ones (64 rows over 1400 keys 29.2 us instead of 26.0), also without a workspace; the bits are the same."""
    dtype, P, heads = torch.bfloat16, 64, 8
    st, q, bidx, lim = make_case(dtype, 128, 1, P, lens=lens, pads=[0] * len(lens))
    q, bidx, lim = (q[:, :, -rows:] / 3).repeat(1, heads, 1, 1).to(DEV), bidx[-rows:].contiguous(), lim[-rows:].contiguous()
    pk, pv = (x.repeat(heads, 1, 1) for x in st.pool_planes())
    table = st.cache.page_table
    wide = torch.cat([table, torch.full_like(table, -1), torch.full_like(table, -1)], 1)
    short = 64 * min(5 + rows * 16 // 1500, 13)

    def run(columns):
        return ops.paged_prefill(q, pk, pv, wide[:, :columns], bidx, lim, P, workspace=False, score_bound=39.0)

    assert wide.shape[1] * P > short and pages <= wide.shape[1]
    ways = [kernels(lambda c=c: run(c)) for c in (pages, wide.shape[1])]
    assert [len(w) for w in ways] == [1, 1]
    assert (FOUR if pages * P <= short else EIGHT) in ways[0][0] and EIGHT in ways[1][0]
    (out, lse), (out2, lse2) = run(pages), run(wide.shape[1])
    assert torch.equal(out, out2) and torch.equal(lse, lse2)


def test_the_drop_in_says_how_long_its_sequences_are():
    """A prompt in a cache whose table has columns for 8192 tokens; the same prompt once a sequence of 6000 tokens is cached."""
    dtype, Hc, D, P, rows = torch.bfloat16, 16, 128, 128, 613
    st = PagedState(19, n_pages=64, page_size=P, max_batch=4, Hc=Hc, D=D, dtype=dtype)
    cache, L = st.cache, 640
    cache.qk_normalised = True
    slot, results = st.add_sequence(rows), []
    q, k, v = (randn(st.gen, (1, Hc, L, D), dtype).to(DEV) for _ in range(3))
    q = q / 3
    live = torch.arange(L, device=DEV)[None] < rows
    bidx, pos = torch.where(live, slot, 0), torch.where(live, torch.arange(L, device=DEV)[None], 0)
    for way in ([FOUR], [EIGHT, "paged_prefill_merge_kernel"]):

        def run():
            mask = cache.create_prefill_blockmask(bidx, torch.full_like(bidx, 9), 1, 2)
            K, V = cache.insert_kv(0, k, v, input_pos=pos, batch_idx=bidx)
            return A.compiled_flex_attn_prefill(q, K, V, block_mask=mask, return_aux=AuxRequest(lse=True))

        seen = [n for n in kernels(run) if "paged_prefill" in n]
        assert len(seen) == len(way) and all(w in n for w, n in zip(way, seen))
        out, aux = run()
        results.append((out, aux.lse))
        if len(results) == 1:
            st.add_sequence(6000)
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
