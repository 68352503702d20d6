"""GPU parity: the decode step as one launch (fp_paged_decode_step).

The last workgroup to leave a partial result merges them, so that a launch has no merge pass.  The pieces and their partial
results are those of the two passes (which the other decode tests hold against the float64 oracle), only the sums over the pieces
run in another order: in fp32 that moves a result by less than n * 2^-23 of the largest term for n pieces (n <= 64 here, and
the weights add up to 1), and the type's rounding comes on top.
"""

import pytest
import torch
from torch.nn.attention.flex_attention import AuxRequest, BlockMask

from falcon_perception_amd import attention as A
from falcon_perception_amd import ops
from tests.gpu_cases import DEV, PagedState, randn
from tests.test_gpu_decode_plan import decode, flat_state, new_plan

pytestmark = pytest.mark.gpu

STEP = {torch.bfloat16: 2.0**-7, torch.float16: 2.0**-10, torch.float32: 0.0}  # distance of two neighbours, relative


def close(got, ref, dtype, n):
    (out, lse), (ro, rl) = got, ref
    bound = 2 * n * 2.0**-23
    assert not (out.isnan() ^ ro.isnan()).any()
    tol = STEP[dtype] * ro.float().abs() + bound * (1 + ro.float().abs().amax(-1, keepdim=True))
    assert ((out.float() - ro.float()).abs() <= tol).all()
    same = torch.isneginf(lse) == torch.isneginf(rl)
    assert same.all() and ((lse - rl).abs().nan_to_num(0.0) <= bound * (1 + rl.abs().nan_to_num(0.0, 0.0, 0.0))).all()


def holds(got, st, q, pos, bidx, ctx, dtype, split_p):
    """`got` against float64 over the pool as it is, each sequence within what its own keys can be off by: a score by 12 roundings of
    sum |q k|, the sums of a lane over n / 16 of n keys by two roundings a key, and as many for pieces, wavefronts and the last
    division as 64 cover; `split_p`: probabilities in two 16-bit parts, 2^-16 of each is left over in bf16.  A key that is missing or
    counted twice, or a piece a few per cent off in weight, is more than that."""
    (out, lse), (pk, pv) = got, st.pool_planes()
    B, Hq, _, D = q.shape
    scale = D**-0.5
    table = st.cache.page_table
    for b in range(B):
        slot, n = int(bidx[b]), min(int(pos[b]) + 1, ctx)
        if n <= 0 or not 0 <= slot < table.shape[0]:
            assert not out[b].any() and torch.isneginf(lse[b]).all(), b
            continue
        t = torch.arange(n, device=DEV)
        slots = table[slot, t // st.P].clamp(min=0) * st.P + t % st.P  # without a page: page 0
        K, V = (x[:, slots].double().repeat_interleave(Hq // x.shape[0], 0) for x in (pk, pv))
        Q = q[b].double()
        s = Q @ K.transpose(1, 2) * scale
        p = torch.softmax(s, -1)
        off = (12 * scale * (Q.abs() @ K.abs().transpose(1, 2)).amax(-1) + n / 8 + 64) * 2.0**-24 + split_p * 2.0**-16
        ref, size = p @ V, p @ V.abs()
        assert ((out[b].double() - ref).abs() <= off[..., None] * size + STEP[dtype] / 2 * ref.abs() + 2.0**-25 * (dtype == torch.float16)).all(), b
        assert ((lse[b].double() - torch.logsumexp(s, -1)).abs() <= 2 * off).all(), b


def inputs(st, B, Hc, G, D, dtype, rep):
    q = randn(st.gen, (B, Hc * G, 1, D), dtype).to(DEV)
    k_new = randn(st.gen, (B, Hc * rep, 1, D), dtype).to(DEV)
    v_new = randn(st.gen, (B, Hc, 1, D), dtype).repeat_interleave(rep, dim=1).to(DEV)
    return q, k_new, v_new


# split by split: one sequence of 64 splits (8 heads: of 32 twice as long ones), of 33, of 17 and of 1, a few of different
# lengths; cut evenly, where the merge pass stays
@pytest.mark.parametrize("cut", ["all", "33", "17", "one", "few", "even"])
@pytest.mark.parametrize("dtype,D,P,G,rep", [
    (torch.bfloat16, 128, 64, 2, 1), (torch.bfloat16, 64, 24, 4, 1), (torch.float32, 64, 16, 1, 1), (torch.float32, 128, 32, 8, 1),
    (torch.float16, 128, 48, 8, 1), (torch.bfloat16, 128, 64, 2, 2), (torch.float16, 64, 64, 1, 1), (torch.bfloat16, 64, 16, 4, 4)],
    ids=str)
def test_one_launch_gives_what_the_two_passes_give(cut, dtype, D, P, G, rep):
    B, Hc, split, ctx = {"all": (1, 8, 64, 4096), "33": (1, 8, 64, 64 * 33), "17": (1, 8, 64, 64 * 17), "one": (1, 8, 64, 128),
                         "few": (7, 4, 128, 1536), "even": (96, 4, 64, 512)}[cut]
    lens = {"all": [4090], "33": [64 * 33 - 1], "17": [64 * 16], "one": [63], "few": [1535, 0, 700, 127, 128, 1, 900], "even": None}[cut]
    st = flat_state(17 + D + G, B, Hc, D, P, ctx, dtype, rep, lens)
    q, k_new, v_new = inputs(st, B, Hc, G, D, dtype, rep)
    pos = torch.tensor(st.lens, dtype=torch.int32, device=DEV)
    bidx = torch.tensor(st.slots, dtype=torch.int64, device=DEV)
    if B > 20:
        pos[5], bidx[9], bidx[11], pos[13] = -1, B + 40, -3, ctx + 7  # no key, foreign slots, beyond the launch's limit
    elif B > 1:
        pos[1], bidx[6] = -1, B + 40
    arrivals = torch.zeros(B * Hc, dtype=torch.int32, device=DEV)
    before = st.cache.kv_cache.clone()
    sinks = torch.linspace(-2, 3, Hc * G, device=DEV)
    for gate in (None, sinks):
        kw = dict(max_context=ctx, split_tokens=split, kv_rep=rep, bidx=bidx, sinks=gate)
        st.cache.kv_cache.copy_(before)
        ref = decode(st, q, pos, k_new=k_new, v_new=v_new, **kw)
        pool = st.cache.kv_cache.clone()
        plan = new_plan()
        decode(st, q, pos, phase="plan", plan=plan, **kw)
        for p in (None, plan, new_plan(0xA5)):
            st.cache.kv_cache.copy_(before)
            got = decode(st, q, pos, k_new=k_new, v_new=v_new, plan=p, arrivals=arrivals, **kw)
            close(got, ref, dtype, 64)
            assert torch.equal(st.cache.kv_cache, pool)
            assert not arrivals.any()
            again = decode(st, q, pos, plan=p, arrivals=arrivals, **kw)  # the rows are in the pool now
            close(again, ref, dtype, 64)
            assert not arrivals.any()


def test_counters_too_small_are_refused():
    st = flat_state(6, 4, 2, 64, 32, 256, torch.float32)
    q, *_ = inputs(st, 4, 2, 1, 64, torch.float32, 1)
    pos = torch.tensor(st.lens, dtype=torch.int32, device=DEV)
    with pytest.raises(RuntimeError, match="arrival counters"):
        decode(st, q, pos, max_context=256, split_tokens=64, arrivals=torch.zeros(8 - 1, dtype=torch.int32, device=DEV))
    with pytest.raises(RuntimeError, match="int32"):
        decode(st, q, pos, max_context=256, split_tokens=64, arrivals=torch.zeros(8, dtype=torch.int64, device=DEV))
    with pytest.raises(RuntimeError, match="both passes"):
        decode(st, q, pos, max_context=256, split_tokens=64, phase="merge", arrivals=torch.zeros(8, dtype=torch.int32, device=DEV))


def test_replays_of_a_captured_step():
    """Layers that share workspace and counters, replayed with the positions advancing in place."""
    dtype, B, Hc, G, D, P, split, ctx = torch.bfloat16, 6, 8, 2, 128, 32, 128, 1024
    st = flat_state(8, B, Hc, D, P, ctx - 40, dtype)
    q, *_ = inputs(st, B, Hc, G, D, dtype, 1)
    pos = torch.tensor(st.lens, dtype=torch.int32, device=DEV)
    arrivals = torch.zeros(B * Hc, dtype=torch.int32, device=DEV)
    ws = torch.empty(ops.decode_workspace_bytes(B, Hc * G, D, ctx, split), dtype=torch.uint8, device=DEV)
    outs = [(torch.empty_like(q), torch.empty((B, Hc * G, 1), device=DEV)) for _ in range(3)]
    bidx = torch.tensor(st.slots, dtype=torch.int64, device=DEV)

    def layers():
        for o, l in outs:
            decode(st, q, pos, bidx=bidx, max_context=ctx, split_tokens=split, workspace=ws, arrivals=arrivals, out=o, lse=l)

    layers()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        layers()
    for _ in range(6):
        ref = decode(st, q, pos, bidx=bidx, max_context=ctx, split_tokens=split)
        graph.replay()
        for got in outs:
            close(got, ref, dtype, 64)
        assert not arrivals.any()
        pos -= 13


# piece by piece: the fewest sequences and few of them, more than 16 pieces' worth of one, some without keys, all shorter than a
# piece, the most sequences; page sizes that are no power of two; the first shapes on the other side of each line
PIECES = {"three": (3, 16, 2048, [1, 2047, 300]), "uneven": (9, 8, 8192, [8190, 0, 63, 64, 127, 4000, 65, 1, 700]),
          "empty": (8, 8, 1536, [-1, 1535, -1, 200, 0, 0, 129, 999]), "short": (40, 8, 1024, None), "most": (48, 4, 1100, None)}


@pytest.mark.parametrize("case", PIECES)
@pytest.mark.parametrize("dtype,D,P,G,rep", [
    (torch.bfloat16, 128, 64, 2, 1), (torch.bfloat16, 64, 24, 4, 1), (torch.float32, 64, 16, 1, 1), (torch.float32, 128, 32, 2, 1),
    (torch.bfloat16, 128, 48, 2, 2), (torch.float16, 64, 128, 1, 1), (torch.bfloat16, 64, 16, 4, 4)], ids=str)
def test_piece_by_piece_gives_what_the_two_passes_give(case, dtype, D, P, G, rep):
    B, Hc, ctx, lens = PIECES[case]
    if lens is None:
        lens = [(37 * i * i + 11 * i) % (250 if case == "short" else ctx - 2) for i in range(B)]
    split = ops.decode_split_tokens(B, Hc, ctx, P)
    assert ops.decode_step_pieces(B, Hc * G, Hc * rep, rep, D, ctx, P, split) > 0
    st = flat_state(31 + D + G, B, Hc, D, P, ctx, dtype, rep, [max(n, 0) for n in lens])
    q, k_new, v_new = inputs(st, B, Hc, G, D, dtype, rep)
    bidx = torch.tensor(st.slots, dtype=torch.int64, device=DEV)
    if B > 20:
        lens[5], lens[13], bidx[9], bidx[11] = -1, ctx + 7, B + 40, -3  # no key, beyond the launch's limit, foreign slots
    before = st.cache.kv_cache.clone()
    arrivals = torch.zeros(B * Hc * 5 + 3, dtype=torch.int32, device=DEV)  # counters five words apart
    kw = dict(max_context=ctx, split_tokens=split, kv_rep=rep, bidx=bidx)
    # the pieces are others than the splits, so the sums over the keys run in another order: n = keys in `close`, which says little of
    # a long sequence; `holds` bounds each by itself
    for pos_type in (torch.int32, torch.int64):
        pos = torch.tensor(lens, dtype=pos_type, device=DEV)
        if pos_type is torch.int64 and B > 20:
            pos[13], pos[5] = 2**40, -(2**40)
        st.cache.kv_cache.copy_(before)
        ref = decode(st, q, pos, k_new=k_new, v_new=v_new, **kw)
        pool = st.cache.kv_cache.clone()
        st.cache.kv_cache.copy_(before)
        got = decode(st, q, pos, k_new=k_new, v_new=v_new, arrivals=arrivals, **kw)
        close(got, ref, dtype, ctx)
        assert torch.equal(st.cache.kv_cache, pool) and not arrivals.any()
        holds(got, st, q, pos, bidx, ctx, dtype, G >= 4 and dtype == torch.bfloat16)


def test_which_launches_go_piece_by_piece():
    def pieces(B, Hc, limit, G=2, D=128, P=64, rep=1):
        return ops.decode_step_pieces(B, Hc * G, Hc * rep, rep, D, limit, P, 0)

    assert [pieces(B, 8, 8192) > 0 for B in (1, 3, 4, 16, 17, 63, 64)] == [False, False, True, True, False, False, False]
    assert pieces(48, 8, 1024) > 0 and pieces(49, 8, 1024) == 0
    assert pieces(2, 16, 8192) == 0 and pieces(3, 16, 8192) > 0 and pieces(7, 4, 8192) == 0 and pieces(8, 4, 8192) > 0
    assert pieces(16, 8, 1024) == 0 and pieces(17, 8, 1024) > 0  # the splits fill the CUs as it is
    assert pieces(8, 8, 8192, G=4) == 0 and pieces(8, 8, 8192, G=4, D=64) > 0  # more than 256 elements a merge
    assert pieces(8, 8, 128) == 0 and pieces(8, 8, 0) == 0  # one split
    with pytest.raises(RuntimeError):
        pieces(0, 8, 8192)


def drop_in_state(B, Hc, D, P, ctx, dtype, layers, lens):
    """A cache with `lens` tokens per sequence in every layer, and the positions and mask of the step after them."""
    st = PagedState(57, n_pages=ctx // P + sum(-(-(n + 4) // P) for n in lens), page_size=P, max_batch=B + 2, Hc=Hc, D=D, dtype=dtype,
                    n_layers=layers)
    for n in lens:
        st.add_sequence(n + 4)
    st.cache.kv_cache.normal_()
    bidx, pos = torch.tensor(st.slots, dtype=torch.int64, device=DEV), torch.tensor(lens, dtype=torch.int32, device=DEV)
    full = st.cache.create_causal_blockmask(B=1, L=ctx)
    row, blk = torch.zeros_like(bidx), (pos // P).long()
    logical = BlockMask.from_kv_blocks(
        full.kv_num_blocks[row, :, blk].view(B, 1, 1), full.kv_indices[row, :, blk].view(B, 1, 1, -1),
        full.full_kv_num_blocks[row, :, blk].view(B, 1, 1), full.full_kv_indices[row, :, blk].view(B, 1, 1, -1),
        BLOCK_SIZE=full.BLOCK_SIZE, mask_mod=lambda b, h, q, kv: q + pos[b] >= kv, seq_lengths=(1, ctx))
    return st, st.cache.convert_logical_block_mask(logical, bidx), bidx, pos


# split by split; piece by piece; on the matrix cores
@pytest.mark.parametrize("layers", [2, 3])
@pytest.mark.parametrize("B,G,D,dtype", [(2, 2, 128, torch.bfloat16), (9, 1, 64, torch.float32), (9, 4, 64, torch.float16)], ids=str)
def test_counters_that_are_not_zero_spoil_one_launch(B, G, D, dtype, layers):
    """Launches that overlapped on one cache, against its contract, may leave counters behind; the layers after the next one and
    every later step are right again."""
    Hc, P, ctx = 8, 64, 4096
    lens = [4000 - 431 * i for i in range(B)]
    lens[1] = 0
    st, mask, bidx, pos = drop_in_state(B, Hc, D, P, ctx, dtype, layers, lens)
    cache = st.cache
    for left_over in (1, 3, 1000):
        sets = cache._decode_arrivals if isinstance(cache._decode_arrivals, tuple) else (cache._decode_arrivals,)
        for t in sets:
            t.fill_(left_over)
        for step in range(2):
            for layer in range(layers):
                q, k, v = (randn(st.gen, (B, h, 1, D), dtype).to(DEV) for h in (Hc * G, Hc, Hc))
                K, V = cache.insert_kv(layer, k, v, input_pos=pos.view(B, 1), batch_idx=bidx)
                out, aux = A.compiled_flex_attn_decode(q, K, V, block_mask=mask, return_aux=AuxRequest(lse=True))
                if step == 0 and layer == 0:
                    continue
                eo, el = ops.paged_decode(q, K[0], V[0], cache.page_table, bidx, pos, P, mask.max_context)
                torch.testing.assert_close(out, eo, rtol=max(2 * STEP[dtype], 1e-5), atol=1e-5)
                torch.testing.assert_close(aux.lse.view(el.shape), el, rtol=1e-5, atol=1e-5)


def test_counters_of_the_next_launch():
    """They are set to 0 for the sequences of the launch, whether a sequence has splits to merge or not, and lie elsewhere."""
    B, Hc, ctx = 4, 2, 256
    st = flat_state(6, B, Hc, 64, 32, ctx, torch.float32, 1, [255, 0, 60, 130])
    q, *_ = inputs(st, B, Hc, 1, 64, torch.float32, 1)
    pos = torch.tensor([255, -1, 60, 130], dtype=torch.int32, device=DEV)
    sets = torch.zeros(3, 24, dtype=torch.int32, device=DEV)  # counters three words apart
    sets[1:] = 7
    kw = dict(max_context=ctx, split_tokens=64, bidx=torch.tensor(st.slots, dtype=torch.int64, device=DEV))
    ref = decode(st, q, pos, **kw)
    got = decode(st, q, pos, arrivals=sets[0], next_arrivals=sets[1], **kw)
    close(got, ref, torch.float32, 64)
    assert not sets[0].any() and not sets[1, ::3].any() and (sets[1].view(8, 3)[:, 1:] == 7).all() and (sets[2] == 7).all()
    for after, match in ((sets[0], "overlap"), (sets.view(-1)[20:44], "overlap"), (sets[1, :8], "like arrivals"), (sets[1].float(), "like arrivals")):
        with pytest.raises(RuntimeError, match=match):
            decode(st, q, pos, arrivals=sets[0], next_arrivals=after, **kw)


@pytest.mark.parametrize("case", [*PIECES, "splits"])
@pytest.mark.parametrize("dtype,D,P,G,rep", [
    (torch.bfloat16, 128, 64, 2, 1), (torch.float32, 64, 16, 1, 1), (torch.float16, 64, 24, 4, 1), (torch.bfloat16, 128, 48, 2, 2)], ids=str)
def test_every_key_counts_once(case, dtype, D, P, G, rep):
    """Keys of equal weight: lse is the logarithm of their number, and element d of a head whose V is 4096 at one key and 0 elsewhere is
    4096 over their number, if that key counts once.  The keys marked are those at multiples of 64 and in front of them, where pieces
    end, the first and the last, then some of the others."""
    B, Hc, ctx, lens = PIECES[case] if case != "splits" else (2, 8, 4096, [4095, 1000])
    if lens is None:
        lens = [(37 * i * i + 11 * i) % (ctx - 2) for i in range(B)]
    split = ops.decode_split_tokens(B, Hc, ctx, P)
    assert (ops.decode_step_pieces(B, Hc * G, Hc * rep, rep, D, ctx, P, split) > 0) == (case != "splits")
    st = flat_state(77, B, Hc, D, P, ctx, dtype, rep, [max(n, 0) for n in lens])
    _, pv = st.pool_planes()
    pv.zero_()
    v_new = torch.zeros(B, Hc * rep, 1, D, dtype=dtype, device=DEV)
    for b, n in enumerate(lens):
        if n < 0:
            continue
        edges = {0, n, *range(64, n + 1, 64), *range(63, n + 1, 64)}
        keys = [*sorted(edges), *(i * 7919 % (n + 1) for i in range(Hc * D))][: Hc * D]
        keys = torch.tensor(keys, device=DEV).view(Hc, D).repeat_interleave(rep, 0)
        slots = st.cache.page_table[st.slots[b], keys // P] * P + keys % P
        h, d = torch.meshgrid(torch.arange(Hc * rep, device=DEV), torch.arange(D, device=DEV), indexing="ij")
        pool_has = keys < n
        pv[h[pool_has], slots[pool_has], d[pool_has]] = 4096.0
        v_new[b, :, 0] = torch.where(pool_has, 0.0, 4096.0)
    q = torch.zeros(B, Hc * G, 1, D, dtype=dtype, device=DEV)
    k_new = randn(st.gen, v_new.shape, dtype).to(DEV)
    pos = torch.tensor(lens, dtype=torch.int32, device=DEV)
    arrivals = torch.zeros(B * Hc, dtype=torch.int32, device=DEV)
    out, lse = decode(st, q, pos, k_new=k_new, v_new=v_new, max_context=ctx, split_tokens=split, kv_rep=rep, arrivals=arrivals)
    n = (pos + 1).double().view(B, 1, 1, 1)
    want = torch.where(n > 0, 4096.0 / n, 0.0)
    assert ((out.double() - want).abs() <= (STEP[dtype] / 2 + 2.0**-21) * want).all()
    assert torch.equal(torch.isneginf(lse), (n[..., 0] <= 0).expand_as(lse))
    assert ((lse.double() - n[..., 0].clamp(min=1).log()).abs() <= 2.0**-20 * (1 + n[..., 0].clamp(min=1).log()))[pos >= 0].all()


def test_more_rows_than_the_cache_has_counters_for():
    """A batch padded far beyond the cache's slots goes in two passes, as does one over pools of another cache."""
    dtype, live, B, Hc, G, D, P, ctx = torch.float16, 3, 1030, 8, 2, 64, 64, 4096
    st, mask, bidx, pos = drop_in_state(live, Hc, D, P, ctx, dtype, 1, [4000, 70, 1500])
    assert B * Hc > max(len(t) for t in st.cache._decode_arrivals)
    logical = mask.logical
    rows = torch.arange(B, device=DEV).clamp(max=live - 1)
    many = BlockMask.from_kv_blocks(*(getattr(logical, n)[rows] for n in ("kv_num_blocks", "kv_indices", "full_kv_num_blocks", "full_kv_indices")),
                                    BLOCK_SIZE=logical.BLOCK_SIZE, mask_mod=logical.mask_mod, seq_lengths=(1, ctx))
    wide = torch.zeros(B, dtype=torch.int64, device=DEV)
    wide[:live] = bidx
    pos = torch.cat([pos, torch.zeros(B - live, dtype=torch.int32, device=DEV)])
    q, k, v = (randn(st.gen, (B, h, 1, D), dtype).to(DEV) for h in (Hc * G, Hc, Hc))
    k[live:], v[live:] = k[live].clone(), v[live].clone()  # all of them the same padding row
    K, V = st.cache.insert_kv(0, k, v, input_pos=pos.view(B, 1), batch_idx=wide)
    for kk, vv in ((K, V), (K.clone(), V.clone())):
        out, aux = A.compiled_flex_attn_decode(q, kk, vv, block_mask=A.PagedDecodeMask(st.cache, many, wide), return_aux=AuxRequest(lse=True))
        eo, el = ops.paged_decode(q, K[0], V[0], st.cache.page_table, wide, pos, P, ctx)
        torch.testing.assert_close(out, eo, rtol=2 * STEP[dtype], atol=1e-5)
        torch.testing.assert_close(aux.lse.view(el.shape), el, rtol=1e-5, atol=1e-5)
