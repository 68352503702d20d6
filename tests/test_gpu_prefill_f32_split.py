"""GPU parity: the fp32 prefill kernel, whose products are sums of six bf16 products (three bf16 numbers to every fp32 number), and
the fp32 matrix instruction it goes back to where a number does not fit that (infinities, NaN, from the largest bf16 on, below 2^-100).

Bound of an output element, from the inputs: the scores are sums of fp32 roundings, fewer than 12 of the size of the
whole, so a probability is off by 12 * 2^-24 * scale * sum |q k| (natural units) and a few roundings of its own; the sums over n
keys and the denominator add at most 2 (n + 8) roundings: (12 scale max_k sum |q k| + 2 n + 16) * 2^-24 * sum p |v|.
"""

import math

import pytest
import torch

from falcon_perception_amd import ops
from tests.gpu_cases import DEV, PagedState

pytestmark = pytest.mark.gpu

LENS = [150, 1, 97, 32, 64, 33]  # rows and keys of each sequence: tiles of 32 and 64 keys, their edges, parts of one


def build(D, G, P, seed=3):
    Hc = 2
    st = PagedState(seed, n_pages=sum(-(-n // P) for n in LENS) + 3, page_size=P, max_batch=len(LENS) + 2, Hc=Hc, D=D, dtype=torch.float32)
    for n in LENS:
        st.add_sequence(n)
    L = sum(LENS)
    k, v = (torch.randn((Hc, L, D), generator=st.gen) for _ in range(2))
    q = torch.randn((Hc * G, L, D), generator=st.gen)
    return st, q, k, v


def run(st, q, k, v, shares):
    L, (Hq, _, D) = q.shape[1], q.shape
    bidx = torch.cat([torch.full((n,), b) for n, b in zip(LENS, st.slots)]).to(torch.int64)
    pos = torch.cat([torch.arange(n) for n in LENS])
    limit = torch.cat([torch.full((n,), n) for n in LENS]).to(torch.int32)  # every row sees all keys of its sequence
    st.cache.insert_kv(0, k[None].to(DEV), v[None].to(DEV), input_pos=pos[None].to(DEV), batch_idx=bidx[None].to(DEV))
    ws = torch.empty(shares * L * Hq * (D * 4 + 8), dtype=torch.uint8, device=DEV) if shares > 1 else False
    out, lse = ops.paged_prefill(q[None].to(DEV), *st.pool_planes(), st.cache.page_table, bidx.to(DEV), limit.to(DEV), st.P, workspace=ws)
    return out[0].cpu().double(), lse[0].cpu().double()


def check(got, q, k, v, skip=()):
    """`skip`: (sequence, output columns or None for all, rows or None) that the caller looks at himself."""
    out, lse = got
    G, D = q.shape[0] // k.shape[0], q.shape[-1]
    scale = 1 / math.sqrt(D)
    start = 0
    for i, n in enumerate(LENS):
        rows = slice(start, start + n)
        start += n
        Q, K, V = q[:, rows].double(), k[:, rows].double().repeat_interleave(G, 0), v[:, rows].double().repeat_interleave(G, 0)
        s = Q @ K.transpose(1, 2) * scale
        p = torch.softmax(s, -1)
        ref, size = p @ V, p @ V.abs()
        weight = 12 * scale * (Q.abs() @ K.abs().transpose(1, 2)).amax(-1, keepdim=True) + 2 * n + 16
        ok = (out[:, rows] - ref).abs() <= weight * 2.0**-24 * size
        ok_lse = (lse[:, rows] - torch.logsumexp(s, -1)).abs() <= weight[..., 0] * 2.0**-24 * 2
        for j, cols, which in skip:
            if j == i:
                r = slice(None) if which is None else which
                ok[:, r, slice(None) if cols is None else cols] = True
                if cols is None:
                    ok_lse[:, r] = True
        assert ok.all() and ok_lse.all(), f"sequence {i}"


@pytest.mark.parametrize("shares", [1, 3])
@pytest.mark.parametrize("D,G,P", [(128, 1, 64), (128, 8, 16), (128, 2, 24), (64, 1, 64), (64, 4, 32), (64, 2, 128)])
def test_values_the_split_holds(D, G, P, shares):
    st, q, k, v = build(D, G, P)
    v *= 2.0 ** torch.linspace(-60, 60, D)  # a column of V has one size, the columns of a tile any
    k[:, ::7] *= 2.0**-40
    q[:, ::5] *= 0.0
    check(run(st, q, k, v, shares), q, k, v)


@pytest.mark.parametrize("shares", [1, 3])
@pytest.mark.parametrize("D,G,P", [(128, 1, 64), (128, 2, 24), (64, 1, 64), (64, 4, 16)])
def test_values_it_does_not_hold(D, G, P, shares):
    st, q, k, v = build(D, G, P)
    a, b = 70, sum(LENS[:2]) + 40  # a key of the first sequence in its third (second) tile, and one of the third sequence
    v[:, a, 3], v[:, a + 2, 4], v[:, a, 5] = math.inf, -math.inf, math.nan
    v[:, 10, 6] = torch.finfo(torch.float32).max
    v[:, : LENS[0], 7] *= 2.0**-110
    k[:, b, 0] = math.nan
    out, lse = run(st, q, k, v, shares)
    first, third = slice(0, LENS[0]), slice(sum(LENS[:2]), sum(LENS[:3]))
    assert (out[:, first, 3] == math.inf).all() and (out[:, first, 4] == -math.inf).all() and out[:, first, 5].isnan().all()
    assert out[:, third].isnan().all() and not lse[:, third].isfinite().any()
    vc = v.clone()
    vc[:, a, 3], vc[:, a + 2, 4], vc[:, a, 5] = 0.0, 0.0, 0.0
    kc = k.clone()
    kc[:, b, 0] = 0.0
    check((out, lse), q, kc, vc, skip=[(0, [3, 4, 5], None), (2, None, None)])


@pytest.mark.parametrize("D,G", [(128, 1), (64, 2)])
def test_query_rows_it_does_not_hold(D, G):
    """One row is not finite, one far out of the range against keys that are as far out on the other side."""
    st, q, k, v = build(D, G, 64)
    q[:, 20, 1] = math.nan
    last = slice(sum(LENS[:5]), None)
    q[:, last] *= 2.0**118
    k[:, last] *= 2.0**-118
    out, lse = run(st, q, k, v, 1)
    assert out[:, 20].isnan().all() and not lse[:, 20].isfinite().any()
    q[:, 20, 1] = 0.0
    check((out, lse), q, k, v, skip=[(0, None, 20)])


@pytest.mark.parametrize("shares", [1, 3])
@pytest.mark.parametrize("D,G,P", [(128, 1, 64), (128, 2, 24), (64, 4, 16)])
def test_a_score_that_overflows_takes_its_own_key_only(D, G, P, shares):
    """Finite numbers whose product is beyond fp32: the score is -inf and its key has no weight, whatever the signs of the products
    of their smaller parts are.  Each factor comes as itself and with another lowest part, so that these have either sign."""
    st, q, k, v = build(D, G, P)
    q[..., 0] = 0.0
    k[..., 0] = 0.0
    big = torch.tensor([3.01e22, 3.0e22, 2.97e22, 1.0e21, 2.0**61, 9.99e30])
    first, third = slice(0, LENS[0]), slice(sum(LENS[:2]), sum(LENS[:3]))
    for rows in (first, third):
        n = rows.stop - rows.start
        k[:, rows.start + 5 : rows.start + 5 + len(big), 0] = big
        q[:, rows, 0] = -(big * 1.001)[torch.arange(n) % len(big)].clamp(min=1e21)
    got = run(st, q, k, v, shares)
    qc, kc = q.clone(), k.clone()  # the same with products that fp32 holds: at -180 and below a key has no weight either
    qc[..., 0] = (q[..., 0] != 0) * -32.0
    kc[..., 0] = (k[..., 0] != 0) * 64.0 * math.sqrt(D / 128)
    check(got, qc, kc, v)


@pytest.mark.parametrize("D,G,P", [(128, 1, 64), (128, 4, 24), (64, 2, 16)])
def test_queries_of_one_sequence_leave_the_others_alone(D, G, P):
    """The rows of several sequences share a workgroup; what the queries of one hold changes no bit of the others."""
    rows = slice(sum(LENS[:2]), sum(LENS[:3]))
    others = torch.ones(sum(LENS), dtype=torch.bool)
    others[rows] = False
    results = []
    for value in (1.0, math.nan, math.inf, 2.0**-110, 1e30):
        st, q, k, v = build(D, G, P)
        q[:, rows] *= value
        out, lse = run(st, q, k, v, 1)
        results.append((out[:, others], lse[:, others]))
    for out, lse in results[1:]:
        assert torch.equal(out, results[0][0]) and torch.equal(lse, results[0][1])


@pytest.mark.parametrize("exact", [False, True], ids=["split", "instruction"])
@pytest.mark.parametrize("D,P", [(128, 32), (128, 24), (64, 64), (64, 8)])
def test_a_key_without_a_page_reads_slot_0(D, P, exact):
    """A limit beyond the pages a sequence has, and beyond the table: every key there is the first row of the pool, on either matrix instruction."""
    Hc, n, more = 2, 75, 30
    mapped = -(-n // P) * P
    st = PagedState(5, n_pages=16, page_size=P, max_batch=3, Hc=Hc, D=D, dtype=torch.float32, max_blocks_per_seq=mapped // P + 1)
    st.add_sequence(n)
    k, v = (torch.randn((Hc, mapped + more, D), generator=st.gen) for _ in range(2))
    q = torch.randn((Hc, n, D), generator=st.gen)
    if exact:
        v[:, 3, 0] = 2.0**-105  # sends the run to the fp32 instruction
    k[:, mapped:], v[:, mapped:] = k[:, mapped : mapped + 1], v[:, mapped : mapped + 1]
    pk, pv = st.pool_planes()
    slots = (st.cache.page_table[st.slots[0], : mapped // P, None] * P + torch.arange(P, device=DEV)).reshape(-1)
    for pool, x in ((pk, k), (pv, v)):
        pool[:, slots], pool[:, 0] = x[:, :mapped].to(DEV), x[:, mapped].to(DEV)
    bidx = torch.full((n,), st.slots[0], dtype=torch.int64, device=DEV)
    limit = torch.full((n,), mapped + more, dtype=torch.int32, device=DEV)
    out, _ = ops.paged_prefill(q[None].to(DEV), pk, pv, st.cache.page_table, bidx, limit, P, workspace=False)
    s = q.double() @ k.double().transpose(1, 2) / math.sqrt(D)
    p = torch.softmax(s, -1)
    weight = 12 / math.sqrt(D) * (q.abs() @ k.abs().transpose(1, 2)).amax(-1, keepdim=True) + 2 * k.shape[1] + 16
    assert ((out[0].cpu().double() - p @ v.double()).abs() <= weight * 2.0**-24 * (p @ v.double().abs())).all()
