"""GPU parity: the matrix-core decode kernel (16-bit caches, four or eight query heads per cache head) against the float64
oracle, at the edges of its stages (16 tokens at head_dim 128, 32 at 64), on pages that hold whole stages and pages that do
not, for every way a launch is cut."""

import numpy as np
import pytest
import torch

from falcon_perception_amd import ops
from oracle import paged_kv_oracle as O
from tests.gpu_cases import DEV, PagedState, f64, randn

pytestmark = pytest.mark.gpu

# A result is rounded once to the type (half a unit in the last place: at most 2^-8 of the value in bf16, 2^-11 in f16).  The probabilities keep 16
# (bf16) or 22 (f16) bits, so the sum before that rounding is off by at most 2^-16 of the largest |v| (below 6 here), and
# the hardware's exp2 and log2 add about 2^-20.
TOL = {torch.bfloat16: (2.0 ** -8 * 1.01, 6 * 2.0 ** -16 + 2e-5), torch.float16: (2.0 ** -11 * 1.01, 6 * 2.0 ** -21 + 2e-5)}

EDGES = [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 257]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("G,P", [(4, 32), (4, 24), (8, 64), (8, 16)])
@pytest.mark.parametrize("cut", ["one split", "split by split", "even"])
@pytest.mark.parametrize("spread", [1.0, 6.0], ids=["scores-N01", "scores-spread"])
def test_matrix_core_decode(dtype, D, G, P, cut, spread):
    Hc = 2
    lens = EDGES if cut != "even" else EDGES * 18  # tokens with the new one; 288 sequences fill the 256 chunks' rows
    split, limit = {"one split": (512, 288), "split by split": (64, 288), "even": (128, 384)}[cut]
    B = len(lens)
    limit = -(-limit // P) * P
    st = PagedState(300 + D + G, n_pages=max(limit // P, sum(-(-L // P) for L in lens)) + 4, page_size=P, max_batch=B + 2,
                    Hc=Hc, D=D, dtype=dtype)
    for L in lens:
        st.add_sequence(L)
    st.prefill_random()
    q = (randn(st.gen, (B, Hc * G, 1, D), torch.float32) * spread).to(dtype).to(DEV)
    k_new, v_new = (randn(st.gen, (B, Hc, 1, D), dtype).to(DEV) for _ in range(2))
    pos = torch.tensor(lens, dtype=torch.int32, device=DEV) - 1
    bidx = torch.tensor(st.slots, dtype=torch.int64, device=DEV)
    pk, pv = st.pool_planes()
    out, lse = ops.paged_decode(q, pk, pv, st.cache.page_table, bidx, pos, P, limit, split_tokens=split, k_new=k_new,
                                v_new=v_new)
    for b, L in enumerate(lens):  # the fresh rows are in their slots
        slot = int(st.cache.page_table[st.slots[b], (L - 1) // P]) * P + (L - 1) % P
        assert torch.equal(pk[:, slot], k_new[b, :, 0]) and torch.equal(pv[:, slot], v_new[b, :, 0])
    eo, el = O.decode_attention(f64(q), f64(pk), f64(pv), st.mirror.page_table, st.slots, np.array(lens) - 1, P)
    rtol, atol = TOL[dtype]
    np.testing.assert_allclose(f64(out), eo, rtol=rtol, atol=atol)
    np.testing.assert_allclose(f64(lse), el, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("D,G", [(128, 8), (64, 4)])
@pytest.mark.parametrize("split", [512, 64])
def test_infinite_scores_and_values(dtype, D, G, split):
    """Keys whose score is -inf (the whole first stage of the first wavefront) weigh nothing, and an infinite V
    element makes its element of the result infinite and no other."""
    Hc, P, L = 2, 64, 200
    st = PagedState(77, n_pages=8, page_size=P, max_batch=2, Hc=Hc, D=D, dtype=dtype)
    st.add_sequence(L)
    st.prefill_random()
    pk, pv = st.pool_planes()
    slots = [int(st.cache.page_table[st.slots[0], t // P]) * P + t % P for t in range(L)]
    q = torch.ones((1, Hc * G, 1, D), dtype=dtype, device=DEV)
    pos = torch.tensor([L - 1], dtype=torch.int32, device=DEV)
    bidx = torch.tensor(st.slots, dtype=torch.int64, device=DEV)
    args = (st.cache.page_table, bidx, pos, P, 256)
    eo, el = O.decode_attention(f64(q), f64(pk[:, slots[32:]]), f64(pv[:, slots[32:]]),
                                np.arange(L - 32).reshape(1, -1), [0], np.array([L - 33]), 1)
    pk[:, slots[:32]] = -float("inf")
    out, lse = ops.paged_decode(q, pk, pv, *args, split_tokens=split)
    rtol, atol = TOL[dtype]
    np.testing.assert_allclose(f64(out), eo, rtol=rtol, atol=atol)
    np.testing.assert_allclose(f64(lse), el, rtol=1e-5, atol=1e-5)
    pv[:, slots[40], 5] = float("inf")
    got, _ = ops.paged_decode(q, pk, pv, *args, split_tokens=split)
    assert (got[..., 5] == float("inf")).all()
    keep = [d for d in range(D) if d != 5]
    assert torch.equal(got[..., keep], out[..., keep])


def one_sequence(dtype, D, G, L, seed=78):
    """A sequence of L tokens; every head's query is sqrt(D) in element 0, so a key's score is its element 0."""
    Hc, P = 2, 64
    st = PagedState(seed, n_pages=8, page_size=P, max_batch=2, Hc=Hc, D=D, dtype=dtype)
    st.add_sequence(L)
    st.prefill_random()
    pk, pv = st.pool_planes()
    slots = [int(st.cache.page_table[st.slots[0], t // P]) * P + t % P for t in range(L)]
    q = torch.zeros((1, Hc * G, 1, D), dtype=dtype, device=DEV)
    q[..., 0] = D ** 0.5
    args = (st.cache.page_table, torch.tensor(st.slots, dtype=torch.int64, device=DEV),
            torch.tensor([L - 1], dtype=torch.int32, device=DEV), P, 256)
    return st, q, pk, pv, slots, args


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("D,G", [(128, 8), (64, 4)])
@pytest.mark.parametrize("L", [1, 17, 200])
@pytest.mark.parametrize("split", [512, 64])
@pytest.mark.parametrize("fused", [False, True], ids=["from-the-pool", "fresh-row"])
def test_an_infinite_value_in_the_last_row(dtype, D, G, L, split, fused):
    """The tokens a stage has room for behind the last row have no weight, and none of its infinity either."""
    st, q, pk, pv, slots, args = one_sequence(dtype, D, G, L)
    fresh = {}
    if fused:
        fresh = dict(k_new=pk[None, :, slots[-1:]].contiguous(), v_new=pv[None, :, slots[-1:]].contiguous())
    out, lse = ops.paged_decode(q, pk, pv, *args, split_tokens=split, **fresh)
    for v in (pv[None, :, slots[-1:]], fresh.get("v_new")):
        if v is not None:
            v[..., 5] = float("inf")
    pv[:, slots[-1], 5] = float("inf")
    got, lse2 = ops.paged_decode(q, pk, pv, *args, split_tokens=split, **fresh)
    keep = [d for d in range(D) if d != 5]
    assert (got[..., 5] == float("inf")).all() and torch.equal(got[..., keep], out[..., keep]) and torch.equal(lse2, lse)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("D,G", [(128, 8), (64, 4)])
@pytest.mark.parametrize("score", [-12.0, -17.5, -24.0, -60.0, -75.0])
def test_an_infinite_value_of_a_key_that_weighs_next_to_nothing(dtype, D, G, score):
    """A probability that the 16-bit type rounds to 0 (below 2^-33 of the largest in f16) is still above 0."""
    st, q, pk, pv, slots, args = one_sequence(dtype, D, G, 200)
    pk[:, slots, 0] = 0.0
    pk[:, slots[3], 0] = score
    out, lse = ops.paged_decode(q, pk, pv, *args, split_tokens=512)
    pv[:, slots[3], 5] = float("-inf")
    got, _ = ops.paged_decode(q, pk, pv, *args, split_tokens=512)
    keep = [d for d in range(D) if d != 5]
    assert (got[..., 5] == float("-inf")).all() and torch.equal(got[..., keep], out[..., keep])
    eo, _ = O.decode_attention(f64(q), f64(pk), np.nan_to_num(f64(pv), neginf=0.0), st.mirror.page_table, st.slots,
                               np.array([199]), 64)
    rtol, atol = TOL[dtype]
    np.testing.assert_allclose(f64(got[..., keep]), eo[..., keep], rtol=rtol, atol=atol)


@pytest.mark.parametrize("D,G", [(128, 8), (64, 4)])
@pytest.mark.parametrize("score", [1.0, 4.0])
def test_the_largest_value_of_the_type(D, G, score):
    """V at the largest bf16 under the key with the largest score, which comes after keys that weigh less: the reference
    point of the exponentials lags, and no product may leave fp32."""
    dtype = torch.bfloat16
    st, q, pk, pv, slots, args = one_sequence(dtype, D, G, 200)
    pk[:, slots, 0] = 0.0
    late = slots[4 * (4096 // (2 * D)) + 2]  # in the second stage of the first wavefront
    pk[:, late, 0] = score
    pv[:, late, 5] = torch.finfo(dtype).max
    pv[:, late, 6] = torch.finfo(dtype).min
    out, _ = ops.paged_decode(q, pk, pv, *args, split_tokens=512)
    eo, _ = O.decode_attention(f64(q), f64(pk), f64(pv), st.mirror.page_table, st.slots, np.array([199]), 64)
    rtol, atol = TOL[dtype]
    np.testing.assert_allclose(f64(out), eo, rtol=rtol + 2.0 ** -16, atol=atol)
