"""The work a serving engine has this package do, as a list of measurable cases.

Every case is one step of a model as an engine runs it: the mask of the step, then for every layer the insert of
the new K/V rows into the page pool and the attention call over the pages.

* a decode step (one new token per sequence) is captured once in a HIP graph per batch bucket and replayed, or run
  eagerly where no graph was captured;
* a prefill step (packed rows of several sequences, each padded to 128 rows) is run eagerly: whole sequences whose
  image span is bidirectional, or chunks of text over a prefix that is cached already.

Rows have the values the path meets in a model: q and k are RMS-normalised rows (norm sqrt(head_dim)), v is N(0, 1),
pages come from a shuffled free list.  Padding rows carry slot 0 and position 0 and are all the same row, as one
padding token at one position is.  Lengths are spread over their range by a fixed low-discrepancy sequence, so
`work` knows them from the case alone; everything else follows from the seed.
"""

import math
import os
import sys

import torch
from torch.nn.attention.flex_attention import AuxRequest, BlockMask

_PACKAGE = os.path.join(os.getcwd(), "falcon-perception_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(1, _PACKAGE)

from falcon_perception_amd import attention  # noqa: E402
from falcon_perception_amd.paged_attention import PagedKVCache  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
SOI, IMG, EOI, TXT, PAD = 1, 2, 3, 4, 0
DEVICE = "cuda"


def _decode(name, *, batch, live, lo, hi, max_context, q_heads, cached_heads, kv_rep, head_dim, page_size, dtype,
            layers, graph, sinks):
    case = dict(kind="decode", batch=batch, live=live, lo=lo, hi=hi, max_context=max_context, q_heads=q_heads,
                cached_heads=cached_heads, kv_rep=kv_rep, head_dim=head_dim, page_size=page_size, dtype=dtype,
                layers=layers, graph=graph, sinks=sinks)
    return case if name is None else dict(name=name, **case)


def _prefill(name, *, sequences, image_lo, image_hi, text_lo, text_hi, whole, q_heads, cached_heads, head_dim,
             page_size, dtype, layers, normalised, rope_heads):
    case = dict(kind="prefill", sequences=sequences, image_lo=image_lo, image_hi=image_hi, text_lo=text_lo,
                text_hi=text_hi, whole=whole, q_heads=q_heads, cached_heads=cached_heads, head_dim=head_dim,
                page_size=page_size, dtype=dtype, layers=layers, normalised=normalised, rope_heads=rope_heads)
    return case if name is None else dict(name=name, **case)


def listed():
    return [
        # One user with one small picture: the latency of a token.  The engine's own cache (one cached head per query
        # head, V heads in identical pairs), its sequence limit of 8192 tokens, the graph of the bucket of one.
        _decode("decode_single", batch=1, live=1, lo=711, hi=711, max_context=8192, q_heads=16, cached_heads=16,
                kv_rep=2, head_dim=128, page_size=128, dtype="bf16", layers=28, graph=True, sinks=False),
        # A moderately busy server: 13 requests in the graph of the bucket of 16, three padded rows.
        _decode("decode_bucket16", batch=16, live=13, lo=350, hi=4620, max_context=8192, q_heads=16, cached_heads=16,
                kv_rep=2, head_dim=128, page_size=128, dtype="bf16", layers=28, graph=True, sinks=False),
        # A full server, one cached head per kv head: 64 sequences of a 1024-token picture and 64 to 3072 tokens.
        _decode("decode_serving", batch=64, live=64, lo=1088, hi=4096, max_context=8192, q_heads=16, cached_heads=8,
                kv_rep=1, head_dim=128, page_size=128, dtype="bf16", layers=8, graph=True, sinks=False),
        # Pages of text read by many users at once: 4096-token pictures and up to 12288 tokens of text, four query
        # heads per kv head; the largest decode step.
        _decode("decode_long", batch=96, live=96, lo=4352, hi=16384, max_context=16384, q_heads=32, cached_heads=8,
                kv_rep=1, head_dim=128, page_size=128, dtype="bf16", layers=2, graph=True, sinks=False),
        # A few long documents through the small variants (head_dim 64) in half precision, pages of 64 tokens.
        _decode("decode_few_long", batch=4, live=4, lo=5003, hi=16001, max_context=16384, q_heads=16, cached_heads=8,
                kv_rep=1, head_dim=64, page_size=64, dtype="f16", layers=28, graph=True, sinks=False),
        # The first thing a user tries: float32 (the engine's default), four short sequences, no graphs.
        _decode("decode_f32_eager", batch=4, live=4, lo=64, hi=512, max_context=4096, q_heads=8, cached_heads=8,
                kv_rep=1, head_dim=64, page_size=64, dtype="f32", layers=28, graph=False, sinks=False),
        # Wide query groups (eight query heads per kv head) with the sink gate in the attention call.
        _decode("decode_group8_sinks", batch=24, live=24, lo=512, hi=8191, max_context=8192, q_heads=64,
                cached_heads=8, kv_rep=1, head_dim=128, page_size=64, dtype="bf16", layers=4, graph=True, sinks=True),
        # One request is admitted: a small picture and its prompt, alone in the step; first-token latency.
        _prefill("prefill_single", sequences=1, image_lo=576, image_hi=576, text_lo=37, text_hi=37, whole=True,
                 q_heads=16, cached_heads=16, head_dim=128, page_size=128, dtype="bf16", layers=28, normalised=True,
                 rope_heads=0),
        # Eight text chunks of 512 rows over cached prefixes of 256 to 4096 tokens; nothing declared about the rows.
        _prefill("prefill_chunks", sequences=8, image_lo=256, image_hi=4096, text_lo=512, text_hi=512, whole=False,
                 q_heads=16, cached_heads=8, head_dim=128, page_size=64, dtype="bf16", layers=8, normalised=False,
                 rope_heads=0),
        # A full admission step of whole sequences on the engine's own cache: the bulk of a picture workload.
        _prefill("prefill_whole", sequences=8, image_lo=256, image_hi=4096, text_lo=512, text_hi=512, whole=True,
                 q_heads=16, cached_heads=16, head_dim=128, page_size=128, dtype="bf16", layers=8, normalised=True,
                 rope_heads=0),
        # The same through the small variants, norm, rotary embedding and insert in one call (8 kv heads).
        _prefill("prefill_whole_rope64", sequences=9, image_lo=300, image_hi=4001, text_lo=17, text_hi=490, whole=True,
                 q_heads=16, cached_heads=16, head_dim=64, page_size=128, dtype="bf16", layers=8, normalised=True,
                 rope_heads=8),
        # Whole sequences in float32, the engine's default type.
        _prefill("prefill_whole_f32", sequences=3, image_lo=500, image_hi=2304, text_lo=41, text_hi=256, whole=True,
                 q_heads=16, cached_heads=16, head_dim=128, page_size=128, dtype="f32", layers=4, normalised=True,
                 rope_heads=0),
    ]


# ---------------------------------------------------------------------------------------------------- drawn cases

def _log(rng, lo, hi):
    """A whole number between lo and hi, even over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# what a drawn case may cost at most: bytes and flops of the largest listed cases
_MOST_BYTES, _MOST_FLOPS = 8.0e9, {"bf16": 4.0e12, "f16": 4.0e12, "f32": 4.0e11}


def draw(rng):
    while True:
        case = _draw_decode(rng) if rng.random() < 0.55 else _draw_prefill(rng)
        w = work(case)
        if w["bytes"] <= _MOST_BYTES and w["flops"] <= _MOST_FLOPS[case["dtype"]]:
            return case


def _draw_heads(rng):
    """(query heads, cached heads, copies of V per group): the engine's cache or one cached head per kv head."""
    kv = rng.choice([4, 8])
    group = rng.choice([1, 2, 2, 2, 4, 8])
    if group == 2 and rng.random() < 0.5:
        return 2 * kv, 2 * kv, 2
    return group * kv, kv, 1


def _draw_decode(rng):
    q_heads, cached_heads, kv_rep = _draw_heads(rng)
    live = _log(rng, 1, 96)
    graph = rng.random() < 0.8
    bucket = live if not graph else (1 << (live - 1).bit_length() if live <= 8 else -(-live // 16) * 16)
    hi = _log(rng, 96, 16000)
    lo = _log(rng, 64, hi) if hi > 64 else hi
    room = 8192 if hi < 8192 else 16384
    return _decode(None, batch=bucket, live=live, lo=lo, hi=hi, max_context=room, q_heads=q_heads,
                   cached_heads=cached_heads, kv_rep=kv_rep, head_dim=rng.choice([64, 128, 128]),
                   page_size=rng.choice([32, 64, 128, 128, 256]), dtype=rng.choice(["bf16", "bf16", "f16", "f32"]),
                   layers=rng.choice([1, 2, 4, 28]), graph=graph, sinks=rng.random() < 0.25)


def _draw_prefill(rng):
    q_heads, cached_heads, _ = _draw_heads(rng)
    head_dim = rng.choice([64, 128, 128])
    whole = rng.random() < 0.65
    image_hi = _log(rng, 64, 4096)
    text_hi = _log(rng, 16, 512) if whole else _log(rng, 64, 1024)
    rope = cached_heads if rng.random() < 0.2 else 0
    if rope and cached_heads == q_heads and rng.random() < 0.7:
        rope = cached_heads // 2
    return _prefill(None, sequences=_log(rng, 1, 12), image_lo=_log(rng, 48, image_hi), image_hi=image_hi,
                    text_lo=_log(rng, 8, text_hi), text_hi=text_hi, whole=whole, q_heads=q_heads,
                    cached_heads=cached_heads, head_dim=head_dim, page_size=rng.choice([32, 64, 128, 128, 256]),
                    dtype=rng.choice(["bf16", "bf16", "bf16", "f16", "f32"]), layers=rng.choice([1, 4, 8, 28]),
                    normalised=rng.random() < 0.6, rope_heads=rope)


# ------------------------------------------------------------------------------------------------------- geometry

def _spread(lo, hi, n, shift=0.0):
    """n whole numbers over [lo, hi], the ends apart by a golden-ratio sequence."""
    return [lo + int((i * 0.6180339887498949 + shift) % 1.0 * (hi - lo + 1)) for i in range(n)]


def _decode_lengths(c):
    """Tokens cached of each live sequence before the step."""
    return [c["hi"] - 1] if c["live"] == 1 else _spread(c["lo"] - 1, c["hi"] - 1, c["live"])


def _prefill_lengths(c):
    """(image tokens, text tokens) of each sequence."""
    n = c["sequences"]
    if n == 1:
        return [(c["image_hi"], c["text_hi"])]
    return list(zip(_spread(c["image_lo"], c["image_hi"], n, 0.3), _spread(c["text_lo"], c["text_hi"], n, 0.7)))


def work(case):
    c = case
    e = 4 if c["dtype"] == "f32" else 2
    D, Hq, Hc, P = c["head_dim"], c["q_heads"], c["cached_heads"], c["page_size"]
    if c["kind"] == "decode":
        contexts = [n + 1 for n in _decode_lengths(c)]
        # K of every cached head, V of every distinct one; the new rows in and into the pool; q, out, lse, page ids
        n_bytes = sum(contexts) * (Hc + Hc // c["kv_rep"]) * D * e
        n_bytes += c["batch"] * (4 * Hc * D * e + 2 * Hq * D * e + 4 * Hq)
        n_bytes += 8 * sum(-(-n // P) for n in contexts)
        return {"bytes": c["layers"] * n_bytes, "flops": c["layers"] * 4 * D * Hq * sum(contexts)}
    n_bytes = pairs = rows = 0
    for image, text in _prefill_lengths(c):
        if c["whole"]:
            rows += image + text
            span = image - 1  # the end-of-image token is no part of the bidirectional span
            pairs += span * span + sum(range(span + 1, image + text + 1))
        else:
            rows += text
            pairs += sum(range(image + 1, image + text + 1))
            n_bytes += 2 * image * Hc * D * e
    if c["rope_heads"]:  # projection rows and angle tables in; K and V rows into the pool
        n_bytes += rows * ((Hq + 2 * c["rope_heads"]) * D * e + (1 + Hq) * 2 * D + 2 * Hc * D * e)
    else:
        n_bytes += rows * (Hq * D * e + 4 * Hc * D * e)
    n_bytes += rows * (Hq * D * e + 4 * Hq)  # out and lse
    return {"bytes": c["layers"] * n_bytes, "flops": c["layers"] * 4 * D * Hq * pairs}


def tolerance(case):
    """About four times what the path was seen to differ from attention over the same stored rows in float64: bf16
    3.3e-3 (largest 2.9e-2), f16 3.0e-4 (9e-4 to 1.5e-3), f32 5.1e-7 (6.3e-6).  Probabilities and results are rounded
    to the model's type, sums are fp32."""
    return dict(_TOLERANCE[case["dtype"]])


_TOLERANCE = {
    "bf16": {"rel": 1.2e-2, "max": 0.1},
    "f16": {"rel": 1.2e-3, "max": 6e-3},
    "f32": {"rel": 2e-6, "max": 3e-5},
}


# --------------------------------------------------------------------------------------------------------- states

class _State:
    pass


def _normalise(x):
    """RMS norm of the last axis in place, a few million rows at a time."""
    flat = x.view(-1, x.shape[-1])
    step = max(1, (1 << 27) // x.shape[-1])
    for s in range(0, flat.shape[0], step):
        part = flat[s:s + step].float()
        flat[s:s + step] = part * part.square().mean(-1, keepdim=True).rsqrt()
    return x


def _rows(gen, shape, dtype, norm):
    x = torch.empty(shape, dtype=dtype, device=DEVICE).normal_(generator=gen)
    return _normalise(x) if norm else x


def _fill_pool(cache, gen, kv_rep):
    """Rows of earlier steps in every page: normalised k, N(0, 1) v (identical inside a group of copies)."""
    pool = cache.kv_cache
    for layer in range(pool.shape[0]):
        _normalise(pool[layer, 0].normal_(generator=gen))
        v = pool[layer, 1, 0]
        if kv_rep == 1:
            v.normal_(generator=gen)
        else:
            groups = v.view(v.shape[0] // kv_rep, kv_rep, *v.shape[1:])
            groups.copy_(torch.empty_like(groups[:, 0]).normal_(generator=gen).unsqueeze(1))


def _copies(x, kv_rep):
    return x if kv_rep == 1 else x.repeat_interleave(kv_rep, dim=2)


def _admit(cache, lengths, seed):
    order = torch.randperm(cache.n_pages - 1, generator=torch.Generator().manual_seed(seed)) + 1
    cache.free_pages = order.tolist()
    slots = []
    for n in lengths:
        slot = cache.allocate()
        cache.reserve(slot, torch.tensor([slot], device=DEVICE), n)
        slots.append(slot)
    return slots


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    return (_prepare_decode if case["kind"] == "decode" else _prepare_prefill)(case, seed, gen)


def _prepare_decode(c, seed, gen):
    s = _State()
    s.decode, s.layers = True, c["layers"]
    dtype, P, B, D = DTYPES[c["dtype"]], c["page_size"], c["batch"], c["head_dim"]
    lengths = _decode_lengths(c)
    pages = 1 + sum(-(-(n + 1) // P) for n in lengths)
    n_pages = max(pages + pages // 8, c["max_context"] // P)
    s.cache = PagedKVCache(n_pages, P, B + 1, c["cached_heads"], D, c["layers"], dtype, device=DEVICE,
                           max_blocks_per_seq=c["max_context"] // P, kv_rep=c["kv_rep"], qk_normalised=True,
                           fuse_decode_append=True)
    slots = _admit(s.cache, [n + 1 for n in lengths], seed)
    _fill_pool(s.cache, gen, c["kv_rep"])
    pad = B - c["live"]
    s.batch_idx = torch.tensor(slots + [0] * pad, dtype=torch.int64, device=DEVICE)
    pos = torch.tensor(lengths + [0] * pad, dtype=torch.int32, device=DEVICE)
    s.input_pos = pos.view(B, 1)
    kv_heads = c["cached_heads"] // c["kv_rep"]
    s.q = _rows(gen, (c["layers"], B, c["q_heads"], 1, D), dtype, True)
    s.k = _rows(gen, (c["layers"], B, c["cached_heads"], 1, D), dtype, True)
    s.v = _copies(_rows(gen, (c["layers"], B, kv_heads, 1, D), dtype, False), c["kv_rep"])
    for x in (s.q, s.k, s.v):
        x[:, c["live"]:] = x[:, :1].clone()
    s.sinks = torch.empty(c["q_heads"], device=DEVICE).uniform_(2.0, 9.0, generator=gen) if c["sinks"] else None
    # the engine slices the block mask of its longest sequence once per step
    whole = s.cache.create_causal_blockmask(B=1, L=c["max_context"])
    block = (pos // P).long()
    row = torch.zeros_like(block)
    s.logical = BlockMask.from_kv_blocks(
        whole.kv_num_blocks[row, :, block].view(B, 1, 1), whole.kv_indices[row, :, block].view(B, 1, 1, -1),
        whole.full_kv_num_blocks[row, :, block].view(B, 1, 1), whole.full_kv_indices[row, :, block].view(B, 1, 1, -1),
        BLOCK_SIZE=whole.BLOCK_SIZE, mask_mod=lambda b, h, q, kv: q + pos[b] >= kv,
        seq_lengths=(1, whole.seq_lengths[1]))
    s.aux = AuxRequest(lse=True)
    s.graph = None
    if c["graph"]:  # captured once per batch bucket after a warm-up step, replayed every step
        _decode_step(s)
        torch.cuda.synchronize()
        s.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s.graph):
            s.results = _decode_step(s)
        torch.cuda.synchronize()
    return s


def _decode_step(s):
    mask = s.cache.convert_logical_block_mask(s.logical, s.batch_idx)
    results = []
    for layer in range(s.layers):
        K, V = s.cache.insert_kv(layer, s.k[layer], s.v[layer], input_pos=s.input_pos, batch_idx=s.batch_idx)
        out, aux = attention.compiled_flex_attn_decode(s.q[layer], K, V, block_mask=mask, return_aux=s.aux,
                                                       sinks=s.sinks)
        results += [out, aux.lse]
    return results


def _prepare_prefill(c, seed, gen):
    s = _State()
    s.decode, s.layers, s.graph = False, c["layers"], None
    dtype, P, D, Hq, Hc = DTYPES[c["dtype"]], c["page_size"], c["head_dim"], c["q_heads"], c["cached_heads"]
    lengths = _prefill_lengths(c)
    n_pages = 8 + sum(-(-(i + t) // P) for i, t in lengths)
    s.cache = PagedKVCache(n_pages, P, c["sequences"] + 1, Hc, D, c["layers"], dtype, device=DEVICE, kv_rep=1,
                           qk_normalised=c["normalised"], fuse_decode_append=True)
    slots = _admit(s.cache, [i + t for i, t in lengths], seed)
    _fill_pool(s.cache, gen, 1)
    ids, bidx, pos = [], [], []
    for slot, (image, text) in zip(slots, lengths):
        if c["whole"]:
            tokens, first = [SOI] + [IMG] * (image - 2) + [EOI] + [TXT] * text, 0
        else:
            tokens, first = [TXT] * text, image
        n, gap = len(tokens), -len(tokens) % 128
        ids += tokens + [PAD] * gap
        bidx += [slot] * n + [0] * gap
        pos += list(range(first, first + n)) + [0] * gap
    s.ids, s.batch_idx, s.input_pos = (torch.tensor([x], dtype=torch.int64, device=DEVICE) for x in (ids, bidx, pos))
    L, layers = len(ids), c["layers"]
    padding = s.batch_idx[0] == 0
    s.rope = c["rope_heads"]
    if s.rope:
        heads = Hq + 2 * s.rope
        qkv = _rows(gen, (layers, 1, L, heads, D), dtype, False)
        qkv[:, :, padding] = qkv[:1, :1, :1].clone()
        s.q, s.k, s.v = qkv.split([Hq, s.rope, s.rope], dim=3)
        angle = torch.empty((1, L, D // 4), device=DEVICE).uniform_(-3.2, 3.2, generator=gen)
        angle2 = torch.empty((1, L, Hq, D // 4), device=DEVICE).uniform_(-3.2, 3.2, generator=gen)
        angle[:, padding], angle2[:, padding] = 0.0, 0.0
        s.freqs, s.freqs_2d = torch.polar(torch.ones_like(angle), angle), torch.polar(torch.ones_like(angle2), angle2)
    else:  # [1, L, H, D] rows of the projection, handed over as [1, H, L, D]
        rows = [_rows(gen, (layers, 1, L, h, D), dtype, norm) for h, norm in ((Hq, True), (Hc, True), (Hc, False))]
        for x in rows:
            x[:, :, padding] = x[:1, :1, :1].clone()
        s.q, s.k, s.v = (x.transpose(2, 3) for x in rows)
    s.aux = AuxRequest(lse=True)
    return s


def _prefill_step(s):
    cache = s.cache
    mask = cache.create_prefill_blockmask(s.batch_idx, s.ids, SOI, EOI)
    results = []
    for layer in range(s.layers):
        if s.rope:
            q, K, V = cache.insert_qkv_norm_rope(layer, s.q[layer], s.k[layer], s.v[layer], s.freqs, s.freqs_2d,
                                                 input_pos=s.input_pos, batch_idx=s.batch_idx)
        else:
            q = s.q[layer]
            K, V = cache.insert_kv(layer, s.k[layer], s.v[layer], input_pos=s.input_pos, batch_idx=s.batch_idx)
        out, aux = attention.compiled_flex_attn_prefill(q, K, V, block_mask=mask, return_aux=s.aux)
        results += [out, aux.lse]
    return results


def run(state):
    """One step of all layers: (out, lse) of every layer, and the page pool with the step's rows in it."""
    if state.graph is not None:
        state.graph.replay()
        return [*state.results, state.cache.kv_cache]
    results = _decode_step(state) if state.decode else _prefill_step(state)
    return [*results, state.cache.kv_cache]
