"""The calls of an eager layer in C++ (csrc/host.cpp): append, decode step and prefill attention from tensors."""

import gc
import sys
import threading
import time

import pytest
import torch

from falcon_perception_amd import _native as N
from falcon_perception_amd import ops
from tests.gpu_cases import DEV, PagedState, randn

pytestmark = pytest.mark.gpu


class Layer:
    """Two sequences in a small cache and the arguments of the three calls, as ops.py and the drop-in give them."""

    def __init__(self, dtype=torch.float32, Hc=2, G=2, D=64, P=16):
        st = self.st = PagedState(71, n_pages=16, page_size=P, max_batch=4, Hc=Hc, D=D, dtype=dtype)
        for n in (40, 25):
            st.add_sequence(n)
        st.prefill_random()
        self.P, self.scale, self.limit = P, D**-0.5, 64
        self.pk, self.pv = st.pool_planes()
        self.table = st.cache.page_table
        self.bidx = torch.tensor(st.slots, dtype=torch.int64, device=DEV)
        self.pos = torch.tensor([39, 24], dtype=torch.int32, device=DEV)
        self.k, self.v = (randn(st.gen, (2, Hc, 1, D), dtype).to(DEV) for _ in range(2))
        self.q = randn(st.gen, (2, Hc * G, 1, D), dtype).to(DEV)
        self.qp = randn(st.gen, (1, Hc * G, 65, D), dtype).to(DEV)
        self.rows = torch.tensor([st.slots[0]] * 40 + [st.slots[1]] * 25, dtype=torch.int64, device=DEV)
        self.limits = torch.cat([torch.arange(1, 41), torch.arange(1, 26)]).to(torch.int32).to(DEV)
        self.arrivals = torch.zeros(64, dtype=torch.int32, device=DEV)
        self.stream = N.raw_stream(self.q.get_device())

    def append(self, **c):
        a = {**vars(self), **c}
        return N.host().append(a["pk"], a["pv"], a["k"], a["v"], a["table"], a["bidx"], a["pos"], self.P, True, False, self.stream)

    def decode(self, **c):
        a = dict(vars(self), ws=None, sinks=None, kn=None, vn=None, plan=None, after=None, split=64)
        a.update(c)
        return N.host().decode(a["q"], a["pk"], a["pv"], a["table"], a["bidx"], a["pos"], self.P, self.limit, self.scale, a["split"],
                               a["ws"], a["sinks"], 1, a["kn"], a["vn"], a["plan"], a["arrivals"], a["after"], self.stream)

    def prefill(self, **c):
        a = dict(vars(self), sinks=None, ws=None, order=None, order_rows=0)
        a.update(c)
        return N.host().prefill(a["qp"], a["pk"], a["pv"], a["table"], a["rows"], a["limits"], self.P, self.scale, a["sinks"], a["ws"],
                                0.0, a["order"], a["order_rows"], self.stream)


@pytest.mark.parametrize("call", ["append", "decode", "prefill"])
def test_other_threads_run_while_a_call_does(call):
    """With a switch interval of minutes a thread runs only when another lets go of the interpreter by itself."""
    layer = Layer()
    run = getattr(layer, call)
    turns, stop = [0], threading.Event()

    def other():
        while not stop.is_set():
            turns[0] += 1
            time.sleep(0)

    thread = threading.Thread(target=other)
    interval = sys.getswitchinterval()
    try:
        sys.setswitchinterval(600.0)
        thread.start()
        while turns[0] == 0:
            time.sleep(0.001)
        gc.collect()
        gc.disable()
        before, results = turns[0], []  # kept: a tensor that goes away lets go of the interpreter, too
        while turns[0] == before and len(results) < 4000:
            results.append(run())
        assert turns[0] > before and None not in results
    finally:
        gc.enable()
        sys.setswitchinterval(interval)
        stop.set()
        thread.join()
        torch.cuda.synchronize()


class Other(torch.Tensor):
    pass


def spread(t):
    """The same values with a gap behind every element of the last axis."""
    return torch.stack([t, t], -1).flatten(-2)[..., ::2]


# what the C++ calls leave to ops.py: (call, argument, the value it is given instead)
LEFT = [
    ("append", "k", spread), ("append", "v", spread), ("append", "v", lambda t: t[:1]), ("append", "v", lambda t: t.half()),
    ("append", "k", lambda t: t.as_subclass(Other)), ("append", "k", lambda t: t.cpu()), ("append", "k", lambda t: t[0]),
    ("append", "pk", lambda t: t.half()), ("append", "pv", lambda t: t.transpose(0, 1)), ("append", "table", lambda t: t.int()),
    ("append", "table", spread), ("append", "bidx", lambda t: t.int()), ("append", "bidx", spread), ("append", "bidx", lambda t: t[:1]),
    ("append", "pos", lambda t: t.float()), ("append", "pos", spread), ("append", "pos", lambda t: t[:1]),
    ("decode", "q", spread), ("decode", "q", lambda t: t.half()), ("decode", "q", lambda t: t[:, :, 0]),
    ("decode", "q", lambda t: t.repeat(1, 1, 2, 1)), ("decode", "q", lambda t: t.as_subclass(Other)), ("decode", "pv", lambda t: t[:, 1:]),
    ("decode", "bidx", lambda t: t.int()), ("decode", "bidx", lambda t: t[:1]), ("decode", "pos", spread), ("decode", "pos", lambda t: t[:1]),
    ("decode", "split", lambda t: 0), ("decode", "ws", lambda t: torch.zeros(64, device=DEV)), ("decode", "plan", lambda t: torch.zeros(64, device=DEV)),
    ("decode", "arrivals", lambda t: t.long()), ("decode", "arrivals", lambda t: None), ("decode", "after", lambda t: torch.zeros(8, dtype=torch.int32, device=DEV)),
    ("decode", "sinks", lambda t: torch.zeros(4, dtype=torch.float64, device=DEV)), ("decode", "sinks", lambda t: torch.zeros(3, device=DEV)),
    ("decode", "sinks", lambda t: torch.zeros(4)), ("decode", "kn", lambda t: torch.zeros(2, 2, 1, 64, device=DEV)),
    ("prefill", "qp", spread), ("prefill", "qp", lambda t: t.repeat(2, 1, 1, 1)), ("prefill", "qp", lambda t: t.half()),
    ("prefill", "rows", lambda t: t.int()), ("prefill", "rows", spread), ("prefill", "limits", lambda t: t.long()),
    ("prefill", "limits", lambda t: t[:5]), ("prefill", "sinks", lambda t: torch.zeros(4, dtype=torch.float64, device=DEV)),
    ("prefill", "ws", lambda t: torch.zeros(64, device=DEV)),
    ("prefill", "order", lambda t: (torch.zeros(1, dtype=torch.int32, device=DEV))),  # without its number of rows
]


@pytest.mark.parametrize("i", range(len(LEFT)))
def test_what_is_not_recognised_is_left_alone(i):
    call, name, other = LEFT[i]
    layer = Layer()
    before = layer.st.cache.kv_cache.clone()
    assert getattr(layer, call)(**{name: other(getattr(layer, name, None))}) is None
    assert torch.equal(layer.st.cache.kv_cache, before)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
def test_results_are_those_of_ops(dtype, monkeypatch):
    layer = Layer(dtype)
    pool = layer.st.cache.kv_cache
    before = pool.clone()
    assert layer.append() is True
    after = pool.clone()
    assert not torch.equal(after, before)
    pool.copy_(before)
    sinks = torch.linspace(-2, 3, 4, device=DEV)
    args = (layer.pk, layer.pv, layer.table)
    ws = torch.empty(ops.decode_workspace_bytes(2, 4, 64, layer.limit, 64), dtype=torch.uint8, device=DEV)
    step = layer.decode(ws=ws if ws.numel() else None, sinks=sinks, kn=layer.k, vn=layer.v, after=torch.ones_like(layer.arrivals))
    assert torch.equal(pool, after)
    n = ops.prefill_tile_rows(65, 4, 2, 64, dtype)  # 0: takes no order
    order = ops.prefill_tile_order(layer.rows, layer.limits, n)[0] if n else None
    rows = layer.prefill(sinks=sinks, order=order, order_rows=n)
    pool.copy_(before)

    class Nothing:  # ops.py by itself
        append = staticmethod(lambda *a: None)

    monkeypatch.setattr(N, "host", lambda: Nothing)
    ops.kv_append(*args[:2], layer.k, layer.v, layer.table, layer.bidx, layer.pos, layer.P, True)
    assert torch.equal(pool, after)
    pool.copy_(before)
    for got, ref in ((step, ops.paged_decode(layer.q, *args, layer.bidx, layer.pos, layer.P, layer.limit, split_tokens=64, sinks=sinks,
                                             k_new=layer.k, v_new=layer.v, arrivals=layer.arrivals)),
                     (rows, ops.paged_prefill(layer.qp, *args, layer.rows, layer.limits, layer.P, sinks=sinks, workspace=False))):
        for x, y in zip(got, ref):
            assert x.shape == y.shape and x.stride() == y.stride() and x.dtype == y.dtype and torch.equal(x, y)
    for change, match in ((dict(v=layer.v[:1]), "same shape"), (dict(table=layer.table.int()), "page_table must be int64"),
                          (dict(pk=layer.pk.double()), "dtype mismatch"), (dict(pk=layer.pk.transpose(0, 1)), "must be contiguous")):
        a = {**vars(layer), **change}
        monkeypatch.undo()
        with pytest.raises(RuntimeError, match=match):
            ops.kv_append(a["pk"], a["pv"], a["k"], a["v"], a["table"], a["bidx"], a["pos"], layer.P, True)


def test_wrong_numbers_of_arguments_are_refused():
    for call in (N.host().append, N.host().decode, N.host().prefill):
        with pytest.raises(TypeError, match="arguments expected"):
            call(1, 2)
