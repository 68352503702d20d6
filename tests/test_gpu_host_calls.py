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
