"""The scratch of attend_slots (partial sums between the two launches of a call of
more than 2^18 keys in all) belongs to one call: calls of other threads on the
same stream, and graphs captured on one stream and replayed side by side, have
their own."""
import threading

import pytest
import torch

from conftest import pkg

AT = pkg("attention")
L = pkg("_lib")
WS = pkg("_workspace")


def _inputs(seed, rows, keys, dev, heads=4, slots=4096):
    g = torch.Generator(device=dev).manual_seed(seed)
    kp, vp = (torch.randn((slots, 1, 128), device=dev, generator=g).to(torch.bfloat16) for _ in range(2))
    req = torch.randperm(slots, device=dev, generator=g).to(torch.int32)
    ids = torch.randint(0, slots, (rows, keys), device=dev, generator=g, dtype=torch.int32)
    q = torch.randn((rows, heads, 128), device=dev, generator=g).to(torch.bfloat16)
    return q, kp, vp, req, ids, 0


def test_a_call_between_the_launches_of_another_has_its_own_scratch(monkeypatch):
    """The second call is made while the first is inside the library, as another
    thread's can be (the binding lets go of the interpreter lock)."""
    if not L.LIB_PATH.exists():
        pkg("build").build()
    ranges = []

    def call(name, *args):
        assert name == "v1_decode_attention_slots_ws"
        at, size = args[-3], args[-2]
        assert at and size == L.lib().v1_decode_attention_slots_workspace(rows, 4, 2048)
        ranges.append((at, at + size))
        if len(ranges) == 1:
            AT.attend_slots(*inputs)

    rows = 136
    inputs = _inputs(1, rows, 2048, "cpu")
    monkeypatch.setattr(L, "call", call)
    monkeypatch.setattr(L, "require_gpu", lambda *tensors: None)
    monkeypatch.setattr(L, "stream_of", lambda t: 0)
    monkeypatch.setattr(WS, "_key", lambda device, tag, stream: ("cpu", 0, tag))
    AT.attend_slots(*inputs)
    (a0, a1), (b0, b1) = ranges
    assert a1 <= b0 or b1 <= a0, "two calls in flight share their scratch"


@pytest.mark.gpu
def test_threads_on_one_stream():
    sets = [_inputs(s, rows, keys, "cuda:0") for s, (rows, keys) in enumerate([(136, 2048), (136, 2048), (600, 512), (300, 1000)])]
    assert all(L.lib().v1_decode_attention_slots_workspace(len(x[0]), 4, x[4].shape[1]) > 0 for x in sets)
    want = [AT.attend_slots(*x) for x in sets]
    torch.cuda.synchronize()
    got, start = [[] for _ in sets], threading.Barrier(len(sets))

    def work(i):
        start.wait()
        for _ in range(40):
            got[i].append(AT.attend_slots(*sets[i]))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sets))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        assert len(g) == 40 and all(torch.equal(x, w) for x in g)


@pytest.mark.gpu
def test_graphs_captured_on_one_stream_replayed_on_two():
    s = torch.cuda.Stream()
    sets = [_inputs(s_, 136, 2048, "cuda:0") for s_ in (1, 2)]
    want = [AT.attend_slots(*x) for x in sets]
    torch.cuda.synchronize()
    graphs, outs = [], []
    with torch.cuda.stream(s):
        AT.attend_slots(*sets[0])
    s.synchronize()
    for x in sets:
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1], stream=s):
            outs.append(AT.attend_slots(*x))
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for _ in range(20):
        for o in outs:
            o.zero_()
        torch.cuda.synchronize()
        for g, t in zip(graphs, streams):
            with torch.cuda.stream(t):
                g.replay()
        AT.attend_slots(*sets[0])  # the program's own work beside them
        torch.cuda.synchronize()
        assert all(torch.equal(o, w) for o, w in zip(outs, want))
