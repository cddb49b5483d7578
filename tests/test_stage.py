"""The staging of a bucketed call's inputs (csrc/stage.hip, runtime.stage_items):
argument checks without a GPU, and on an MI355X the copies, zeros and lengths
against torch for sources of every route (device fp32 at any alignment, other
types, strided, host memory); and the order of a runtime's calls over streams,
on the host against a model of streams and events."""

from __future__ import annotations

import contextlib
import ctypes

import pytest
import torch


@pytest.mark.parametrize("over,code", [
    (dict(dst=None), -1), (dict(counts=None), -1), (dict(values=None), -1), (dict(src=None, dst=None, out=None), -1),
    (dict(B=0), -2), (dict(m=30), -2), (dict(counts=[41, 1]), -2), (dict(counts=[1, -1]), -2), (dict(n=8), -2),
    (dict(dst=24), -4), (dict(src=18), -4),
])
def test_stage_rejects_bad_arguments(sidon, over, code):
    a = dict(src=16, n=64, dst=32, m=40, counts=[40, 9], out=48, values=[3, 4], B=2)
    a.update(over)
    counts = (ctypes.c_int64 * 2)(*a["counts"]) if a["counts"] else None
    values = (ctypes.c_int * 2)(*a["values"]) if a["values"] else None
    lib = sidon._lib.load()
    assert lib.sidon_stage_items(a["src"], a["n"], a["dst"], a["m"], counts, a["out"], values, None, None, a["B"],
                                 None) == code
    assert lib.sidon_last_error().decode()


class _Stream:
    """What a stream's work comes after: ``seen`` holds the pieces of work that
    are done when its next piece starts."""

    def __init__(self):
        self.seen = set()

    def wait_event(self, event):
        self.seen |= event

    def wait_stream(self, other):
        self.seen |= other.seen

    def record_event(self):
        return frozenset(self.seen)


class _Device:
    """Stands in for torch.cuda, the encoder and the front end of a runtime on the host."""

    device = torch.device("cpu")
    features = hidden = 4

    def __init__(self, monkeypatch, runtime):
        self.streams = {name: _Stream() for name in ("default", "a", "b")}
        self.at, self.work, self.capturing, self.unordered = "default", 0, False, []
        for name, value in (("current_stream", lambda device=None: self.streams[self.at]),
                            ("default_stream", lambda device=None: self.streams["default"]),
                            ("is_current_stream_capturing", lambda: self.capturing)):
            monkeypatch.setattr(torch.cuda, name, value)
        monkeypatch.setattr(runtime, "_on_device", lambda device: contextlib.nullcontext())
        monkeypatch.setattr(runtime, "stage_items", lambda *args: self.launch())

    def launch(self):
        """A piece of work that touches the runtime's buffers, on the current stream."""
        stream = self.streams[self.at]
        if len(stream.seen) < self.work:
            self.unordered.append((self.work, self.at))
        stream.seen.add(self.work)
        self.work += 1

    def workspace(self, *sizes):
        self.launch()      # a buffer is cleared
        return {}

    def __call__(self, *args, **kwargs):
        self.launch()


@pytest.mark.parametrize("order", ["default a", "a default", "a b", "b a b", "default default a", "a a b default b",
                                   "default a default b", "b default a"])
def test_runtime_orders_its_calls_and_its_construction(sidon, monkeypatch, order):
    """Built on the first stream named and called on the others in turn: every
    piece of work on the shared buffers, the constructor's clears among it,
    comes after all earlier ones, whatever streams they are on."""
    dev = _Device(monkeypatch, sidon.runtime)
    dev.at, *calls = order.split()
    rt = sidon.runtime.EncoderRuntime(dev, max_batch=1, max_seconds=2, use_graph=False, frontend=dev)
    built = dev.work
    for dev.at in calls:
        rt.run(torch.zeros(1, 60, 4))
    assert dev.work == built + 2 * len(calls) and not dev.unordered


def test_runtime_refuses_a_capturing_stream(sidon, monkeypatch):
    """Before it enqueues or records anything; the next call outside the capture
    is a call like any other."""
    dev = _Device(monkeypatch, sidon.runtime)
    rt = sidon.runtime.EncoderRuntime(dev, max_batch=1, max_seconds=2, use_graph=False, frontend=dev)
    built, dev.at, dev.capturing = dev.work, "a", True
    for call in (lambda: rt.run(torch.zeros(1, 60, 4)), lambda: rt.run_wave(torch.zeros(1, 16000))):
        with pytest.raises(RuntimeError, match="captured"):
            call()
    assert dev.work == built and not dev.streams["a"].seen
    dev.capturing = False
    rt.run(torch.zeros(1, 60, 4))
    assert dev.work == built + 2 and not dev.unordered


@pytest.mark.gpu
@pytest.mark.parametrize("batch,n,m", [(1, 1, 4), (1, 1023, 1024), (3, 1025, 1100), (2, 4000, 4000), (130, 37, 40)])
@pytest.mark.parametrize("route", ["device", "offset", "double", "strided", "host"])
def test_stage_items_copy_pad_and_set(sidon, batch, n, m, route):
    dev = torch.device("cuda:0")
    gen = torch.Generator().manual_seed(batch + n)
    data = torch.randn(batch, n, generator=gen)
    src = {"device": lambda: data.to(dev),
           "offset": lambda: torch.cat([torch.zeros(1), data.reshape(-1)]).to(dev)[1:].view(batch, n),
           "double": lambda: data.double().to(dev),
           "strided": lambda: torch.stack([data, data], dim=2).to(dev)[:, :, 0],
           "host": lambda: data.clone()}[route]()
    counts = [max(0, n - 3 * b) for b in range(batch)]
    dst = torch.full((batch, m), 9.0, device=dev)
    outs = [torch.full((batch + 1,), -1, dtype=torch.int32, device=dev) for _ in range(2)]
    sidon.runtime.stage_items(src, counts, dst, [(outs[0], counts), (outs[1], range(batch))])
    if route == "host":
        src.fill_(float("nan"))  # the caller may reuse it at once
    want = torch.zeros(batch, m)
    for b, c in enumerate(counts):
        want[b, :c] = data[b, :c]
    assert torch.equal(dst.cpu(), want)
    assert outs[0].tolist() == counts + [-1] and outs[1].tolist() == list(range(batch)) + [-1]


def _runtime(sidon, max_seconds, **kw):
    """A two-layer encoder's runtime on the GPU."""
    from make_encoder_golden import encoder_weights

    enc = sidon.encoder.HipEncoder(sidon.encoder.pack_weights(encoder_weights(2, 2, seed=9)), torch.device("cuda:0"))
    return sidon.runtime.EncoderRuntime(enc, max_batch=1, max_seconds=max_seconds, **kw)


@pytest.mark.gpu
def test_runtime_call_in_a_capture_leaves_both_usable(sidon):
    rt = _runtime(sidon, 12)
    feats, count = torch.randn(1, 97, 160).cuda(), torch.zeros(4, device="cuda")
    alone = rt.run(feats).clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        count.add_(1)
        with pytest.raises(RuntimeError, match="captured"):
            rt.run(feats)
    for rep in range(3):
        graph.replay()
        assert torch.equal(rt.run(feats), alone) and (count == rep + 1).all()


@pytest.mark.gpu
@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("first,second", [(0, 1), (1, 0), (1, 2)])
def test_runtime_call_waits_for_the_one_before(sidon, use_graph, first, second):
    """A long call on one stream (0: the default one) and at once a short one on
    another, nothing between them: the short one, which shares the long one's
    buffers, equals the same call made alone."""
    rt = _runtime(sidon, 96, use_graph=use_graph)
    gen = torch.Generator().manual_seed(1)
    long, short = (torch.randn(1, n, 160, generator=gen).cuda() for n in (4800, 97))
    rt.run(long)
    alone = rt.run(short).clone()
    streams = [torch.cuda.default_stream(), torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for _ in range(3):
        with torch.cuda.stream(streams[first]):
            rt.run(long)
        with torch.cuda.stream(streams[second]):
            got = rt.run(short).clone()
        torch.cuda.synchronize()
        assert torch.equal(got, alone)
