"""The staging of a bucketed call's inputs (csrc/stage.hip, runtime.stage_items):
argument checks without a GPU, and on an MI355X the copies, zeros and lengths
against torch for sources of every route (device fp32 at any alignment, other
types, strided, host memory)."""

from __future__ import annotations

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


@pytest.mark.gpu
def test_runtime_calls_from_several_streams_do_not_overlap(sidon):
    """One runtime called from the default stream and from two others in turn,
    with no synchronisation between the calls: every result, copied on its own
    stream, equals the same call made alone."""
    import sys

    from conftest import GOLDEN

    sys.path.insert(0, str(GOLDEN))
    from make_encoder_golden import encoder_weights

    dev = torch.device("cuda:0")
    enc = sidon.encoder.HipEncoder(sidon.encoder.pack_weights(encoder_weights(2, 2, seed=9)), dev)
    rt = sidon.runtime.EncoderRuntime(enc, max_batch=1, max_seconds=12)
    gen = torch.Generator().manual_seed(1)
    feats = [torch.randn(1, n, 160, generator=gen).to(dev) for n in (480, 301, 480, 97, 600, 599)]
    alone = []
    for f in feats:
        alone.append(rt.run(f).clone())
        torch.cuda.synchronize()
    streams = [torch.cuda.current_stream(dev), torch.cuda.Stream(dev), torch.cuda.Stream(dev)]
    for rep in range(3):
        got = []
        for i, f in enumerate(feats):
            with torch.cuda.stream(streams[(i + rep) % 3]):
                got.append(rt.run(f).clone())
                # the next call may start as soon as this one's buffer is read
                for s in streams:
                    s.wait_stream(streams[(i + rep) % 3])
        torch.cuda.synchronize()
        for a, b in zip(got, alone):
            assert torch.equal(a, b), rep
