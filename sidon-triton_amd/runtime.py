"""Bucketed HIP-graph runtime for the encoder.

Mirrors the encoder side of src/sidon_triton/runtime.py:

  * flat max-size device buffers (features, valid frames, hidden) re-viewed
    per (batch, bucket), allocated once (:140-156 of ``EngineSet``);
  * a chunk runs zero-padded to its bucket with its true length passed
    alongside, so every chunk of a bucket shares one captured graph: 1 s
    buckets up to 32 s, 4 s buckets above, capped at the maximum (:366-372;
    here in 50 Hz frames: 50-frame steps up to 1600 frames, 200-frame steps
    above);
  * graphs keyed by (batch, bucket), captured after a warm-up on a side
    stream, drawing from one shared memory pool, least recently used evicted
    past ``max_graphs`` (:374-401, via ``graphs.BucketGraphs``);
  * all work enqueued on the caller's current stream (the reference's on a
    compute stream of its own, :27, :360): handing a call to another stream and
    back left the GPU idle for 100 us, which is 15% of a 3 s chunk's call.
    Calls from several streams are ordered one after another, since they share
    the buffers.

The valid rows of a bucketed run equal an exact-length run: the front end
takes its statistics over the true frames only, the attention masks the
padded keys, the depthwise conv is causal and every other op is row-wise.

Two entries: ``run`` takes 160-channel features (bucketed in frames);
``run_wave`` takes 16 kHz waveforms and runs the fbank front end and the
encoder in one graph per (batch, bucket), bucketed in samples exactly as
runtime.py:366-372 does.  The decoder is not part of this runtime.
"""

from __future__ import annotations

import contextlib
import ctypes

import torch

from . import _lib
from .encoder import HipEncoder
from .flexrel import _on_device, _stream_handle
from .frontend import BUCKET_QUANTUM, Fbank, num_features
from .graphs import BucketGraphs

FRAME_RATE = 50                 # encoder frames per second
FINE_BUCKET_FRAMES = 50         # 1 s
FINE_LIMIT_FRAMES = 32 * 50     # 32 s
COARSE_BUCKET_FRAMES = 4 * 50   # 4 s
IN_RATE = 16_000
FINE_BUCKET_SAMPLES = IN_RATE           # 1 s
FINE_LIMIT_SAMPLES = 32 * IN_RATE       # 32 s
COARSE_BUCKET_SAMPLES = 4 * IN_RATE     # 4 s
MIN_SEQ = 2


def bucket_frames(frames: int, max_frames: int) -> int:
    """Bucket length (frames) of a chunk with ``frames`` valid frames."""
    if frames < 1:
        raise ValueError("a chunk needs at least one frame")
    step = FINE_BUCKET_FRAMES if frames <= FINE_LIMIT_FRAMES else COARSE_BUCKET_FRAMES
    return min(max_frames, -(-frames // step) * step)


def bucket_samples(samples: int, max_samples: int) -> int:
    """Bucket length (samples, a multiple of 320) of a chunk of ``samples``
    samples (runtime.py:366-372)."""
    if samples < 1:
        raise ValueError("a chunk needs at least one sample")
    step = FINE_BUCKET_SAMPLES if samples <= FINE_LIMIT_SAMPLES else COARSE_BUCKET_SAMPLES
    return min(max_samples, -(-samples // step) * step)


def stage_items(src: torch.Tensor, counts, dst: torch.Tensor, outs) -> None:
    """dst[b] = src[b, :counts[b]] and zeros after it, and for each (out, values)
    of ``outs`` (at most two) out[b] = values[b], on the current stream.  src
    [B, ...] (any device and type), dst [B, ...] fp32 contiguous on the device, out
    int32 [B] on the device, values host ints.  One launch, enqueued without
    waiting for the stream's earlier work, when src is a contiguous fp32 tensor
    of dst's device; a host src is copied before the call returns, so the caller
    may overwrite it, and that copy does wait for the stream."""
    batch = dst.shape[0]
    n, m = src[0].numel(), dst[0].numel()
    direct = src.device == dst.device and src.dtype == torch.float32 and src.is_contiguous() and m % 4 == 0
    if not direct:
        flat = dst.view(batch, m)
        flat[:, :n].copy_(src.reshape(batch, n), non_blocking=src.device.type != "cpu")
        for b, count in enumerate(counts):
            if count < m:
                flat[b, count:].zero_()
    args = []
    for out, values in outs:
        args += [out.data_ptr(), (ctypes.c_int * batch)(*values)]
    args += [None, None] * (2 - len(outs))
    lib = _lib.load()
    with _on_device(dst.device):
        rc = lib.sidon_stage_items(src.data_ptr() if direct else None, n, dst.data_ptr() if direct else None, m,
                                   (ctypes.c_int64 * batch)(*counts), *args, batch, _stream_handle(dst.device))
    _lib.check("sidon_stage_items", rc)


class EncoderRuntime:
    """Encoder calls on bucketed, graph-captured, fixed-address buffers."""

    def __init__(self, encoder: HipEncoder, max_batch: int = 1, max_seconds: float = 96.0,
                 use_graph: bool = True, max_graphs: int = 48, frontend: Fbank | None = None) -> None:
        self.encoder = encoder
        self.max_batch = int(max_batch)
        self.max_seq = int(max_seconds * FRAME_RATE)
        if self.max_seq < MIN_SEQ:
            raise ValueError("max_seconds is too short")
        device = encoder.device
        b, s = self.max_batch, self.max_seq
        self.features = torch.zeros(b * s * encoder.features, device=device)
        self.lens = torch.zeros(b, dtype=torch.int32, device=device)
        self.hidden = torch.zeros(b * s * encoder.hidden, device=device)
        self.workspace = encoder.workspace(b * s)
        self.use_graph = use_graph
        self.graphs = BucketGraphs(max_graphs)
        self.frontend = frontend
        self.max_samples = self.max_seq * BUCKET_QUANTUM
        if frontend is not None:
            self.wave = torch.zeros(b * self.max_samples, device=device)
            self.wave_valid = torch.zeros(b, dtype=torch.int32, device=device)
            self.fbank_workspace = frontend.workspace(b, self.max_samples)
        # The buffers' clears above come before the first call too.
        self._mark(torch.cuda.current_stream(device), torch.cuda.default_stream(device))

    def _mark(self, stream, default) -> None:
        """Later calls wait for what ``stream`` holds now: by an event, or, for
        the default stream, which lives as long as the process, by that stream."""
        self._on_default = stream == default
        self._done = None if self._on_default else stream.record_event()

    @contextlib.contextmanager
    def _ordered(self):
        """The call inside runs after the runtime's construction and its earlier
        calls, whatever streams those ran on.  A capturing stream is refused
        before anything is enqueued: a recording would hold this call's lengths,
        and an event of a capture cannot be waited for outside of it."""
        device = self.encoder.device
        stream, default = torch.cuda.current_stream(device), torch.cuda.default_stream(device)
        with _on_device(device):
            # (the default stream never is, and asking costs the host 12 us)
            if stream != default and torch.cuda.is_current_stream_capturing():
                raise RuntimeError("a runtime's calls cannot be captured into a graph: it keeps graphs of its own")
            if self._done is not None:
                stream.wait_event(self._done)
            elif self._on_default and stream != default:
                stream.wait_stream(default)
            try:
                yield
            finally:
                self._mark(stream, default)

    def bucket(self, frames: int) -> int:
        return bucket_frames(frames, self.max_seq)

    def _views(self, batch: int, length: int):
        enc = self.encoder
        feats = self.features[:batch * length * enc.features].view(batch, length, enc.features)
        hidden = self.hidden[:batch * length * enc.hidden].view(batch, length, enc.hidden)
        return feats, hidden

    def _enqueue(self, batch: int, length: int) -> None:
        feats, hidden = self._views(batch, length)
        self.encoder(feats, self.lens[:batch], out=hidden, workspace=self.workspace)

    def run(self, features: torch.Tensor, frames=None) -> torch.Tensor:
        """features [B, n, F] (any device; fp32) with ``frames`` valid frames
        per item (a sequence of ints, None: all n) -> hidden [B, n, C], a view
        of the runtime's buffer valid until the next call.  Enqueued on the
        current stream."""
        batch, n, nfeat = features.shape
        if not 1 <= batch <= self.max_batch:
            raise ValueError(f"batch {batch} outside [1, {self.max_batch}]")
        if nfeat != self.encoder.features:
            raise ValueError(f"features must have {self.encoder.features} channels")
        frames = [n] * batch if frames is None else [int(f) for f in frames]
        if len(frames) != batch or min(frames) < MIN_SEQ or max(frames) > n:
            raise ValueError(f"frames {frames} must lie in [{MIN_SEQ}, {n}]")
        if n > self.max_seq:
            raise ValueError(f"{n} frames exceed the runtime's maximum of {self.max_seq}")
        length = self.bucket(n)
        with self._ordered():
            feats, hidden = self._views(batch, length)
            stage_items(features, [n * nfeat] * batch, feats, [(self.lens, frames)])
            if self.use_graph:
                self.graphs.run((batch, length), lambda: self._enqueue(batch, length))
            else:
                self._enqueue(batch, length)
        return hidden[:, :n]

    def _enqueue_wave(self, batch: int, samples: int) -> None:
        length = samples // BUCKET_QUANTUM
        feats, hidden = self._views(batch, length)
        wave = self.wave[:batch * samples].view(batch, samples)
        self.frontend(wave, self.wave_valid[:batch], out=feats, workspace=self.fbank_workspace)
        self.encoder(feats, self.lens[:batch], out=hidden, workspace=self.workspace)

    def run_wave(self, wave: torch.Tensor, samples=None) -> torch.Tensor:
        """wave [B, n] 16 kHz fp32 (any device) with ``samples`` true samples
        per item (None: all n) -> hidden [B, num_features(n), C], a view of the
        runtime's buffer valid until the next call; item b's first
        num_features(samples[b]) rows are its valid frames.  Front end and
        encoder run as one graph per (batch, bucket)."""
        if self.frontend is None:
            raise RuntimeError("this runtime was built without a front end")
        batch, n = wave.shape
        if not 1 <= batch <= self.max_batch:
            raise ValueError(f"batch {batch} outside [1, {self.max_batch}]")
        samples = [n] * batch if samples is None else [int(x) for x in samples]
        if len(samples) != batch or max(samples) > n or min(num_features(x) for x in samples) < MIN_SEQ:
            raise ValueError(f"samples {samples} must lie in [1, {n}] and give >= {MIN_SEQ} frames")
        if n > self.max_samples:
            raise ValueError(f"{n} samples exceed the runtime's maximum of {self.max_samples}")
        bucket = bucket_samples(n, self.max_samples)
        with self._ordered():
            view = self.wave[:batch * bucket].view(batch, bucket)
            stage_items(wave, samples, view,
                        [(self.wave_valid, samples), (self.lens, [num_features(x) for x in samples])])
            if self.use_graph:
                self.graphs.run(("wave", batch, bucket), lambda: self._enqueue_wave(batch, bucket))
            else:
                self._enqueue_wave(batch, bucket)
        _, hidden = self._views(batch, bucket // BUCKET_QUANTUM)
        return hidden[:, :num_features(n)]
