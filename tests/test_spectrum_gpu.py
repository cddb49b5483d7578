"""The front end's one-call form (csrc/fbank.hip: float64 FFT per frame, merge in
the normalizing blocks) at the sizes where it can go wrong: the shortest chunk,
frame counts that are no multiple of a block's, one statistics tile and many, a
chunk that starts off a 16-byte boundary, and frames whose quiet bins lie far
below their loud ones (needs an MI355X)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle.frontend_oracle as fo

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _chunks(batch, samples, valid, seed):
    """Noise under a loud low tone that fades in and out: up to ~100 dB between
    a frame's bins."""
    rng = np.random.default_rng(seed)
    t = np.arange(samples) / 16000.0
    out = np.zeros((batch, samples), np.float32)
    for b in range(batch):
        x = 0.6 * np.sin(2 * np.pi * (150 + 40 * b) * t) * (0.5 + 0.5 * np.sin(2 * np.pi * 3 * t)) ** 4
        x = x + 1e-5 * rng.standard_normal(samples) + 0.02
        out[b, :valid[b]] = x[:valid[b]]
    return out


@pytest.mark.parametrize("samples,valid,offset", [
    (640, [640], 0), (640, [400, 641 - 1], 1), (960, [800], 0), (3200, [3200, 1777, 560], 3), (16000, [15999], 0),
    (20480, [20480], 0), (40960, [40959, 30000], 1), (320 * 1300, [320 * 1300 - 77], 2)])
def test_features_match_float64(sidon, samples, valid, offset):
    host = _chunks(len(valid), samples, valid, samples)
    flat = torch.zeros(host.size + offset, device=DEV)
    flat[offset:] = torch.from_numpy(host).to(DEV).reshape(-1)
    chunk = flat[offset:].view(len(valid), samples)
    fb = sidon.frontend.Fbank(DEV)
    got = fb(chunk, torch.tensor(valid, dtype=torch.int32, device=DEV)).double().cpu().numpy()
    assert got.shape == (len(valid), samples // 320, 160)
    for b, n in enumerate(valid):
        want = fo.fbank_exact(host[b, :n])
        rows = want.shape[0]
        # log mel is fp32 of a float64 power: 2^-24 x its size (at most 30), over
        # the bin's deviation, which the normalization divides by
        logmel = fo.frame_features(np.pad(host[b, :n].astype(np.float64), 160), fo.num_frames(n))
        dev = np.tile(np.sqrt(logmel.var(axis=0, ddof=1) + fo.VAR_EPS), 2)
        tol = 16 * 2.0 ** -24 * (30 / dev + np.abs(want))
        assert (np.abs(got[b, :rows] - want) <= tol).all()
        assert not got[b, rows:].any()
