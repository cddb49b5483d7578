"""The front end's one-call form (csrc/fbank.hip: float64 FFT per frame, merge in
the normalizing blocks) at the sizes where it can go wrong: the shortest chunk,
frame counts that are no multiple of a block's, one statistics tile and many, a
chunk that starts off a 16-byte boundary, and frames whose quiet bins lie far
below their loud ones; and its parts as calls of their own (needs an MI355X)."""

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


def _check_features(got, host, valid):
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
    _check_features(got, host, valid)


@pytest.mark.parametrize("at", [0, 159, 5000, 5001, 14999])
@pytest.mark.parametrize("values", [[float("inf")], [float("-inf")], [float("inf")] * 3, [3e38]])
def test_an_infinite_sample_shows_in_its_item_alone(sidon, at, values):
    """Infinite, or too large for an fp32 power: its item's features are NaN (as
    float64 torch gives them), the other item's the same bits as without it."""
    host = torch.from_numpy(_chunks(2, 16000, [15000, 15000], 9)).to(DEV)
    lens = torch.tensor([15000, 15000], dtype=torch.int32, device=DEV)
    fb = sidon.frontend.Fbank(DEV)
    want = fb(host, lens)
    assert torch.isfinite(want).all()
    host[0, at:min(at + len(values), 15000)] = torch.tensor(values, device=DEV)[:15000 - at]
    got, frames = fb(host, lens), fo.num_frames(15000)
    assert got[0].reshape(-1, 80)[:frames].isnan().all() and torch.equal(got[1], want[1])
    assert torch.equal(got[0].reshape(-1, 80)[frames:], want[0].reshape(-1, 80)[frames:])


@pytest.mark.parametrize("samples,valid,offset", [
    (640, [640], 0), (960, [800, 960], 1), (1600, [1600, 1111, 560], 2), (32000, [31999], 3), (32000, [32000, 20001], 0)])
def test_features_in_parts_match_float64(sidon, samples, valid, offset):
    """frames, the product with ``frame_transform``, logmel and normalize as calls of
    their own: the framing exact, the log mel within fp32 of the spectrum it is
    given, the features as the one call's are held to."""
    host = _chunks(len(valid), samples, valid, samples + 1)
    batch, frames = len(valid), samples // 160
    flat = torch.zeros(host.size + offset, device=DEV)
    flat[offset:] = torch.from_numpy(host).to(DEV).reshape(-1)
    fb, lib, stream = sidon.frontend.Fbank(DEV), sidon._lib.load(), torch.cuda.current_stream().cuda_stream
    rows = torch.full((batch * frames + 1, 400), 7.0, device=DEV)
    sidon._lib.check("frames", lib.sidon_fbank_frames(flat[offset:].data_ptr(), rows.data_ptr(), batch, samples, stream))
    padded = torch.nn.functional.pad(torch.from_numpy(host), (160, 160))
    want = padded.unfold(1, 400, 160)[:, :frames].reshape(batch * frames, 400)
    assert torch.equal(rows[:-1].cpu(), want) and (rows[-1] == 7).all()

    spec = (rows[:-1].double() @ sidon.frontend.frame_transform().to(DEV).double()).float()
    logmel = torch.full((batch * frames + 1, 80), 7.0, device=DEV)
    sidon._lib.check("logmel", lib.sidon_fbank_logmel(
        spec.data_ptr(), fb.mel_w.data_ptr(), fb.mel_lo.data_ptr(), fb.mel_len.data_ptr(), fb.mel_w.shape[1],
        logmel.data_ptr(), batch * frames, stream))
    power = spec[:, :257].double() ** 2 + spec[:, 257:].double() ** 2
    mel = power.cpu() @ torch.from_numpy(sidon.frontend.mel_banks())
    want = torch.log(mel.clamp_min(fo.MEL_FLOOR))
    # a positive sum of up to 16 terms of four roundings each, then the log's
    assert ((logmel[:-1].double().cpu() - want).abs() <= 2.0 ** -24 * (24 + 4 * want.abs())).all()
    assert (logmel[-1] == 7).all()

    nbytes = lib.sidon_fbank_workspace_bytes(batch, frames)
    work, out = torch.full((nbytes // 4 + 64,), 7.0, device=DEV), torch.empty(batch, frames // 2, 160, device=DEV)
    lens = torch.tensor(valid, dtype=torch.int32, device=DEV)
    sidon._lib.check("normalize", lib.sidon_fbank_normalize(
        logmel.data_ptr(), lens.data_ptr(), work.data_ptr(), nbytes, out.data_ptr(), batch, frames, stream))
    assert (work[-64:] == 7).all()
    _check_features(out.double().cpu().numpy(), host, valid)
