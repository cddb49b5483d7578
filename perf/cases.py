"""The workloads whose speed matters to a user of this package, as data.

Every case calls the package's public entry points on inputs made from a seed,
at the sizes of the w2v-BERT encoder it is built for (hidden 1024, 16 heads,
feed-forward 4096, convolution of 31 taps, 8 layers): 50 frames a second,
chunks of 1 s to 96 s, run at whole buckets (1 s steps up to 32 s, 4 s steps
above) with their true length inside the bucket.

``listed()`` names the fixed cases, ``draw(rng)`` gives another one of the same
ranges, ``prepare`` / ``run`` make and run a case, ``work`` counts what it
cannot do without, ``exact`` computes it in 64 bits with plain torch and
``tolerance`` says how far two correct implementations may be apart.

The kinds of work:

  attention  8 layers of the fused-QKV attention as one captured graph, the
             valid lengths written before each replay
  views      one eager attention call on [B, H, L, 64] views of three separate
             projections, as the module drop-in makes it
  block      8 attention sub-blocks (norm, QKV, attention, out-projection) on
             the residual stream, one captured graph
  ffn        one feed-forward half step between its two norms, eager, each
             projection on the kernel that the package's own rule prefers
  conv       the convolution module's GLU + depthwise conv + norm + SiLU, eager
  fbank      the front end alone, eager, on caller-kept workspaces
  encoder    the whole encoder through the bucket runtime, from features
  wave       front end and encoder through the bucket runtime, from waveforms
"""

from __future__ import annotations

import importlib
import math

import torch

HEADS = 16
DIM = 64
HIDDEN = HEADS * DIM
INTER = 4096
TAPS = 31
LAYERS = 8
FEATURES = 160
LEFT, RIGHT, POSITIONS = 64, 8, 73
RATE = 16_000
EPS = 1e-5


# ---- cases ------------------------------------------------------------------------


def listed():
    return [
        # A short utterance (3 s bucket), attention alone: 8 launches of a few
        # microseconds each, where latency and launches count.
        {"name": "attention 3 s", "kind": "attention", "batch": 1, "length": 150, "frames": 139, "shortest": 139},
        # A 30 s chunk, its true length inside the bucket.
        {"name": "attention 30 s", "kind": "attention", "batch": 1, "length": 1500, "frames": 1463, "shortest": 1463},
        # The longest chunk the reference runs: the package's headline shape.
        {"name": "attention 96 s", "kind": "attention", "batch": 1, "length": 4800, "frames": 4800, "shortest": 4800},
        # A ragged batch of utterances through the module drop-in's layout, an
        # odd length.
        {"name": "views 4 x 517", "kind": "views", "batch": 4, "heads": 16, "length": 517, "frames": 517,
         "shortest": 211},
        # The attention half of a layer on a chunk of no round length.
        {"name": "block 1037", "kind": "block", "batch": 1, "length": 1037, "frames": 1037, "shortest": 1037},
        # A feed-forward half step of a one-minute chunk.
        {"name": "ffn 3000", "kind": "ffn", "rows": 3000},
        # The convolution module over a small batch of odd length.
        {"name": "conv 3 x 1463", "kind": "conv", "batch": 3, "length": 1463},
        # The front end of a full chunk that is not full to its end.
        {"name": "fbank 96 s", "kind": "fbank", "batch": 1, "bucket": 96 * RATE, "samples": 96 * RATE - 12_345,
         "shortest": 96 * RATE - 12_345},
        # Streaming-sized chunk through the whole encoder: weights dominate.
        {"name": "encoder 3 s", "kind": "encoder", "batch": 1, "frames": 139, "shortest": 139},
        # The common chunk of interactive use.
        {"name": "encoder 15 s", "kind": "encoder", "batch": 1, "frames": 750, "shortest": 750},
        # A ragged batch of utterances.
        {"name": "encoder 4 x 8 s", "kind": "encoder", "batch": 4, "frames": 391, "shortest": 163},
        # The largest call: a full 96 s chunk from its waveform.
        {"name": "wave 96 s", "kind": "wave", "batch": 1, "samples": 96 * RATE - 4_321, "shortest": 96 * RATE - 4_321},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _bucket(frames):
    step = 50 if frames <= 1600 else 200
    return -(-frames // step) * step


def draw(rng):
    """One more case of the same ranges: up to 4800 frames (96 s) in all, in 1 to
    8 items, of any length from half a second."""
    kind = rng.choice(["attention", "attention", "views", "block", "ffn", "ffn", "conv", "fbank", "encoder", "encoder",
                       "encoder", "wave"])
    frames = _log(rng, 25, 4800)
    batch = min(rng.choice([1, 1, 1, 2, 3, 4, 8]), max(1, 4800 // _bucket(frames)))
    shortest = frames if batch == 1 else max(2, int(frames * rng.uniform(0.25, 1.0)))
    if kind == "attention":
        return {"kind": kind, "batch": batch, "length": _bucket(frames), "frames": frames, "shortest": shortest}
    if kind == "views":
        return {"kind": kind, "batch": batch, "heads": rng.choice([4, 8, 16, 16]), "length": frames,
                "frames": frames, "shortest": shortest}
    if kind == "block":
        return {"kind": kind, "batch": batch, "length": frames, "frames": frames, "shortest": shortest}
    if kind == "ffn":
        return {"kind": kind, "rows": _log(rng, 25, 4800)}
    if kind == "conv":
        return {"kind": kind, "batch": batch, "length": frames}
    if kind == "encoder":
        return {"kind": kind, "batch": batch, "frames": frames, "shortest": shortest}
    samples = 320 * frames - rng.randrange(320)
    shortest = samples if batch == 1 else 320 * shortest - rng.randrange(320)
    if kind == "fbank":
        return {"kind": kind, "batch": batch, "bucket": 320 * _bucket(frames), "samples": samples,
                "shortest": shortest}
    return {"kind": kind, "batch": batch, "samples": samples, "shortest": shortest}


def _lengths(longest, shortest, batch):
    """The items' true lengths, evenly from the longest to the shortest."""
    if batch == 1:
        return [longest]
    return [longest - round((longest - shortest) * b / (batch - 1)) for b in range(batch)]


# ---- inputs -----------------------------------------------------------------------


class _Rand:
    """Seeded normal tensors on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, scale=1.0):
        return torch.randn(*shape, generator=self.gen, device="cuda") * scale

    def norm(self, n):
        return (1.0 + self.normal(n, scale=0.1), self.normal(n, scale=0.1), EPS)


def _layer(r):
    """One layer's packed weights (fp16 GEMM operands, fp32 norms, taps and
    biases), random-init at the architecture's scales; the running biases are
    those of a first layer."""
    def h(*shape, scale=0.02):
        return r.normal(*shape, scale=scale).half()

    p = {name: r.norm(HIDDEN) for name in ("ffn1_ln", "attn_ln", "conv_ln", "dw_ln", "ffn2_ln", "final_ln")}
    p.update({
        "ffn1_w1": h(INTER, HIDDEN), "ffn1_b1": h(INTER), "ffn1_w2": h(HIDDEN, INTER, scale=0.01),
        "qkv_w": h(3 * HIDDEN, HIDDEN), "qkv_b": h(3 * HIDDEN), "rel": h(POSITIONS, DIM), "out_w": h(HIDDEN, HIDDEN),
        "pw1_w": h(2 * HIDDEN, HIDDEN), "dwt": r.normal(TAPS, HIDDEN, scale=0.1), "pw2_w": h(HIDDEN, HIDDEN),
        "ffn2_w1": h(INTER, HIDDEN), "ffn2_b1": h(INTER), "ffn2_w2": h(HIDDEN, INTER, scale=0.01),
    })
    b1, b2, b4 = (r.normal(HIDDEN, scale=0.02) for _ in range(3))
    p["cum_bias"] = (b1, b1 + b2, b1 + b2 + b4)
    return p


def _packed(r):
    return {"heads": HEADS, "fp_ln": r.norm(FEATURES), "fp_w": r.normal(HIDDEN, FEATURES, scale=0.02),
            "fp_b": r.normal(HIDDEN, scale=0.02), "layers": [_layer(r) for _ in range(LAYERS)]}


def _speech(r, batch, samples, lens):
    """Waveforms with the level swings of speech: a few harmonics of a moving
    pitch under a slow envelope, over a noise floor, zero past each length."""
    t = torch.arange(samples, device="cuda", dtype=torch.float64) / RATE
    out = torch.zeros(batch, samples, device="cuda")
    for b in range(batch):
        pitch, rate, phase = (float(v) for v in r.normal(3).abs().cpu())
        f0 = 90.0 + 60.0 * pitch
        turn = 2 * math.pi * (f0 * t + 0.8 * torch.sin(2 * math.pi * 0.7 * t))
        voice = sum(torch.sin(k * turn) / k for k in range(1, 9))
        envelope = (0.5 - 0.5 * torch.cos(2 * math.pi * (1.5 + rate) * t + phase)) ** 2
        out[b] = (0.08 * voice * envelope).float() + r.normal(samples, scale=0.004)
        out[b, lens[b]:] = 0.0
    return out


def _inputs(case, seed):
    """The case's inputs and weights, from the seed alone."""
    r, kind = _Rand(seed), case["kind"]
    d = {}
    if kind == "attention":
        rows = case["batch"] * case["length"]
        d["qkv"] = [r.normal(rows, 3 * HIDDEN).half() for _ in range(LAYERS)]
        d["rel"] = [r.normal(POSITIONS, DIM, scale=0.02).half() for _ in range(LAYERS)]
    elif kind == "views":
        shape = (case["batch"], case["length"], case["heads"] * DIM)
        d["q"], d["k"], d["v"] = (r.normal(*shape).half() for _ in range(3))
        d["rel"] = r.normal(POSITIONS, DIM, scale=0.02).half()
    elif kind == "block":
        d["x"] = r.normal(case["batch"] * case["length"], HIDDEN)
        d["layers"] = []
        bias = torch.zeros(HIDDEN, device="cuda")
        for _ in range(LAYERS):
            bias = bias + r.normal(HIDDEN, scale=0.02)
            d["layers"].append({"attn_ln": r.norm(HIDDEN), "qkv_w": r.normal(3 * HIDDEN, HIDDEN, scale=0.02).half(),
                                "qkv_b": r.normal(3 * HIDDEN, scale=0.02).half(),
                                "rel": r.normal(POSITIONS, DIM, scale=0.02).half(),
                                "out_w": r.normal(HIDDEN, HIDDEN, scale=0.02).half(), "cum_bias": bias})
    elif kind == "ffn":
        d["x"] = r.normal(case["rows"], HIDDEN)
        d["before"], d["after"] = r.norm(HIDDEN), r.norm(HIDDEN)
        d["w1"], d["b1"] = r.normal(INTER, HIDDEN, scale=0.02).half(), r.normal(INTER, scale=0.02).half()
        d["w2"], d["b2"] = r.normal(HIDDEN, INTER, scale=0.01).half(), r.normal(HIDDEN, scale=0.02)
    elif kind == "conv":
        d["h"] = r.normal(case["batch"] * case["length"], 2 * HIDDEN, scale=0.7).half()
        d["taps"], d["norm"] = r.normal(TAPS, HIDDEN, scale=0.1), r.norm(HIDDEN)
    elif kind == "fbank":
        d["lens"] = _lengths(case["samples"], case["shortest"], case["batch"])
        d["wave"] = _speech(r, case["batch"], case["bucket"], d["lens"])
    else:
        d["packed"] = _packed(r)
        if kind == "encoder":
            d["lens"] = _lengths(case["frames"], case["shortest"], case["batch"])
            d["features"] = r.normal(case["batch"], case["frames"], FEATURES)
        else:
            d["lens"] = _lengths(case["samples"], case["shortest"], case["batch"])
            d["wave"] = _speech(r, case["batch"], case["samples"], d["lens"])
    return d


# ---- the calls --------------------------------------------------------------------


def _package():
    return importlib.import_module("sidon-triton_amd")


def prepare(case, seed):
    pkg, kind, d = _package(), case["kind"], _inputs(case, seed)
    state = {"kind": kind, "case": case, "pkg": pkg, "in": d}
    if kind in ("attention", "views", "block"):
        lens = _lengths(case["frames"], case["shortest"], case["batch"])
        state["valid"] = torch.tensor(lens, dtype=torch.int32, device="cuda")
    if kind == "attention":
        rows = case["batch"] * case["length"]
        state["lens"] = torch.full((case["batch"],), case["length"], dtype=torch.int32, device="cuda")
        state["out"] = [torch.empty(rows, HIDDEN, dtype=torch.float16, device="cuda") for _ in range(LAYERS)]
        attention = pkg.encoder_attention.flexrel_attention
        qkv, rel, lens, out, batch = d["qkv"], d["rel"], state["lens"], state["out"], case["batch"]

        def enqueue():
            for i in range(LAYERS):
                attention(qkv[i], batch, HEADS, rel[i], lens, out=out[i])

        state["enqueue"], state["graphs"] = enqueue, pkg.graphs.BucketGraphs()
        state["graphs"].capture("layers", enqueue)
    elif kind == "views":
        shape = (case["batch"], case["length"], case["heads"], DIM)
        state["views"] = [d[name].view(shape).transpose(1, 2) for name in "qkv"]
    elif kind == "block":
        rows = case["batch"] * case["length"]
        half = {"dtype": torch.float16, "device": "cuda"}
        state["x"] = d["x"].clone()
        buffers = {"xn": torch.empty(rows, HIDDEN, **half), "qkv": torch.empty(rows, 3 * HIDDEN, **half),
                   "ctx": torch.empty(rows, HIDDEN, **half)}
        x, layers, batch, valid = state["x"], d["layers"], case["batch"], state["valid"]

        def enqueue():
            pkg.encoder_block.attention_blocks(x, layers, batch, HEADS, valid, buffers)

        state["enqueue"], state["graphs"] = enqueue, pkg.graphs.BucketGraphs()
        state["graphs"].capture("blocks", enqueue)
    elif kind == "ffn":
        rows = case["rows"]
        state["xn"] = torch.empty(rows, HIDDEN, dtype=torch.float16, device="cuda")
        state["h"] = torch.empty(rows, INTER, dtype=torch.float16, device="cuda")
    elif kind == "conv":
        state["out"] = torch.empty(case["batch"] * case["length"], HIDDEN, dtype=torch.float16, device="cuda")
    elif kind == "fbank":
        state["fbank"] = pkg.frontend.Fbank("cuda")
        state["valid"] = torch.tensor(d["lens"], dtype=torch.int32, device="cuda")
        state["workspace"] = state["fbank"].workspace(case["batch"], case["bucket"])
        state["out"] = torch.empty(case["batch"], case["bucket"] // 320, FEATURES, device="cuda")
    else:
        encoder = pkg.encoder.HipEncoder(d.pop("packed"), "cuda")
        frontend = pkg.frontend.Fbank("cuda") if kind == "wave" else None
        state["runtime"] = pkg.runtime.EncoderRuntime(encoder, max_batch=case["batch"], max_seconds=96.0,
                                                      frontend=frontend)
        run(state)  # a server warms the buckets that it serves: the bucket's graph is there before the first call
    return state


def run(state):
    pkg, kind, d = state["pkg"], state["kind"], state["in"]
    if kind == "attention":
        state["lens"].copy_(state["valid"])
        state["graphs"].run("layers", state["enqueue"])
        return state["out"]
    if kind == "views":
        return pkg.flexrel.flexrel_attention(*state["views"], d["rel"], lens=state["valid"])
    if kind == "block":
        state["x"].copy_(d["x"])
        state["graphs"].run("blocks", state["enqueue"])
        return state["x"]
    if kind == "ffn":
        ops, x, rows = pkg.conformer, d["x"], state["case"]["rows"]
        xn = pkg.encoder_block.res_norm(x, norm2=d["before"], write_x=False, xn=state["xn"])
        linear = ops.linear_silu if ops.linear_silu_preferred(rows, INTER, HIDDEN, x.device) else ops.linear_silu_lt
        h = linear(xn, d["w1"], d["b1"], out=state["h"])
        if ops.residual_gemm_preferred(rows, HIDDEN, INTER, x.device):
            ops.residual_gemm(x, h, d["w2"])
        else:
            torch.addmm(x, h, d["w2"].t(), out_dtype=torch.float32, out=x)
        xn = pkg.encoder_block.res_norm(x, bias=d["b2"], norm2=d["after"], write_x=False, xn=state["xn"])
        return [x, xn]
    if kind == "conv":
        return pkg.conformer.glu_causal_dw_norm(d["h"], state["case"]["batch"], d["taps"], *d["norm"],
                                                out=state["out"])
    if kind == "fbank":
        return state["fbank"](d["wave"], state["valid"], out=state["out"], workspace=state["workspace"])
    if kind == "encoder":
        hidden = state["runtime"].run(d["features"], d["lens"])
        return [hidden[b, :n] for b, n in enumerate(d["lens"])]  # an item's valid frames: nothing else is meant
    hidden = state["runtime"].run_wave(d["wave"], d["lens"])
    return [hidden[b, :_frames(n)] for b, n in enumerate(d["lens"])]


def _frames(samples):
    """Encoder frames of a waveform: 400-sample windows every 160 samples over
    the waveform padded by 160 on each side, stacked in pairs."""
    return ((samples + 320 - 400) // 160 + 1 + 1) // 2


# ---- what a pass cannot do without ------------------------------------------------


def _attention_flops(batch, heads, length, lens):
    return sum(heads * (4.0 * length * n * DIM + 2.0 * length * POSITIONS * DIM) for n in lens)


def _encoder_work(batch, length, lens):
    rows = batch * length
    weights = 2 * INTER * HIDDEN * 2 + 3 * HIDDEN * HIDDEN + HIDDEN * HIDDEN + 2 * HIDDEN * HIDDEN + HIDDEN * HIDDEN
    flops = 2.0 * rows * (FEATURES * HIDDEN + LAYERS * (weights + TAPS * HIDDEN))
    flops += LAYERS * _attention_flops(batch, HEADS, length, lens)
    return {"bytes": 2.0 * LAYERS * weights + 4.0 * rows * (FEATURES + HIDDEN), "flops": flops}


def work(case):
    kind = case["kind"]
    if kind in ("attention", "views", "block"):
        batch, length = case["batch"], case["length"]
        lens = _lengths(case["frames"], case["shortest"], batch)
        rows = batch * length
        if kind == "attention":
            return {"bytes": LAYERS * rows * 4 * HIDDEN * 2.0,
                    "flops": LAYERS * _attention_flops(batch, HEADS, length, lens)}
        if kind == "views":
            return {"bytes": rows * 4 * case["heads"] * DIM * 2.0,
                    "flops": _attention_flops(batch, case["heads"], length, lens)}
        gemms = 4 * HIDDEN * HIDDEN
        return {"bytes": LAYERS * gemms * 2.0 + rows * HIDDEN * 8.0,
                "flops": LAYERS * (2.0 * rows * gemms + _attention_flops(batch, HEADS, length, lens))}
    if kind == "ffn":
        return {"bytes": 2 * HIDDEN * INTER * 2.0 + case["rows"] * HIDDEN * (4.0 + 4.0 + 2.0),
                "flops": 4.0 * case["rows"] * HIDDEN * INTER}
    if kind == "conv":
        rows = case["batch"] * case["length"]
        return {"bytes": rows * 3 * HIDDEN * 2.0, "flops": rows * HIDDEN * 2.0 * TAPS}
    if kind == "fbank":
        frames = case["batch"] * case["bucket"] // 160
        # A 512-point real transform, the power, 80 triangles and the statistics.
        return {"bytes": case["batch"] * case["bucket"] * 4.0 + frames * 80 * 4.0,
                "flops": frames * (2.5 * 512 * 9 + 3 * 257 + 4 * 257 + 8 * 80)}
    if kind == "encoder":
        lens = _lengths(case["frames"], case["shortest"], case["batch"])
        return _encoder_work(case["batch"], case["frames"], lens)
    lens = [_frames(n) for n in _lengths(case["samples"], case["shortest"], case["batch"])]
    return _encoder_work(case["batch"], max(lens), lens)


def tolerance(case):
    """About four times what each path is off its 64-bit value: fp16 products
    with fp32 sums, and fp16 rounding between the stages of a layer; the front
    end is fp32 throughout."""
    return {
        "attention": {"rel": 1.2e-3, "max": 8e-3},
        "views": {"rel": 1.2e-3, "max": 8e-3},
        "block": {"rel": 1.8e-4, "max": 1e-3},
        "ffn": {"rel": 9e-4, "max": 3e-3},
        "conv": {"rel": 1.2e-3, "max": 9e-3},
        "fbank": {"rel": 1e-5, "max": 1e-4},
        "encoder": {"rel": 2.4e-3, "max": 1.5e-2},
        "wave": {"rel": 2.4e-3, "max": 1.5e-2},
    }[case["kind"]]


# ---- the same in 64 bits ----------------------------------------------------------


def _ln(x, norm):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], norm[0].double(), norm[1].double(), norm[2])


def _silu(x):
    return x * torch.sigmoid(x)


def _linear(x, w):
    return x @ w.double().t()


def _attend(q, k, v, rel, valid):
    """One head: q, k, v [L, 64] in 64 bits, keys past ``valid`` left out."""
    length = q.shape[0]
    keys = torch.arange(valid, device=q.device)
    table = q @ rel.double().t()
    out = torch.empty_like(q)
    for at in range(0, length, 1200):
        rows = torch.arange(at, min(at + 1200, length), device=q.device)
        place = (keys[None, :] - rows[:, None]).clamp(-LEFT, RIGHT) + LEFT
        s = (q[rows] @ k[:valid].t() + table[rows].gather(1, place)) / 8.0
        out[rows] = torch.softmax(s, dim=1) @ v[:valid]
    return out


def _attend_rows(qkv, batch, heads, rel, lens):
    """Fused rows [B*L, 3*H*64] -> context rows [B*L, H*64]."""
    rows, hid = qkv.shape[0], heads * DIM
    length = rows // batch
    out = torch.empty(rows, hid, dtype=torch.float64, device=qkv.device)
    for b in range(batch):
        item = qkv[b * length:(b + 1) * length].double()
        for h in range(heads):
            q, k, v = (item[:, i * hid + h * DIM:i * hid + (h + 1) * DIM].contiguous() for i in range(3))
            out[b * length:(b + 1) * length, h * DIM:(h + 1) * DIM] = _attend(q, k, v, rel, lens[b])
    return out


def _conv(h, batch, taps, norm):
    g = h[:, :HIDDEN] * torch.sigmoid(h[:, HIDDEN:])
    g = torch.nn.functional.pad(g.view(batch, -1, HIDDEN), (0, 0, TAPS - 1, 0))
    length = g.shape[1] - (TAPS - 1)
    y = sum(taps[k].double() * g[:, k:k + length] for k in range(TAPS))
    return _silu(_ln(y.reshape(batch * length, HIDDEN), norm))


def _encode(features, packed):
    """One item [n, 160] -> [n, 1024].  The running biases come off again as the
    stream is summed without them."""
    x = _linear(_ln(features.double(), packed["fp_ln"]), packed["fp_w"]) + packed["fp_b"].double()
    n = x.shape[0]
    for p in packed["layers"]:
        b1, b2, b4 = (b.double() for b in p["cum_bias"])
        x = x + _linear(_silu(_linear(_ln(x, p["ffn1_ln"]), p["ffn1_w1"]) + p["ffn1_b1"].double()), p["ffn1_w2"])
        qkv = _linear(_ln(x + b1, p["attn_ln"]), p["qkv_w"]) + p["qkv_b"].double()
        x = x + _linear(_attend_rows(qkv, 1, HEADS, p["rel"], [n]), p["out_w"])
        c = _conv(_linear(_ln(x + b2, p["conv_ln"]), p["pw1_w"]), 1, p["dwt"], p["dw_ln"])
        x = x + _linear(c, p["pw2_w"])
        h = _silu(_linear(_ln(x + b2, p["ffn2_ln"]), p["ffn2_w1"]) + p["ffn2_b1"].double())
        x = _ln(x + _linear(h, p["ffn2_w2"]) + b4, p["final_ln"])
    return x


def _fbank(wave):
    """One waveform (its true samples) -> [frames, 160] features."""
    x = torch.nn.functional.pad(wave.double(), (160, 160)) * 2.0 ** 15
    frames = x.unfold(0, 400, 160).clone()
    frames = frames - frames.mean(dim=1, keepdim=True)
    before = torch.cat([frames[:, :1], frames[:, :-1]], dim=1)
    i = torch.arange(400, dtype=torch.float64, device=x.device)
    window = (0.5 - 0.5 * torch.cos(2 * math.pi * i / 399)) ** 0.85
    frames = (frames - 0.97 * before) * window
    angle = 2 * math.pi * torch.outer(i, torch.arange(257, dtype=torch.float64, device=x.device)) / 512
    power = (frames @ torch.cos(angle)) ** 2 + (frames @ torch.sin(angle)) ** 2

    def mel(f):
        return 1127.0 * torch.log(1.0 + f / 700.0)

    lo, hi = (mel(torch.tensor(f, dtype=torch.float64, device=x.device)) for f in (20.0, 8000.0))
    edge = lo + (hi - lo) / 81 * torch.arange(82, dtype=torch.float64, device=x.device)
    bins = mel(torch.linspace(0.0, 8000.0, 257, dtype=torch.float64, device=x.device))[:, None]
    up = (bins - edge[:-2]) / (edge[1:-1] - edge[:-2])
    down = (edge[2:] - bins) / (edge[2:] - edge[1:-1])
    y = torch.log((power @ torch.minimum(up, down).clamp_min(0.0)).clamp_min(1.192092955078125e-07))
    y = (y - y.mean(dim=0)) / torch.sqrt(y.var(dim=0, unbiased=True) + 1e-7)
    if y.shape[0] % 2:
        y = torch.cat([y, torch.ones_like(y[:1])])
    return y.reshape(-1, FEATURES)


def exact(case, seed):
    kind, d = case["kind"], _inputs(case, seed)
    if kind in ("attention", "views", "block"):
        lens = _lengths(case["frames"], case["shortest"], case["batch"])
    if kind == "attention":
        return [_attend_rows(d["qkv"][i], case["batch"], HEADS, d["rel"][i], lens) for i in range(LAYERS)]
    if kind == "views":
        batch, length, heads = case["batch"], case["length"], case["heads"]
        qkv = torch.cat([d[name].view(batch * length, heads * DIM) for name in "qkv"], dim=1)
        return _attend_rows(qkv, batch, heads, d["rel"], lens).view(batch, length, heads, DIM).transpose(1, 2)
    if kind == "block":
        x, bias = d["x"].double(), torch.zeros(HIDDEN, dtype=torch.float64, device="cuda")
        for p in d["layers"]:
            qkv = _linear(_ln(x + bias, p["attn_ln"]), p["qkv_w"]) + p["qkv_b"].double()
            x = x + _linear(_attend_rows(qkv, case["batch"], HEADS, p["rel"], lens), p["out_w"])
            bias = p["cum_bias"].double()
        return x + bias
    if kind == "ffn":
        x = d["x"].double()
        h = _silu(_linear(_ln(x, d["before"]), d["w1"]) + d["b1"].double())
        x = x + _linear(h, d["w2"])
        return [x, _ln(x + d["b2"].double(), d["after"])]
    if kind == "conv":
        return _conv(d["h"].double(), case["batch"], d["taps"], d["norm"])
    if kind == "fbank":
        out = torch.zeros(case["batch"], case["bucket"] // 320, FEATURES, dtype=torch.float64, device="cuda")
        for b, n in enumerate(d["lens"]):
            got = _fbank(d["wave"][b, :n])
            out[b, :got.shape[0]] = got
        return out
    if kind == "encoder":
        return [_encode(d["features"][b, :n], d["packed"]) for b, n in enumerate(d["lens"])]
    return [_encode(_fbank(d["wave"][b, :n]), d["packed"]) for b, n in enumerate(d["lens"])]
