"""The tiled GEMM kernel (csrc/gemm_tile.h) through each of its epilogues, at
sizes that reach every tile shape the rule of csrc/gemm.hip picks for the
encoder's projections on 256 compute units (test_tiles_host.py holds the lists
below to that), one row past and before tile edges, and at fewer K slices than
ring buffers; and the norm that adds a split projection's partial sums (needs an
MI355X)."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


# (rows, columns, K) by epilogue.
LINEAR = [
    (1, 64, 64), (31, 128, 64), (33, 64, 128), (65, 192, 192), (97, 4096, 256), (129, 4096, 320), (333, 4096, 128),
    (400, 4096, 1024), (500, 3072, 1024), (577, 3072, 1024), (577, 4096, 1024), (750, 3072, 1024), (751, 4096, 1024),
    (1000, 4096, 192), (1463, 3072, 1024), (1601, 3072, 1024), (2000, 4096, 128), (2303, 4096, 1024),
    (3000, 3072, 192), (9000, 1024, 64)]
GLU = [(m, 2048, k) for m, k in (
    (1, 64), (33, 128), (300, 1024), (650, 1024), (900, 192), (1000, 1024), (1463, 256), (1601, 1024), (2500, 128),
    (3000, 1024), (3600, 192), (4200, 1024), (1025, 1024), (1279, 1024))]
PARTS = [(1, 64, 128), (33, 1024, 4096), (97, 1024, 4096), (150, 1024, 4096), (200, 1024, 4096), (300, 1024, 4096),
         (577, 1024, 4096), (751, 1024, 4096), (1463, 1024, 4096), (150, 1024, 1024), (400, 1024, 1024),
         (2500, 1024, 4096), (130, 1024, 4096), (257, 1024, 4096), (479, 1024, 4096), (500, 1024, 4096),
         (865, 1024, 4096), (1121, 1024, 4096), (1599, 1024, 4096), (2047, 1024, 4096)]
WIDE = [(2305, 4096, 1024), (2561, 4096, 1024), (3841, 4096, 1024), (4095, 4096, 1024), (4097, 4096, 1024),
        (4799, 4096, 1024)]
RESIDUAL = [(m, 1024, k) for k, rows in (
    (1024, (33, 511, 513, 1025, 1537, 1599, 1601, 1700, 2049, 2200, 2561, 3000, 3500, 4097, 4799)),
    (4096, (150, 1000, 1100, 1537, 1601, 2049, 2081, 2500, 3073, 4097))) for m in rows]


def _operands(m, n, k, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(m, k, generator=gen, device=DEV).half()
    w = (torch.randn(n, k, generator=gen, device=DEV) / k ** 0.5).half()
    return x, w, gen


def _sums(x, w):
    """The float64 products, and a bound on the error of fp32 sums in any order."""
    exact = x.double() @ w.double().t()
    return exact, x.shape[1] * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())


def _block_layer(gen):
    return {"attn_ln": (torch.ones(1024, device=DEV), torch.zeros(1024, device=DEV), 1e-5),
            "qkv_w": (torch.randn(3072, 1024, generator=gen, device=DEV) * 0.02).half(),
            "qkv_b": torch.zeros(3072, dtype=torch.float16, device=DEV),
            "rel": torch.zeros(73, 64, dtype=torch.float16, device=DEV),
            "out_w": (torch.randn(1024, 1024, generator=gen, device=DEV) * 0.02).half(),
            "cum_bias": torch.zeros(1024, device=DEV)}


@pytest.mark.parametrize("m,n,k", LINEAR)
def test_linear_matches_float64(sidon, m, n, k):
    """Bias, SiLU of the fp32 sum, one rounding: within half an fp16 step of the
    float64 value plus the fp32 sums' own bound (the SiLU's slope is below
    1.1); columns beside a strided output stay untouched."""
    assert sidon._lib.load().sidon_gemm_half_preferred(m, n, k)
    x, w, gen = _operands(m, n, k, m + n + k)
    b = (torch.randn(n, generator=gen, device=DEV) * 0.1).half()
    exact, bound = _sums(x, w)
    exact = exact + b.double()
    for act in (False, True):
        wide = torch.full((m + 1, n + 16), 7.0, dtype=torch.float16, device=DEV)
        out = sidon.conformer.linear_silu_lt(x, w, b, out=wide[:m, 8:n + 8], act=act)
        want = torch.nn.functional.silu(exact) if act else exact
        tol = 2.0 ** -11 * want.abs() + 1.1 * bound + 2.0 ** -20 * want.abs() + 2.0 ** -24
        assert ((out.double() - want).abs() <= tol).all(), (act, float(((out.double() - want).abs() - tol).max()))
        assert (wide[:, :8] == 7).all() and (wide[:, n + 8:] == 7).all() and (wide[m] == 7).all()


@pytest.mark.parametrize("m,n,k", WIDE)
def test_linear_silu_matches_float64(sidon, m, n, k):
    """The form with two roundings: the sum to fp16, within half a step plus the fp32
    sums' bound, and its SiLU (slope below 1.1) once more."""
    x, w, gen = _operands(m, n, k, m + n + k)
    b = (torch.randn(n, generator=gen, device=DEV) * 0.1).half()
    exact, bound = _sums(x, w)
    exact = exact + b.double()
    off = 2.0 ** -11 * exact.abs() + bound + 2.0 ** -24
    wide = torch.full((m + 1, n + 16), 7.0, dtype=torch.float16, device=DEV)
    out = sidon.conformer.linear_silu(x, w, b, out=wide[:m, 8:n + 8], act=False)
    assert ((out.double() - exact).abs() <= off).all()
    out = sidon.conformer.linear_silu(x, w, b, out=wide[:m, 8:n + 8])
    want = torch.nn.functional.silu(exact)
    assert ((out.double() - want).abs() <= 1.1 * off + (2.0 ** -11 + 2.0 ** -20) * want.abs() + 2.0 ** -24).all()
    assert (wide[:, :8] == 7).all() and (wide[:, n + 8:] == 7).all() and (wide[m] == 7).all()


@pytest.mark.parametrize("m,n,k", RESIDUAL)
def test_residual_gemm_matches_float64(sidon, m, n, k):
    """Into random values, each lane adding the ones it loaded: the sums' bound and
    one more fp32 rounding; rows and columns beside the stream stay untouched."""
    x, w, gen = _operands(m, n, k, m + k)
    exact, bound = _sums(x, w)
    buf = torch.randn(m + 1, n + 16, generator=gen, device=DEV)
    old = buf.clone()
    sidon.conformer.residual_gemm(buf[:m, 8:n + 8], x, w)
    want = old[:m, 8:n + 8].double() + exact
    assert ((buf[:m, 8:n + 8].double() - want).abs() <= bound + 2.0 ** -24 * want.abs()).all()
    buf[:m, 8:n + 8] = old[:m, 8:n + 8]
    assert torch.equal(buf, old)


@pytest.mark.parametrize("m,n,k", GLU)
def test_linear_glu_is_the_projection_then_the_glu(sidon, m, n, k):
    """Bit for bit what the projection followed by the GLU kernel gives: the
    same sums in the same order, the same roundings."""
    x, w, _ = _operands(m, n, k, m + k)
    h = torch.empty(m, n, dtype=torch.float16, device=DEV)
    want = sidon.conformer.glu(sidon.conformer.linear_silu(x, w, None, out=h, act=False))
    assert torch.equal(sidon.conformer.linear_glu(x, w), want)


def test_linear_glu_narrow_and_strided(sidon):
    x, w, _ = _operands(70, 192, 192, 3)          # C = 96, one wavefront's columns past a power of two
    wide = torch.full((70, 112), 7.0, dtype=torch.float16, device=DEV)
    got = sidon.conformer.linear_glu(x, w, out=wide[:, 8:104])
    h = (x.double() @ w.double().t()).half().double()
    want = h[:, :96] * torch.sigmoid(h[:, 96:])
    assert ((got.double() - want).abs() <= 2.0 ** -9 * want.abs() + 2.0 ** -12).all()
    assert (wide[:, :8] == 7).all() and (wide[:, 104:] == 7).all()


@pytest.mark.parametrize("m,n,k", PARTS)
def test_partials_add_up_and_join_the_stream(sidon, m, n, k):
    """The partial tiles' sum against float64, twice with the same bits; a
    buffer of ``partial_values`` holds them; the norm adds them to the stream."""
    x, w, gen = _operands(m, n, k, m + n + k)
    exact, bound = _sums(x, w)
    part = torch.full((sidon.conformer.partial_values(m, n),), float("nan"), device=DEV)
    got = sidon.conformer.residual_partials(x, w, part)
    assert got.shape[0] == sidon.conformer.residual_splits(m, n, k, DEV) and got.shape[0] >= 1
    assert ((got.double().sum(0) - exact).abs() <= bound + 1e-12).all()
    again = sidon.conformer.residual_partials(x, w, torch.empty_like(part))
    assert torch.equal(again, got)
    stream = torch.randn(m, n, generator=gen, device=DEV)
    want = stream.double() + exact
    sidon.encoder_block.res_norm_parts(stream, got)
    # the sum of up to 9 fp32 terms: each addition rounds values below the bound
    scale = got.double().abs().sum(0) + want.abs()
    assert ((stream.double() - want).abs() <= bound + 9 * 2.0 ** -24 * scale).all()


@pytest.mark.parametrize("rows,cols,splits", [(1, 4, 1), (3, 100, 2), (5, 1024, 8), (2, 1028, 3), (7, 2048, 5)])
@pytest.mark.parametrize("first", [False, True])
def test_res_norm_parts_matches_float64(sidon, rows, cols, splits, first):
    gen = torch.Generator(device=DEV).manual_seed(rows + cols)

    def r(*shape):
        return torch.randn(*shape, generator=gen, device=DEV)

    x, part, bias = r(rows, cols), r(splits, rows, cols), r(cols)
    norms = [(1 + 0.1 * r(cols), 0.1 * r(cols), 1e-5) for _ in range(2)]
    summed = x.double() + part.double().sum(0)

    def ln(v, p):
        return torch.nn.functional.layer_norm(v, (cols,), p[0].double(), p[1].double(), p[2])

    stored = ln(summed + bias.double(), norms[0]) if first else summed
    normed = ln(stored if first else summed + bias.double(), norms[1])
    got = x.clone()
    xn = sidon.encoder_block.res_norm_parts(got, part, bias=bias, norm1=norms[0] if first else None, norm2=norms[1])
    # fp32 arithmetic on values of a few units; the fp16 output rounds once more
    assert ((got.double() - stored).abs() <= 2e-5 * (1 + stored.abs())).all()
    assert ((xn.double() - normed).abs() <= 2.0 ** -11 * normed.abs() + 4e-5).all()


def test_split_projections_replay_like_eager(sidon):
    """A captured projection, partial sums and norm, replayed three times with
    eager work between, equal the eager calls."""
    x, w, gen = _operands(150, 1024, 4096, 5)
    ln = (torch.ones(1024, device=DEV), torch.zeros(1024, device=DEV), 1e-5)
    start = torch.randn(150, 1024, generator=gen, device=DEV)
    part = torch.empty(sidon.conformer.partial_values(150, 1024), device=DEV)
    stream, xn = start.clone(), torch.empty(150, 1024, dtype=torch.float16, device=DEV)

    def step():
        sidon.encoder_block.res_norm_parts(stream, sidon.conformer.residual_partials(x, w, part), norm2=ln, xn=xn)

    step()
    want, want_n = stream.clone(), xn.clone()
    graphs = sidon.graphs.BucketGraphs()
    graphs.capture("step", step)
    for rep in range(3):
        stream.copy_(start)
        xn.zero_()
        part.zero_()
        graphs.run("step", step)
        torch.cuda.synchronize()
        assert torch.equal(stream, want) and torch.equal(xn, want_n), rep
        _ = (start * 2).sum().item()


def test_residual_gemm_takes_a_contiguous_or_a_strided_stream(sidon):
    """K = 4096 into a contiguous stream and into a strided one."""
    x, w, gen = _operands(201, 1024, 4096, 6)
    exact, bound = _sums(x, w)
    for ld in (1024, 1040):
        buf = torch.randn(202, ld, generator=gen, device=DEV)
        old = buf.clone()
        sidon.conformer.residual_gemm(buf[:201, :1024], x, w)
        want = old[:201, :1024].double() + exact
        scale = want.abs() + exact.abs() + 1
        assert ((buf[:201, :1024].double() - want).abs() <= bound + 9 * 2.0 ** -24 * scale).all()
        assert torch.equal(buf[201], old[201]) and torch.equal(buf[:, 1024:], old[:, 1024:])


@pytest.mark.parametrize("rows", [25, 150, 750, 1024])
def test_residual_projections_take_no_memory(sidon, rows):
    """``residual_gemm`` at any K, the attention sub-blocks on buffers for all
    their results and an encoder on its workspace allocate nothing, as a capture
    begun outside torch needs; without buffers the sub-blocks give the same bits."""
    from make_encoder_golden import encoder_weights

    def allocated():
        return torch.cuda.memory_stats(DEV)["allocation.all.allocated"]

    x, w, gen = _operands(rows, 1024, 4096, rows)
    stream = torch.randn(rows, 1024, generator=gen, device=DEV)
    before = allocated()
    sidon.conformer.residual_gemm(stream, x, w)
    sidon.conformer.residual_gemm(stream, x[:, :1024], w[:, :1024])
    assert allocated() == before

    half = dict(dtype=torch.float16, device=DEV)
    layers = [_block_layer(gen) for _ in range(2)]
    buffers = {"xn": torch.empty(rows, 1024, **half), "qkv": torch.empty(rows, 3072, **half),
               "ctx": torch.empty(rows, 1024, **half)}
    start = stream.clone()
    want = sidon.encoder_block.attention_blocks(start.clone(), layers, 1, 16, None)
    before = allocated()
    sidon.encoder_block.attention_blocks(stream, layers, 1, 16, None, buffers)
    assert allocated() == before and torch.equal(stream, want)
    # sums in another order, within a part of one fp16 step of the stream
    part = torch.full((sidon.conformer.partial_values(rows, 1024),), float("nan"), device=DEV)
    split = start.clone()
    before = allocated()
    sidon.encoder_block.attention_blocks(split, layers, 1, 16, None, {**buffers, "part": part})
    assert allocated() == before and float((split - want).norm() / want.norm()) <= 2.0 ** -11

    packed = sidon.encoder.pack_weights(encoder_weights(2, 2, seed=9))
    for own in (None, True):
        enc = sidon.encoder.HipEncoder(packed, DEV, own_residual=own)
        feats = torch.randn(1, rows, 160, generator=gen, device=DEV)
        lens, out = torch.full((1,), rows, dtype=torch.int32, device=DEV), torch.empty(1, rows, enc.hidden, device=DEV)
        ws = enc.workspace(rows)
        enc(feats, lens, out=out, workspace=ws)       # the libraries' own first call
        before = allocated()
        enc(feats, lens, out=out, workspace=ws)
        assert allocated() == before


@pytest.mark.parametrize("rows,n,k,in_place,split", [
    (150, 1024, 4096, 1, True), (512, 512, 4096, 1, True), (150, 1024, 2048, 1, True), (25, 1024, 1024, 1, True),
    (5120, 1024, 1024, 1, False), (5121, 1024, 1024, 0, False), (100, 1024, 192, 0, False)])
def test_residual_route(sidon, rows, n, k, in_place, split):
    """Split where a buffer is there and the cost rule splits, else in place up to
    5 * 2^20 outputs, else the library."""
    ops = sidon.conformer
    assert ops.residual_gemm_preferred(rows, n, k, DEV) == bool(in_place)
    assert ops.residual_splits(rows, n, k, DEV, part=False) == in_place
    assert ops.residual_splits(rows, n, k, DEV) in (range(2, 9) if split else (in_place,))


def _check_conv(sidon, batch, t, c, taps_n):
    gen = torch.Generator(device=DEV).manual_seed(t + c)
    h = torch.randn(batch * t, 2 * c, generator=gen, device=DEV).half()
    taps = torch.randn(taps_n, c, generator=gen, device=DEV) * 0.2
    w, b = 1 + 0.1 * torch.randn(c, generator=gen, device=DEV), 0.1 * torch.randn(c, generator=gen, device=DEV)
    g = sidon.conformer.glu(h)
    wide = torch.full((batch * t + 1, c), 7.0, dtype=torch.float16, device=DEV)
    got = sidon.conformer.causal_dw_norm(g, batch, taps, w, b, 1e-5, out=wide[:batch * t])
    assert torch.equal(sidon.conformer.glu_causal_dw_norm(h, batch, taps, w, b, 1e-5), got)
    assert (wide[batch * t] == 7).all()
    x = torch.nn.functional.pad(g.double().view(batch, t, c), (0, 0, taps_n - 1, 0))
    y = sum(taps[k].double() * x[:, k:k + t] for k in range(taps_n)).reshape(batch * t, c)
    y = torch.nn.functional.silu(torch.nn.functional.layer_norm(y, (c,), w.double(), b.double(), 1e-5))
    # fp32 sums and norm of values of a few units, one rounding to fp16
    assert ((got.double() - y).abs() <= 2.0 ** -11 * y.abs() + 3e-5).all()


@pytest.mark.parametrize("batch,t,c", [(1, 1, 2), (1, 150, 1024), (2, 250, 1024), (1, 500, 130), (3, 333, 1024),
                                       (1, 1500, 1024), (4, 400, 1024), (1, 3001, 1024), (1, 4999, 64),
                                       (2, 700, 1026), (1, 3000, 2048)])
def test_conv_module_at_every_block_size(sidon, batch, t, c):
    """Frame counts that pick each number of frames per block, ragged last
    blocks, channel counts that leave a wavefront part empty, both widths of a
    block: from h and from g alike, bit for bit, and against float64 torch."""
    _check_conv(sidon, batch, t, c, 31)


@pytest.mark.parametrize("taps,t,c", [(31, 4799, 1536), (31, 3001, 1030), (31, 4801, 2048), (31, 3001, 1540),
                                      (31, 400, 1200), (15, 4799, 1100), (15, 3001, 2046), (15, 4900, 1600),
                                      (7, 4800, 1026), (3, 3000, 1538), (3, 150, 2048)])
def test_conv_module_past_1024_channels(sidon, taps, t, c):
    """20, 16, 8 and 4 frames per block on up to 12 and up to 16 wavefronts, with the
    frames ahead of the products refilled as they are taken, or 8 at a time."""
    _check_conv(sidon, 1, t, c, taps)


@pytest.mark.parametrize("rows", [150, 1100])
@pytest.mark.parametrize("layout", ["columns", "rows of 1028"])
def test_projections_take_weights_of_any_layout(sidon, rows, layout):
    """Weights that the tiled kernel's 16-byte copies cannot read (stored
    transposed, or with rows no multiple of 16 bytes apart) go through
    torch.addmm: ``linear`` within its rounding, the attention sub-blocks as on
    packed weights up to the fp16 roundings between the stages, each a part of
    one fp16 step of the stream."""
    def laid(w):
        if layout == "columns":
            return w.t().contiguous().t()
        return torch.nn.functional.pad(w, (0, 4))[:, :w.shape[1]]

    x, w, gen = _operands(rows, 3072, 1024, rows)
    b = (torch.randn(3072, generator=gen, device=DEV) * 0.1).half()
    exact, bound = _sums(x, w)
    exact = exact + b.double()
    assert not sidon.conformer.tile_operand(laid(w)) and not sidon.conformer.linear_glu_fits(x, laid(w))
    out = sidon.conformer.linear(x, laid(w), b, torch.empty(rows, 3072, dtype=torch.float16, device=DEV))
    assert ((out.double() - exact).abs() <= 2.0 ** -10 * exact.abs() + bound + 2.0 ** -24).all()

    layers = []
    for _ in range(2):
        layers.append({"attn_ln": (torch.ones(1024, device=DEV), torch.zeros(1024, device=DEV), 1e-5),
                       "qkv_w": (torch.randn(3072, 1024, generator=gen, device=DEV) * 0.02).half(), "qkv_b": b,
                       "rel": (torch.randn(73, 64, generator=gen, device=DEV) * 0.02).half(),
                       "out_w": (torch.randn(1024, 1024, generator=gen, device=DEV) * 0.02).half(),
                       "cum_bias": torch.randn(1024, generator=gen, device=DEV) * 0.02})
    stream = torch.randn(rows, 1024, generator=gen, device=DEV)
    want = sidon.encoder_block.attention_blocks(stream.clone(), layers, 1, 16, None)
    odd = [{**p, "qkv_w": laid(p["qkv_w"]), "out_w": laid(p["out_w"])} for p in layers]
    got = sidon.encoder_block.attention_blocks(stream.clone(), odd, 1, 16, None)
    assert float((got - want).norm() / want.norm()) <= 2.0 ** -11


@pytest.mark.parametrize("form", ["bias off 8 bytes", "output over x", "output over w"])
def test_linear_leaves_to_torch_what_the_kernel_cannot_read(sidon, monkeypatch, form):
    """Not to the library behind ``linear_silu_lt``, whose first call must not be
    captured: bit for bit torch.addmm."""
    monkeypatch.setattr(sidon.conformer, "linear_silu_lt", None)
    x, w, gen = _operands(200, 1024, 1024, 7)
    b = torch.randn(1026, generator=gen, device=DEV).half()
    want = torch.addmm(b[1:1025] if "bias" in form else b[:1024], x, w.t())
    if "bias" in form:
        got = sidon.conformer.linear(x, w, b[1:1025], torch.empty_like(want))
        assert torch.equal(got, want)
    else:
        seen = []
        monkeypatch.setattr(torch, "addmm", lambda *args, out: seen.append(out))
        sidon.conformer.linear(x, w, b[:1024], x if "x" in form else w[:200])
        assert len(seen) == 1


@pytest.mark.parametrize("rows", [150, 1100])
@pytest.mark.parametrize("name", ["x", "qkv_w", "qkv_b", "out_w"])
def test_sub_blocks_refuse_what_autograd_would_follow(sidon, rows, name):
    """The results go into given tensors: as torch.addmm(out=) does, the call
    raises where a gradient or a tangent would be dropped (its form with an fp32
    output takes a weight that requires one), and runs without gradients as on
    plain tensors."""
    from torch.autograd import forward_ad

    gen = torch.Generator(device=DEV).manual_seed(rows)
    layers = [_block_layer(gen) for _ in range(2)]
    start = torch.randn(rows, 1024, generator=gen, device=DEV)

    def call(change):
        x, p = start.clone(), dict(layers[0])
        if name == "x":
            x = change(x)
        else:
            p[name] = change(p[name])
        return sidon.encoder_block.attention_blocks(x, [p, layers[1]], 1, 16, None)

    def tracked(t):
        return t.clone().requires_grad_()

    want = call(lambda t: t)
    if name == "out_w":
        assert float((call(tracked).detach() - want).norm() / want.norm()) <= 2.0 ** -11
    else:
        with pytest.raises(RuntimeError, match="automatic differentiation"):
            call(tracked)
    with torch.no_grad():
        assert torch.equal(call(tracked), want)
    with forward_ad.dual_level(), pytest.raises(NotImplementedError, match="forward AD"):
        call(lambda t: forward_ad.make_dual(t, torch.ones_like(t)))
    assert torch.equal(call(lambda t: torch.nn.Parameter(t, requires_grad=False)), want)


@pytest.mark.parametrize("rows", [150, 1100])
def test_residual_gemm_refuses_operands_in_the_stream(sidon, rows):
    """On the split route and in place alike; touching ranges do not overlap."""
    buf = torch.zeros(rows * 1024 + rows * 2048 + 64, device=DEV)
    x = buf[:rows * 1024].view(rows, 1024)
    w = torch.zeros(1024, 4096, dtype=torch.float16, device=DEV)
    with pytest.raises(RuntimeError, match="overlap"):
        sidon.conformer.residual_gemm(x, buf[rows * 1024 - 4:][:rows * 2048].view(torch.float16).view(rows, 4096), w)
    sidon.conformer.residual_gemm(x, buf[rows * 1024:][:rows * 2048].view(torch.float16).view(rows, 4096), w)
    assert (buf == 0).all()


@pytest.mark.parametrize("rows,cols", [(1, 256), (5, 1024), (7, 1020), (3, 2048), (3000, 1024)])
@pytest.mark.parametrize("form", ["first norm", "last norm", "last bias"])
def test_res_norm_at_the_ends_of_a_stack(sidon, rows, cols, form):
    """The forms compiled for whole 256-column chunks, and the general form beside
    them (1020 columns), against float64."""
    gen = torch.Generator(device=DEV).manual_seed(rows + cols)
    x = torch.randn(rows, cols, generator=gen, device=DEV)
    bias = torch.randn(cols, generator=gen, device=DEV)
    w, b = (1 + 0.1 * torch.randn(cols, generator=gen, device=DEV)), 0.1 * torch.randn(cols, generator=gen, device=DEV)
    res_norm, got = sidon.encoder_block.res_norm, x.clone()

    def ln(v):
        return torch.nn.functional.layer_norm(v, (cols,), w.double(), b.double(), 1e-5)

    if form == "first norm":
        xn = res_norm(got, norm2=(w, b, 1e-5), write_x=False)
        want = ln(x.double())
        # fp32 arithmetic on values of a few units; the fp16 output rounds once more
        assert torch.equal(got, x) and xn.dtype == torch.float16
        assert ((xn.double() - want).abs() <= 2.0 ** -11 * want.abs() + 4e-5).all()
    elif form == "last norm":
        res_norm(got, bias=bias, norm1=(w, b, 1e-5))
        want = ln((x + bias).double())
        assert ((got.double() - want).abs() <= 2e-5 * (1 + want.abs())).all()
    else:
        res_norm(got, bias=bias)
        assert torch.equal(got, x + bias)
