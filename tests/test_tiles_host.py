"""Argument checks of the tiled GEMM's and the one-call front end's entry points: fake aligned addresses,
each case wrong in one argument, refused before any HIP call; and that the sizes of test_tiles_gpu.py
reach every tile that the GEMM's rule picks (no GPU needed)."""

from __future__ import annotations

import ctypes

import pytest
import torch


@pytest.mark.parametrize("over,code", [
    (dict(x=None), -1), (dict(y=None), -1), (dict(C=48), -2), (dict(C=0), -2), (dict(K=96), -2), (dict(M=0), -2),
    (dict(ldx=1000), -3), (dict(ldy=1023), -3), (dict(ldw=1028), -3), (dict(x=24), -4), (dict(y=40), -4),
    (dict(M=1 << 21, ldx=1024), -2), (dict(x=1 << 30, y=(1 << 30) + 64), -2), (dict(w=1 << 30, y=(1 << 30) + 64), -2),
])
def test_glu_projection_rejects_bad_arguments(sidon, over, code):
    a = dict(x=1 << 40, ldx=1024, w=1 << 41, ldw=1024, y=1 << 42, ldy=1024, M=750, C=1024, K=1024)
    a.update(over)
    lib = sidon._lib.load()
    assert lib.sidon_gemm_glu(a["x"], a["ldx"], a["w"], a["ldw"], a["y"], a["ldy"], a["M"], a["C"], a["K"],
                              None) == code
    assert lib.sidon_last_error().decode()


def test_glu_projection_declines_operands_of_4_gib(sidon):
    """So that the encoder's pointwise conv takes its general route there."""
    def rows(m, ld=1024):
        return torch.empty(m, ld, dtype=torch.float16, device="meta")[:, :1024]

    fits = sidon.conformer.linear_glu_fits
    assert fits(rows((1 << 21) - 1), rows(2048)) and fits(rows(1024, 1 << 20), rows(2048))
    assert not fits(rows(1 << 21), rows(2048)) and not fits(rows(750), rows(2048, 1 << 20))


@pytest.mark.parametrize("over", [
    dict(N=96), dict(K=96), dict(M=0), dict(M=3100), dict(ldx=1000), dict(ldx=1028), dict(ldw=1020), dict(ldy=3068),
    dict(ldy=3076), dict(x=(1 << 40) + 8), dict(w=(1 << 41) + 8), dict(y=(1 << 42) + 8), dict(bias=(1 << 43) + 4),
    dict(bias=(1 << 43) + 2), dict(ldx=1 << 22), dict(ldw=1 << 20), dict(y=(1 << 40) + 4096), dict(y=(1 << 41) - 4096),
])
def test_projection_takes_only_what_the_kernel_reads(sidon, over):
    """The answer that sends a call to the tiled kernel: each case wrong in one
    argument (sizes, strides, alignment of each operand and of the bias, spans of
    4 GiB, an output over an operand); the plain call, an 8-byte bias and touching
    ranges are taken, few outputs only of a K up to 2048."""
    def takes(**over):
        a = dict(x=1 << 40, ldx=1024, w=1 << 41, ldw=1024, bias=1 << 43, y=1 << 42, ldy=3072, M=750, N=3072, K=1024)
        a.update(over)
        return sidon._lib.load().sidon_gemm_half_takes(a["x"], a["ldx"], a["w"], a["ldw"], a["bias"], a["y"],
                                                       a["ldy"], a["M"], a["N"], a["K"])

    assert takes(K=2048, ldx=2048, ldw=2048) == takes(M=86, K=4096, ldx=4096, ldw=4096) == 1
    assert takes(M=85, K=4096, ldx=4096, ldw=4096) == takes(M=85, K=2112, ldx=2112, ldw=2112) == 0
    assert takes() == takes(bias=(1 << 43) + 8) == takes(bias=None) == takes(y=(1 << 40) + 750 * 2048) == 1
    assert takes(**over) == 0


@pytest.mark.parametrize("over,code", [
    (dict(part=None), -1), (dict(N=96), -2), (dict(K=192), -2), (dict(M=0), -2), (dict(ldx=4000), -3),
    (dict(ldw=4100), -3), (dict(x=8), -4), (dict(part=8), -4),
])
def test_partial_projection_rejects_bad_arguments(sidon, over, code):
    a = dict(x=1 << 40, ldx=4096, w=1 << 41, ldw=4096, part=1 << 42, elems=1 << 40, M=750, N=1024, K=4096)
    a.update(over)
    lib = sidon._lib.load()
    assert lib.sidon_gemm_part(a["x"], a["ldx"], a["w"], a["ldw"], a["part"], a["elems"], a["M"], a["N"], a["K"],
                               None) == code
    assert lib.sidon_last_error().decode()


@pytest.mark.parametrize("over,code", [
    (dict(x=None), -1), (dict(part=None), -1), (dict(n2_w=None), -1), (dict(xn=None), -1), (dict(splits=0), -2),
    (dict(splits=9), -2), (dict(C=1022), -2), (dict(C=2052), -2), (dict(R=0), -2), (dict(part=8), -4),
    (dict(xn=4), -4),
])
def test_norm_of_partials_rejects_bad_arguments(sidon, over, code):
    a = dict(x=16, part=32, splits=4, n2_w=48, n2_b=64, xn=80, R=10, C=1024)
    a.update(over)
    lib = sidon._lib.load()
    assert lib.sidon_res_norm_parts(a["x"], a["part"], a["splits"], None, None, None, 0.0, a["n2_w"], a["n2_b"], 1e-5,
                                    a["xn"], a["R"], a["C"], None) == code
    assert lib.sidon_last_error().decode()


def test_partial_rows_bound_every_smaller_call(sidon):
    """The workspace rule is monotone and never below the rows themselves."""
    rows = [sidon._lib.load().sidon_gemm_part_rows(m) for m in (1, 150, 4800, 8192, 8193, 50000)]
    assert rows == sorted(rows) and rows[0] == 8192 and rows[-1] == 50000


@pytest.mark.parametrize("over,code", [
    (dict(chunk=None), -1), (dict(roots=None), -1), (dict(feats=None), -1), (dict(B=0), -2), (dict(S=1000), -2),
    (dict(S=160), -2), (dict(max_len=0), -2), (dict(max_len=258), -2), (dict(nbytes=64), -2), (dict(feats=112), -2),
    (dict(B=1 << 20, nbytes=1 << 40), -2), (dict(roots=8), -4), (dict(window=8), -4),
])
def test_front_end_rejects_bad_arguments(sidon, over, code):
    a = dict(chunk=16, valid=32, window=48, roots=64, mel_w=80, mel_lo=96, mel_len=96, max_len=16, logmel=112,
             work=128, nbytes=1 << 30, feats=144, B=1, S=1536000)
    a.update(over)
    lib = sidon._lib.load()
    assert lib.sidon_fbank_features(a["chunk"], a["valid"], a["window"], a["roots"], a["mel_w"], a["mel_lo"],
                                    a["mel_len"], a["max_len"], a["logmel"], a["work"], a["nbytes"], a["feats"],
                                    a["B"], a["S"], None) == code
    assert lib.sidon_last_error().decode()


def _tiles(lib, sizes, epilogue):
    """(rows, columns, K split or not) of the tiles that run ``sizes`` on 256 compute units."""
    bm, bn, reached = ctypes.c_int(), ctypes.c_int(), set()
    for m, n, k in sizes:
        splits = lib.sidon_gemm_choice(m, n, k, epilogue, 8 if epilogue == 2 else 1, 256, bm, bn)
        assert splits >= 1
        reached.add((bm.value, bn.value, splits > 1))
    return reached


# epilogue, (N, K, rows): the encoder's projections over chunks up to 96 s and
# batches past that, as far as each one's route goes (the partial sums' single
# ranges are the in-place epilogue's rows).
@pytest.mark.parametrize("epilogue,projections,lists", [
    (0, [(3072, 1024, 3072), (4096, 1024, 9600)], ["LINEAR", "WIDE"]), (1, [(2048, 1024, 9600)], ["GLU"]),
    (2, [(1024, 1024, 512), (1024, 4096, 2560)], ["PARTS"]), (3, [(1024, 1024, 5120), (1024, 4096, 5120)], ["RESIDUAL"]),
])
def test_every_tile_of_the_projections_is_tested(sidon, epilogue, projections, lists):
    """A refit of the cost rule that moves a shape shows here."""
    import test_tiles_gpu

    lib = sidon._lib.load()
    wanted = _tiles(lib, [(m, n, k) for n, k, rows in projections for m in range(1, rows + 1)], epilogue)
    tested = _tiles(lib, [size for name in lists for size in getattr(test_tiles_gpu, name)], epilogue)
    assert wanted <= tested, sorted(wanted - tested)


@pytest.mark.parametrize("args", [(0, 64, 64, 0, 1, 256), (1, 96, 64, 0, 1, 256), (1, 64, 96, 0, 1, 256),
                                  (1, 64, 64, 4, 1, 256), (1, 64, 64, -1, 1, 256), (1, 64, 64, 0, 2, 256),
                                  (1, 64, 64, 2, 9, 256), (1, 64, 64, 2, 0, 256), (1, 64, 64, 0, 1, 0)])
def test_choice_of_no_such_call(sidon, args):
    assert sidon._lib.load().sidon_gemm_choice(*args, None, None) == 0
