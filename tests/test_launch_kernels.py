"""Which kernels each plan's device-resident launches run
(relx_launch_kernels), for every form of tests/test_ragged.py and
tests/permute_cases.py: a rule that sent a shape to another kernel than the
one these files mean to test fails here."""
import ctypes

import numpy as np
import pytest

from sym_amd import _native as N
from sym_amd import encoder as EN
from sym_amd import pyreloc as P
from sym_amd import workloads as W
from tests import permute_cases as PC
from tests import test_ragged as R

# Per group of test_ragged.py: the kernels that its plans run, every one of
# them. Parameters that run along neither the rows nor the columns leave the
# rows and permute-direct kernels; a vector of q or of a pixel group that a
# wider type does not fill, or planes that fill little of a tile, leave the
# tile and interleave ones.
GROUP_KERNELS = {
    "transpose": {"ragged_transpose", "element"},
    "element": {"element"},
    "permute": {"permute_shift", "permute_div", "permute"},
    "image": {"ragged_interleave", "interleave"},
    "rows": {"rows", "element"},
    "flat": {"flat", "stream"},
}


def _kernels(blob, symbols=None, params=None):
    return P.launch_kernels(P.Bound(P.Plan(blob), symbols or {}, params or {}))


@pytest.mark.parametrize("kind", sorted(GROUP_KERNELS))
def test_kernels_of_the_ragged_groups(kind):
    seen = set()
    for k, case, make in R.GROUPS:
        if k != kind:
            continue
        mine = set()
        for name, blob, _ in make(case):
            got = _kernels(blob)
            assert len(got) == 1 and got[0].split()[0] in GROUP_KERNELS[kind], (name, got)
            mine.add(got[0].split()[0])
        if kind == "rows":
            assert "rows" in mine, case
        if kind == "transpose" and case[1] * case[2] >= 500 and min(case[1:]) >= 9:
            assert mine == {"ragged_transpose"} or case == (2, 35, 15), case
        seen |= mine
    assert seen == GROUP_KERNELS[kind]


@pytest.mark.parametrize("case", PC.cases(), ids=[c[0] for c in PC.cases()])
def test_kernels_of_the_permutes(case):
    """Shifts where every division is one; divisions where only they are
    missing (24 heads, D = 96); the general body where the parameters do not
    run along H."""
    name, blob, _, direct = case
    want = "permute_shift" if direct else "permute" if " per D" in name or " per S" in name or "batch" in name \
        else "permute_div"
    assert [k.split()[0] for k in _kernels(blob)] == [want]


def test_random_permutes_take_every_body():
    assert {_kernels(blob)[0].split()[0] for _, blob, _ in PC.random_cases(200)} == \
        {"permute_shift", "permute_div", "permute"}


def _head_quant(heads):
    return [EN.Cast("float32", "exact"),
            EN.Quantize(EN.InlineParam(tuple(0.01 + 0.001 * i for i in range(heads)), "float32", 1), axis=1)]


# [B, S, H, D] -> [B, H, S, D]: the body and the block (heads by rows of S).
# Blocks of 256 vectors and more, and blocks that fill three quarters of the
# lanes and store whole lines, keep their power-of-two pair of H and S.
PERMUTES = [((8, 1024, 7, 256), "float32", None, "permute 7x1"), ((8, 1024, 7, 256), "float16", None, "permute_div 7x2"),
            ((16, 1024, 32, 96), "float32", None, "permute_div 8x1"), ((16, 1024, 32, 96), "float16", None, "permute_div 16x1"),
            ((16, 1024, 32, 96), "float16", _head_quant(32), "permute_div 16x4"),
            ((128, 196, 12, 64), "float32", None, "permute 12x2"), ((128, 196, 12, 64), "float32", [EN.Cast("float16")], "permute 12x2"),
            ((128, 197, 12, 64), "float32", None, "permute_div 12x1"), ((128, 197, 12, 64), "float16", None, "permute_div 12x8"),
            ((8, 1024, 40, 128), "float32", None, "permute_shift 8x1"), ((8, 1024, 40, 128), "float16", _head_quant(40), "permute_shift 8x2"),
            ((8, 512, 3, 1024), "float32", [EN.Cast("float16")], "permute 3x1"), ((8, 1024, 16, 80), "int8", None, "permute_div 16x4"),
            ((33, 999, 8, 128), "float16", _head_quant(8), "permute_div 8x2"), ((32, 1000, 8, 128), "float16", None, "permute_shift 8x4"),
            ((8, 4096, 32, 128), "float16", _head_quant(32), "permute_shift 16x1")]


@pytest.mark.parametrize("shape,dtype,ops,want", PERMUTES, ids=["%s %s %s" % (s, d, w) for s, d, _, w in PERMUTES])
def test_permute_blocks(shape, dtype, ops, want):
    assert _kernels(EN.encode(list(shape), dtype, [EN.Transpose((0, 2, 1, 3))] + (ops or [])).blob) == [want]


DEQ = EN.Dequantize(EN.InlineParam((0.03125,)))
F16 = EN.Cast("float16")
# Transposes of the last two axes: tiles from 384 elements each on average
# (256 where an element is dequantized), one vector of q and six c.
TRANSPOSES = [((64, 12, 12), "float32", [], "element"), ((64, 16, 16), "float32", [], "element"),
              ((64, 16, 24), "float32", [], "ragged_transpose"), ((64, 16, 23), "float32", [F16], "element"),
              ((64, 24, 40), "float32", [], "ragged_transpose"), ((64, 6, 640), "float16", [], "ragged_transpose"),
              ((64, 6, 641), "float16", [], "element"), ((64, 1000, 6), "float32", [], "element"),
              ((64, 9, 6), "float32", [], "element"), ((64, 6, 16), "int8", [], "element"),
              ((64, 16, 16), "int8", [DEQ, F16], "ragged_transpose"), ((64, 15, 17), "int8", [DEQ], "element"),
              ((64, 16, 16), "int8", [], "element"), ((64, 5, 640), "int8", [DEQ], "element"),
              ((64, 65, 65), "float32", [], "ragged_transpose"), ((64, 33, 17), "float32", [], "ragged_transpose")]


@pytest.mark.parametrize("shape,dtype,ops,want", TRANSPOSES, ids=["%s %s %d" % (s, d, len(o)) for s, d, o, _ in TRANSPOSES])
def test_planes_that_fill_little_of_a_tile(shape, dtype, ops, want):
    plan = EN.encode(list(shape), dtype, ops + [EN.Transpose((0, 2, 1))])
    assert _kernels(plan.blob) == [want]


def test_small_planes_under_swapped_outer_axes():
    for dtype, ops in (("float32", []), ("float32", [F16]), ("int8", [])):
        plan = EN.encode([64, 64, 8, 8, 8], dtype, [EN.Transpose((0, 4, 2, 1, 3))] + ops)
        assert _kernels(plan.blob) == ["element"]


def test_kernels_of_the_workloads():
    assert _kernels(W.c1_plan().blob, {"s0": 64 * 4096}) == ["transpose"]
    assert _kernels(W.c2_plan(n=3).blob) == ["interleave"]
    assert _kernels(W.c3_plan().blob, {"s0": 4096, "s1": 11008},
                    W.param("scale", np.ones(11008, np.float32))) == ["transpose"]
    assert _kernels(W.c4_plan().blob, {"s0": 512, "s1": 256}, W.param("scale", np.ones(512, np.float32))) == ["stream"]
    assert _kernels(W.c5_plan().blob, {"B": 2, "S": 64}, W.param("scale", np.ones(32, np.float32))) == \
        ["permute_shift 16x1"]


# (table dtype, result dtype, elements of a row, kernel) on either side of each
# length from which rows move in cut 16-byte items
GATHERS = [("int8", "int8", 15, "gather"), ("int8", "int8", 17, "gather_cut"), ("int8", "int8", 30, "gather"),
           ("int8", "int8", 31, "gather_cut"), ("int8", "int8", 34, "gather_cut"), ("int8", "int8", 764, "gather"),
           ("int8", "int8", 772, "gather_cut"), ("int8", "int8", 1001, "gather_cut"), ("int8", "int8", 1024, "gather"),
           ("float16", "float16", 15, "gather"), ("float16", "float16", 17, "gather_cut"),
           ("float32", "float32", 33, "gather"), ("float32", "float32", 191, "gather"),
           ("float32", "float32", 193, "gather_cut"), ("float32", "float32", 194, "gather"),
           ("float32", "float16", 7, "gather"), ("float32", "float16", 9, "gather_cut"),
           ("float16", "float32", 501, "gather")]


def _gather_kernels(rows, d, src, count, dst):
    blob = EN.encode_index_select([rows, d], src, count, "int64", dst)
    idx = (np.arange(count) % rows).astype("<i8")
    return P.launch_kernels(P.bind_indexed(P.load_indexed_plan(blob), {}, ("int64", [count], idx.tobytes())))


@pytest.mark.parametrize("src,dst,d,want", GATHERS, ids=["%s-%s %d" % g[:3] for g in GATHERS])
def test_kernels_of_a_row_gather(src, dst, d, want):
    assert _gather_kernels(64, d, src, 8, dst) == [want]


def test_word_rows_that_a_selection_reads_again_keep_whole_items():
    for d, count, want in ((251, 64, "gather_cut"), (251, 65, "gather"), (999, 65, "gather"), (1001, 65, "gather_cut")):
        assert _gather_kernels(64, d, "float32", count, "float32") == [want], (d, count)


def test_refusals():
    b = P.Bound(P.Plan(EN.encode([8, 64], "float32", [EN.Cast("float16")]).blob), {}, {})
    assert P.launch_kernels(b, 0) == ["stream"] and P.launch_kernels(b, 1) == ["stream"]
    for k in (-1, 2):
        with pytest.raises(P.BindError, match="invalid_boundary"):
            P.launch_kernels(b, k)
    err, out = N.relx_err(), ctypes.create_string_buffer(4)
    assert N.lib().relx_launch_kernels(b._h, 0, out, 4, ctypes.byref(err)) != 0
    assert N.lib().relx_launch_kernels(b._h, 0, None, 4, ctypes.byref(err)) != 0
    assert N.lib().relx_launch_kernels(None, 0, out, 4, ctypes.byref(err)) != 0


# Launches of 96 MiB and more whose result rows share lines: tiles 128 wide
# where the planes are wider than a 64 x 64 tile along c
LARGE = [((32768, 24, 40), "float32", [], "ragged_transpose"), ((8192, 63, 65), "float32", [], "ragged_transpose"),
         ((8192, 65, 65), "float32", [], "ragged_transpose_large"), ((32, 2047, 513), "float32", [F16], "ragged_transpose_large"),
         ((32, 2048, 513), "float32", [F16], "ragged_transpose"), ((2, 2047, 513), "float32", [F16], "ragged_transpose"),
         ((1, 8001, 8001), "int8", [], "ragged_transpose_large"), ((500000, 20, 60), "int8", [], "ragged_transpose")]


@pytest.mark.parametrize("shape,dtype,ops,want", LARGE, ids=["%s %s" % (s, d) for s, d, _, _ in LARGE])
def test_large_tiles_need_wide_planes(shape, dtype, ops, want):
    plan = EN.encode(list(shape), dtype, ops + [EN.Transpose((0, 2, 1))])
    assert _kernels(plan.blob) == [want]


# Whole-tile transposes that keep their source in the Infinity Cache: from
# four to two bytes, sources of at most 64 MiB
KEEP = [((16, 1024, 768), "float32", [F16], True), ((16, 1024, 1024), "float32", [EN.Cast("bfloat16")], True),
        ((16, 1024, 1088), "float32", [F16], False), ((2, 4096, 4096), "float32", [F16], False),
        ((16, 1024, 768), "float32", [EN.Quantize(EN.InlineParam((0.03125,)))], False),
        ((16, 1024, 768), "float16", [EN.Cast("float32", "exact"), EN.Quantize(EN.InlineParam((0.03125,)))], False),
        ((16, 1024, 768), "float32", [], False), ((16, 1024, 768), "float16", [EN.Cast("float32", "exact")], False)]


@pytest.mark.parametrize("shape,dtype,ops,keep", KEEP, ids=["%s %s %d" % (s, d, i) for i, (s, d, _, _) in enumerate(KEEP)])
def test_transposes_that_keep_their_source(shape, dtype, ops, keep):
    plan = EN.encode(list(shape), dtype, ops + [EN.Transpose((0, 2, 1))])
    assert _kernels(plan.blob) == ["transpose_keep" if keep else "transpose"]


def _scale(n):
    return EN.InlineParam(tuple(0.01 + 0.001 * (i % 50) for i in range(n)), "float32", 1)


# Large aligned transposes [r, q] whose last tiles are cut: one ragged launch,
# or whole tiles and ragged strips (a channel per element of unaligned rows;
# one-byte rows 8 KiB apart to f32)
CUT = [((4112, 11008), "int8", 0, "float16", ["transpose", "ragged_transpose"]),
       ((4112, 11008), "int8", 1, "float16", ["ragged_transpose_large"]),
       ((4128, 11008), "int8", 0, "float16", ["ragged_transpose"]),
       ((2064, 2064), "int8", 0, "float16", ["ragged_transpose"]),
       ((8208, 8192), "float32", 0, "int8", ["transpose", "ragged_transpose"]),
       ((4112, 8192), "int8", 1, "float32", ["transpose", "ragged_transpose"]),
       ((1040, 8192), "int8", 1, "float32", ["ragged_transpose"]),
       ((4112, 6144), "int8", 1, "float32", ["ragged_transpose"]),
       ((4112, 8192), "int8", 1, "float16", ["ragged_transpose_large"]),
       ((7001, 7003), "int8", 0, "float16", ["ragged_transpose"])]


@pytest.mark.parametrize("shape,dtype,axis,out,want", CUT, ids=["%s %s %d %s" % c[:4] for c in CUT])
def test_cut_tiles_of_large_transposes(shape, dtype, axis, out, want):
    sc = _scale(shape[axis])
    ops = [EN.Quantize(sc, axis=axis)] if out == "int8" else [EN.Dequantize(sc, axis=axis)]
    plan = EN.encode(list(shape), dtype, ops + ([F16] if out == "float16" else []) + [EN.Transpose((1, 0))])
    assert _kernels(plan.blob) == want
    assert P.verify_launches(P.Bound(P.Plan(plan.blob), {}, {}), 0, 1 << 30) >= len(want)
