"""Relayouts whose extents and row alignments fit no whole tile or vector:
every launch verified on the CPU, and on the GPU every result byte against
the oracle (uploaded at two chunk sizes, device-resident and device -> host),
with guard bytes around each result."""
import numpy as np
import pytest

from oracle import relx_oracle as O
from sym_amd import encoder as EN
from sym_amd import pyreloc as P

GUARD = 64


def _scale(n, rng):
    return EN.InlineParam(tuple(float(v) for v in rng.uniform(0.004, 0.05, n)), "float32", 1)


def _zp(n, rng):
    return EN.InlineParam(tuple(int(v) for v in rng.integers(-9, 10, n)), "int32", 1)


def _chains(shape, axis, rng):
    """(source dtype, ops) of each value chain; per-channel ones along `axis`
    (per tensor when None)."""
    def sc():
        return _scale(shape[axis], rng) if axis is not None else EN.InlineParam((0.03125,), "float32", 0)

    zp = _zp(shape[axis], rng) if axis is not None else EN.InlineParam((-3,), "int32", 0)
    return [("int8", []), ("float16", []), ("float32", []),
            ("float32", [EN.Cast("float16")]), ("float32", [EN.Cast("bfloat16")]),
            ("float16", [EN.Cast("float32", "exact")]),
            ("int8", [EN.Dequantize(sc(), zero_point=zp, axis=axis)]),
            ("int8", [EN.Dequantize(sc(), axis=axis), EN.Cast("float16")]),
            ("float32", [EN.Quantize(sc(), axis=axis)]),
            ("float16", [EN.Cast("float32", "exact"), EN.Quantize(sc(), axis=axis)]),
            # bf16 sources, and chains without a compile-time kernel body
            ("bfloat16", [EN.Cast("float32", "exact")]),
            ("int8", [EN.Dequantize(sc(), zero_point=zp, axis=axis), EN.Cast("bfloat16")]),
            ("bfloat16", [EN.Cast("float32", "exact"), EN.Quantize(sc(), axis=axis)])]


def _source(shape, dtype, rng):
    if dtype == "int8":
        return rng.integers(-128, 128, shape, dtype=np.int8)
    narrow = "float32" if dtype == "bfloat16" else dtype
    x = (rng.standard_normal(shape) * 3).astype(narrow)
    x.reshape(-1)[:: 97] = np.resize(np.array([np.nan, np.inf, -np.inf, -0.0, 6e4, 1e-7], narrow),
                                     x.reshape(-1)[::97].size)
    return (x.view(np.uint32) >> 16).astype(np.uint16) if dtype == "bfloat16" else x


# (rows, cols) [batch] around the tile widths: one row of a vector less or
# more than a tile, extents of the smallest tile launch, several tiles
TRANSPOSES = [(None, 16, 16), (None, 17, 31), (None, 63, 65), (None, 64, 130), (None, 129, 127),
              (None, 257, 190), (3, 33, 67), (2, 128, 129),
              # either side of the smallest c and q that take tiles; the others
              # run element-wise
              (None, 5, 40), (None, 6, 40), (2, 40, 3), (None, 130, 4), (None, 70, 7), (None, 70, 8),
              (2, 35, 15),
              # either side of the fewest elements that a tile may hold, with
              # the narrowest tiles along c and along q
              (None, 6, 640), (None, 640, 6), (3, 16, 24), (3, 16, 23), (None, 64, 8), (2, 9, 57)]


def transpose_cases(case):
    batch, r, q = case
    rng = np.random.default_rng(r * 1000 + q)
    shape, perm = ((r, q), (1, 0)) if batch is None else ((batch, r, q), (0, 2, 1))
    for axis in [None] + list(range(len(shape))):
        for dtype, ops in _chains(shape, axis, rng):
            if axis is not None and not any(isinstance(o, (EN.Dequantize, EN.Quantize)) for o in ops):
                continue
            plan = EN.encode(list(shape), dtype, ops + [EN.Transpose(perm)])
            yield "%s %s axis %s %s" % (dtype, shape, axis, [type(o).__name__ for o in ops]), plan.blob, \
                _source(shape, dtype, rng)


# (shape, pads as (axis, lo, hi), outer permutation): pads that begin and end
# inside a vector, rows of one vector and of one element more, padded outer
# axes, odd rows under swapped outer axes
ROWS = [((5, 16), ((1, 0, 1),), None), ((7, 17), ((1, 3, 0),), None), ((33, 1003), ((1, 0, 21),), None),
        ((9, 130), ((1, 5, 7),), None), ((6, 65), ((0, 1, 2), (1, 1, 0)), None), ((1, 300), ((1, 2, 3),), None),
        ((3, 4, 5, 35), (), (0, 2, 1, 3)), ((3, 5, 67), (), (1, 0, 2)), ((2, 3, 5, 21), ((3, 1, 1),), None)]


def rows_cases(case):
    shape, pads, perm = case
    rng = np.random.default_rng(sum(shape))
    for axis in [None] + list(range(len(shape))):
        for dtype, ops in _chains(shape, axis, rng):
            params = any(isinstance(o, (EN.Dequantize, EN.Quantize)) for o in ops)
            if axis is not None and not params:
                continue
            layout = [EN.Pad(a, lo, hi, 3 if dtype == "int8" else 1.5) for a, lo, hi in pads]
            layout += [EN.Transpose(perm)] if perm else []
            # a fill cannot cross a per-channel stage: the pad follows it
            ops = layout + ops if axis is None else ops + layout
            try:
                plan = EN.encode(list(shape), dtype, ops)
            except EN.EncodeError:
                continue
            yield "%s %s axis %s %s" % (dtype, shape, axis, [type(o).__name__ for o in ops]), plan.blob, \
                _source(shape, dtype, rng)


# flat tensors: channels of rows shorter and longer than a vector that start
# inside one, one channel per column with the wrap inside a vector, tails of
# every length class
FLAT = [(3, 17), (37, 16), (50, 21), (129, 67), (11, 4099), (1, 1027), (2053, 33)]


def flat_cases(shape):
    rng = np.random.default_rng(shape[0] * 31 + shape[1])
    for axis in (None, 0, 1):
        for dtype, ops in _chains(shape, axis, rng):
            plan = EN.encode(list(shape), dtype, ops)
            yield "%s %s axis %s %s" % (dtype, shape, axis, [type(o).__name__ for o in ops]), plan.blob, \
                _source(shape, dtype, rng)


# ([batch..., C, H, W], leading and trailing channel pad) to two, four or
# eight interleaved channels: pixel counts that cut the last pixel group at
# every place, one group, planes of one batch entry after another
IMAGES = [((2, 3, 3, 5), (0, 1)), ((3, 1, 17, 19), (1, 0)), ((1, 3, 4, 4), (1, 0)), ((2, 5, 9, 11), (1, 2)),
          ((5, 4, 25, 41), (0, 0)), ((2, 2, 3, 7, 13), (0, 1)), ((4, 7, 3, 7), (0, 1)), ((1, 2, 1, 1027), (0, 0))]


def image_cases(case):
    shape, (lo, hi) = case
    rng = np.random.default_rng(sum(shape))
    n = len(shape)
    perm = tuple(range(n - 3)) + (n - 2, n - 1, n - 3)
    for dtype, ops in _chains(shape, None, rng):
        layout = ([EN.Pad(n - 3, lo, hi, 3 if dtype == "int8" else 1.5)] if lo + hi else []) + [EN.Transpose(perm)]
        plan = EN.encode(list(shape), dtype, layout + ops)
        yield "%s %s %s" % (dtype, shape, [type(o).__name__ for o in ops]), plan.blob, _source(shape, dtype, rng)


# [B, S, H, D] -> [B, H, S, D]: heads and head dims whose blocks are no power
# of two, and sequence lengths that cut the last block of rows
PERMUTES = [(2, 5, 12, 64), (1, 7, 40, 128), (3, 13, 32, 96), (2, 9, 8, 128), (1, 333, 16, 64), (2, 2, 6, 32)]


def permute_cases(shape):
    rng = np.random.default_rng(sum(shape))
    out = [shape[i] for i in (0, 2, 1, 3)]
    for axis in (None, 1, 2):
        for dtype, ops in _chains(out, axis, rng):
            if axis is not None and not any(isinstance(o, (EN.Dequantize, EN.Quantize)) for o in ops):
                continue
            plan = EN.encode(list(shape), dtype, [EN.Transpose((0, 2, 1, 3))] + ops)
            yield "%s %s axis %s %s" % (dtype, shape, axis, [type(o).__name__ for o in ops]), plan.blob, \
                _source(shape, dtype, rng)


# Plans that no vector or tile kernel takes (rows and extents below a vector,
# channel maps along a merged axis, pads beside a transpose), one element at a
# time: (shape, perm, pads, reshape)
ELEMENTS = [((3, 5, 2, 7), (2, 0, 3, 1), (), None), ((40, 3), None, ((0, 1, 2), (1, 0, 1)), None),
            ((9, 33), (1, 0), ((0, 2, 1),), None), ((4, 6, 10), (1, 0, 2), (), (24, 10)),
            ((2, 3, 2, 3, 2, 3), (5, 3, 1, 4, 2, 0), (), None)]


def element_cases(case):
    shape, perm, pads, to = case
    rng = np.random.default_rng(sum(shape))
    for axis in [None] + list(range(len(shape))):
        for dtype, ops in _chains(shape, axis, rng):
            if axis is not None and not any(isinstance(o, (EN.Dequantize, EN.Quantize)) for o in ops):
                continue
            layout = ([EN.Transpose(perm)] if perm else [])
            layout += [EN.Pad(a, lo, hi, 3 if dtype == "int8" else 1.5) for a, lo, hi in pads]
            layout += [EN.Reshape(to)] if to else []
            ops = layout + ops if axis is None else ops + layout
            try:
                plan = EN.encode(list(shape), dtype, ops)
            except EN.EncodeError:
                continue
            yield "%s %s axis %s %s" % (dtype, shape, axis, [type(o).__name__ for o in ops]), plan.blob, \
                _source(shape, dtype, rng)


GROUPS = [("transpose", c, transpose_cases) for c in TRANSPOSES]
GROUPS += [("element", c, element_cases) for c in ELEMENTS]
GROUPS += [("permute", c, permute_cases) for c in PERMUTES]
GROUPS += [("image", c, image_cases) for c in IMAGES]
GROUPS += [("rows", c, rows_cases) for c in ROWS]
GROUPS += [("flat", c, flat_cases) for c in FLAT]
IDS = ["%s %s" % (k, c) for k, c, _ in GROUPS]


@pytest.mark.parametrize("group", GROUPS, ids=IDS)
def test_launches_verify(group):
    _, case, make = group
    for name, blob, x in make(case):
        b = P.Bound(P.Plan(blob), {}, {})
        for k in range(b.info.host_stages_max + 1):
            for chunk in (0, 4096, 1 << 14):
                assert P.verify_launches(b, k, chunk) >= 1, name


def _want(blob, x):
    with np.errstate(all="ignore"):
        if P.Plan(blob).typed:
            return O.run_typed(blob, {}, {}, x).tobytes()
    return O.execute_layout(O.bind(O.decode_plan(blob), {}), x.tobytes())


@pytest.mark.gpu
@pytest.mark.parametrize("group", GROUPS, ids=IDS)
def test_results_on_the_gpu(group):
    torch = pytest.importorskip("torch")
    _, case, make = group
    with P.Context(0) as ctx:
        for name, blob, x in make(case):
            print("[gpu-case]", name, flush=True)
            want = _want(blob, x)
            n = len(want)
            b = P.Bound(P.Plan(blob), {}, {})
            buf = torch.empty(n + 2 * GUARD, dtype=torch.uint8, device="cuda")
            out = buf[GUARD:GUARD + n]
            src = torch.from_numpy(np.ascontiguousarray(x).view(np.uint8).reshape(-1).copy())
            dev = src.cuda()
            stream = torch.cuda.current_stream().cuda_stream

            def check(what):
                torch.cuda.synchronize()
                got = buf.cpu().numpy()
                assert got[GUARD:GUARD + n].tobytes() == want, (name, what)
                assert (got[:GUARD] == 0xA5).all() and (got[GUARD + n:] == 0xA5).all(), (name, what)

            for chunk in (0, 4096):
                buf.fill_(0xA5)
                ctx.execute_h2d(b, src.data_ptr(), src.numel(), out.data_ptr(), n, host_stages=0,
                                chunk_bytes=chunk, caller_stream=stream)
                check("upload, chunk %d" % chunk)
            buf.fill_(0xA5)
            ctx.relayout_device(b, dev.data_ptr(), out.data_ptr(), stream=stream)
            check("device")
            host = np.full(n, 0xA5, np.uint8)
            ctx.execute_d2h(b, dev.data_ptr(), dev.numel(), host.ctypes.data, n, chunk_bytes=4096,
                            source_pinned=0, caller_stream=stream)
            assert host.tobytes() == want, (name, "d2h")


# (table dtype, result dtype, row elements): rows of one 16-byte item, of one
# element more and less than items, and on either side of each length from
# which rows move in cut items
GATHERS = [("int8", "int8", (15, 16, 17, 31, 33, 127, 764, 772, 1001)),
           ("float16", "float16", (7, 8, 9, 15, 17, 63, 501)),
           ("float32", "float32", (5, 31, 32, 33, 63, 191, 193, 1001)), ("float32", "float16", (7, 8, 9, 11, 33, 1001)),
           ("float16", "float32", (3, 9, 33, 501))]


@pytest.mark.gpu
@pytest.mark.parametrize("src,dst,widths", GATHERS, ids=["%s-%s" % g[:2] for g in GATHERS])
def test_row_gathers_on_the_gpu(src, dst, widths):
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(len(widths))
    with P.Context(0) as ctx:
        # selections of more and of fewer rows than the table has
        for d, rows, count in [(d, rows, 333) for d in widths for rows in (211, 401)]:
            x = _source((rows, d), src, rng)
            idx = rng.integers(0, rows, count).astype("<i8")
            idx[:2] = (rows - 1, 0)
            blob = EN.encode_index_select([rows, d], src, count, "int64", dst)
            b = P.bind_indexed(P.load_indexed_plan(blob), {}, ("int64", [count], idx.tobytes()))
            with np.errstate(all="ignore"):
                want = (O.narrow_f32_f16_bits(x.view(np.uint32)) if (src, dst) == ("float32", "float16") else
                        O.widen_f16_f32_bits(x.view(np.uint16)) if src != dst else x)[idx].tobytes()
            sw, rw = x.itemsize, len(want) // (count * d)
            for shift in (0, 1):
                print("[gpu-case]", src, dst, d, "shift", shift, flush=True)
                table = torch.zeros(x.nbytes + 64, dtype=torch.uint8, device="cuda")
                table[shift * sw:shift * sw + x.nbytes].copy_(torch.from_numpy(x.view(np.uint8).reshape(-1)))
                out = torch.full((len(want) + 64,), 0xA5, dtype=torch.uint8, device="cuda")
                ctx.index_select_device(b, table.data_ptr() + shift * sw, x.nbytes,
                                        out.data_ptr() + shift * rw, len(want),
                                        stream=torch.cuda.current_stream().cuda_stream)
                torch.cuda.synchronize()
                got = out.cpu().numpy()
                assert got[shift * rw:shift * rw + len(want)].tobytes() == want, (src, dst, d, shift)
                assert (got[:shift * rw] == 0xA5).all() and (got[shift * rw + len(want):] == 0xA5).all()


@pytest.mark.gpu
def test_a_bound_plan_keeps_no_block_of_a_closed_context():
    """One bound plan with per-channel parameters run by more contexts than it
    keeps parameter blocks for, each closed before the next is made, then by
    two contexts that are open together: every result equals the oracle's."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(5)
    x = rng.integers(-128, 128, (96, 257), dtype=np.int8)
    plan = EN.encode([96, 257], "int8", [EN.Dequantize(_scale(257, rng), zero_point=_zp(257, rng), axis=1),
                                         EN.Cast("float16"), EN.Transpose((1, 0))])
    want = _want(plan.blob, x)
    b = P.Bound(P.Plan(plan.blob), {}, {})
    dev = torch.from_numpy(x.view(np.uint8).reshape(-1).copy()).cuda()
    stream = torch.cuda.current_stream().cuda_stream

    def run(ctx):
        out = torch.full((len(want),), 0xA5, dtype=torch.uint8, device="cuda")
        for _ in range(2):
            ctx.relayout_device(b, dev.data_ptr(), out.data_ptr(), stream=stream)
        ctx.synchronize()
        torch.cuda.synchronize()
        assert out.cpu().numpy().tobytes() == want

    for _ in range(7):
        with P.Context(0) as ctx:
            run(ctx)
            # other parameter blocks of the same size where a freed one was
            torch.full((4096,), 0x7F, dtype=torch.uint8, device="cuda")
    with P.Context(0) as first, P.Context(0) as second:
        for ctx in (first, second, first, second):
            run(ctx)


# Transposes just above the size from which unaligned result rows take large
# tiles (other kernel bodies with other LDS pitches, streaming loads), both
# edges cut: one per source width and chain, parameters along either axis (a
# channel per element of a row takes small tiles, or with aligned source rows
# whole tiles and strips, as one-byte rows 8 KiB apart do to f32).
LARGE = [((1, 7103, 7107), "int8", None, None), ((1, 5801, 5803), "int8", 0, "float16"),
         ((1, 5801, 5803), "int8", 1, "float16"), ((1, 4493, 4493), "int8", 1, "float32"),
         ((1, 4493, 4493), "int8", 0, "float32"), ((1, 5021, 5023), "float16", None, None),
         ((1, 3551, 3549), "float32", None, None), ((3, 2369, 2371), "float32", None, "float16"),
         ((3, 2369, 2371), "float32", None, "bfloat16"), ((1, 4112, 11008), "int8", 0, "float16"),
         ((1, 4112, 8192), "int8", 1, "float32")]


def _large_plan(shape, dtype, axis, out, rng):
    ops = []
    if axis is not None:
        n = shape[1 + axis]
        ops = [EN.Dequantize(_scale(n, rng), zero_point=_zp(n, rng), axis=1 + axis)]
    if out in ("float16", "bfloat16"):
        ops.append(EN.Cast(out))
    return EN.encode(list(shape), dtype, ops + [EN.Transpose((0, 2, 1))]), ops


@pytest.mark.parametrize("case", LARGE, ids=[str(c) for c in LARGE])
def test_large_tile_launches_verify(case):
    plan, _ = _large_plan(*case, np.random.default_rng(1))
    b = P.Bound(P.Plan(plan.blob), {}, {})
    shape, dtype, axis, out = case
    if shape[2] % 16 == 0:
        want = ["transpose", "ragged_transpose"]
    else:
        want = ["ragged_transpose" if axis == 0 else "ragged_transpose_large"]
    assert P.launch_kernels(b) == want
    assert P.verify_launches(b, 0, 1 << 30) >= 1


@pytest.mark.gpu
@pytest.mark.parametrize("case", LARGE, ids=[str(c) for c in LARGE])
def test_large_tiles_on_the_gpu(case):
    """Bit for bit against torch: the moves are moves, (x - zero point) * scale
    and the narrowing round once each in both."""
    torch = pytest.importorskip("torch")
    shape, dtype, axis, out = case
    plan, ops = _large_plan(*case, np.random.default_rng(1))
    b = P.Bound(P.Plan(plan.blob), {}, {})
    g = torch.Generator(device="cuda").manual_seed(3)
    if dtype == "int8":
        x = torch.randint(-128, 128, shape, dtype=torch.int8, device="cuda", generator=g)
    else:
        x = torch.randn(shape, dtype=getattr(torch, dtype), device="cuda", generator=g)
    want = x
    if axis is not None:
        view = [1, 1, 1]
        view[1 + axis] = -1
        sc, zp = (torch.tensor(p.values, dtype=t, device="cuda").view(view)
                  for p, t in ((ops[0].scale, torch.float32), (ops[0].zero_point, torch.int32)))
        want = (x.to(torch.int32) - zp).float() * sc
    if out in ("float16", "bfloat16"):
        want = want.to(getattr(torch, out))
    want = want.transpose(1, 2).contiguous().view(torch.uint8).view(-1)
    buf = torch.full((want.numel() + 2 * GUARD,), 0xA5, dtype=torch.uint8, device="cuda")
    with P.Context(0) as ctx:
        ctx.relayout_device(b, x.data_ptr(), buf.data_ptr() + GUARD, stream=torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
    assert torch.equal(buf[GUARD:-GUARD], want)
    assert bool((buf[:GUARD] == 0xA5).all()) and bool((buf[-GUARD:] == 0xA5).all())


# One case per kernel that takes buffers at any address, and one per kernel
# whose launches then run element-wise
SHIFTED = [("transpose", (3, 33, 67), transpose_cases), ("transpose", (None, 6, 640), transpose_cases),
           ("rows", ROWS[2], rows_cases), ("rows", ROWS[6], rows_cases), ("image", IMAGES[1], image_cases),
           ("image", IMAGES[2], image_cases), ("flat", (50, 21), flat_cases), ("flat", (37, 16), flat_cases),
           ("permute", (2, 5, 12, 64), permute_cases), ("element", ELEMENTS[0], element_cases)]


@pytest.mark.gpu
@pytest.mark.parametrize("group", SHIFTED, ids=["%s %s" % (k, c) for k, c, _ in SHIFTED])
def test_shifted_buffers_on_the_gpu(group):
    """Device-resident sources and results that start one element, and one
    byte, past a 64-byte boundary: the same bytes, and none around them."""
    torch = pytest.importorskip("torch")
    _, case, make = group
    with P.Context(0) as ctx:
        for name, blob, x in make(case):
            print("[gpu-case]", name, flush=True)
            want = _want(blob, x)
            n = len(want)
            b = P.Bound(P.Plan(blob), {}, {})
            src = torch.from_numpy(np.ascontiguousarray(x).view(np.uint8).reshape(-1).copy()).cuda()
            for s_at, d_at in ((x.itemsize, b.element_size), (1, 1), (0, 1), (1, 0)):
                dev = torch.full((src.numel() + 2 * GUARD,), 0x5A, dtype=torch.uint8, device="cuda")
                dev[GUARD + s_at:GUARD + s_at + src.numel()].copy_(src)
                buf = torch.full((n + 2 * GUARD,), 0xA5, dtype=torch.uint8, device="cuda")
                at = GUARD + d_at
                ctx.relayout_device(b, dev.data_ptr() + GUARD + s_at, buf.data_ptr() + at,
                                    stream=torch.cuda.current_stream().cuda_stream)
                torch.cuda.synchronize()
                got = buf.cpu().numpy()
                assert got[at:at + n].tobytes() == want, (name, s_at, d_at)
                assert (got[:at] == 0xA5).all() and (got[at + n:] == 0xA5).all(), (name, s_at, d_at)
