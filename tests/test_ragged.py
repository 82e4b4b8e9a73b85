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
            ("float16", [EN.Cast("float32", "exact"), EN.Quantize(sc(), axis=axis)])]


def _source(shape, dtype, rng):
    if dtype == "int8":
        return rng.integers(-128, 128, shape, dtype=np.int8)
    x = rng.standard_normal(shape) * 3
    x.reshape(-1)[:: 97] = np.resize([np.nan, np.inf, -np.inf, -0.0, 1e30, 1e-30], x.reshape(-1)[::97].size)
    return x.astype(dtype)


# (rows, cols) [batch] around the tile widths: one row of a vector less or
# more than a tile, extents of the smallest tile launch, several tiles
TRANSPOSES = [(None, 16, 16), (None, 17, 31), (None, 63, 65), (None, 64, 130), (None, 129, 127),
              (None, 257, 190), (3, 33, 67), (2, 128, 129)]


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


GROUPS = [("transpose", c, transpose_cases) for c in TRANSPOSES]
IDS = ["%s %s" % (k, "x".join(str(v) for v in c if v is not None)) for k, c, _ in GROUPS]


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
