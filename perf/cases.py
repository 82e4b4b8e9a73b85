"""Performance cases of the relocation library's public entry points.

A case is one call of a program that loads plans: a relayout of a tensor that
is already on the GPU (`Context.relayout_device`), a row gather from a table
on the GPU (`Context.index_select_device`), an upload of a host tensor
(`execute_transfer` for layout plans, `execute_dispatch` for typed ones), or
an eviction of a GPU tensor to the host (`execute_dispatch`, "d2h"). Each
recipe is one that the package's workloads, tests or benchmark run, at their
sizes and at the odd ones that real shapes bring: a sequence length, an image
side, a vocabulary or a feature count is rarely a multiple of a tile.

Results are bit-exact by contract, so every tolerance is "exact".
"""
import math

import numpy as np
import torch

from sym_amd import encoder as EN
from sym_amd import pyreloc as P
from sym_amd import workloads as W

DEVICE = 0
STAGING_THREADS = 8
WIDTH = {"float32": 4, "float16": 2, "bfloat16": 2, "int8": 1}

# One retained context and one set of transfer resources per process, as a
# program that makes many calls keeps them.
_shared = {}


def _resources():
    if "dispatch" not in _shared:
        _shared["dispatch"] = P.Resources(DEVICE)
        _shared["transfer"] = P.TransferResourceCache(max_retained_bytes=1 << 30)
    return _shared


def listed():
    return [
        # The smallest call: a few hundred values of host memory through the
        # split + transpose plan of the README. Latency of the whole call.
        {"name": "split upload 192", "recipe": "split", "path": "upload", "n": 192, "pinned": False},
        # The same plan over a large f32 vector that is on the GPU.
        {"name": "split 16M", "recipe": "split", "path": "device", "n": 16777216},
        # A batch of images made channels-last, padded to four channels, in
        # half precision, as a vision model's input stage wants it.
        {"name": "image 32x224", "recipe": "image", "path": "device", "b": 32, "c": 3, "h": 224, "w": 224},
        # A quantized weight [in, out] dequantized per output channel and
        # transposed to [out, in] halves: a whole projection matrix.
        {"name": "weight 4096x11008", "recipe": "weight", "path": "device", "k": 4096, "n": 11008,
         "out": "float16"},
        # The same fetch to f32 for a smaller matrix whose sides are odd, as
        # of a vocabulary or a pruned layer.
        {"name": "weight 1027x4099", "recipe": "weight", "path": "device", "k": 1027, "n": 4099,
         "out": "float32"},
        # An expert's weight [out, in] dequantized per row, layout kept.
        {"name": "expert 14336x4096", "recipe": "expert", "path": "device", "k": 14336, "n": 4096},
        # A key/value cache block [B, S, heads, dim] made head-major and
        # quantized per head: the package's largest device-resident workload.
        {"name": "kv 8x4096", "recipe": "kv", "path": "device", "b": 8, "s": 4096, "heads": 32, "dim": 128},
        # Activations [B, S, H] transposed to [B, H, S] and narrowed to
        # bf16, at a sequence length of a real batch.
        {"name": "activation 16x1001x770", "recipe": "activation", "path": "device", "b": 16, "s": 1001,
         "h": 770, "out": "bfloat16"},
        # Feature rows padded to the alignment of the next layer's kernel and
        # quantized per tensor.
        {"name": "rows 8000x1003", "recipe": "rows", "path": "device", "n": 8000, "d": 1003},
        # An embedding lookup narrowed to halves, table on the GPU.
        {"name": "gather 64Kx1024", "recipe": "gather", "path": "device", "rows": 262144, "d": 1024,
         "count": 65536, "pair": "float32:float16"},
        # A cache block that comes back from page-locked host memory.
        {"name": "kv upload 8x1024", "recipe": "kv", "path": "upload", "b": 8, "s": 1024, "heads": 32,
         "dim": 128, "pinned": True},
        # A cache block that leaves for pageable host memory.
        {"name": "kv evict 8x1024", "recipe": "kv", "path": "evict", "b": 8, "s": 1024, "heads": 32,
         "dim": 128, "pinned": False},
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _side(rng, lo, hi, align):
    """A matrix side: a multiple of `align` half of the time, any number else."""
    v = _log(rng, lo, hi)
    return v if rng.random() < 0.5 else max(align, (v + align // 2) // align * align)


def draw(rng):
    """One more case of the listed ranges: device-resident recipes two times
    in three, transfers of up to 64 MiB of wire else."""
    kind = rng.choice(["split", "image", "weight", "expert", "kv", "activation", "rows", "gather"])
    case = {"recipe": kind, "path": "device"}
    # device-resident calls move at most the largest listed relayout's
    # elements, transfers a quarter of that
    most = 1 << 27
    if kind != "gather" and rng.random() < 0.33:
        case["path"] = rng.choice(["upload", "evict"]) if kind == "kv" else "upload"
        case["pinned"] = rng.random() < 0.5
        most = 1 << 23
    if kind == "split":
        case["n"] = 64 * _log(rng, 2, min(most, 1 << 24) // 64)
    elif kind == "image":
        c = rng.choice([1, 3, 3, 3, 7])
        h = rng.choice([32, 96, 224, 225, 256, 299, 384, 417])
        case.update(b=_log(rng, 1, max(1, min(64, most // 8 // (c * h * h)))), c=c, h=h, w=h)
    elif kind in ("weight", "expert"):
        k = _side(rng, 256, 8192, 128)
        case.update(k=k, n=_side(rng, 256, max(256, min(16384, most // 2 // k)), 128))
        if kind == "weight":
            case["out"] = rng.choice(["float16", "float32"])
    elif kind == "kv":
        heads, dim = rng.choice([(32, 128), (8, 128), (40, 128), (16, 64), (12, 64), (32, 96)])
        b = _log(rng, 1, 64)
        case.update(b=b, s=_log(rng, 1, max(1, min(4096, most // (b * heads * dim)))), heads=heads, dim=dim)
    elif kind == "activation":
        b, s = _log(rng, 1, 32), _side(rng, 16, 2048, 64)
        case.update(b=b, s=s, h=_side(rng, 64, max(64, min(4096, most // 4 // (b * s))), 64),
                    out=rng.choice(["bfloat16", "float16"]))
    elif kind == "rows":
        n = _log(rng, 16, 16384)
        case.update(n=n, d=_side(rng, 64, max(64, min(8192, most // 4 // n)), 64))
    else:
        d = _log(rng, 4, 2048)
        count = _log(rng, 256, min(1 << 19, (1 << 26) // d))
        case.update(rows=min(1 << 19, 4 * count), d=d, count=count,
                    pair=rng.choice(["float32:float16", "float16:float32", "int8:int8", "float32:float32"]))
    return case


# ------------------------------------------------------------------ recipes


def _shapes(case):
    """(source shape, source dtype, result shape, result dtype)."""
    r = case["recipe"]
    if r == "split":
        return (case["n"],), "float32", (64, case["n"] // 64), "float32"
    if r == "image":
        b, c, h, w = case["b"], case["c"], case["h"], case["w"]
        return (b, c, h, w), "float32", (b, h, w, c + 1), "float16"
    if r == "weight":
        return (case["k"], case["n"]), "int8", (case["n"], case["k"]), case["out"]
    if r == "expert":
        return (case["k"], case["n"]), "int8", (case["k"], case["n"]), "float16"
    if r == "kv":
        b, s, heads, dim = case["b"], case["s"], case["heads"], case["dim"]
        return (b, s, heads, dim), "float16", (b, heads, s, dim), "int8"
    if r == "activation":
        b, s, h = case["b"], case["s"], case["h"]
        return (b, s, h), "float32", (b, h, s), case["out"]
    if r == "rows":
        n, d = case["n"], case["d"]
        return (n, d), "float32", (n, (d + 63) // 64 * 64), "int8"
    src, dst = case["pair"].split(":")
    return (case["rows"], case["d"]), src, (case["count"], case["d"]), dst


def _channels(case):
    """Entries of the recipe's scale table (0: none, or one inline)."""
    return {"weight": case.get("n"), "expert": case.get("k"), "kv": case.get("heads")}.get(case["recipe"], 0) or 0


ROWS_SCALE = 0.03125


def _plan(case):
    """(plan, symbol values) of the recipe; the plans are symbolic where the
    package's workloads are."""
    r = case["recipe"]
    if r == "split":
        return P.load_plan(W.c1_plan().blob), {"s0": case["n"]}
    if r == "image":
        return P.load_typed_plan(W.c2_plan(case["b"], case["c"], case["h"], case["w"]).blob), {}
    if r == "weight":
        if case["out"] == "float16":
            blob = W.c3_plan().blob
        else:
            scale = EN.BindingParam("scale", "float32", ("s1",))
            blob = EN.encode(["s0", "s1"], "int8",
                             [EN.Dequantize(scale, axis=1), EN.Transpose((1, 0))]).blob
        return P.load_typed_plan(blob), {"s0": case["k"], "s1": case["n"]}
    if r == "expert":
        return P.load_typed_plan(W.c4_plan().blob), {"s0": case["k"], "s1": case["n"]}
    if r == "kv":
        return P.load_typed_plan(W.c5_plan(case["heads"], case["dim"]).blob), {"B": case["b"], "S": case["s"]}
    shape, dt, result, out = _shapes(case)
    if r == "activation":
        ops = [EN.Transpose((0, 2, 1)), EN.Cast(out)]
    else:
        ops = [EN.Pad(1, 0, result[1] - shape[1], 0.0), EN.Quantize(EN.InlineParam((ROWS_SCALE,)))]
    return P.load_typed_plan(EN.encode(list(shape), dt, ops).blob), {}


def _inputs(case, seed):
    """(source on the GPU, scale table or None): standard normal activations
    and images, int8 weights over their range with scales of their size."""
    g = torch.Generator(device="cuda:%d" % DEVICE)
    g.manual_seed(int(seed))
    shape, dt, _, _ = _shapes(case)
    dev = "cuda:%d" % DEVICE
    if dt == "int8":
        x = torch.randint(-127, 128, shape, dtype=torch.int8, device=dev, generator=g)
    else:
        x = torch.randn(shape, dtype=getattr(torch, dt), device=dev, generator=g)
    n = _channels(case)
    lo, hi = (0.02, 0.05) if case["recipe"] == "kv" else (1e-3, 2e-2)
    scale = torch.rand(n, device=dev, generator=g) * (hi - lo) + lo if n else None
    return x, scale


def _indices(case, seed):
    return np.random.default_rng(int(seed)).integers(0, case["rows"], case["count"]).astype("<i8")


def _view(t):
    size = t.element_size()
    if t.device.type == "cpu":
        return P.BufferView(t.data_ptr(), t.numel() * size, 0, list(t.shape), list(t.stride()), size, "host")
    return P.BufferView(t.data_ptr(), t.numel() * size, 0, list(t.shape), list(t.stride()), size, "cuda",
                        t.device.index)


def _host(t, pinned):
    h = torch.empty(t.shape, dtype=t.dtype, pin_memory=bool(pinned))
    h.copy_(t)
    return h


def prepare(case, seed):
    """The plan and its parameters, the source where the program has it, and,
    for device-resident calls, the binding and the result's buffer."""
    res = _resources()
    x, scale = _inputs(case, seed)
    _, _, result, out = _shapes(case)
    dtype = getattr(torch, out)
    s = {"path": case["path"], "recipe": case["recipe"], "result": result, "dtype": dtype,
         "ctx": res["dispatch"], "cache": res["transfer"]}
    if case["recipe"] == "gather":
        shape, src, _, dst = _shapes(case)
        blob = EN.encode_index_select(list(shape), src, case["count"], "int64", dst)
        idx = _indices(case, seed)
        s["bound"] = P.bind_indexed(P.load_indexed_plan(blob), {}, ("int64", [case["count"]], idx.tobytes()))
    else:
        s["plan"], s["symbols"] = _plan(case)
        s["params"] = W.param("scale", scale.cpu().numpy()) if scale is not None else {}
    if case["path"] == "device":
        if case["recipe"] == "split":
            s["bound"] = P.bind(s["plan"], s["symbols"])
        elif case["recipe"] != "gather":
            s["bound"] = P.bind_typed(s["plan"], s["symbols"], s["params"])
        s["src"] = x
        s["out"] = torch.empty(result, dtype=dtype, device=x.device)
    elif case["path"] == "upload":
        s["src"] = _host(x, case["pinned"])
    else:
        s["src"] = x
        s["out"] = torch.empty(result, dtype=dtype, pin_memory=case["pinned"])
    return s


def run(state):
    s = state
    stream = torch.cuda.current_stream().cuda_stream
    src = s["src"]
    if s["path"] == "device":
        out = s["out"]
        if s["recipe"] == "gather":
            s["ctx"].index_select_device(s["bound"], src.data_ptr(), src.numel() * src.element_size(),
                                         out.data_ptr(), out.numel() * out.element_size(), stream=stream)
        else:
            s["ctx"].relayout_device(s["bound"], src.data_ptr(), out.data_ptr(), stream=stream)
        return out
    if s["path"] == "evict":
        bound = P.bind_typed(s["plan"], s["symbols"], s["params"])
        req = P.prepare_dispatch(bound, _view(src), _view(s["out"]), "d2h")
        P.execute_dispatch(req, caller_stream=stream, resources=s["ctx"], gather_threads=STAGING_THREADS)
        return s["out"]
    out = torch.empty(s["result"], dtype=s["dtype"], device="cuda:%d" % DEVICE)
    if s["recipe"] == "split":
        bound = P.bind(s["plan"], s["symbols"])
        req = P.make_transfer(bound, _view(src), _view(out), "h2d")
        P.execute_transfer(req, caller_stream=stream, gather_threads=STAGING_THREADS, resources=s["cache"],
                           owners=(src, out))
    else:
        bound = P.bind_typed(s["plan"], s["symbols"], s["params"])
        req = P.prepare_dispatch(bound, _view(src), _view(out), "h2d")
        P.execute_dispatch(req, caller_stream=stream, resources=s["ctx"], gather_threads=STAGING_THREADS)
    return out


def work(case):
    shape, dt, result, out = _shapes(case)
    if case["recipe"] == "gather":
        read = case["count"] * (case["d"] * WIDTH[dt] + 4)
    else:
        read = math.prod(shape) * WIDTH[dt] + 4 * _channels(case)
    return {"bytes": read + math.prod(result) * WIDTH[out], "flops": 0}


def tolerance(case):
    """Every result is bit-exact by the library's contract: each stage keeps
    its own rounding, layout moves bits."""
    return "exact"


def _quantized(x, scale):
    return torch.clamp(torch.round(x / scale), -128, 127)


def exact(case, seed):
    x, scale = _inputs(case, seed)
    r = case["recipe"]
    if r == "gather":
        idx = torch.from_numpy(_indices(case, seed)).to(x.device)
        return x[idx].double()
    x = x.double()
    scale = scale.double() if scale is not None else None
    if r == "split":
        return x.view(-1, 64).t().contiguous()
    if r == "image":
        return torch.nn.functional.pad(x, (0, 0, 0, 0, 0, 1)).permute(0, 2, 3, 1).contiguous()
    if r == "weight":
        return (x * scale).t().contiguous()
    if r == "expert":
        return x * scale[:, None]
    if r == "kv":
        return _quantized(x.permute(0, 2, 1, 3), scale[:, None, None]).contiguous()
    if r == "activation":
        return x.permute(0, 2, 1).contiguous()
    result = _shapes(case)[2]
    return _quantized(torch.nn.functional.pad(x, (0, result[1] - x.shape[1])), ROWS_SCALE)
