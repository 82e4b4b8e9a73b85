"""The host stages' vector loops against the oracle's stage arithmetic: every
length around the vector widths at every start, special values, ties, and a
sweep over the binary32 encodings."""
import numpy as np
import pytest

from oracle import relx_oracle as O
from sym_amd import encoder as EN
from sym_amd import pyreloc as P

SPECIAL = np.array([0x00000000, 0x80000000, 0x00000001, 0x807fffff, 0x7f800000, 0xff800000, 0x7f800001,
                    0x7fc00000, 0xffc12345, 0x7fffffff, 0xff80ffff, 0x7f7fffff, 0x3f808000, 0x3f818000,
                    0x3f80ffff, 0x477fe000, 0x33000000], np.uint32)


def _values(n, seed, scale):
    rng = np.random.default_rng(seed)
    bits = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    x = bits.view(np.float32).copy()
    x[1::3] = (rng.integers(-300, 300, x[1::3].size) * np.float32(0.5) * np.float32(scale))
    k = min(n, SPECIAL.size)
    x.view(np.uint32)[:k] = SPECIAL[:k]
    return x


@pytest.mark.parametrize("op,dtype", [(EN.Cast("bfloat16"), np.uint16), (EN.Cast("float16"), np.uint16),
                                      (EN.Quantize(EN.InlineParam((0.03125,))), np.uint8),
                                      (EN.Quantize(EN.InlineParam((0.0371,))), np.uint8)],
                         ids=["bf16", "f16", "quant", "quant inexact"])
def test_host_stage_equals_the_oracle(op, dtype):
    scale = op.scale.values[0] if isinstance(op, EN.Quantize) else 1.0
    for n in list(range(1, 70)) + [1 << 18]:
        blob = EN.encode([n], "float32", [op]).blob
        b = P.Bound(P.Plan(blob), {}, {})
        x = _values(n, n, scale)
        with np.errstate(all="ignore"):
            want = O.run_typed(blob, {}, {}, x).tobytes()
        got = np.full(n + 8, 0xA5A5 & np.iinfo(dtype).max, dtype)
        P.host_stage(b, 1, x.ctypes.data, got.ctypes.data, threads=3)
        assert got[:n].tobytes() == want, n
        assert (got[n:] == (0xA5A5 & np.iinfo(dtype).max)).all(), n
