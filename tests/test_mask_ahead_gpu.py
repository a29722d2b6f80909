"""Attention masks whose quads are loaded ahead of their use (MaskAhead), at any
alignment: against the same mask with a key stride of two, which is read one
element at a time where it is used. The arithmetic is the same, so are the bits.
"""

import ctypes

import numpy as np
import pytest

from test_sdpa_gpu import _dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tn():
    import torchnative_amd as tn

    print("device:", tn._hip_probe(), flush=True)
    return tn


@pytest.mark.parametrize("dtype,kind", [("bfloat16", "float32"), ("bfloat16", "bfloat16"), ("float16", "float16"),
                                        ("float16", "bool"), ("float32", "float32"), ("float32", "bool")])
@pytest.mark.parametrize("D,L,S,causal", [(64, 70, 131, False), (64, 1, 1, False), (128, 65, 66, True),
                                          (128, 33, 1027, False), (96, 40, 129, True), (256, 35, 63, False)])
@pytest.mark.parametrize("lead,gap", [(0, 0), (1, 0), (3, 2), (2, 5)])
def test_any_alignment_gives_the_element_loads_bits(tn, dtype, kind, D, L, S, causal, lead, gap):
    """`lead` elements before the mask's base, `gap` between its rows."""
    from torchnative_amd import _lib as LB

    B, Hq, Hkv = 2, 2, 1
    rng = np.random.default_rng(D + L + S)
    q, k, v = (_dev(tn, dtype, rng.standard_normal(s)) for s in ((B, Hq, L, D), (B, Hkv, S, D), (B, Hkv, S, D)))
    row = S + gap
    n = lead + B * L * row
    m = rng.random(n) < 0.7 if kind == "bool" else rng.standard_normal(n)
    if kind != "bool":
        m[rng.random(n) < 0.2] = -np.inf
    out = []
    for step in (1, 2):
        wide = np.zeros(n * step, m.dtype)
        wide[::step] = m
        md = tn.tensor(wide, device="hip") if kind == "bool" else _dev(tn, kind, wide)
        es = {"bool": 1, "float32": 4}.get(kind, 2)
        o = _dev(tn, dtype, np.zeros((B, Hq, L, D)))
        lse = _dev(tn, "float32", np.zeros((B, Hq, L)))
        strides = (ctypes.c_int64 * 4)(L * row * step, 0, row * step, step)
        code = {"float32": LB.TN_F32, "bfloat16": LB.TN_BF16, "float16": LB.TN_F16, "bool": LB.TN_BOOL}
        LB.check(LB.lib().tn_sdpa_fwd(None, code[dtype], q.data_ptr(), k.data_ptr(), v.data_ptr(), B, Hq, Hkv, L, S, D,
                                  md.data_ptr() + lead * step * es, code[kind], strides, int(causal), float("nan"),
                                  o.data_ptr(), lse.data_ptr()))
        out.append((o.numpy(), lse.numpy()))
    assert S == 1 or np.isfinite(out[0][1]).mean() > 0.5
    for a, b in zip(out[0], out[1]):
        assert a.tobytes() == b.tobytes()
