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


@pytest.mark.parametrize("dtype,kind", [("bfloat16", None), ("float16", "bool"), ("float16", "float16"),
                                        ("bfloat16", "float32")])
@pytest.mark.parametrize("B,Hq,Hkv,L,S", [(8, 9, 3, 250, 100), (1, 90, 45, 129, 70), (4, 20, 5, 257, 65)])
def test_wide_blocks(tn, dtype, kind, B, Hq, Hkv, L, S):
    """Head dim 128, unmasked by causality, more 64-query blocks than compute units
    but fewer 128-query ones: rows of the eight-wave workgroups against the same
    rows called a sequence at a time, which the four-wave ones run unsplit."""
    from torchnative_amd import _lib as LB

    D = 128
    rng = np.random.default_rng(L + S)
    q, k, v = (rng.standard_normal(s) for s in ((B, Hq, L, D), (B, Hkv, S, D), (B, Hkv, S, D)))
    m = None
    if kind:
        m = rng.random((B, 1, L, S)) < 0.7 if kind == "bool" else rng.standard_normal((B, 1, L, S))
    code = {"float32": LB.TN_F32, "bfloat16": LB.TN_BF16, "float16": LB.TN_F16, "bool": LB.TN_BOOL}

    def run(b, h):  # sequences b, query heads h (whole groups)
        hk = slice(h.start // (Hq // Hkv), h.stop // (Hq // Hkv))
        qd, kd, vd = (_dev(tn, dtype, np.ascontiguousarray(x)) for x in (q[b, h], k[b, hk], v[b, hk]))
        n, nh = qd.shape[0], qd.shape[1]
        mp, strides = None, None
        if m is not None:
            md = tn.tensor(m[b].copy(), device="hip") if kind == "bool" else _dev(tn, kind, m[b])
            mp, strides = md.data_ptr(), (ctypes.c_int64 * 4)(L * S, 0, S, 1)
        o, lse = _dev(tn, dtype, np.zeros((n, nh, L, D))), _dev(tn, "float32", np.zeros((n, nh, L)))
        LB.check(LB.lib().tn_sdpa_fwd(None, code[dtype], qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), n, nh,
                                      kd.shape[1], L, S, D, mp, code[kind] if kind else 0, strides, 0, float("nan"),
                                      o.data_ptr(), lse.data_ptr()))
        return o.numpy(), lse.numpy()

    whole = run(slice(0, B), slice(0, Hq))
    for b in (0, B - 1):
        for h in (0, Hkv - 1):
            hs = slice(h * (Hq // Hkv), (h + 1) * (Hq // Hkv))
            part = run(slice(b, b + 1), hs)
            for x, y in zip(whole, part):
                assert np.ascontiguousarray(x[b, hs]).tobytes() == y[0].tobytes()
