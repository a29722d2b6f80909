"""Attention at head dims other than 64 and 128, and with a negative scale, on
the 16-bit matrix cores (flash_any.hip), at the edges of its tiles: row blocks
of 32 and 64, ring stages of 128 keys (64 at head dims past 128), every padded
width of the head dim, split keys and their merge.

Tolerance: the rule of test_sdpa_gpu.py with the P-narrowing term divided by
2^8 (bf16) or 2^9 (f16) and the subnormal term by 2^6: the kernel multiplies V
by both halves of P = hi + lo, so P is off by at most 2^-16 (2^-20) of itself,
and f16 probabilities carry a factor of 2^6.
"""

import ctypes

import numpy as np
import pytest

import oracle as O

from test_sdpa_gpu import OP, _bound, _dev, _narrow, _vsum

pytestmark = pytest.mark.gpu
FRAC = {"bfloat16": 2.0 ** -8, "float16": 2.0 ** -9}


@pytest.fixture(scope="module")
def tn():
    import torchnative_amd as tn

    print("device:", tn._hip_probe(), flush=True)
    return tn


def _compare(dtype, got, lse, qw, kw, vw, causal=False, mask=None, scale=None, nan=None):
    Hq, L = qw.shape[1:3]
    with np.errstate(invalid="ignore"):
        r32, l32 = O.sdpa(qw, kw, vw, is_causal=causal, mask=mask, scale=scale, threads=16)
        r64, l64 = O.sdpa(qw, kw, vw, is_causal=causal, mask=mask, scale=scale, threads=16, dtype=np.float64)
        pav, _ = O.sdpa(qw, kw, np.abs(vw), is_causal=causal, mask=mask, scale=scale, threads=16, dtype=np.float64)
    vsum = _vsum(vw, Hq, L, causal, mask) if dtype == "float16" else None
    rows = np.zeros(qw.shape[:3], bool) if nan is None else nan
    assert np.array_equal(np.isnan(got).any(-1), rows) and np.array_equal(np.isnan(lse), rows)
    k = ~rows
    tol = _bound(r32[k], r64[k], pav[k] * FRAC[dtype], got=got[k], kind=dtype,
                 vsum=None if vsum is None else vsum[k] * 2.0 ** -6)
    worst = float(np.max(np.abs(got[k] - _narrow(dtype, r32)[k]) / tol))
    assert worst <= 1.0, f"{worst:.3g}x the bound"
    lworst = float(np.max(np.abs(lse[k].astype(np.float64) - l32[k]) / _bound(l32[k], l64[k])))
    assert lworst <= 1.0, f"lse {lworst:.3g}x the bound"


def _inputs(tn, dtype, B, Hq, Hkv, L, S, D, seed):
    rng = np.random.default_rng(seed)
    t = [_dev(tn, dtype, rng.standard_normal(s)) for s in ((B, Hq, L, D), (B, Hkv, S, D), (B, Hkv, S, D))]
    return t, [x.numpy().astype(np.float64) for x in t]


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("shape", [
    # B, Hq, Hkv, L, S, D
    (1, 1, 1, 1, 1, 8), (2, 2, 1, 31, 33, 24), (1, 2, 2, 32, 127, 32), (1, 3, 1, 33, 128, 40), (1, 2, 2, 64, 129, 48),
    (1, 2, 1, 65, 257, 56), (1, 2, 2, 100, 100, 72), (2, 4, 2, 130, 64, 80), (1, 2, 2, 96, 300, 96),
    (1, 2, 2, 70, 70, 104), (1, 2, 2, 40, 200, 120), (1, 1, 1, 66, 130, 136), (1, 2, 2, 33, 65, 192),
    (1, 2, 1, 80, 200, 256)])
@pytest.mark.parametrize("causal", [False, True])
def test_rows_keys_and_head_dims(tn, shape, dtype, causal):
    B, Hq, Hkv, L, S, D = shape
    (q, k, v), (qw, kw, vw) = _inputs(tn, dtype, *shape, seed=L + S + D)
    o, lse = tn._aten_dispatch(OP, q, k, v, 0.0, causal)
    _compare(dtype, o.numpy().astype(np.float64), lse.numpy(), qw, kw, vw, causal)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("D", [64, 128, 80])
def test_negative_scale(tn, dtype, D):
    (q, k, v), (qw, kw, vw) = _inputs(tn, dtype, 1, 4, 2, 90, 150, D, seed=D)
    o, lse = tn._aten_dispatch(OP, q, k, v, 0.0, False, scale=-0.3)
    _compare(dtype, o.numpy().astype(np.float64), lse.numpy(), qw, kw, vw, scale=-0.3)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("shape,causal", [((1, 2, 1, 5, 2100, 96), False), ((1, 1, 1, 70, 1500, 256), False),
                                          ((1, 2, 2, 600, 600, 32), True)])
def test_split_keys_and_their_merge(tn, shape, causal, dtype):
    """Few rows over long keys: several splits per row block, causal ones with
    splits that hold no key."""
    (q, k, v), (qw, kw, vw) = _inputs(tn, dtype, *shape, seed=sum(shape))
    o, lse = tn._aten_dispatch(OP, q, k, v, 0.0, causal)
    _compare(dtype, o.numpy().astype(np.float64), lse.numpy(), qw, kw, vw, causal)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("kind", ["f32", "same", "bool"])
@pytest.mark.parametrize("D,S", [(72, 61), (96, 1030), (256, 130)])
def test_masks(tn, dtype, kind, D, S):
    """Additive and bool masks read in place, odd key lengths (unaligned mask
    rows), the type's lowest value, a row that sees nothing, keys hidden at the
    front of a stage."""
    B, Hq, Hkv, L = 2, 2, 1, 35
    (q, k, v), (qw, kw, vw) = _inputs(tn, dtype, B, Hq, Hkv, L, S, D, seed=S)
    rng = np.random.default_rng(S + D)
    nan = np.zeros((B, Hq, L), bool)
    nan[:, :, 7] = True
    if kind == "bool":
        m = rng.random((B, 1, L, S)) < 0.6
        m[:, :, :, 0] = True
        m[:, :, 9, :S - 1] = False
        m[:, :, 9, S - 1] = True
        m[:, :, 7] = False
        o = tn.scaled_dot_product_attention(q, k, v, attn_mask=tn.tensor(m, device="hip"), enable_gqa=True)
        add = np.where(np.broadcast_to(m, (B, Hq, L, S)), 0.0, -np.inf)
        got, lse = o.numpy().astype(np.float64), None
    else:
        mt = "float32" if kind == "f32" else dtype
        m = rng.standard_normal((L, S))
        m[9, : S - 1] = -3.0e38 if mt != "float16" else -65504.0
        m[7] = -np.inf
        md = _dev(tn, mt, m)
        add = np.ascontiguousarray(np.broadcast_to(md.numpy().astype(np.float64), (B, Hq, L, S)))
        o, lse = tn._aten_dispatch(OP, q, k, v, 0.0, False, attn_mask=md)
        got, lse = o.numpy().astype(np.float64), lse.numpy()
    if lse is None:
        with np.errstate(invalid="ignore"):
            lse = O.sdpa(qw, kw, vw, mask=add, threads=16)[1].astype(np.float32)
    _compare(dtype, got, lse, qw, kw, vw, mask=np.ascontiguousarray(add), nan=nan)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("Hq,Hkv,D,lens,cap", [
    (8, 1, 96, [1, 128, 129, 300], 300), (6, 2, 80, [3000], 3100), (33, 1, 72, [40, 700], 701), (4, 4, 256, [0, 65], 65),
    (64, 1, 32, [513], 600)])
def test_decode(tn, dtype, Hq, Hkv, D, lens, cap):
    """Grouped heads as rows, lengths from the device, past the cache's filled
    rows NaN (they must not reach the result), both entries the same bits."""
    from torchnative_amd import _lib as L

    B = len(lens)
    rng = np.random.default_rng(D)
    q = _dev(tn, dtype, rng.standard_normal((B, Hq, D)))
    kc, vc = (rng.standard_normal((B, Hkv, cap, D)) for _ in range(2))
    for b, n in enumerate(lens):
        kc[b, :, n:] = np.nan
        vc[b, :, n:] = np.nan
    k, v = _dev(tn, dtype, kc), _dev(tn, dtype, vc)
    ln = tn.tensor(np.asarray(lens, np.int32), device="hip")
    o, lse = tn.sdpa_decode(q, k, v, ln, max(lens))
    o2, l2 = tn.empty((B, Hq, D), dtype, "hip"), tn.empty((B, Hq), "float32", "hip")
    code = L.TN_BF16 if dtype == "bfloat16" else L.TN_F16
    L.check(L.lib().tn_sdpa_decode_noalloc(None, code, q.data_ptr(), k.data_ptr(), v.data_ptr(), B, Hq, Hkv, cap, D,
                                           ln.data_ptr(), max(lens), float("nan"), o2.data_ptr(), l2.data_ptr()))
    assert o.bits().tobytes() == o2.bits().tobytes() and lse.numpy().tobytes() == l2.numpy().tobytes()
    qw, kw, vw = (t.numpy().astype(np.float64) for t in (q, k, v))
    got, gl = o.numpy().astype(np.float64), lse.numpy()
    for b, n in enumerate(lens):
        if n == 0:
            assert np.isnan(got[b]).all() and np.isneginf(gl[b]).all()
            continue
        _compare(dtype, got[b][None, :, None], gl[b][None, :, None], qw[b][None, :, None], kw[b:b + 1, :, :n],
                 vw[b:b + 1, :, :n])


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("shape,causal,scale", [
    # B, Hq, Hkv, L, S, D: rows and key groups, split keys, the decode entry (L 1), a negative scale
    ((1, 2, 2, 70, 200, 96), False, None), ((2, 2, 1, 90, 90, 72), True, None), ((1, 1, 1, 33, 40, 256), False, None),
    ((1, 2, 1, 5, 2100, 80), False, None), ((2, 8, 2, 1, 1500, 96), False, None), ((1, 2, 2, 40, 70, 64), False, -0.2)])
def test_infinite_values(tn, shape, causal, scale, dtype):
    """V infinite in single keys of some columns: every row that gives the key
    a probability gets that infinity, both signs in a column NaN, as f32
    probabilities do, however small the probability (about 1e-28 here); the other
    columns keep their bits."""
    B, Hq, Hkv, L, S, D = shape
    rng = np.random.default_rng(S)
    q, k, v = (rng.standard_normal(s) for s in ((B, Hq, L, D), (B, Hkv, S, D), (B, Hkv, S, D)))
    # key 0 far below the other keys: a score of -64 (-51 with the negative scale)
    q[..., 0], k[:, :, 1:, 0] = 32.0, 0.0
    k[:, :, 0, 0] = -2.0 * np.sqrt(D) if scale is None else 8.0
    inf = v.copy()
    inf[:, :, 0, 3], inf[:, :, 0, 5], inf[:, :, min(S - 1, 37) if not causal else 0, 7] = np.inf, -np.inf, np.inf
    if not causal:
        inf[:, :, S // 2, 9], inf[:, :, S // 2 + 1, 9] = np.inf, -np.inf
    cols = [3, 5, 7] + ([] if causal else [9])
    qd, kd = _dev(tn, dtype, q), _dev(tn, dtype, k)
    outs = []
    for val in (inf, v):
        vd = _dev(tn, dtype, val)
        if L == 1:
            ln = tn.tensor(np.full(B, S, np.int32), device="hip")
            o, _ = tn.sdpa_decode(_dev(tn, dtype, q[:, :, 0]), kd, vd, ln, S)
            outs.append(o.numpy().reshape(B, Hq, 1, D))
        else:
            o, _ = tn._aten_dispatch(OP, qd, kd, vd, 0.0, causal, scale=scale)
            outs.append(o.numpy())
    rest = [c for c in range(D) if c not in cols]
    assert np.isfinite(outs[1]).all() and np.array_equal(outs[0][..., rest], outs[1][..., rest])
    with np.errstate(invalid="ignore"):
        want = O.sdpa(*(t.numpy().astype(np.float64) for t in (qd, kd)), _dev(tn, dtype, inf).numpy().astype(np.float64),
                      is_causal=causal, scale=scale, threads=16)[0]
    assert np.array_equal(outs[0][..., cols], want[..., cols].astype(outs[0].dtype), equal_nan=True)
    assert np.isposinf(want[..., 3]).all() and np.isneginf(want[..., 5]).all()


@pytest.mark.parametrize("dtype,shape,causal,scale,masked", [
    # every padded width, one and two row halves; a mask; causal splits without a key; 64 and 128 by the scale's sign
    ("bfloat16", (1, 2, 1, 5, 2100, 96), False, None, False), ("float16", (1, 2, 1, 40, 1100, 32), False, None, True),
    ("float16", (1, 1, 1, 70, 1500, 128), False, -0.1, True), ("bfloat16", (1, 2, 2, 600, 600, 80), True, None, False),
    ("bfloat16", (2, 1, 1, 7, 900, 64), False, -0.2, False), ("bfloat16", (1, 1, 1, 30, 800, 256), False, None, True),
    ("float16", (1, 2, 2, 33, 513, 200), False, None, False)])
def test_captured_without_a_workspace_gives_the_same_bits(tn, dtype, shape, causal, scale, masked):
    """A call that splits its keys, captured on a stream that holds no
    workspace (nothing may be allocated then): one workgroup takes its rows'
    splits in turn; three replays on changing inputs, the eager call's bits
    and within the bound."""
    from torchnative_amd import _lib as L

    f = L.lib()
    B, Hq, Hkv, Lq, S, D = shape
    code, sc = (L.TN_BF16 if dtype == "bfloat16" else L.TN_F16), float("nan") if scale is None else scale
    (q, k, v), _ = _inputs(tn, dtype, *shape, seed=3)
    add = np.random.default_rng(4).standard_normal((Lq, S)) if masked else None
    md = _dev(tn, "float32", add) if masked else None
    strides = (ctypes.c_int64 * 4)(0, 0, S, 1)
    outs = [(tn.empty((B, Hq, Lq, D), dtype, "hip"), tn.empty((B, Hq, Lq), "float32", "hip")) for _ in range(2)]

    def call(stream, out, lse):
        L.check(f.tn_sdpa_fwd(stream, code, q.data_ptr(), k.data_ptr(), v.data_ptr(), B, Hq, Hkv, Lq, S, D,
                              md.data_ptr() if masked else None, L.TN_F32 if masked else 0, strides if masked else None,
                              int(causal), sc, out.data_ptr(), lse.data_ptr()))

    s = ctypes.c_void_p()
    L.check(f.tn_stream_create(ctypes.byref(s)))
    try:
        L.check(f.tn_stream_begin_capture(s))
        call(s, *outs[0])
        g = ctypes.c_void_p()
        L.check(f.tn_stream_end_capture(s, ctypes.byref(g)))
        for i in range(3):
            (q2, k2, v2), w = _inputs(tn, dtype, *shape, seed=20 + i)
            for a, b in ((q, q2), (k, k2), (v, v2)):
                L.check(f.tn_memcpy_d2d(a.data_ptr(), b.data_ptr(), a.nbytes, s))
            L.check(f.tn_graph_launch(s, g))
            L.check(f.tn_stream_synchronize(s))
            call(None, *outs[1])
            tn.synchronize()
            (o, lse), (o2, l2) = outs
            assert o.bits().tobytes() == o2.bits().tobytes() and lse.numpy().tobytes() == l2.numpy().tobytes()
            mask = None if md is None else np.ascontiguousarray(
                np.broadcast_to(md.numpy().astype(np.float64), (B, Hq, Lq, S)))
            _compare(dtype, o.numpy().astype(np.float64), lse.numpy(), *w, causal=causal, mask=mask, scale=scale)
        L.check(f.tn_graph_destroy(g))
    finally:
        L.check(f.tn_stream_destroy(s))
