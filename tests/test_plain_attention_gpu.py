"""The plain attention kernel (k_attn_any) on every path that still reaches it:
16-bit head dims that are no multiple of 8, f32 ones that are no multiple of 4,
16-bit rows off 16 bytes, f32 calls at small head dims with few keys, and its
decode form (lengths, truncation, empty sequences).

Tolerance: the rule of test_sdpa_gpu.py; probabilities are f32 here for every
dtype, so the P-narrowing and subnormal terms of 16-bit inputs are left out.
"""

import numpy as np
import pytest

import oracle as O

from test_sdpa_gpu import OP, _bound, _dev, _narrow

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tn():
    import torchnative_amd as tn

    print("device:", tn._hip_probe(), flush=True)
    return tn


def _compare(dtype, got, lse, q, k, v, nan=None, **kw):
    with np.errstate(invalid="ignore"):
        r32, l32 = O.sdpa(q, k, v, threads=16, **kw)
        r64, l64 = O.sdpa(q, k, v, threads=16, dtype=np.float64, **kw)
    rows = np.zeros(q.shape[:3], bool) if nan is None else nan
    assert np.array_equal(np.isnan(got).any(-1), rows)
    keep = ~rows
    zero = np.zeros_like(r64[keep])
    tol = _bound(r32[keep], r64[keep], zero, got=got[keep], kind=dtype, vsum=zero if dtype == "float16" else None)
    assert float(np.max(np.abs(got[keep] - _narrow(dtype, r32)[keep]) / tol)) <= 1.0
    if lse is not None:
        assert np.array_equal(np.isnan(lse), rows)
        assert float(np.max(np.abs(lse[keep].astype(np.float64) - l32[keep]) / _bound(l32[keep], l64[keep]))) <= 1.0


def _inputs(tn, dtype, B, Hq, Hkv, L, S, D, seed):
    rng = np.random.default_rng(seed)
    t = [_dev(tn, dtype, rng.standard_normal(s)) for s in ((B, Hq, L, D), (B, Hkv, S, D), (B, Hkv, S, D))]
    return t, [x.numpy().astype(np.float64) for x in t]


HEAD_DIMS = [("bfloat16", 20), ("float16", 20), ("float32", 30), ("float16", 250), ("float32", 7)]


@pytest.mark.parametrize("dtype,D", HEAD_DIMS)
@pytest.mark.parametrize("causal,scale", [(False, None), (True, None), (False, -0.3), (True, -0.3)])
def test_prefill(tn, dtype, D, causal, scale):
    for shape in ((2, 4, 2, 35, 70, D), (1, 2, 1, 64, 33, D)):
        (q, k, v), w = _inputs(tn, dtype, *shape, seed=sum(shape))
        o, lse = tn._aten_dispatch(OP, q, k, v, 0.0, causal, scale=scale)
        _compare(dtype, o.numpy().astype(np.float64), lse.numpy(), *w, is_causal=causal, scale=scale)


@pytest.mark.parametrize("dtype,D", HEAD_DIMS)
@pytest.mark.parametrize("kind", ["f32", "same", "bool"])
def test_masks(tn, dtype, D, kind):
    """An additive or bool mask under a negative scale as under the default
    one, a row that sees nothing, one whose keys but the last are hidden (but
    the first and last in an additive mask)."""
    B, Hq, Hkv, L, S = 2, 2, 1, 37, 41
    (q, k, v), w = _inputs(tn, dtype, B, Hq, Hkv, L, S, D, seed=D)
    rng = np.random.default_rng(D + 1)
    nan = np.zeros((B, Hq, L), bool)
    nan[:, :, 7] = True
    if kind == "bool":
        m = rng.random((L, S)) < 0.6
        m[:, 0], m[7], m[9, : S - 1], m[9, S - 1] = True, False, False, True
        o = tn.scaled_dot_product_attention(q, k, v, attn_mask=tn.tensor(m, device="hip"), enable_gqa=True)
        add = np.ascontiguousarray(np.broadcast_to(np.where(m, 0.0, -np.inf), (B, Hq, L, S)))
        _compare(dtype, o.numpy().astype(np.float64), None, *w, nan=nan, mask=add)
        return
    mt = "float32" if kind == "f32" else dtype
    m = rng.standard_normal((L, S))
    m[7] = -np.inf
    m[9, 1:S - 1] = -65504.0 if mt == "float16" else -3.0e38
    md = _dev(tn, mt, m)
    add = np.ascontiguousarray(np.broadcast_to(md.numpy().astype(np.float64), (B, Hq, L, S)))
    for scale, causal in ((None, False), (-0.3, False), (None, True)):
        o, lse = tn._aten_dispatch(OP, q, k, v, 0.0, causal, attn_mask=md, scale=scale)
        _compare(dtype, o.numpy().astype(np.float64), lse.numpy(), *w, nan=nan, mask=add, scale=scale,
                 is_causal=causal)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("D", [96, 64])
def test_rows_off_sixteen_bytes(tn, dtype, D):
    """Every tensor one element past an aligned address. Head dim 64 with a
    negative scale (a positive one is refused there)."""
    from torchnative_amd import _lib as L

    B, Hq, Hkv, Lq, S = 1, 4, 2, 33, 65
    scale = float("nan") if D == 96 else -0.2
    shapes = ((B, Hq, Lq, D), (B, Hkv, S, D), (B, Hkv, S, D))
    rng = np.random.default_rng(D)
    bufs = [_dev(tn, dtype, rng.standard_normal(int(np.prod(s)) + 1)) for s in shapes]
    w = [b.numpy().astype(np.float64)[1:].reshape(s) for b, s in zip(bufs, shapes)]
    out, lse = tn.empty((int(np.prod(shapes[0])) + 1,), dtype, "hip"), tn.empty((B, Hq, Lq), "float32", "hip")
    es, code = {"bfloat16": (2, L.TN_BF16), "float16": (2, L.TN_F16), "float32": (4, L.TN_F32)}[dtype]
    ptr = [b.data_ptr() + es for b in bufs]
    L.check(L.lib().tn_sdpa_fwd(None, code, *ptr, B, Hq, Hkv, Lq, S, D, None, 0, None, 0, scale, out.data_ptr() + es,
                                lse.data_ptr()))
    tn.synchronize()
    got = out.numpy().astype(np.float64)[1:].reshape(shapes[0])
    _compare(dtype, got, lse.numpy(), *w, scale=None if D == 96 else scale)


@pytest.mark.parametrize("B,Hq,L,S,D", [
    # either side of the line to the padded f32 kernel: one or two tiles of 32 keys, one round of workgroups and two
    (1, 4, 1, 1, 4), (1, 4, 7, 16, 8), (1, 4, 33, 64, 8), (1, 4, 33, 65, 8), (1, 4, 33, 100, 8), (1, 2, 33, 32, 24),
    (1, 2, 33, 33, 24), (8, 32, 1, 200, 8), (8, 32, 2, 200, 16), (16, 32, 1, 64, 8), (16, 32, 1, 33, 12),
    (1, 2, 33, 32, 28)])
def test_small_head_dims_in_f32(tn, B, Hq, L, S, D):
    (q, k, v), w = _inputs(tn, "float32", B, Hq, Hq, L, S, D, seed=S + D)
    add = np.random.default_rng(S).standard_normal((L, S))
    md = _dev(tn, "float32", add)
    for causal, mask in ((False, None), (True, None), (False, md)):
        o, lse = tn._aten_dispatch(OP, q, k, v, 0.0, causal, attn_mask=mask)
        full = None if mask is None else np.ascontiguousarray(
            np.broadcast_to(md.numpy().astype(np.float64), (B, Hq, L, S)))
        _compare("float32", o.numpy().astype(np.float64), lse.numpy(), *w, is_causal=causal, mask=full)


@pytest.mark.parametrize("dtype,D", HEAD_DIMS)
@pytest.mark.parametrize("scale", [None, -0.2])
def test_decode(tn, dtype, D, scale):
    """Ragged and zero lengths, a length past max_len (truncated there), large
    values past it, grouped heads."""
    B, Hq, Hkv, cap, lens, max_len = 4, 6, 2, 90, [1, 0, 33, 90], 64
    rng = np.random.default_rng(D)
    q = _dev(tn, dtype, rng.standard_normal((B, Hq, D)))
    kc, vc = (rng.standard_normal((B, Hkv, cap, D)) for _ in range(2))
    for b, n in enumerate(lens):
        kc[b, :, min(n, max_len):] = vc[b, :, min(n, max_len):] = 1e4
    k, v = _dev(tn, dtype, kc), _dev(tn, dtype, vc)
    o, lse = tn.sdpa_decode(q, k, v, tn.tensor(np.asarray(lens, np.int32), device="hip"), max_len, scale=scale)
    qw, kw, vw = (t.numpy().astype(np.float64) for t in (q, k, v))
    got, gl = o.numpy().astype(np.float64), lse.numpy()
    for b, n in enumerate(lens):
        n = min(n, max_len)
        if n == 0:
            assert np.isnan(got[b]).all() and np.isneginf(gl[b]).all()
            continue
        _compare(dtype, got[b][None, :, None], gl[b][None, :, None], qw[b][None, :, None], kw[b:b + 1, :, :n],
                 vw[b:b + 1, :, :n], scale=scale)
