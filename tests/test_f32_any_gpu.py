"""f32 attention at head dims other than 64 and 128 and with a negative scale:
the padded flash kernel (k_fa_f32) and the decode kernel (decode_any.hip), at
the edges of their tiles: row blocks of 128, key tiles of 64, 32 and 16, every
padded width, row groups of 8 to 64 lanes, splits and their merge.

Tolerance: the f32 rule of test_sdpa_gpu.py (`_bound`).
"""

import ctypes

import numpy as np
import pytest

import oracle as O

from test_sdpa_gpu import OP, _bound, _dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tn():
    import torchnative_amd as tn

    print("device:", tn._hip_probe(), flush=True)
    return tn


def _compare(got, lse, q, k, v, causal=False, mask=None, scale=None):
    r32, l32 = O.sdpa(q, k, v, is_causal=causal, mask=mask, scale=scale, threads=16)
    r64, l64 = O.sdpa(q, k, v, is_causal=causal, mask=mask, scale=scale, threads=16, dtype=np.float64)
    assert float(np.max(np.abs(got - r32) / _bound(r32, r64))) <= 1.0
    assert float(np.max(np.abs(lse.astype(np.float64) - l32) / _bound(l32, l64))) <= 1.0


def _inputs(tn, B, Hq, Hkv, L, S, D, seed):
    rng = np.random.default_rng(seed)
    t = [_dev(tn, "float32", rng.standard_normal(s)) for s in ((B, Hq, L, D), (B, Hkv, S, D), (B, Hkv, S, D))]
    return t, [x.numpy().astype(np.float64) for x in t]


@pytest.mark.parametrize("shape", [
    # B, Hq, Hkv, L, S, D
    (1, 1, 1, 1, 1, 4), (2, 2, 1, 127, 63, 20), (1, 2, 2, 129, 65, 36), (1, 2, 2, 128, 64, 60), (1, 3, 1, 130, 33, 72),
    (2, 4, 2, 100, 300, 96), (1, 2, 1, 260, 260, 124), (1, 2, 2, 65, 17, 132), (1, 2, 1, 140, 140, 256),
    (1, 1, 1, 5, 3000, 80), (3, 4, 1, 300, 300, 32), (1, 2, 2, 64, 64, 30),
    (1, 1, 1, 1, 1, 32), (1, 2, 1, 130, 200, 4)])  # the plain kernel: head dims 30, and 4 over one key
@pytest.mark.parametrize("causal", [False, True])
def test_rows_keys_and_head_dims(tn, shape, causal):
    (q, k, v), w = _inputs(tn, *shape, seed=sum(shape))
    o, lse = tn._aten_dispatch(OP, q, k, v, 0.0, causal)
    _compare(o.numpy().astype(np.float64), lse.numpy(), *w, causal=causal)


@pytest.mark.parametrize("D,causal", [(64, True), (128, False), (96, False), (200, True)])
@pytest.mark.parametrize("scale", [-0.3, 0.0])
def test_negative_and_zero_scale_with_a_mask(tn, D, causal, scale):
    B, Hq, Hkv, L, S = 1, 4, 2, 130, 131
    (q, k, v), w = _inputs(tn, B, Hq, Hkv, L, S, D, seed=D)
    m = np.random.default_rng(D).standard_normal((L, S))
    m[9, 1:] = -3.0e38
    md = _dev(tn, "float32", m)
    add = np.ascontiguousarray(np.broadcast_to(md.numpy().astype(np.float64), (B, Hq, L, S)))
    for mask, a in ((None, None), (md, add)):
        o, lse = tn._aten_dispatch(OP, q, k, v, 0.0, causal, attn_mask=mask, scale=scale)
        _compare(o.numpy().astype(np.float64), lse.numpy(), *w, causal=causal, mask=a, scale=scale)


@pytest.mark.parametrize("Hq,Hkv,D,lens,cap", [
    (1, 1, 4, [1, 7], 9), (8, 2, 32, [63, 64, 65], 65), (6, 2, 60, [300, 0], 300), (5, 1, 96, [16, 17], 20),
    (4, 4, 96, [3000], 3100), (2, 1, 132, [9, 700], 701), (12, 3, 256, [0, 513], 600)])
def test_decode(tn, Hq, Hkv, D, lens, cap):
    """Past the cache's filled rows NaN (they must not reach the result), both
    entries the same bits, an empty sequence NaN with lse -inf."""
    from torchnative_amd import _lib as L

    B = len(lens)
    rng = np.random.default_rng(D)
    q = _dev(tn, "float32", rng.standard_normal((B, Hq, D)))
    kc, vc = (rng.standard_normal((B, Hkv, cap, D)) for _ in range(2))
    for b, n in enumerate(lens):
        kc[b, :, n:] = np.nan
        vc[b, :, n:] = np.nan
    k, v = _dev(tn, "float32", kc), _dev(tn, "float32", vc)
    ln = tn.tensor(np.asarray(lens, np.int32), device="hip")
    o, lse = tn.sdpa_decode(q, k, v, ln, max(lens))
    o2, l2 = tn.empty((B, Hq, D), "float32", "hip"), tn.empty((B, Hq), "float32", "hip")
    L.check(L.lib().tn_sdpa_decode_noalloc(None, L.TN_F32, q.data_ptr(), k.data_ptr(), v.data_ptr(), B, Hq, Hkv, cap, D,
                                           ln.data_ptr(), max(lens), float("nan"), o2.data_ptr(), l2.data_ptr()))
    assert o.numpy().tobytes() == o2.numpy().tobytes() and lse.numpy().tobytes() == l2.numpy().tobytes()
    qw, kw, vw = (t.numpy().astype(np.float64) for t in (q, k, v))
    got, gl = o.numpy().astype(np.float64), lse.numpy()
    for b, n in enumerate(lens):
        if n == 0:
            assert np.isnan(got[b]).all() and np.isneginf(gl[b]).all()
            continue
        _compare(got[b][None, :, None], gl[b][None, :, None], qw[b][None, :, None], kw[b:b + 1, :, :n],
                 vw[b:b + 1, :, :n])


def test_captured_without_a_workspace(tn):
    """A prompt whose blocks are cut, captured on a stream that holds no
    workspace (nothing may be allocated then), runs on the plain kernel; three
    replays on changing inputs within the bound."""
    from torchnative_amd import _lib as L

    f = L.lib()
    shape = (1, 2, 1, 150, 150, 96)
    B, Hq, Hkv, Lq, S, D = shape
    (q, k, v), _ = _inputs(tn, *shape, seed=3)
    out, lse = tn.empty((B, Hq, Lq, D), "float32", "hip"), tn.empty((B, Hq, Lq), "float32", "hip")
    s = ctypes.c_void_p()
    L.check(f.tn_stream_create(ctypes.byref(s)))
    try:
        L.check(f.tn_stream_begin_capture(s))
        L.check(f.tn_sdpa_fwd(s, L.TN_F32, q.data_ptr(), k.data_ptr(), v.data_ptr(), B, Hq, Hkv, Lq, S, D, None, 0, None,
                              0, float("nan"), out.data_ptr(), lse.data_ptr()))
        g = ctypes.c_void_p()
        L.check(f.tn_stream_end_capture(s, ctypes.byref(g)))
        for i in range(3):
            (q2, k2, v2), w = _inputs(tn, *shape, seed=20 + i)
            for a, b in ((q, q2), (k, k2), (v, v2)):
                L.check(f.tn_memcpy_d2d(a.data_ptr(), b.data_ptr(), a.nbytes, s))
            L.check(f.tn_graph_launch(s, g))
            L.check(f.tn_stream_synchronize(s))
            _compare(out.numpy().astype(np.float64), lse.numpy(), *w)
        L.check(f.tn_graph_destroy(g))
    finally:
        L.check(f.tn_stream_destroy(s))
