"""Calls whose workgroups hold 2^32 threads and more, which no single dimension
of a grid takes (wg_grid, tn_common.h): the dense linear of rows in any
alignment, the q4_0 linear of one row tile, attention over very many heads.
Only some columns or all of a cheap result are checked; the rest of the weight
is whatever the allocation held.
"""

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tn():
    import torchnative_amd as tn

    print("device:", tn._hip_probe(), flush=True)
    return tn


def _put(ptr, a):
    from torchnative_amd import _lib as L

    a = np.ascontiguousarray(a)
    L.check(L.lib().tn_memcpy_h2d(ptr, a.ctypes.data, a.nbytes, None))


def _get(ptr, count, dtype):
    from torchnative_amd import _lib as L

    a = np.empty(count, dtype)
    L.check(L.lib().tn_memcpy_d2h(a.ctypes.data, ptr, a.nbytes, None))
    return a


def test_dense_linear(tn):
    """[17, 1] x [2^29 + 20, 1] f16: 2^24 + 2 workgroups of 256."""
    from torchnative_amd import _lib as L

    m, n, c = 17, 2 ** 29 + 20, 1000
    rng = np.random.default_rng(1)
    x = rng.standard_normal((m, 1)).astype(np.float32)
    w, y = tn.empty((n, 1), "float16", "hip"), tn.empty((m, n), "float32", "hip")
    xd = tn.tensor(x, device="hip")
    parts = {0: None, n // 2: None, n - c: None}
    for p in parts:
        parts[p] = rng.standard_normal((c, 1)).astype(np.float16)
        _put(w.data_ptr() + 2 * p, parts[p])
    L.check(L.lib().tn_dense_linear(None, xd.data_ptr(), m, 1, w.data_ptr(), L.TN_F16, n, None, y.data_ptr()))
    tn.synchronize()
    for p, v in parts.items():
        for r in (0, 15, 16):
            got = _get(y.data_ptr() + 4 * (r * n + p), c, np.float32)
            assert np.array_equal(got, (x[r] * v.astype(np.float32)[:, 0]).astype(np.float32)), (p, r)


def test_q4_linear(tn):
    """One row that is not 16-byte aligned (it runs on the GEMM), 2^30 + 200
    columns of one block: 2^24 + 4 workgroups of 256."""
    from torchnative_amd import _lib as L

    n, k, c = 2 ** 30 + 200, 32, 640
    rng = np.random.default_rng(2)
    buf = tn.tensor(rng.standard_normal(k + 1).astype(np.float32), device="hip")
    x = buf.numpy()[1:].reshape(1, k)
    qs, d = tn.empty((n, 16), "uint8", "hip"), tn.empty((n,), "float16", "hip")
    y = tn.empty((n,), "bfloat16", "hip")
    parts = {0: None, n // 2 // 64 * 64: None, n - c: None}
    for p in parts:
        parts[p] = O.synth_q4_0_weight(c, k, 0.01, p % 1000)
        raw = np.frombuffer(parts[p], np.uint8).reshape(c, 18)
        _put(qs.data_ptr() + 16 * p, raw[:, 2:])
        _put(d.data_ptr() + 2 * p, raw[:, :2])
    L.check(L.lib().tn_q4_0_linear(None, buf.data_ptr() + 4, L.TN_F32, 1, k, qs.data_ptr(), d.data_ptr(), n, None,
                                   y.data_ptr(), L.TN_BF16))
    tn.synchronize()
    for p, blob in parts.items():
        want = O.bf16_from_f32(O.q4_0_linear(x, blob, c, threads=4))
        assert np.array_equal(_get(y.data_ptr() + 2 * p, c, np.uint16), want[0]), p


def test_attention_at_other_head_dims(tn):
    """65535 sequences of 257 heads, one key each: 16.8 million workgroups of
    256, and every output is its sequence's value."""
    from torchnative_amd import _lib as L

    B, H, D = 65535, 257, 8
    v = np.random.default_rng(3).standard_normal((B, 1, D)).astype(np.float32)
    vd = tn.tensor(v, dtype="bfloat16", device="hip")
    q, out = tn.empty((B, H, D), "bfloat16", "hip"), tn.empty((B, H, D), "bfloat16", "hip")
    q.zero_()
    L.check(L.lib().tn_sdpa_fwd(None, L.TN_BF16, q.data_ptr(), vd.data_ptr(), vd.data_ptr(), B, H, 1, 1, 1, D, None, 0,
                                None, 0, float("nan"), out.data_ptr(), None))
    tn.synchronize()
    assert np.array_equal(out.bits(), np.broadcast_to(vd.bits(), (B, H, D)))
