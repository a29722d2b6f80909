"""The q4_0 / q8_0 linear of more rows than the GEMV takes (qgemm.hip), bit for
bit against the oracle at the edges of its tile shapes: row tiles of 16, column
tiles of 16 in workgroups of 32 and 64, stages of 4 and 8 blocks in rings of 3
and 4, each of the four tile shapes the launch picks by the number of tiles,
scales over every f16 regime (the q4_0 path carries 16 S and d_x / 16), and
activations and planes that start at any element.
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


def _blob(fmt, n, k, seed):
    return (O.synth_q4_0_weight if fmt == "q4_0" else O.synth_q8_0_weight)(n, k, 0.01, seed)


def _linear(fmt):
    return O.q4_0_linear if fmt == "q4_0" else O.q8_0_linear


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0"])
@pytest.mark.parametrize("m,n,k", [
    # one row tile, 64 columns a workgroup: 1 to 33 blocks over stages of 8 in a ring of 4
    (5, 1, 32), (16, 63, 64), (9, 64, 224), (16, 65, 256), (7, 130, 288), (16, 40, 1024), (8, 33, 1056),
    # few tiles, 32 x 32: row and column remainders, stages of 8 in a ring of 3
    (17, 16, 32), (32, 31, 512), (33, 100, 736), (63, 32, 768), (64, 33, 800),
    # 2561 to 6144 tiles, stages of 4 in a ring of 4
    (20, 20600, 32), (33, 13700, 160), (50, 12000, 544),
    # more, 2 x 2 tiles, stages of 4 in a ring of 3
    (128, 12304, 32), (130, 11000, 128), (400, 4000, 416)])
def test_tile_shapes_bit_for_bit(tn, fmt, m, n, k):
    rng = np.random.default_rng(m + n + k)
    x = (rng.standard_normal((m, k)) * 1.3).astype(np.float32)
    x[m // 2] = 0.0
    blob = _blob(fmt, n, k, m + 100)
    bias = rng.standard_normal(n).astype(np.float32) if n % 2 else None
    want = _linear(fmt)(x, blob, n, bias=bias, threads=16)
    q = tn._quantized_from_blob(blob, (n, k), fmt, device="hip")
    b = tn.tensor(bias, device="hip") if bias is not None else None
    got = tn._quantized_linear(tn.tensor(x, device="hip"), q, b).numpy()
    assert got.tobytes() == want.tobytes(), np.argwhere(got != want)[:5]
    # bf16 in and out
    xb = tn.tensor(x, dtype="bfloat16", device="hip")
    want = _linear(fmt)(xb.numpy(), blob, n, bias=bias, threads=16)
    assert np.array_equal(tn._quantized_linear(xb, q, b, out_dtype="bfloat16").bits(), O.bf16_from_f32(want))


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0"])
def test_scales_across_every_f16_regime(tn, fmt):
    """Every finite f16 weight scale; activation scales from zero through the
    subnormals to the f16 maximum, and one that overflows to inf."""
    k, nb, size = 1024, 32, 18 if fmt == "q4_0" else 34
    bits = np.arange(65536, dtype=np.uint32).astype(np.uint16)
    finite = bits[(bits & 0x7C00) != 0x7C00]
    n = len(finite) // nb
    rng = np.random.default_rng(43)
    blob = np.zeros((n * nb, size), np.uint8)
    blob[:, :2] = finite[: n * nb].view(np.uint8).reshape(-1, 2)
    blob[:, 2:] = rng.integers(0, 256, size=(n * nb, size - 2), dtype=np.uint8)
    blob = blob.tobytes()
    q = tn._quantized_from_blob(blob, (n, k), fmt, device="hip")
    x = rng.standard_normal((6, k)).astype(np.float32)
    targets = [0.0, 1e-9, 2.9e-8, 5.9604645e-08, 8.9e-8, 6.097e-05, 6.1035156e-05, 6.104e-05, 1.0, 65504.0, 65519.0,
               65519.996]
    for i, t in enumerate(targets):
        blk = x[0, 32 * i:32 * (i + 1)]
        x[0, 32 * i:32 * (i + 1)] = (blk / np.max(np.abs(blk)) * np.float32(t * 127.0)).astype(np.float32)
    x[1, :32] *= np.float32(1e7)  # amax / 127 > 65520: the scale rounds to inf
    want = _linear(fmt)(x, blob, n, threads=16)
    got = tn._quantized_linear(tn.tensor(x, device="hip"), q).numpy()
    keep = [0, 2, 3, 4, 5]
    assert got[keep].tobytes() == want[keep].tobytes()
    assert not np.isfinite(want[1]).any() and np.array_equal(got[1], want[1], equal_nan=True)


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0"])
def test_operands_at_any_element(tn, fmt):
    """bf16 and f32 rows one element past an aligned address."""
    from torchnative_amd import _lib

    rng = np.random.default_rng(5)
    m, n, k = 21, 50, 320
    blob = _blob(fmt, n, k, 6)
    q = tn._quantized_from_blob(blob, (n, k), fmt, device="hip")
    fn = getattr(_lib.lib(), f"tn_{fmt}_linear")
    for dt, code, es in (("float32", _lib.TN_F32, 4), ("bfloat16", _lib.TN_BF16, 2)):
        buf = tn.tensor(rng.standard_normal(m * k + 1).astype(np.float32), dtype=dt, device="hip")
        x = buf.numpy()[1:].reshape(m, k)
        y = tn.empty((m, n), "float32", "hip")
        _lib.check(fn(None, buf.data_ptr() + es, code, m, k, *q._planes(), n, None, y.data_ptr(), _lib.TN_F32))
        assert y.numpy().tobytes() == _linear(fmt)(x, blob, n, threads=8).tobytes(), dt


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0"])
@pytest.mark.parametrize("m,n,k,off,xoff", [
    # both tile shapes of such a plane (up to 6144 tiles, and more), stages in rings of 4 and 3: one block, less than
    # a ring, remainders; one to four rows with an unaligned x; a row past the GEMV's limits
    (21, 50, 320, 8, 0), (7, 33, 32, 1, 1), (64, 70, 544, 4, 0), (5, 40, 128, 2, 0), (130, 11000, 160, 8, 1),
    (400, 4000, 416, 3, 0), (1, 40, 320, 8, 1), (4, 33, 64, 1, 1), (2, 5, 40960, 12, 0)])
def test_code_plane_at_any_byte(tn, fmt, m, n, k, off, xoff):
    from torchnative_amd import _lib

    rng = np.random.default_rng(m + n + off)
    blob = _blob(fmt, n, k, 6)
    q = tn._quantized_from_blob(blob, (n, k), fmt, device="hip")
    buf = tn.tensor(rng.standard_normal(m * k + xoff).astype(np.float32), device="hip")
    codes = q._qs.numpy().view(np.uint8).reshape(-1)
    moved = tn.tensor(np.concatenate([np.full(off, 0x5A, np.uint8), codes, np.full(16 - off, 0xA5, np.uint8)]), device="hip")
    y = tn.empty((m, n), "float32", "hip")
    _lib.check(getattr(_lib.lib(), f"tn_{fmt}_linear")(None, buf.data_ptr() + 4 * xoff, _lib.TN_F32, m, k,
                                                      moved.data_ptr() + off, q._d.data_ptr(), n, None, y.data_ptr(),
                                                      _lib.TN_F32))
    want = _linear(fmt)(buf.numpy()[xoff:].reshape(m, k), blob, n, threads=16)
    assert y.numpy().tobytes() == want.tobytes()


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0"])
def test_large_products_of_two_to_four_rows(tn, fmt):
    """m n past the line where they leave the GEMV: the oracle's bits, and the
    same bits from a captured call on a stream without a workspace, which
    stays on the GEMV (three replays)."""
    import ctypes

    from torchnative_amd import _lib as L

    f = L.lib()
    k, n = 1024, 20000
    blob = _blob(fmt, n, k, 9)
    q = tn._quantized_from_blob(blob, (n, k), fmt, device="hip")
    for m in (2, 3, 4):
        x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
        xd, y = tn.tensor(x, device="hip"), tn.empty((m, n), "float32", "hip")
        want = _linear(fmt)(x, blob, n, threads=16)
        assert tn._quantized_linear(xd, q).numpy().tobytes() == want.tobytes()
        s, g = ctypes.c_void_p(), ctypes.c_void_p()
        L.check(f.tn_stream_create(ctypes.byref(s)))
        try:
            L.check(f.tn_stream_begin_capture(s))
            L.check(getattr(f, f"tn_{fmt}_linear")(s, xd.data_ptr(), L.TN_F32, m, k, *q._planes(), n, None, y.data_ptr(),
                                                   L.TN_F32))
            L.check(f.tn_stream_end_capture(s, ctypes.byref(g)))
            for _ in range(3):
                y.zero_()
                tn.synchronize()
                L.check(f.tn_graph_launch(s, g))
                L.check(f.tn_stream_synchronize(s))
                assert y.numpy().tobytes() == want.tobytes()
            L.check(f.tn_graph_destroy(g))
        finally:
            L.check(f.tn_stream_destroy(s))
