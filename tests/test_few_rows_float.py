"""Float outputs of 1-32 rows: the same bits whichever plan runs (GEMM tiles, int32 sums and a dequantising launch,
the GEMVs' own epilogues, padded copies), as the exact int32 product scaled once and rounded once per output, and
under graph capture before the stream owns any buffers."""
import numpy as np
import pytest

import ternixengine_amd as tx
from ternixengine_amd import hip_runtime as hr

F32 = np.float32
# aligned short and long K, N/4 % 64 != 0, K % 64 != 0, ragged; rows at the edges of the rules
SHAPES = [(m, k, n) for k, n in ((512, 512), (4096, 1024), (1024, 832), (1040, 768), (659, 516), (2061, 1028))
          for m in (1, 3, 4, 8, 9, 16, 17, 32)]


def _bufs(rng, m, k, n):
    a = rng.integers(-128, 128, size=(m, k), dtype=np.int8)
    wp = rng.integers(0, 256, size=(k, n // 4), dtype=np.uint8)
    rs = rng.uniform(0.5, 2.0, m).astype(F32)
    return a, wp, rs, [hr.DeviceBuffer.from_array(x) for x in (a, wp, rs)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_dequant_and_swiglu_plans(oracle, shape):
    lib = tx._load()
    m, k, n = shape
    print(f"M={m} K={k} N={n}", flush=True)
    a, wp, rs, (da, dw, drs) = _bufs(np.random.default_rng(sum(shape)), m, k, n)
    c = oracle.mm("scalar_mt", a, wp, n)
    y = c.astype(F32) * (rs * F32(0.25))[:, None]
    for offset in (0, 4):  # Y aligned to 16 bytes, or not
        dy = hr.DeviceBuffer(4 * m * n + 64)
        dy.upload(np.full(m * n + 16, 7, F32))
        assert lib.ternix_hip_mul_mat_ternary_dequant(da.value, dw.value, dy.value + offset, m, k, n, drs.value, 0.25, None) == 0
        hr.synchronize()
        got = dy.download(F32, (m * n + 16,))
        np.testing.assert_array_equal(got[offset // 4:offset // 4 + m * n].reshape(m, n), y)
        assert (got[offset // 4 + m * n:] == 7).all()
    dh, dy, dsc = hr.DeviceBuffer(2 * m * n), hr.DeviceBuffer(4 * m * n), hr.DeviceBuffer(4 * m * n)
    # with and without scratch: the product dequantised, then the standalone SwiGLU, bit for bit
    assert lib.ternix_hip_mul_mat_ternary_dequant(da.value, dw.value, dy.value, m, k, n, drs.value, 1e-4, None) == 0
    assert lib.ternix_hip_swiglu(dh.value, dy.value, m * n, None) == 0
    hr.synchronize()
    ref = dh.download(F32, (m, n // 2))
    for scratch in (dsc.value, None):
        dh.upload(np.full(m * (n // 2), 7, F32))
        assert lib.ternix_hip_mul_mat_ternary_swiglu(da.value, dw.value, dh.value, m, k, n, drs.value, 1e-4, scratch, None) == 0
        hr.synchronize()
        np.testing.assert_array_equal(dh.download(F32, (m, n // 2)), ref)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(4, 4096, 1024), (16, 512, 512), (8, 659, 516), (32, 2061, 1028)], ids=lambda s: "x".join(map(str, s)))
def test_dequant_first_call_inside_capture(oracle, shape):
    """A fresh stream's first call is captured: no allocation then, other plans, the same results on each replay,
    and after an eager call on the stream has created its buffers."""
    lib = tx._load()
    m, k, n = shape
    print(f"capture M={m} K={k} N={n}", flush=True)
    a, wp, rs, (da, dw, drs) = _bufs(np.random.default_rng(sum(shape) + 1), m, k, n)
    y = oracle.mm("scalar_mt", a, wp, n).astype(F32) * (rs * F32(0.25))[:, None]
    dy, s = hr.DeviceBuffer(4 * m * n), hr.Stream()

    def call():
        assert lib.ternix_hip_mul_mat_ternary_dequant(da.value, dw.value, dy.value, m, k, n, drs.value, 0.25, s.handle) == 0

    before = lib.ternix_hip_debug_alloc_count()
    g = hr.Graph(s, call)
    assert lib.ternix_hip_debug_alloc_count() == before
    for rep in range(3):
        dy.upload(np.full(m * n, 7, F32))
        g.launch()
        s.synchronize()
        np.testing.assert_array_equal(dy.download(F32, (m, n)), y)
        dy.upload(np.full(m * n, 7, F32))
        call()
        s.synchronize()
        np.testing.assert_array_equal(dy.download(F32, (m, n)), y)
    lib.ternix_hip_release_stream(s.handle)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(17, 512, 768), (32, 2048, 1024), (32, 2176, 256), (16, 512, 768)], ids=lambda s: "x".join(map(str, s)))
def test_tile64_few_rows_float(oracle, shape):
    """Tile-64 weights, either side of the rules for the GEMM's 32-row tiles: the row-major layout's bits."""
    lib = tx._load()
    m, k, n = shape
    print(f"tile-64 M={m} K={k} N={n}", flush=True)
    a, wp, rs, (da, dw, drs) = _bufs(np.random.default_rng(sum(shape)), m, k, n)
    dt, dy = hr.DeviceBuffer(wp.nbytes), hr.DeviceBuffer(4 * m * n)
    assert tx.interleave_tile64_device(dt.value, dw.value, k, n) == 0
    assert lib.ternix_hip_mul_mat_ternary_tile64_dequant(da.value, dt.value, dy.value, m, k, n, drs.value, 0.25, None) == 0
    hr.synchronize()
    ref = oracle.mm("scalar_mt", a, wp, n).astype(F32) * (rs * F32(0.25))[:, None]
    np.testing.assert_array_equal(dy.download(F32, (m, n)), ref)
