"""gemm_pipe_kernel: every tile shape, at the edges of its tiles and stages, against the oracle, bit-exact.

Edges: rows and columns one short of, at and one past a tile; k-ranges that end inside a 128- or 256-row stage
(the last stage then starts inside the one before it and masks the rows already done); splits whose last range
is shorter; outputs of fewer columns than the padded weights; float outputs; a 4-byte aligned C."""
import numpy as np
import pytest

import ternixengine_amd as tx
from ternixengine_amd import hip_runtime as hr

TILES = 7
SHAPES = [(31, 256, 64), (33, 272, 128), (64, 400, 192), (65, 1040, 320), (129, 2576, 576), (200, 640, 1088)]


@pytest.fixture
def lib():
    lib = tx._load()
    lib.ternix_hip_debug_reset()
    yield lib
    lib.ternix_hip_debug_reset()


def _call(lib, fn, a, wp, n, offset=0, extra=()):
    m, k = a.shape
    da, db, dc = hr.DeviceBuffer.from_array(a), hr.DeviceBuffer.from_array(wp), hr.DeviceBuffer(4 * m * n + 64)
    dc.upload(np.full(m * n + 16, -7, np.int32))
    assert fn(da.value, db.value, dc.value + offset, m, k, n, *extra, None) == 0
    hr.synchronize()
    out = dc.download(np.int32, (m * n + 16,))
    o = offset // 4
    assert (out[:o] == -7).all() and (out[o + m * n:] == -7).all(), "wrote outside C"
    return out[o:o + m * n].reshape(m, n)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(TILES))
@pytest.mark.parametrize("splits", [1, 3])
def test_gemm_tile_edges(lib, oracle, tile, splits):
    rng = np.random.default_rng(tile)
    for m, k, n in SHAPES:
        print(f"tile {tile} splits {splits} M={m} K={k} N={n}", flush=True)
        a = rng.integers(-128, 128, size=(m, k), dtype=np.int8)
        wp = rng.integers(0, 256, size=(k, n // 4), dtype=np.uint8)  # the code 10 among them
        ref = oracle.mm("scalar_mt", a, wp, n)
        assert lib.ternix_hip_debug_set(b"gemm_bm", -1, tile, -1, -1) == 0
        assert lib.ternix_hip_debug_set(b"gemm_splits", splits, -1, -1, -1) == 0
        for offset in (0, 4):
            assert (_call(lib, lib.ternix_hip_mul_mat_ternary_gemm, a, wp, n, offset) == ref).all(), (m, k, n, offset)
        rs = rng.uniform(0.5, 2.0, m).astype(np.float32)
        drs = hr.DeviceBuffer.from_array(rs)
        if m > 32:
            y = _call(lib, lib.ternix_hip_mul_mat_ternary_dequant, a, wp, n, 0, (drs.value, 0.25))
            scale = (rs * np.float32(0.25)).astype(np.float32)
            np.testing.assert_array_equal(y.view(np.float32), ref.astype(np.float32) * scale[:, None])


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(33, 255, 68), (40, 100, 36), (65, 1001, 516), (129, 4093, 260), (260, 300, 1028)])
def test_padded_copy_writes_the_real_columns(lib, oracle, shape):
    m, k, n = shape
    rng = np.random.default_rng(m)
    a = rng.integers(-128, 128, size=(m, k), dtype=np.int8)
    wp = rng.integers(0, 256, size=(k, n // 4), dtype=np.uint8)
    ref = oracle.mm("scalar_mt", a, wp, n)
    for offset in (0, 4):
        assert (_call(lib, lib.ternix_hip_mul_mat_ternary, a, wp, n, offset) == ref).all(), offset
    rs = rng.uniform(0.5, 2.0, m).astype(np.float32)
    drs = hr.DeviceBuffer.from_array(rs)
    y = _call(lib, lib.ternix_hip_mul_mat_ternary_dequant, a, wp, n, 0, (drs.value, 0.25))
    np.testing.assert_array_equal(y.view(np.float32), ref.astype(np.float32) * (rs * np.float32(0.25))[:, None])


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [7, 8])
@pytest.mark.parametrize("splits", [1, 3])
def test_ragged_tiles_read_in_place(lib, oracle, tile, splits):
    """The ragged forms: sizes and addresses off every boundary, the smallest K and N they take, last stages and
    column tiles that overlap their neighbours, operands that end where their buffers do."""
    rng = np.random.default_rng(tile)
    for m, k, n, ao, wo in ((1, 256, 256, 0, 0), (31, 257, 260, 1, 3), (33, 511, 516, 2, 0), (65, 1001, 508, 3, 1),
                            (129, 769, 1028, 0, 2), (40, 2049, 2044, 1, 1)):
        print(f"ragged tile {tile} splits {splits} M={m} K={k} N={n} A+{ao} W+{wo}", flush=True)
        a = rng.integers(-128, 128, size=(m, k), dtype=np.int8)
        wp = rng.integers(0, 256, size=(k, n // 4), dtype=np.uint8)
        ref = oracle.mm("scalar_mt", a, wp, n)
        da = hr.DeviceBuffer.from_array(np.concatenate([np.zeros(ao, np.int8), a.reshape(-1)]))
        dw = hr.DeviceBuffer.from_array(np.concatenate([np.zeros(wo, np.uint8), wp.reshape(-1)]))
        dc = hr.DeviceBuffer(4 * m * n + 64)
        assert lib.ternix_hip_debug_set(b"gemm_bm", -1, tile, -1, -1) == 0
        assert lib.ternix_hip_debug_set(b"gemm_splits", splits, -1, -1, -1) == 0
        dc.upload(np.full(m * n + 16, -7, np.int32))
        assert lib.ternix_hip_mul_mat_ternary_gemm(da.value + ao, dw.value + wo, dc.value, m, k, n, None) == 0
        hr.synchronize()
        got = dc.download(np.int32, (m * n + 16,))
        assert (got[:m * n].reshape(m, n) == ref).all() and (got[m * n:] == -7).all(), (m, k, n)


@pytest.mark.gpu
def test_ragged_plans_first_call_inside_capture(oracle):
    """A ragged call whose plan splits K, captured on a fresh stream (no workspace: one split), then eager."""
    lib = tx._load()
    m, k, n = 65, 4093, 1028
    rng = np.random.default_rng(5)
    a, wp = rng.integers(-128, 128, size=(m, k), dtype=np.int8), rng.integers(0, 256, size=(k, n // 4), dtype=np.uint8)
    ref = oracle.mm("scalar_mt", a, wp, n)
    da, dw, dc, s = hr.DeviceBuffer.from_array(a), hr.DeviceBuffer.from_array(wp), hr.DeviceBuffer(4 * m * n), hr.Stream()

    def call():
        assert lib.ternix_hip_mul_mat_ternary(da.value, dw.value, dc.value, m, k, n, s.handle) == 0

    g = hr.Graph(s, call)
    for run in (g.launch, call, g.launch):
        dc.upload(np.full(m * n, -7, np.int32))
        run()
        s.synchronize()
        assert (dc.download(np.int32, (m, n)) == ref).all()
    lib.ternix_hip_release_stream(s.handle)


def test_gemm_plans_split_whole_blocks(lib):
    """Every plan over a range of sizes is described, and its workspace fits its splits (no launch)."""
    import ctypes
    buf = ctypes.create_string_buffer(192)
    for m in (33, 65, 130, 512, 1000, 4096):
        for k in (128, 256, 272, 2000, 4096, 6912, 16400, 140000):
            for n in (64, 256, 832, 4096, 13824):
                assert lib.ternix_hip_plan_describe(1 << 20, 1 << 24, m, k, n, buf, len(buf)) == 0, (m, k, n)
                need = lib.ternix_hip_mul_mat_ternary_workspace_size(m, k, n)
                plan = buf.value.decode()
                if plan.startswith("gemm_pipe_kernel") and "splits=" in plan:
                    s = int(plan.split("splits=")[1].split()[0])
                    assert need == 4 * s * m * n and 2 <= s <= 16, (plan, need)
