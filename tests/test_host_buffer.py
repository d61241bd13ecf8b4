"""The host-pointer call's device buffer, kept between calls: growing and shrinking needs, several threads at once,
release, a rejected call in between, and needs past what is kept, all exact."""
import threading

import numpy as np
import pytest

import ternixengine_amd as tx


@pytest.mark.gpu
def test_host_calls_share_one_buffer(oracle):
    lib = tx._load()
    rng = np.random.default_rng(0)
    cases = []
    for m, k, n in ((1, 64, 64), (3, 1000, 516), (16, 2560, 1024), (1, 0, 64), (2, 4096, 4096), (1, 64, 64)):
        a = rng.integers(-128, 128, size=(m, k), dtype=np.int8)
        wp = rng.integers(0, 256, size=(k, n // 4), dtype=np.uint8)
        cases.append((a, wp, oracle.mm("scalar_mt", a, wp, n)))
    for a, wp, ref in cases:
        assert (tx.ternary_matmul(a, wp) == ref).all(), a.shape
        with pytest.raises(RuntimeError):
            tx.ternary_matmul(a[:1], wp, impl="hip_tiled")  # one row: rejected
    before = lib.ternix_hip_debug_alloc_count()
    for a, wp, ref in cases:
        assert (tx.ternary_matmul(a, wp) == ref).all(), a.shape
    assert lib.ternix_hip_debug_alloc_count() == before  # all of them fit what is kept
    errors = []

    def work(seed):
        order = np.random.default_rng(seed).permutation(len(cases) * 5) % len(cases)
        for i in order:
            a, wp, ref = cases[i]
            if not (tx.ternary_matmul(a, wp) == ref).all():
                errors.append((seed, a.shape))

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[:4]
    assert lib.ternix_hip_release_stream(None) == 0
    a, wp, ref = cases[2]
    assert (tx.ternary_matmul(a, wp) == ref).all()
    m, k, n = 4096, 256, 4096  # 64 MiB of C alone: a buffer of its own
    a = rng.integers(-128, 128, size=(m, k), dtype=np.int8)
    wp = rng.integers(0, 256, size=(k, n // 4), dtype=np.uint8)
    assert (tx.ternary_matmul(a, wp) == oracle.mm("scalar_mt", a, wp, n)).all()
