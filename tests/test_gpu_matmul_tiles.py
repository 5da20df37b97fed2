"""yx_matmul_bf16_dev beyond one row tile: passes of many rows (LDS tiles of 128 x 256, 128 x
128, 64 x 128 and 64 x 64, some split along k) and few rows against many weight rows (the
streaming kernel), at the edges of tiles, stages and splits, against the CPU backend's
restatement (crates/yaxus-backend-cpu/src/lib.rs:234-248, 314-345)."""

import numpy as np
import pytest

from oracle.attn import matmul_bf16, normal

pytestmark = pytest.mark.gpu


def _bf16_bits(a):
    u = np.ascontiguousarray(a, dtype=np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def _matmul(hip, x, w):
    dx = hip.tensor(x.shape).upload(x)
    dw = hip.tensor(w.shape, np.uint16).upload(w)
    try:
        a = hip.matmul_bf16(dx, dw)
        b = hip.matmul_bf16(dx, dw)  # again: the arrival counters are back at zero
        got, again = a.numpy(), b.numpy()
        a.free()
        b.free()
    finally:
        dx.free()
        dw.free()
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32))
    return got


def _bound(x, w):
    # Exact products, f32 sums in another order than the oracle's: each of the two within
    # k 2^-24 of the magnitudes' sum.
    wf = (w.astype(np.uint32) << 16).view(np.float32)
    return 2 * x.shape[1] * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(wf).astype(np.float64).T)


@pytest.mark.parametrize("t,k,n", [
    (33, 72, 2728),      # 64 x 64, k no multiple of a stage, an odd number of stages
    (100, 8, 1300),      # one stage of 8 k
    (515, 520, 516),     # 64 x 64 split along k, partial tiles on both sides
    (17, 512, 5000),     # fewer rows than a tile, more weight rows than rows
    (700, 1032, 1500),   # split along k with a tail
    (1100, 96, 1030),    # 64 x 128, n even but no multiple of 4 (narrow stores)
    (64, 2048, 4100),    # 64 x 128 split
    (1030, 264, 4099),   # 128-row tiles, n odd
    (2049, 40, 2050),
    (16, 1024, 8192), (1, 2048, 8200), (7, 1536, 8209), (16, 2560, 16400), (3, 2048, 33000),  # streaming
    (5, 3072, 8300), (9, 264, 9000),  # few rows, k the streaming kernel is not built for
])
def test_matmul_matches_the_cpu_backend(hip, t, k, n):
    x = normal(t * k, 31, t * 7 + n).reshape(t, k)
    w = _bf16_bits(normal(n * k, 32, k + n).reshape(n, k))
    got = _matmul(hip, x, w)
    assert np.all(np.abs(got.astype(np.float64) - matmul_bf16(x, w)) <= _bound(x, w))


@pytest.mark.parametrize("t,k,n", [(130, 264, 2000), (4, 1024, 8192)])
def test_matmul_carries_infinities_and_nan(hip, t, k, n):
    """One infinite and one NaN activation: the row's outputs are what the CPU gives
    (infinities of the weight's sign, NaN), the other rows' stay finite and right; values
    near FLT_MAX, whose rounded-up bf16 part would be infinite, stay finite."""
    x = normal(t * k, 41, 0).reshape(t, k)
    w = _bf16_bits(normal(n * k, 42, 0).reshape(n, k) * np.float32(2.0 ** -10))
    w[:, 5] = np.where(np.arange(n) % 2, _bf16_bits(np.float32(0.5)), _bf16_bits(np.float32(-0.5)))
    x[0, ::2] = np.float32(3.4e38)
    x[2, 5] = np.inf
    x[t - 1, 3] = np.nan
    got = _matmul(hip, x, w)
    with np.errstate(over="ignore", invalid="ignore"):
        want = matmul_bf16(x, w)
    fine = [i for i in range(t) if i not in (2, t - 1)]
    assert np.array_equal(got[2], want[2]) and np.isinf(got[2]).all()
    assert np.isnan(got[t - 1]).all()
    assert np.all(np.abs(got[fine].astype(np.float64) - want[fine]) <= _bound(x[fine], w))


def test_streamed_rows_do_not_depend_on_the_pass(hip):
    """A row of at most 16 has the same bits whatever other rows share its pass."""
    k, n = 1024, 8200
    x = normal(16 * k, 31, 5).reshape(16, k)
    w = _bf16_bits(normal(n * k, 32, 6).reshape(n, k))
    full = _matmul(hip, x, w)
    for start, rows in [(0, 1), (15, 1), (2, 3), (8, 7)]:
        part = _matmul(hip, x[start:start + rows], w)
        assert np.array_equal(part.view(np.uint32), full[start:start + rows].view(np.uint32)), (start, rows)


@pytest.mark.parametrize("t,k,n,rows_kernel", [
    (256, 512, 512, True), (17, 768, 4096, True), (128, 64, 1536, True), (32, 1024, 6144, True),
    (20, 1024, 4096, True), (256, 1536, 512, False), (64, 1024, 3072, False), (512, 512, 544, False),
])
def test_small_products_keep_the_kernel_that_starts_sooner(hip, t, k, n, rows_kernel):
    """Just above two 16 x 16 tiles per CU, short sums: LDS tiles take up to 1.55 times as long."""
    x, w, out = hip.tensor((t, k)), hip.tensor((n, k), np.uint16), hip.tensor((t, n))
    try:
        hip.matmul_bf16(x, w, out=out)
        assert (hip.stat("matmul_kernel") == 1) == rows_kernel
    finally:
        for b in (x, w, out):
            b.free()
