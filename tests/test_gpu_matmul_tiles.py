"""yx_matmul_bf16_dev beyond one row tile: passes of many rows (LDS tiles of 128 x 256, 128 x
128, 64 x 128 and 64 x 64, whole and split along k) and few rows against many weight rows (the
streaming kernel), at the edges of tiles, stages and splits, against the CPU backend's
restatement (crates/yaxus-backend-cpu/src/lib.rs:234-248, 314-345) and 64 bits. Each case
names the kernel and the split that the automatic choice takes on 256 CUs, so that a retuned
choice cannot drop one unseen."""

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


ROWS, STREAM, T128x256, T128x128, T64x128, T64x64 = range(1, 7)  # yx_ctx_get_stat's matmul_kernel


@pytest.mark.parametrize("t,k,n,kernel,parts", [
    (33, 72, 2728, ROWS, 1),
    (100, 8, 1300, ROWS, 1),
    (45, 72, 9211, T64x64, 1),       # k no multiple of a stage, an odd number of stages, n odd
    (200, 8, 2100, T64x64, 1),       # one stage of 8 k
    (515, 520, 516, T64x64, 2),      # partial tiles on both sides
    (33, 1096, 4333, T64x64, 4),
    (499, 2056, 249, T64x64, 8),
    (1100, 96, 1030, T64x128, 1),    # n even but no multiple of 4 (narrow stores)
    (700, 1032, 1500, T64x128, 1),   # a k tail
    (21, 1288, 8235, T64x128, 2),
    (64, 2048, 4100, T64x128, 4),
    (60, 8200, 2100, T64x128, 8),
    (17, 512, 5000, ROWS, 1),        # fewer rows than a tile, more weight rows than rows
    (300, 72, 8369, T128x128, 1),
    (601, 2056, 2047, T128x128, 2),
    (77, 3352, 4191, T128x128, 4),
    (1030, 264, 4099, T128x256, 1),
    (2049, 40, 2050, T128x256, 1),
    (1029, 2056, 2050, T128x256, 2),
    (71, 3672, 8230, T128x256, 4),
    (16, 1024, 8192, STREAM, 1), (1, 2048, 8200, STREAM, 1), (7, 1536, 8209, STREAM, 1),
    (16, 2560, 16400, STREAM, 1), (3, 2048, 33000, STREAM, 1),
    (5, 3072, 8300, ROWS, 1), (9, 264, 9000, ROWS, 1),  # k the streaming kernel is not built for
])
def test_matmul_matches_the_cpu_backend(hip, t, k, n, kernel, parts):
    x = normal(t * k, 31, t * 7 + n).reshape(t, k)
    w = _bf16_bits(normal(n * k, 32, k + n).reshape(n, k))
    got = _matmul(hip, x, w)
    assert (hip.stat("matmul_kernel"), hip.stat("matmul_k_parts")) == (kernel, parts)
    bound = _bound(x, w)
    some = np.unique(np.linspace(0, t - 1, 48).astype(int))  # the oracle takes a second per 1.3e9 products
    assert np.all(np.abs(got[some].astype(np.float64) - matmul_bf16(x[some], w)) <= bound[some])
    # Against 64 bits: f32 sums are 0.4e-7 to 3.6e-7 off here, x without its third part 1e-5.
    exact = x.astype(np.float64) @ (w.astype(np.uint32) << 16).view(np.float32).astype(np.float64).T
    assert np.all(np.abs(got - exact) <= bound)
    assert np.linalg.norm(got - exact) < 5e-7 * np.linalg.norm(exact)
    if kernel == STREAM:  # the bits of the kernel of 16 x 16 tiles without a split of k
        try:
            hip.set_option("matmul_k_split", 1)
            rows = _matmul(hip, x, w)
        finally:
            hip.set_option("matmul_k_split", 0)
        assert hip.stat("matmul_kernel") == ROWS
        assert np.array_equal(got.view(np.uint32), rows.view(np.uint32))


@pytest.mark.parametrize("t,k,n,kernel,parts", [
    (130, 264, 4000, T64x64, 1), (4, 1024, 8192, STREAM, 1), (601, 2056, 2047, T128x128, 2),
    (1029, 2056, 2050, T128x256, 2), (21, 1288, 8235, T64x128, 2),
])
def test_matmul_carries_infinities_and_nan(hip, t, k, n, kernel, parts):
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
    assert (hip.stat("matmul_kernel"), hip.stat("matmul_k_parts")) == (kernel, parts)
    some = [0, 1, 2, *range(3, t - 1, 1 + t // 48), t - 1]
    with np.errstate(over="ignore", invalid="ignore"):
        want = dict(zip(some, matmul_bf16(x[some], w)))
    assert np.array_equal(got[2], want[2]) and np.isinf(got[2]).all()
    assert np.isnan(got[t - 1]).all()
    assert np.isfinite(np.delete(got, (2, t - 1), 0)).all()
    for i in some:
        if i not in (2, t - 1):
            assert np.all(np.abs(got[i].astype(np.float64) - want[i]) <= _bound(x[i:i + 1], w)[0])


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
    (603, 408, 387, True), (112, 952, 1210, True), (1826, 408, 102, True), (232, 624, 923, True),
    (259, 968, 600, True), (1964, 968, 112, False), (3000, 1000, 144, False),
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
