"""f32 arena: rows whose every score is far below zero or far above it (down to f32's range),
in decode items and in both forms of the prefill tiles."""

import numpy as np
import pytest

from tests.scenario import D, Scenario

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [2.0 ** 90, 2.0 ** 100, 2.0 ** 115])
@pytest.mark.parametrize("waves", [0, 8, 4])  # 0: decode items
def test_scores_near_the_ends_of_the_range(hip, waves, size):
    """One key per row counts: its score leads the others by far more than 2^7, so the row's
    output is that key's V. Scores of +-size and +-2 size, the rows' first keys among them."""
    hq, hkv, rows, prior = 8, 2, 40, 200
    n = rows + prior
    sc = Scenario(hip, pages=n // 16 + 4, page=16, hkv=hkv, pool_seed=3, f32=True)
    try:
        seq = sc.cache.new_seq()
        pr = sc.run_pass([(seq, n)])
        rng = np.random.default_rng(3)
        k = np.zeros((n, hkv, D), np.float32)
        root = np.float32(np.sqrt(size * np.sqrt(np.float32(D))))
        k[:, :, 9] = -2 * root          # every score below zero ..
        lead = rng.integers(0, n, 6)
        lead[0] = 0                     # (the only key of row 0)
        k[lead, :, 9] = -root           # .. but these higher
        v = sc.draw(n * hkv * D).reshape(n, hkv, D)
        q = np.zeros((n, hq, D), np.float32)
        q[:, :, 9] = root
        q[:, 1::2, 9] = -root           # odd heads: scores above zero, where -2 root leads
        hip.append(sc.kv, 0, k, v)
        hip.set_option("prefill_min_rows", 1 if waves else 1 << 20)
        if waves:
            hip.set_option("prefill_f32_waves", waves)
        got = hip.attend(sc.kv, 0, q.reshape(n, -1), hq).reshape(n, hq, D)
        want = np.empty_like(got, dtype=np.float64)
        keys = np.arange(n)
        for i in range(n):
            for h in range(hq):
                seen = k[:i + 1, h // 4, 9].astype(np.float64) * q[i, h, 9]
                best = keys[:i + 1][seen == seen.max()]
                want[i, h] = v[best, h // 4].astype(np.float64).mean(0)
        assert np.abs(got - want).max() < 2e-6
    finally:
        hip.set_option("prefill_min_rows", 0)
        hip.set_option("prefill_f32_waves", 0)
        sc.kv.destroy()


@pytest.mark.parametrize("tiles", [0, 1])
def test_values_near_the_end_of_the_range(hip, tiles):
    """V of 2^119, and keys whose scores grow by less than a tile's maximum lags behind
    (2^8): the weights stay below 1 as on the CPU backend, so 240 keys' sum is finite."""
    hq, hkv, n = 8, 2, 240
    sc = Scenario(hip, pages=n // 16 + 4, page=16, hkv=hkv, pool_seed=3, f32=True)
    try:
        seq = sc.cache.new_seq()
        pr = sc.run_pass([(seq, n)])
        k = np.zeros((n, hkv, D), np.float32)
        k[64:, :, 9] = 5 * np.sqrt(np.float32(D))
        v = (1 + np.abs(sc.draw(n * hkv * D).reshape(n, hkv, D)) / 8) * np.float32(2.0 ** 119)
        q = np.zeros((n, hq, D), np.float32)
        q[:, :, 9] = 1
        q = q.reshape(n, -1)
        hip.append(sc.kv, 0, k, v)
        sc.orc[0].store(pr.meta.kv_slot, k.reshape(n, -1), v.reshape(n, -1))
        hip.set_option("prefill_min_rows", 1 if tiles else 1 << 20)
        got = hip.attend(sc.kv, 0, q, hq)
        want = sc.orc[0].attend_f64(q, hq, pr.meta.pos, pr.meta.pt_off, pr.meta.pages)
        assert np.abs(got - want).max() < 2e-6 * 2.0 ** 119
    finally:
        hip.set_option("prefill_min_rows", 0)
        sc.kv.destroy()
