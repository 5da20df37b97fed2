"""Keys and values that are NaN or infinite: where the CPU backend's result is NaN
(crates/yaxus-backend-cpu/src/lib.rs:389-427: a NaN or +inf score makes the row's sum NaN)
the device's is, in every kernel and however the keys are split over waves and chunks."""

import numpy as np
import pytest

from tests.scenario import D, Scenario, close

pytestmark = pytest.mark.gpu

DEFAULTS = {"attn_max_chunk_blocks": 1 << 20, "attn_decode_shape": 0, "prefill_min_rows": 0,
            "prefill_f32_waves": 0, "attn_cascade": 1}


@pytest.mark.parametrize("what,bad", [("k", np.nan), ("k", np.inf), ("v", np.nan), ("v", -np.inf)])
@pytest.mark.parametrize("lens,rows,forked,f32,options", [
    ([600, 32, 1500, 3000], 1, False, False, {}),
    ([600, 32, 1500, 3000], 1, False, False, {"attn_max_chunk_blocks": 8}),
    ([600, 32, 1500, 3000], 1, False, False, {"attn_decode_shape": 1, "attn_max_chunk_blocks": 40}),
    ([600, 32, 1500, 3000], 1, False, False, {"attn_decode_shape": 2, "attn_max_chunk_blocks": 16}),
    ([600, 32, 1500, 3000], 5, False, False, {"attn_max_chunk_blocks": 16}),
    ([1700, 1024, 2100, 1600], 1, True, False, {}),
    ([600, 32, 1500, 3000], 1, False, True, {"attn_max_chunk_blocks": 16}),
    ([64, 3000, 4096], 64, False, False, {"prefill_min_rows": 1}),
    ([64, 3000, 4096], 64, False, True, {"prefill_min_rows": 1}),
    ([64, 3000, 4096], 64, False, True, {"prefill_min_rows": 1, "prefill_f32_waves": 4}),
])
def test_bad_key_or_value_reaches_the_result(hip, lens, rows, forked, f32, options, what, bad):
    hq, hkv, page = 16, 4, 16
    sc = Scenario(hip, pages=sum(n + rows for n in lens) // page + 16, page=page, hkv=hkv, pool_seed=7, f32=f32)

    def extend(items, at):
        """New tokens for each sequence; key at[s] (counted from the pass's first) of KV head 1 + s % 3 is bad."""
        pr = sc.run_pass(items)
        n = len(pr.meta.pos)
        k, v = (sc.draw(n * hkv * D).reshape(n, hkv, D) for _ in range(2))
        r0 = 0
        for i, (_, cnt) in enumerate(items):
            if at[i] is not None:
                (k if what == "k" else v)[r0 + at[i], 1 + i % 3, 5] = bad
            r0 += cnt
        hip.append(sc.kv, 0, k, v)
        sc.orc[0].store(pr.meta.kv_slot, k.reshape(n, -1), v.reshape(n, -1))
        return pr

    try:
        base = 1024
        if forked:
            first = sc.cache.new_seq()
            extend([(first, base)], [77])
            seqs = [sc.cache.fork(first, base, []) for _ in lens]
            for i, (s, n) in enumerate(zip(seqs, lens)):
                if n > base:
                    extend([(s, n - base)], [None if i == 0 else (n - base) // 2])
        else:
            seqs = [sc.cache.new_seq() for _ in lens]
            for i, (s, n) in enumerate(zip(seqs, lens)):
                extend([(s, n)], [[0, None, n // 2, n - 1][i]])
        # The second sequence's bad key is its pass's first: alone in its block, and in
        # decode alone in its wave.
        pr = extend([(s, rows) for s in seqs], [0 if i == 1 and what == "k" else None for i in range(len(seqs))])
        t = len(pr.meta.pos)
        q = sc.draw(t * hq * D).reshape(t, hq, D)
        q[:, :, 5] = np.abs(q[:, :, 5]) + np.float32(0.1)  # an infinite K scores +inf
        q = q.reshape(t, -1)
        with np.errstate(invalid="ignore"):
            want = sc.orc[0].attend(q, hq, pr.meta.pos, pr.meta.pt_off, pr.meta.pages)
        assert not np.isfinite(want).all() and np.isfinite(want).any()
        for key, value in options.items():
            hip.set_option(key, value)
        split0 = hip.stat("prefill_split_tiles")
        got = hip.attend(sc.kv, 0, q, hq)
        assert "prefill_min_rows" not in options or hip.stat("prefill_split_tiles") > split0
        fine = np.isfinite(want)
        assert np.array_equal(np.isfinite(got), fine)
        if f32 or what == "k":  # an infinite binary16 V times a weight's low part is NaN
            assert np.array_equal(np.isnan(got), np.isnan(want))
        assert close(got[fine], want[fine]).all()
    finally:
        for key in options:
            hip.set_option(key, DEFAULTS[key])
        sc.kv.destroy()
