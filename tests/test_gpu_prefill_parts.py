"""The f32 arena's prefill tiles of 128 logical rows, which multiply bf16 parts of the f32
values, against the tiles of 64 (f32 products): ordinary values, magnitudes that parts
still serve, and those handed over to f32 products (infinities, large K or q, small V)."""

import numpy as np
import pytest

from tests.scenario import D, Scenario
from yaxus_amd._lib import check_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ks,qs,vs,scale,bad,window", [
    (1.0, 1.0, 1.0, None, None, 0),
    (1.0, 1.0, 1.0, None, None, 129),
    (1.0, 1.0, 1.0, -0.11, None, 0),          # the smallest score leads
    (1.0, 1.0, 1.0, 0.0, None, 0),            # equal weights
    (2.0**60, 2.0**-60, 2.0**100, None, None, 0),
    (2.0**-60, 2.0**60, 2.0**-80, None, None, 0),
    (2.0**100, 2.0**-100, 1.0, None, None, 0),   # K above what parts serve
    (2.0**-100, 2.0**100, 1.0, None, None, 33),  # q above
    (2.0**-100, 2.0**-10, 1.0, 2.0**107, None, 0),  # the scale above
    (1.0, 1.0, 2.0**-120, None, None, 0),        # V below
    (1.0, 1.0, 1.0, None, ("k", np.inf), 0),
    (1.0, 1.0, 1.0, None, ("v", -np.inf), 40),
    (1.0, 1.0, 1.0, None, ("v", np.nan), 40),
    (1.0, 1.0, 2.0**105, None, None, 0),
])
def test_parts_match_f32_products(hip, ks, qs, vs, scale, bad, window):
    hq, hkv, rows = 8, 2, [1000, 37, 1]  # split tiles, a ragged tile, one row
    sc = Scenario(hip, pages=sum(-(-r // 32) for r in rows) + 4, page=32, hkv=hkv, pool_seed=5, f32=True)
    try:
        seqs = [sc.cache.new_seq() for _ in rows]
        pr = sc.run_pass(list(zip(seqs, rows)))
        t = len(pr.meta.pos)
        k, v = (sc.draw(t * hkv * D).reshape(t, hkv, D) for _ in range(2))
        q = sc.draw(t * hq * D).reshape(t, hq * D) * np.float32(qs)
        k = k * np.float32(ks)
        v = v / np.abs(v).max() * np.float32(vs)
        if bad:
            {"k": k, "v": v}[bad[0]][500, 1, 77] = bad[1]
        hip.set_option("prefill_min_rows", 1)
        out = {}
        for waves in (8, 4):
            hip.set_option("prefill_f32_waves", waves)
            split0 = hip.stat("prefill_split_tiles")
            out[waves] = hip.attend_append(sc.kv, 0, k, v, q, hq, window=window, scale=scale)
            assert hip.stat("prefill_split_tiles") > split0 or window
        a, b = (np.asarray(x, np.float64) for x in (out[8], out[4]))
        assert np.array_equal(np.isnan(a), np.isnan(b))
        assert np.array_equal(np.isinf(a), np.isinf(b))
        assert (bad is not None) == bool((~np.isfinite(b)).any())
        # A score's rounding (128 products of unit size) and an output's, each a few 2^-24 of
        # the largest value, on either side.
        ok = np.isfinite(a)
        assert np.abs(a[ok] - b[ok]).max() < 4e-6 * vs
        assert np.linalg.norm(a[ok] / vs - b[ok] / vs) < 2e-6 * np.linalg.norm(b[ok] / vs)
    finally:
        hip.set_option("prefill_min_rows", 0)
        hip.set_option("prefill_f32_waves", 0)
        sc.kv.destroy()


def _mantissas(rng, shape, low):
    """Values in [1, 2) whose lower 16 bits are all but the largest (low), or zero."""
    u = (0x3F80 + rng.integers(0, 128, shape)).astype(np.uint32) << 16
    if low:
        u |= (0xFF00 + rng.integers(0, 256, shape)).astype(np.uint32)
    return u.view(np.float32)


@pytest.mark.parametrize("ctx", [64, 1000])
def test_parts_leave_nothing_out_on_one_side(hip, ctx):
    """Values just below a bf16 step, where the products of small parts that are left out
    are largest. In scores: keys with such values against keys that are bf16 exactly, told
    apart by V = +-1, so that a loss of one kind shows in every output; not further off 64
    bits than f32 products. In V: the mean error below 2^-26 of the values, the largest that
    one output's left-out products may reach."""
    hq, hkv, rows = 8, 2, 64
    rng = np.random.default_rng(1)
    even = (np.arange(ctx) % 2 == 0)[:, None, None]
    kv = (ctx, hkv, D)
    worst = _mantissas(rng, kv, True)
    passes = [(np.where(even, worst, _mantissas(rng, kv, False)), np.broadcast_to(np.where(even, 1.0, -1.0), kv),
               _mantissas(rng, (rows, hq * D), True)),
              (rng.standard_normal(kv), worst, rng.standard_normal((rows, hq * D)))]
    err = {}
    for i, (k, v, q) in enumerate(passes):
        for waves in (8, 4):
            sc = Scenario(hip, pages=ctx // 32 + 8, page=32, hkv=hkv, pool_seed=5, f32=True)
            try:
                seq = sc.cache.new_seq()
                pr = sc.run_pass([(seq, ctx)])
                k, v, q = (np.ascontiguousarray(x, np.float32) for x in (k, v, q))
                hip.append(sc.kv, 0, k, v)
                sc.orc[0].store(pr.meta.kv_slot, k.reshape(ctx, -1), v.reshape(ctx, -1))
                pr.meta.pos, pr.meta.pt_off, pr.meta.kv_slot, pr.meta.ids = (
                    x[-rows:] for x in (pr.meta.pos, pr.meta.pt_off, pr.meta.kv_slot, pr.meta.ids))
                hip.begin_pass(pr.meta)
                hip.set_option("prefill_min_rows", 1)
                hip.set_option("prefill_f32_waves", waves)
                got = hip.attend(sc.kv, 0, q, hq)
                want = sc.orc[0].attend_f64(q, hq, pr.meta.pos, pr.meta.pt_off, pr.meta.pages)
                err[i, waves] = got - want
            finally:
                hip.set_option("prefill_min_rows", 0)
                hip.set_option("prefill_f32_waves", 0)
                sc.kv.destroy()
    assert np.linalg.norm(err[0, 8]) <= np.linalg.norm(err[0, 4])
    assert abs(err[1, 8].mean()) < 2.0 ** -26  # V is in [1, 2)


@pytest.mark.parametrize("low", [-90, -108, -112, -118])
def test_small_values_beside_large_ones(hip, low):
    """V whose upper dims are 2^low of the lower ones, in a tile with both: each output as
    exact as f32 products give it."""
    hq, hkv, rows = 8, 2, 300
    sc = Scenario(hip, pages=rows // 32 + 8, page=32, hkv=hkv, pool_seed=5, f32=True)
    try:
        seq = sc.cache.new_seq()
        pr = sc.run_pass([(seq, rows)])
        k, v = (sc.draw(rows * hkv * D).reshape(rows, hkv, D) for _ in range(2))
        v[:, :, 64:] *= np.float32(2.0) ** low
        q = sc.draw(rows * hq * D).reshape(rows, hq * D)
        hip.append(sc.kv, 0, k, v)
        sc.orc[0].store(pr.meta.kv_slot, k.reshape(rows, -1), v.reshape(rows, -1))
        want = sc.orc[0].attend_f64(q, hq, pr.meta.pos, pr.meta.pt_off, pr.meta.pages)
        hip.set_option("prefill_min_rows", 1)
        got = hip.attend(sc.kv, 0, q, hq)
        for half in (slice(0, 64), slice(64, 128)):
            a, b = (x.reshape(rows, hq, D)[..., half].astype(np.float64) * 2.0 ** -low for x in (got, want))
            # f32 products are 1.4e-7 off; parts that lose V's low bits 2.5e-7 (2^-112), 9e-6 (2^-118).
            assert np.linalg.norm(a - b) < 2e-7 * np.linalg.norm(b)
    finally:
        hip.set_option("prefill_min_rows", 0)
        sc.kv.destroy()


@pytest.mark.parametrize("rows,prior,hq,hkv", [
    (8, 4096, 16, 4),    # tiles with a quarter of their rows, partial slots of 32
    (5, 1500, 12, 4),    # 15 logical rows: stays decode items
    (11, 2000, 12, 4),   # 33
])
def test_few_rows_per_tile(hip, rows, prior, hq, hkv):
    """Passes with few rows after a long context (partial slots of the rows in use): the
    automatic choice, decode items and tiles against the oracle's f64 form."""
    sc = Scenario(hip, pages=4 * (-(-(rows + prior) // 64)) + 4, page=64, hkv=hkv, pool_seed=9, f32=True)
    try:
        seqs = [sc.cache.new_seq() for _ in range(4)]
        sc.prefill({s: prior - 7 * i for i, s in enumerate(seqs)})
        pr = sc.run_pass([(s, rows) for s in seqs])
        sc.store(pr)
        t = len(pr.meta.pos)
        q = sc.draw(t * hq * D).reshape(t, hq * D)
        auto = hip.attend(sc.kv, 0, q, hq)
        hip.set_option("prefill_min_rows", 1 << 20)
        items = hip.attend(sc.kv, 0, q, hq)
        hip.set_option("prefill_min_rows", 1)
        tiles = hip.attend(sc.kv, 0, q, hq)
        want = sc.orc[0].attend_f64(q, hq, pr.meta.pos, pr.meta.pt_off, pr.meta.pages)
        for x in (auto, items, tiles):
            assert np.abs(x - want).max() < 1e-5
    finally:
        hip.set_option("prefill_min_rows", 0)
        sc.kv.destroy()


@pytest.mark.parametrize("batch,rows,prior", [
    (16, 8, 4096),    # tiles of 32 logical rows: 256 partial slots, more than whole tiles' scratch
    (1, 32, 28000),   # tiles whose partials don't fit: decode items
])
def test_no_alloc_entry_takes_them(hip, batch, rows, prior):
    """Passes that decode items serve within the fixed scratch keep being served there."""
    hq, hkv = 16, 4
    sc = Scenario(hip, pages=batch * -(-(rows + prior) // 128) + 4, page=128, hkv=hkv, pool_seed=2, f32=True)
    tensors = []
    try:
        seqs = [sc.cache.new_seq() for _ in range(batch)]
        sc.prefill({s: prior for s in seqs}, chunk=8192)
        pr = sc.run_pass([(s, rows) for s in seqs])
        t = len(pr.meta.pos)
        for n in (hkv, hkv, hq):
            tensors.append(hip.tensor((t, n * D)).upload(sc.draw(t * n * D).reshape(t, n * D)))
        k, v, q = tensors
        outs = []
        for fn in (hip.L.yx_attention_append_dev, hip.L.yx_attention_append_noalloc):
            o = hip.tensor((t, hq * D))
            tensors.append(o)
            check_hip(fn(hip.ctx, sc.kv.h, 0, k.ptr, v.ptr, q.ptr, o.ptr, hq, hkv, 0,
                         float(np.float32(1.0) / np.sqrt(np.float32(D)))))
            hip.sync()
            outs.append(o.numpy())
        assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    finally:
        for x in tensors:
            x.free()
        sc.kv.destroy()
