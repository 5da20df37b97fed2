"""Decode and verify passes of many sequences of different lengths: more work items than
CUs, which the work list cuts into one round or dispatches longest first (all heads of an
item in turn), against the oracle and against a split forced by an option."""

import numpy as np
import pytest

from yaxus_amd.kv import PassMeta

from tests.scenario import D, Scenario, close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,rows,lo,hi,hq,hkv,page,window,f32", [
    (70, 1, 200, 420, 8, 4, 16, 0, False),     # more (sequence, head) pairs than CUs: longest first
    (66, 1, 1, 900, 16, 4, 32, 300, False),    # with a window, from one key on
    (34, 1, 100, 1400, 16, 8, 128, 0, False),
    (40, 3, 50, 1500, 16, 8, 16, 0, False),    # verify: two tiles
    (18, 2, 300, 2600, 8, 4, 16, 0, False),
    (70, 1, 100, 300, 8, 4, 16, 0, True),      # the f32 arena
    (3, 1, 5000, 9000, 8, 1, 16, 0, False),
])
def test_ragged_pass(hip, batch, rows, lo, hi, hq, hkv, page, window, f32):
    rng = np.random.default_rng(batch * 1000 + hi)
    lens = [int(x) for x in np.exp(rng.uniform(np.log(lo), np.log(hi), batch))]
    need = sum(-(-(n + rows) // page) for n in lens)
    sc = Scenario(hip, pages=need + 8, page=page, hkv=hkv, pool_seed=batch, f32=f32)
    try:
        seqs = [sc.cache.new_seq() for _ in lens]
        sc.prefill(dict(zip(seqs, lens)))
        pr = sc.run_pass([(s, rows) for s in seqs])
        t = len(pr.meta.pos)
        k, v = (sc.draw(t * hkv * D).reshape(t, hkv, D) for _ in range(2))
        q = sc.draw(t * hq * D).reshape(t, hq * D)
        got = hip.attend_append(sc.kv, 0, k, v, q, hq, window=window)
        again = hip.attend(sc.kv, 0, q, hq, window=window)
        assert np.array_equal(got.view(np.uint32), again.view(np.uint32))
        sc.orc[0].store(pr.meta.kv_slot, k.reshape(t, -1), v.reshape(t, -1))
        want = sc.orc[0].attend(q, hq, pr.meta.pos, pr.meta.pt_off, pr.meta.pages, window=window)
        assert close(got, want).all(), f"max abs err {np.abs(got - want).max()}"
        hip.set_option("attn_max_chunk_blocks", 8)  # another split of the same keys
        other = hip.attend(sc.kv, 0, q, hq, window=window)
        assert np.abs(got - other).max() < 1e-5
    finally:
        hip.set_option("attn_max_chunk_blocks", 1 << 20)
        sc.kv.destroy()


@pytest.mark.parametrize("chunks,priors,hq,hkv,window,f32", [
    ([512], [6000], 24, 4, 0, False),       # tiles of 60 logical rows in several rounds of chunks
    ([512], [3000], 24, 4, 1024, False),    # one round: two chunks per tile
    ([200, 200], [900, 5200], 16, 4, 0, False),
    ([256], [2900], 24, 4, 0, True),        # the f32 arena
])
def test_prefill_chunks_of_long_tiles(hip, chunks, priors, hq, hkv, window, f32):
    """Prefill tiles split along keys where chunks of the average load would leave a second,
    mostly empty round: against the oracle, the unsplit pass and call to call."""
    sc = Scenario(hip, pages=sum(-(-(a + b) // 64) for a, b in zip(chunks, priors)) + 8, page=64, hkv=hkv,
                  pool_seed=3, f32=f32)
    try:
        seqs = [sc.cache.new_seq() for _ in chunks]
        sc.prefill(dict(zip(seqs, priors)))
        pr = sc.run_pass(list(zip(seqs, chunks)))
        sc.store(pr)
        rows = len(pr.meta.pos)
        q = sc.draw(rows * hq * D).reshape(rows, hq * D)
        split0 = hip.stat("prefill_split_tiles")
        got = hip.attend(sc.kv, 0, q, hq, window=window)
        assert hip.stat("prefill_split_tiles") > split0
        again = hip.attend(sc.kv, 0, q, hq, window=window)
        assert np.array_equal(got.view(np.uint32), again.view(np.uint32))
        hip.set_option("prefill_split", 0)
        whole = hip.attend(sc.kv, 0, q, hq, window=window)
        assert np.abs(got - whole).max() < 2e-5
        some = np.r_[0:8, rows // 2 - 4:rows // 2 + 4, rows - 8:rows]  # the oracle on a part of the rows
        want = sc.orc[0].attend(q[some], hq, pr.meta.pos[some], pr.meta.pt_off[some], pr.meta.pages, window=window)
        assert close(got[some], want).all() and np.abs(got[some] - want).max() < 2e-5
    finally:
        hip.set_option("prefill_split", 1)
        sc.kv.destroy()


def _forks(batch, rows, ctx, prefix, page):
    """The metadata of `rows` rows for each of `batch` sequences after ctx keys, the first
    `prefix` of them on shared pages: (pool pages, pass)."""
    shared, own = prefix // page, -(-(ctx + rows) // page) - prefix // page
    tables = [np.r_[0:shared, shared + i * own:shared + (i + 1) * own].astype(np.uint32) for i in range(batch)]
    p = np.arange(ctx, ctx + rows, dtype=np.uint32)
    return shared + batch * own, PassMeta(
        ids=np.zeros(batch * rows, np.uint32), pos=np.tile(p, batch),
        kv_slot=np.concatenate([t[p // page] * np.uint32(page) + p % page for t in tables]),
        pt_off=np.repeat(np.arange(batch, dtype=np.uint32) * len(tables[0]), rows), pages=np.concatenate(tables))


@pytest.mark.parametrize("batch,rows,ctx,prefix,hq,hkv,f32,items", [
    (74, 7, 1250, 0, 16, 4, False, 296),       # shorter chunks estimated 1% better, 14% slower
    (134, 1, 1230, 0, 14, 2, False, 268),      # a few items beyond one round
    (22, 2, 2461, 2432, 40, 8, True, 352),     # f32 forks that read each other's pages
    (60, 8, 3600, 0, 40, 8, False, None),      # whole prefill tiles in one round
])
def test_work_lists_stay_whole_where_a_cut_does_not_pay(hip, batch, rows, ctx, prefix, hq, hkv, f32, items):
    """Passes that a longer or shorter chunk length made slower keep the plain split's items."""
    pool, meta = _forks(batch, rows, ctx, prefix, 32)
    kv = hip.new_kv(1, pool, 32, hkv, D, f32=f32)
    try:
        hip.begin_pass(meta)
        split0 = hip.stat("prefill_split_tiles")
        hip.attend(kv, 0, np.zeros((batch * rows, hq * D), np.float32), hq)
        if items is None:
            assert hip.stat("prefill_split_tiles") == split0
        else:
            assert hip.stat("decode_items") == items
    finally:
        kv.destroy()
