"""HIP-graph replay of the attention launches (how bench.py times them, and how an
engine would replay a step): every replay gives the eager call's bits, with eager
launches and synchronisations of the program between the replays. The split-K arrival
counters are left at zero by the kernels themselves, so no memset is captured."""

import numpy as np
import pytest

from tests.scenario import D, Scenario

pytestmark = pytest.mark.gpu


def _forks(sc, prefix, suffixes):
    base = sc.cache.new_seq()
    sc.prefill({base: prefix})
    seqs = []
    for _ in suffixes:
        copies = []
        seqs.append(sc.cache.fork(base, prefix, copies))
        sc.hip.copy_pages(sc.kv, copies)
    sc.prefill({s: n for s, n in zip(seqs, suffixes) if n})
    return seqs


def _case(hip, kind):
    hkv = 4
    f32 = kind == "f32"
    sc = Scenario(hip, pages=800, page=16, hkv=hkv, pool_seed=41, layers=2, f32=f32)
    if kind == "cascade":
        seqs = _forks(sc, 1200, [100, 900, 30, 2000])
        k = 1
    else:
        seqs = [sc.cache.new_seq() for _ in range(5)]
        sc.prefill(dict(zip(seqs, [4095, 1000, 17, 2500, 300])))
        k = {"decode": 1, "verify": 5, "prefill": 64, "f32": 1}[kind]
    pr = sc.run_pass([(s, k) for s in seqs])
    return sc, pr


@pytest.mark.parametrize("kind", ["decode", "cascade", "verify", "prefill", "f32"])
def test_graph_replays_match_eager(hip, kind):
    hq = 16
    sc, pr = _case(hip, kind)
    rows = len(pr.meta.pos)
    hkv = sc.hkv
    q = hip.tensor((rows, hq * D))
    k = hip.tensor((rows, hkv * D))
    v = hip.tensor((rows, hkv * D))
    outs = [hip.tensor((rows, hq * D)) for _ in range(2)]
    for i, t in enumerate((q, k, v)):
        hip.fill_normal(t.ptr, t.nbytes // 4, False, 77, i << 32)

    def step():
        hip.attend_append(sc.kv, 0, k, v, q, hq, out=outs[0])
        hip.attend(sc.kv, 1, q, hq, window=700, out=outs[1])

    step()
    hip.sync()
    eager = [o.numpy() for o in outs]
    hip.graph_begin()
    step()
    hip.graph_end()
    for rep in range(3):
        for o in outs:
            hip.fill_normal(o.ptr, o.nbytes // 4, False, 99, rep << 32)  # eager work between
        hip.sync()
        hip.graph_launch()
        hip.sync()
        for i, o in enumerate(outs):
            got = o.numpy()
            assert np.array_equal(got.view(np.uint32), eager[i].view(np.uint32)), f"replay {rep}, layer {i}"
        step()  # an eager step between replays as well
        hip.sync()
    for t in (q, k, v, *outs):
        t.free()
    sc.kv.destroy()


def _matmul_operands(hip, t, k, n):
    x, w, out = hip.tensor((t, k)), hip.tensor((n, k), np.uint16), hip.tensor((t, n))
    hip.fill_normal(x.ptr, t * k, False, 5, t)
    w.upload(np.random.default_rng(n).integers(0x3C00, 0x3E00, (n, k)).astype(np.uint16))
    return x, w, out


@pytest.mark.parametrize("t", [80, 600, 1030])  # tiles of three shapes, k split in four and in two
def test_matmul_of_many_rows_is_captured_without_an_earlier_call(t):
    from yaxus_amd.backend import HipBackend

    hip = HipBackend(0)
    try:
        x, w, out = _matmul_operands(hip, t, 2048, 2048)
        hip.graph_begin()
        hip.matmul_bf16(x, w, out=out)
        hip.graph_end()
        got = []
        for rep in range(3):
            hip.fill_normal(out.ptr, out.nbytes // 4, False, 99, rep << 32)
            hip.sync()
            hip.graph_launch()
            got.append(out.numpy())
            hip.fill_normal(out.ptr, out.nbytes // 4, False, 98, rep << 32)
            hip.matmul_bf16(x, w, out=out)
            assert np.array_equal(got[-1].view(np.uint32), out.numpy().view(np.uint32)), f"replay {rep}"
    finally:
        hip.close()


def test_matmul_of_many_rows_leaves_graphs_valid():
    from yaxus_amd.backend import HipBackend

    hip = HipBackend(0)
    try:
        few, many = _matmul_operands(hip, 8, 2048, 2048), _matmul_operands(hip, 1030, 2048, 2048)
        hip.matmul_bf16(few[0], few[1], out=few[2])
        want = few[2].numpy()
        hip.graph_begin()
        hip.matmul_bf16(few[0], few[1], out=few[2])
        hip.graph_end()
        hip.matmul_bf16(many[0], many[1], out=many[2])
        hip.fill_normal(few[2].ptr, few[2].nbytes // 4, False, 99, 0)
        hip.graph_launch()
        assert np.array_equal(few[2].numpy().view(np.uint32), want.view(np.uint32))
    finally:
        hip.close()
