"""Kernel A's half units on routed layers (hidden 4096): the bits of whole
units, with the routing on the device and given, with the shared expert among
the slots, eagerly and in graph replays with eager work between them."""
import numpy as np
import pytest

import kq_synth as S
from katali_hip import Q4_K, Q6_K

pytestmark = pytest.mark.gpu

# ffn, n_expert, n_sel, shared: 272, 288 and 288 units on 256 CUs
CASES = [(4352, 4, 2, False), (4608, 3, 1, True), (1024, 12, 9, False)]


@pytest.mark.parametrize("ffn,n_exp,k,shared", CASES)
def test_half_units_routed(hip, oracle, monkeypatch, ffn, n_exp, k, shared):
    print(f"[moe_half_routed] ffn={ffn} k={k} shared={shared}", flush=True)
    hidden, slots = 4096, k + shared
    rng = np.random.default_rng(ffn + k)

    def mats(n):
        return [hip.to_device(S.matrix(rng, t, n * r, c)) for t, r, c in ((Q4_K, ffn, hidden), (Q4_K, ffn, hidden),
                                                                         (Q6_K, hidden, ffn))]
    dw, dsh = mats(n_exp), mats(1) if shared else None
    desc = hip.moe_desc(hidden, ffn, n_exp, *dw, down_type=Q6_K, shared=dsh)
    x = hip.to_device(S.activation(rng, hidden))
    logits = rng.standard_normal(n_exp).astype(np.float32)
    dl = hip.to_device(logits)
    ids, wts = oracle.router_topk(logits, k)
    di, dwt = hip.to_device(ids), hip.to_device(wts)
    out = {}
    for mode in ("whole", "half"):
        if mode == "whole":
            monkeypatch.setenv("KATALI_HIP_HALF_UNITS", "0")
        else:
            monkeypatch.delenv("KATALI_HIP_HALF_UNITS", raising=False)
        for form, route in (("logits", hip.moe_route(k, logits=dl)), ("given", hip.moe_route(k, ids=di, weights=dwt))):
            y, gu, hq = hip.alloc(hidden * 4), hip.alloc(slots * 2 * ffn * 4), hip.alloc(slots * ffn // 32 * 36)
            for _ in range(3):
                hip.moe_layer_debug(desc, route, y, gu, hq, x=x)
            hip.sync()
            out[mode, form] = (y.download(np.uint32), gu.download(np.uint32), hq.download(np.uint8))
    for key in (("half", "logits"), ("whole", "given"), ("half", "given")):
        for a, b, what in zip(out["whole", "logits"], out[key], ("y", "gate/up", "h blocks")):
            assert np.array_equal(a, b), (key, what)
    route, y = hip.moe_route(k, logits=dl), hip.alloc(hidden * 4)
    hip.moe_layer(desc, route, y, x=x)
    hip.sync()
    hip.graph_begin()
    hip.moe_layer(desc, route, y, x=x)
    gr = hip.graph_end()
    try:
        for rep in range(4):
            hip.memset(y, 0, hidden * 4)
            hip.graph_launch(gr)
            hip.sync()
            assert np.array_equal(y.download(np.uint32), out["half", "logits"][0]), rep
            hip.moe_layer(desc, route, y, x=x)   # eager work between replays
            hip.sync()
            assert np.array_equal(y.download(np.uint32), out["half", "logits"][0]), rep
    finally:
        hip.graph_destroy(gr)


@pytest.mark.parametrize("ffn,n_exp,k,shared", [CASES[0], (12288, 1, 0, True)])
def test_half_units_off_where_nothing_waits(hip, monkeypatch, ffn, n_exp, k, shared):
    """KATALI_HIP_TEST_SKEW=1 sets block 0's counter odd, so its first
    workgroup waits for the second and that wait runs to its bound (about a
    second) and expires. KATALI_HIP_XCD=0, a reported expiry and
    katali_hip_one_launch(0) promise kernels that wait for nothing: there the
    skew changes nothing."""
    import katali_hip as K
    print(f"[moe_half_waits] ffn={ffn} k={k} shared={shared}", flush=True)
    hidden = 4096

    def mats(n):
        bufs = []
        for t, r, c in ((Q4_K, ffn, hidden), (Q4_K, ffn, hidden), (Q6_K, hidden, ffn)):
            nb = n * r * (c // 256)
            bufs.append(hip.alloc(nb * K.BLOCK_BYTES[t]))
            hip.synth_fill(t, bufs[-1], nb, n + r + t)
        return bufs
    desc = hip.moe_desc(hidden, ffn, n_exp, *mats(n_exp), down_type=Q6_K, shared=mats(1) if shared else None)
    rng = np.random.default_rng(ffn)
    x = hip.to_device(S.activation(rng, hidden))
    dl = hip.to_device(rng.standard_normal(n_exp).astype(np.float32))
    route, y = hip.moe_route(k, logits=dl) if k else hip.moe_route(0), hip.alloc(hidden * 4)

    def run():
        hip.moe_layer(desc, route, y, x=x)
        hip.sync()
        return y.download(np.uint32)
    ref = run()
    monkeypatch.setenv("KATALI_HIP_TEST_SKEW", "1")
    try:
        monkeypatch.setenv("KATALI_HIP_XCD", "0")
        assert np.array_equal(run(), ref)
        monkeypatch.delenv("KATALI_HIP_XCD")
        hip.one_launch(0)
        assert np.array_equal(run(), ref)
        hip.one_launch(1)
        with pytest.raises(K.HipError) as err:   # the hook does reach half units
            run()
        assert err.value.rc == K.E_TIMEOUT, err.value
        monkeypatch.delenv("KATALI_HIP_TEST_SKEW")
        assert not hip.one_launch(-1)
        assert np.array_equal(run(), ref)
    finally:
        hip.one_launch(1)
    for _ in range(3):
        assert np.array_equal(run(), ref)


# ffn, experts (all selected), half units: 896 units are the most on 256 CUs
# that half units split more evenly; 1056 split so too, but pass the 1024
# counters of the exchange and stay whole
MANY = [(14336, 2, True), (8448, 4, False)]


@pytest.mark.parametrize("ffn,k,halves", MANY)
def test_half_units_many_blocks(hip, oracle, monkeypatch, ffn, k, halves):
    """Counters and tagged words of high block numbers, in the library's
    exchange area and in the allocation-free entry's own."""
    import katali_hip as K
    print(f"[moe_half_many] ffn={ffn} k={k}", flush=True)
    hidden, units = 4096, k * ffn // 32
    bufs = []
    for t, r, c in ((Q4_K, ffn, hidden), (Q4_K, ffn, hidden), (Q6_K, hidden, ffn)):
        nb = k * r * (c // 256)
        bufs.append(hip.alloc(nb * K.BLOCK_BYTES[t]))
        hip.synth_fill(t, bufs[-1], nb, k + r + t)
    desc = hip.moe_desc(hidden, ffn, k, *bufs, down_type=Q6_K)
    rng = np.random.default_rng(ffn)
    x = hip.to_device(S.activation(rng, hidden))
    route = hip.moe_route(k, logits=hip.to_device(rng.standard_normal(k).astype(np.float32)))
    y, gu, hq = hip.alloc(hidden * 4), hip.alloc(k * 2 * ffn * 4), hip.alloc(units * 36)

    def run():
        for _ in range(3):
            hip.moe_layer_debug(desc, route, y, gu, hq, x=x)
        hip.sync()
        return y.download(np.uint32), gu.download(np.uint32), hq.download(np.uint8)
    monkeypatch.setenv("KATALI_HIP_HALF_UNITS", "0")
    want = run()
    monkeypatch.delenv("KATALI_HIP_HALF_UNITS")
    for a, b, what in zip(want, run(), ("y", "gate/up", "h blocks")):
        assert np.array_equal(a, b), what
    h = hq.download(np.uint8).reshape(units, 36)
    gq = gu.download(np.float32).reshape(k, 2, ffn)
    assert np.isfinite(gq).all() and h[:, 4:].any(axis=1).all()   # every block was written
    hip.graph_begin()
    hip.moe_layer_noalloc(desc, route, y, x=x)
    gr = hip.graph_end()
    try:
        for rep in range(3):
            for entry in (hip.moe_layer, hip.moe_layer_noalloc, None):
                hip.memset(y, 0, hidden * 4)
                hip.graph_launch(gr) if entry is None else entry(desc, route, y, x=x)
                hip.sync()
                assert np.array_equal(y.download(np.uint32), want[0]), (rep, entry)
    finally:
        hip.graph_destroy(gr)
    if halves:   # the hook sets block 0's counter off: half units did run if a wait expires
        monkeypatch.setenv("KATALI_HIP_TEST_SKEW", "1")
        try:
            with pytest.raises(K.HipError) as err:
                hip.moe_layer(desc, route, y, x=x)
                hip.sync()   # clears the exchange area
            assert err.value.rc == K.E_TIMEOUT, err.value
        finally:
            hip.one_launch(1)
