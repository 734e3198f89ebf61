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
