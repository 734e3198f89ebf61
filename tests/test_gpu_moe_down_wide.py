"""Kernel B for long down rows: every split of a pair's items on lanes (16, 32
and 64 lanes, whole and padded), more slots than waves, runs of 1 to 8 rows per
workgroup and h up to the LDS limit. (Runs that do not divide the rows need
another CU count than the device's: tests/test_plan_rules.py checks their plans.)

The down projection alone is compared: the oracle's from the GPU's own h
blocks, so the difference is the order of fp32 sums (1e-5 as in the layer's
other tests; about 2^-24 times the square root of the 500 terms of the longest
row is expected).
"""
import numpy as np
import pytest

import kq_synth as S
from katali_hip import Q4_K, Q6_K

pytestmark = pytest.mark.gpu

CASES = [
    # hidden, ffn, n_expert, n_sel, shared, down_type
    (1024, 1280, 12, 9, False, Q4_K),    # 32 lanes, more slots than kernel B's variants take
    (512, 4096, 10, 10, True, Q4_K),     # 32 lanes x 4 items
    (256, 1536, 18, 16, True, Q6_K),     # 16 lanes, 17 slots
    (256, 4352, 4, 2, False, Q6_K),      # 64 lanes, 17 blocks: padded
    (2048, 4608, 8, 6, False, Q6_K),
    (512, 6912, 3, 3, True, Q4_K),       # 64 lanes x 4 items
    (1024, 8192, 8, 8, False, Q4_K),
    (256, 12288, 2, 0, True, Q6_K),      # the shared expert alone (a dense FFN)
    (512, 13824, 3, 2, False, Q6_K),
    (256, 16384, 2, 1, False, Q6_K),     # the longest rows
    (256, 16384, 2, 1, False, Q4_K),
    (256, 14336, 8, 8, False, Q4_K),     # h near the LDS limit
    (4096, 4352, 2, 2, False, Q6_K),     # 8 rows per workgroup
    (4096, 4608, 2, 2, True, Q4_K),
    (1024, 4352, 4, 2, False, Q6_K),     # the fewest rows that take it at two slots, padded
    (1024, 13824, 2, 2, False, Q6_K),
]


@pytest.mark.parametrize("case", CASES, ids=[f"h{c[0]}_f{c[1]}_k{c[3]}{'_sh' if c[4] else ''}"
                                             f"{'_q4' if c[5] == Q4_K else '_q6'}" for c in CASES])
def test_wide_down(hip, oracle, case):
    hidden, ffn, n_exp, k, shared, dt = case
    print(f"[moe_down_wide] case={case}", flush=True)
    rng = np.random.default_rng(hidden + ffn + k)
    gate, up = S.matrix(rng, Q4_K, n_exp * ffn, hidden), S.matrix(rng, Q4_K, n_exp * ffn, hidden)
    down = S.matrix(rng, dt, n_exp * hidden, ffn)
    sh = (S.matrix(rng, Q4_K, ffn, hidden), S.matrix(rng, Q4_K, ffn, hidden), S.matrix(rng, dt, hidden, ffn)) if shared else None
    x = S.activation(rng, hidden)
    dw = [hip.to_device(m) for m in (gate, up, down)]
    dsh = [hip.to_device(m) for m in sh] if shared else None
    dx, slots = hip.to_device(x), k + shared
    desc = hip.moe_desc(hidden, ffn, n_exp, *dw, down_type=dt, shared=dsh)
    odesc = oracle.moe_desc(hidden, ffn, n_exp, gate, up, down, down_type=dt, shared=(ffn, *sh) if shared else None)
    if k:
        logits = rng.standard_normal(n_exp).astype(np.float32)
        ids, wts = oracle.router_topk(logits, k)
        dl = hip.to_device(logits)
        route = hip.moe_route(k, logits=dl)
    else:
        ids, wts, route = np.zeros(0, np.int32), np.zeros(0, np.float32), hip.moe_route(0)
    y = hip.alloc((hidden + 1) * 4)
    y.upload(np.full(hidden + 1, 3.5, np.float32))
    hq, gu = hip.alloc(slots * ffn // 32 * 36), hip.alloc(slots * 2 * ffn * 4)
    hip.moe_layer_debug(desc, route, y, gu, hq, x=dx)
    hip.sync()
    got = y.download(np.float32)
    assert got[hidden] == 3.5
    want = oracle.moe_down_q8(odesc, ids, wts, hq.download(np.uint8))
    r = np.linalg.norm(got[:hidden] - want) / np.linalg.norm(want)
    assert r <= 1e-5, r
    hip.moe_layer(desc, route, y, x=dx)
    hip.sync()
    assert np.array_equal(y.download(np.uint32)[:hidden], got[:hidden].view(np.uint32))
