"""Dense GEMV over every way a row's items spread on lanes: padded rows (items
past the row's end), each number of items per lane and batch, more than one
batch, workgroups that loop over their rows, and ragged row counts.

Sums: a row of n fp32 terms added in any order differs from the exact sum by at
most about n * 2^-24 of the sum of magnitudes, and by 2^-24 * sqrt(n) in the
usual case; at 32768 columns (1024 terms of 32 or 64 values each) that is 2e-6,
and the tolerance is 1e-5 of the result as in the other GEMV tests.
"""
import numpy as np
import pytest

import kq_synth as S
from katali_hip import Q4_K, Q6_K

pytestmark = pytest.mark.gpu

SHAPES = [
    (Q4_K, 37, 768), (Q6_K, 37, 768),        # 24 and 12 items: S 8 x 3, 4 x 3
    (Q4_K, 21, 1792), (Q6_K, 21, 1792),      # padded by 1/7
    (Q4_K, 35, 2304), (Q6_K, 35, 2304),      # 72 items on 16 x 5; 36 on 16 x 3
    (Q4_K, 9, 4352), (Q6_K, 9, 4352),        # 136 on 32 x 5; 68 on 32 x 3
    (Q4_K, 13, 6912), (Q6_K, 13, 6912),      # 64 x 4, 64 x 2
    (Q4_K, 5, 8448), (Q6_K, 5, 8448),        # 64 x 5; 132 items padded to 192
    (Q4_K, 11, 12544), (Q6_K, 11, 12544),    # 64 x 7, 64 x 4
    (Q4_K, 3, 16384), (Q6_K, 3, 16384),      # one full batch
    (Q4_K, 5, 16640), (Q6_K, 5, 16640),      # two batches, the second padded
    (Q4_K, 2, 32768), (Q6_K, 2, 32768),      # the longest row
    (Q4_K, 9731, 2560), (Q6_K, 4099, 3584),  # workgroups loop over their rows
    (Q6_K, 17, 13824),
]


@pytest.mark.parametrize("t,rows,cols", SHAPES, ids=[f"{'q4k' if s[0] == Q4_K else 'q6k'}_{s[1]}x{s[2]}" for s in SHAPES])
def test_gemv_row_spread(hip, oracle, t, rows, cols):
    print(f"[gemv_spread] type={t} rows={rows} cols={cols}", flush=True)
    rng = np.random.default_rng(rows * 13 + cols)
    w, x = S.matrix(rng, t, rows, cols), S.activation(rng, cols)
    xq = oracle.quantize_q8_1(x)
    wd, xd, xqd = hip.to_device(w), hip.to_device(x), hip.to_device(xq)
    ys = [hip.alloc((rows + 1) * 4) for _ in range(3)]
    for y in ys:
        y.upload(np.full(rows + 1, 7.25, np.float32))
    hip.matvec(t, wd, rows, cols, xd, ys[0])
    hip.matvec_dp4a(t, wd, rows, cols, xd, ys[1])
    hip.matvec_q8(t, wd, rows, cols, xqd, ys[2])
    f32, dp4a, q8 = (y.download(np.float32) for y in ys)
    for got in (f32, dp4a, q8):
        assert got[rows] == 7.25   # nothing past the last row
    for got, want in ((f32, oracle.matvec_f32x(t, w, rows, cols, x)), (q8, oracle.matvec_q8(t, w, rows, cols, xq))):
        d = np.linalg.norm(got[:rows] - want) / np.linalg.norm(want)
        assert d <= 1e-5, d
    assert np.array_equal(dp4a.view(np.uint32), q8.view(np.uint32))
    # one launch over two matrices keeps the single GEMV's bits
    for act, one in ((False, f32), (True, dp4a)):
        y = hip.alloc(rows * 4)
        n2 = min(rows, 3)
        y2 = hip.alloc(n2 * 4)
        hip.matvec_multi([t, t], [wd, wd], [rows, n2], cols, xd, [y, y2], dp4a=act)
        assert np.array_equal(y.download(np.uint32), one[:rows].view(np.uint32))
        assert np.array_equal(y2.download(np.uint32), one[:n2].view(np.uint32))


def test_gemv_multi_large_and_small(hip):
    """Matrices large enough for the least padded spread, beside small ones in one launch."""
    for cols, mats in ((5120, [(Q4_K, 20000), (Q6_K, 700)]), (2560, [(Q6_K, 50000), (Q4_K, 33)])):
        print(f"[gemv_multi_large] cols={cols} mats={mats}", flush=True)
        xd = hip.alloc(cols * 4)
        hip.synth_normal(xd, cols, 5)
        wds = []
        for i, (t, r) in enumerate(mats):
            wds.append(hip.alloc(r * cols // 256 * (144 if t == Q4_K else 210)))
            hip.synth_fill(t, wds[-1], r * cols // 256, 40 + i)
        for dp4a in (False, True):
            ys = [hip.alloc(r * 4) for _, r in mats]
            hip.matvec_multi([t for t, _ in mats], wds, [r for _, r in mats], cols, xd, ys, dp4a=dp4a)
            for (t, r), wd, y in zip(mats, wds, ys):
                one = hip.alloc(r * 4)
                (hip.matvec_dp4a if dp4a else hip.matvec)(t, wd, r, cols, xd, one)
                assert np.array_equal(y.download(np.uint32), one.download(np.uint32))
