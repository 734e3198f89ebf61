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


# The workgroups that gemv_grid picks on 256 CUs, by waves per CU
GRIDS = [
    (Q4_K, 6143, 4096),    # 12: workgroups of 4 waves; quantizing one of 8 per CU
    (Q4_K, 11001, 2048),   # 10.7: of 4 waves
    (Q4_K, 40003, 2048),   # 39: as many of 4 as fit; quantizing two of 8
    (Q6_K, 14333, 2560),   # 14: of 4 waves; quantizing two of 8
    (Q6_K, 20003, 2560),   # 19.5: of 4 waves past 16
    (Q6_K, 25603, 3072),   # 25: of 4 waves; quantizing two of 8
    (Q6_K, 40003, 2560),   # the least padded spread, four of 4 waves
    (Q6_K, 2501, 14336),   # 9.8: one of 8 waves; fp32 two of 6
    (Q6_K, 5633, 20480),   # 22: the same with five items a lane
]


@pytest.mark.parametrize("t,rows,cols", GRIDS, ids=[f"{'q4k' if s[0] == Q4_K else 'q6k'}_{s[1]}x{s[2]}" for s in GRIDS])
def test_gemv_workgroups(hip, t, rows, cols):
    """Every row has the bits it has in a launch of few rows (up to 4 waves per
    CU), however the workgroups share them. At 40003 x 2560 the spread differs
    too, so there the order of the fp32 sums differs (1e-5 as above)."""
    print(f"[gemv_workgroups] type={t} rows={rows} cols={cols}", flush=True)
    rb, few = cols // 256 * (144 if t == Q4_K else 210), 1000

    class At:   # rows from `first` on
        def __init__(self, buf, first):
            self.ptr = buf.ptr + first * rb
    xd, xqd = hip.alloc(cols * 4), hip.alloc(cols // 32 * 36)
    hip.synth_normal(xd, cols, 3)
    hip.quantize_q8_1(xd, cols, xqd)
    wd = hip.alloc(rows * rb)
    hip.synth_fill(t, wd, rows * cols // 256, rows)
    y, part = hip.alloc((rows + 1) * 4), hip.alloc(few * 4)
    for call, x in ((hip.matvec, xd), (hip.matvec_dp4a, xd), (hip.matvec_q8, xqd)):
        y.upload(np.full(rows + 1, 7.25, np.float32))
        call(t, wd, rows, cols, x, y)
        got = y.download(np.float32)
        assert got[rows] == 7.25
        for r0 in range(0, rows, few):
            n = min(few, rows - r0)
            call(t, At(wd, r0), n, cols, x, part)
            want = part.download(np.float32, n)
            if (t, rows, cols) == (Q6_K, 40003, 2560):
                assert np.linalg.norm(got[r0:r0 + n] - want) <= 1e-5 * np.linalg.norm(want), r0
            else:
                assert np.array_equal(got[r0:r0 + n].view(np.uint32), want.view(np.uint32)), (call.__name__, r0)


def test_gemv_multi_three_per_cu(hip):
    """Quantizing, 38 waves per CU: three workgroups of 8 waves, which loop."""
    print("[gemv_multi_three_per_cu]", flush=True)
    cols, mats = 5120, [(Q4_K, 8191), (Q4_K, 1023), (Q6_K, 1021)]
    xd = hip.alloc(cols * 4)
    hip.synth_normal(xd, cols, 5)
    wds = [hip.alloc(r * cols // 256 * (144 if t == Q4_K else 210)) for t, r in mats]
    for i, ((t, r), wd) in enumerate(zip(mats, wds)):
        hip.synth_fill(t, wd, r * cols // 256, 60 + i)
    ys = [hip.alloc((r + 1) * 4) for _, r in mats]
    for (t, r), y in zip(mats, ys):
        y.upload(np.full(r + 1, 7.25, np.float32))
    hip.matvec_multi([t for t, _ in mats], wds, [r for _, r in mats], cols, xd, ys, dp4a=True)
    for (t, r), wd, y in zip(mats, wds, ys):
        one, got = hip.alloc(r * 4), y.download(np.float32)
        hip.matvec_dp4a(t, wd, r, cols, xd, one)
        assert got[r] == 7.25 and np.array_equal(got[:r].view(np.uint32), one.download(np.uint32))
