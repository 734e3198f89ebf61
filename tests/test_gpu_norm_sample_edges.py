"""RMSNorm at the edges of its register variants (1024, 2048, 4096 and 8192
elements, the loop above) and with shared buffers, and argmax at the edges of
its workgroups and load batches: exact results, so compared bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1023, 1024, 1025, 2049, 4097, 8191, 8192, 8193])
def test_norm_edges(hip, oracle, n):
    print(f"[norm_edges] n={n}", flush=True)
    rng = np.random.default_rng(n)
    x, d, w = (rng.standard_normal(n).astype(np.float32) for _ in range(3))
    xd, dd, wd, out = hip.to_device(x), hip.to_device(d), hip.to_device(w), hip.alloc((n + 1) * 4)
    out.upload(np.full(n + 1, 9.5, np.float32))
    hip.rmsnorm(xd, wd, n, 1e-6, out)
    got = out.download(np.float32)
    assert got[n] == 9.5
    assert np.array_equal(got[:n].view(np.uint32), oracle.rmsnorm(x, w, 1e-6).view(np.uint32))
    want_x, want = oracle.add_rmsnorm(x, d, 0.5, w, 1e-6)
    hip.add_rmsnorm(xd, dd, 0.5, wd, n, 1e-6, out)
    assert np.array_equal(xd.download(np.uint32, n), want_x.view(np.uint32))
    assert np.array_equal(out.download(np.uint32, n), want.view(np.uint32))
    # delta is x itself: the residual doubles
    xd = hip.to_device(x)
    want_x, want = oracle.add_rmsnorm(x, x, 1.0, w, 1e-6)
    hip.add_rmsnorm(xd, xd, 1.0, wd, n, 1e-6, out)
    assert np.array_equal(xd.download(np.uint32, n), want_x.view(np.uint32))
    assert np.array_equal(out.download(np.uint32, n), want.view(np.uint32))
    # the weights are x itself: read behind the residual step
    xd = hip.to_device(x)
    sx = (x + d).astype(np.float32)
    hip.add_rmsnorm(xd, dd, 1.0, xd, n, 1e-6, out)
    assert np.array_equal(out.download(np.uint32, n), oracle.rmsnorm(sx, sx, 1e-6).view(np.uint32))


@pytest.mark.parametrize("n", [1, 63, 256, 257, 1023, 1024, 1025, 4096, 4097, 65535, 65536, 67583, 262144, 262145,
                               524288, 524289, 600001])
def test_argmax_edges(hip, n):
    print(f"[argmax_edges] n={n}", flush=True)
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n).astype(np.float32)
    out = hip.alloc(4)

    def check(v):
        hip.argmax(hip.to_device(v), n, out)
        ok = np.where(v > -np.finfo(np.float32).max, v, -np.inf)
        best = int(np.argmax(ok)) if np.any(ok > -np.inf) else 0   # the first maximum; NaN compares false
        assert int(out.download(np.int32)[0]) == best
    check(x)
    for at in {0, n - 1, n // 2, max(0, n - 257)}:
        v = x.copy()
        v[at] = 50.0
        check(v)
        v[min(n - 1, at + 300)] = 50.0   # a tie: the lower index
        check(v)
    v = np.full(n, -np.finfo(np.float32).max, np.float32)
    check(v)
    v[n - 1] = np.nan
    check(v)
    v[n // 2] = -np.inf
    check(v)
    v = np.zeros(n, np.float32)
    v[: n // 2] = -0.0   # equal to +0
    check(v)
