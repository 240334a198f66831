"""The host-buffer integer matmul at sizes around its launches' edges: runs of equal shapes split
three to a launch, codes of every 16-bit value, widths off every vector size, rows past one tile."""
import numpy as np
import pytest

from test_gpu_parity import Dev, eng  # noqa: F401  (module fixture)

pytestmark = pytest.mark.gpu

# (rows, [(K, N) per projection])
CASES = [(5, [(64, 64)]), (5, [(7, 9)] * 2), (24, [(1024, 1024)] * 3), (9, [(100, 33)] * 4 + [(101, 33)] * 2),
         (33, [(1031, 500), (1031, 500), (64, 70), (1031, 500)]), (130, [(515, 300)] * 5), (6, [(4100, 50)]),
         (300, [(2050, 7200)])]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_seam_shapes(eng, case):  # noqa: F811
    rows, shapes = CASES[case]
    print(f"seam rows={rows} shapes={shapes}", flush=True)
    rng = np.random.default_rng(case)
    ws = [rng.integers(-1, 2, (n, k)).astype(np.int8) for k, n in shapes]
    xs = [rng.integers(-32768, 32768, (rows, k)).astype(np.int32) for k, _ in shapes]
    pids = [eng.register_proj(w, 1.0) for w in ws]
    for _ in range(2):  # the second call reuses the staging of the first
        got = eng.ternary_matmul_host(pids, xs)
        for w, x, g in zip(ws, xs, got):
            want = (x.astype(np.float64) @ w.T.astype(np.float64)).astype(np.int64)  # |sums| < 2^53: exact
            np.testing.assert_array_equal(g, want.astype(np.int32))
        xs = [x[::-1].copy() for x in xs]
    for p in pids:
        eng.proj_release(p)


def test_long_rows(eng):  # noqa: F811
    """Rows whose planes do not fit LDS, two projections of one shape (the second's planes and tail
    codes follow the first's), through the host seam and on device buffers."""
    b, K, N = 5, 82005, 20
    print(f"seam long rows {b} x {K} x {N}", flush=True)
    rng = np.random.default_rng(K)
    ws = [rng.integers(-1, 2, (N, K)).astype(np.int8) for _ in range(2)]
    xs = [rng.integers(-2000, 2001, (b, K)).astype(np.int32) for _ in range(2)]
    want = [(x.astype(np.float64) @ w.T.astype(np.float64)).astype(np.int32) for x, w in zip(xs, ws)]  # exact below 2^53
    pids = [eng.register_proj(w, 10.0) for w in ws]
    for got, wz in zip(eng.ternary_matmul_host(pids, xs), want):
        np.testing.assert_array_equal(got, wz)
    dx, dacc = Dev(eng, xs[1]), Dev(eng, shape=(b, N), dtype=np.int32)
    eng.ternary_matmul(pids[1], dx.ptr, dacc.ptr, b)
    eng.sync()
    np.testing.assert_array_equal(dacc.get(), want[1])
    for p in pids:
        eng.proj_release(p)
