"""The host-buffer integer matmul at sizes around its launches' edges: runs of equal shapes split
three to a launch, codes of every 16-bit value, widths off every vector size, rows past one tile."""
import numpy as np
import pytest

from test_gpu_parity import eng  # noqa: F401  (module fixture)

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
