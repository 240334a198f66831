"""BitLinear at widths and row addresses that fit no vector load or tile, against the CPU
restatement, bit for bit: the float4-free row prologue, the tail terms and the partial tiles of
the integer matrix-core epilogues."""
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import assert_bitexact
from test_gpu_parity import Dev, eng  # noqa: F401  (module fixture)

pytestmark = pytest.mark.gpu

FLOAT, FIXED, INT8 = 0, 1, 2

# (rows, K, N): K % 8 from 0 to 7, one and two units per thread of the few-row prologue, one to
# four of the many-row one, rows below, at and above a row tile
SHAPES = [(2, 9, 33), (3, 1025, 70), (5, 4098, 64), (8, 1031, 130), (13, 516, 95), (31, 2047, 1333), (33, 130, 6000),
          (48, 1030, 200), (64, 300, 2100), (65, 1027, 64), (100, 1031, 1333), (130, 8190, 40), (300, 255, 500),
          (520, 1029, 36), (530, 2046, 36), (515, 4099, 36), (514, 6911, 36), (513, 8187, 36), (514, 5632, 36)]


# both sides of the integer modes' choice between dot products and matrix cores, one to four rows
FEW = [(1, 1023, 40), (1, 1025, 40), (1, 1026, 16390), (1, 1032, 16390), (1, 2559, 40), (1, 2561, 40), (1, 2570, 16390),
       (1, 2576, 16390), (1, 4098, 16390), (1, 13900, 8200), (2, 511, 70), (2, 512, 70), (2, 513, 70), (2, 514, 16390),
       (2, 520, 16390), (2, 560, 70), (3, 120, 70), (3, 127, 70), (3, 136, 70), (3, 343, 70), (4, 66, 70), (4, 64, 70),
       (4, 257, 70), (3, 66, 49160)]


@pytest.mark.parametrize("mode", [FLOAT, FIXED, INT8])
@pytest.mark.parametrize("rows,K,N", SHAPES + FEW)
def test_bitlinear_odd(eng, oracle, rows, K, N, mode):  # noqa: F811
    print(f"odd rows={rows} K={K} N={N} mode={mode}", flush=True)
    rng = np.random.default_rng(rows + 3 * K + 5 * N + mode)
    x = (rng.standard_normal((rows, K)) * 2).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(K)).astype(np.float32)
    wq = rng.integers(-1, 2, (N, K)).astype(np.int8)
    sw = float(np.float32(1.0 / 0.0157))
    want = oracle.bitlinear(x, nw, wq, sw, 1e-6, mode)
    pid = eng.register_proj(wq, sw, nw)
    for off in (0, 1):  # the rows one float past an aligned address
        buf = np.zeros(rows * K + off, np.float32)
        buf[off:] = x.ravel()
        dx, dout = Dev(eng, buf), Dev(eng, shape=(rows, N))
        dacc = Dev(eng, shape=(rows, N), dtype=np.int32)
        for acc in ((None,) if mode == FLOAT else (dacc.ptr, None)):
            eng.bitlinear(pid, dx.ptr + 4 * off, dout.ptr, rows, mode=mode, acc=acc)
            eng.sync()
            assert_bitexact(dout.get(), want["out"], f"out offset {off}")
        if mode != FLOAT:
            np.testing.assert_array_equal(dacc.get(), want["acc"])
    eng.proj_release(pid)


# (rows, K, N) around the plan's limits on splitting K: 144 stages of 64 elements (K 9216, then
# chains in steps of 16 positions) with at most 40 rows of eight 64 x 128 tiles or 16 of 14, and 216
# stages (K 13824) whatever the tiles; partial tiles, tails, and the 64- and 128-row tiles split
SPLIT = [(2, 9223, 70), (3, 9224, 70), (40, 9230, 1024), (41, 9230, 1024), (17, 9345, 1025), (16, 9345, 1030), (16, 9345, 1800), (40, 13831, 40),
         (5, 13832, 40), (40, 14003, 333), (100, 16384, 64), (200, 13900, 700)]


@pytest.mark.parametrize("mode", [FIXED, INT8])
@pytest.mark.parametrize("rows,K,N", SPLIT)
def test_bitlinear_split_k(eng, oracle, rows, K, N, mode):  # noqa: F811
    """Long rows whose K is split over blocks: outputs and accumulators, through the context's
    workspace and, with a smaller second call on what the first left, the static scratch."""
    print(f"split rows={rows} K={K} N={N} mode={mode}", flush=True)
    rng = np.random.default_rng(rows + K + N + mode)
    x = (rng.standard_normal((rows, K)) * 2).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(K)).astype(np.float32)
    wq = rng.integers(-1, 2, (N, K)).astype(np.int8)
    sw = float(np.float32(1.0 / 0.0157))
    want = oracle.bitlinear(x, nw, wq, sw, 1e-6, mode)
    pid = eng.register_proj(wq, sw, nw)
    dx, dout, dacc = Dev(eng, x), Dev(eng, shape=(rows, N)), Dev(eng, shape=(rows, N), dtype=np.int32)
    for fn in (eng.bitlinear, eng.bitlinear_noalloc):
        for n in (rows, max(2, rows // 2)):
            for acc in (dacc.ptr, None):
                fn(pid, dx.ptr, dout.ptr, n, mode=mode, acc=acc)
                eng.sync()
                assert_bitexact(dout.get()[:n], want["out"][:n], f"out of {n} rows")
            np.testing.assert_array_equal(dacc.get()[:n], want["acc"][:n])
    eng.proj_release(pid)


@pytest.mark.parametrize("mode", [FIXED, INT8])
@pytest.mark.parametrize("hidden,inter,layers", [(16, 9232, 2), (9232, 32, 1)])
def test_model_split_k(tmp_path, oracle, hidden, inter, layers, mode):
    """Prompts whose residual or whose swiglu-pair GEMM splits K: logits of every position."""
    from matmulfreellmcpu_amd import Engine, make_blob, read_blob
    print(f"split model hidden={hidden} mode={mode}", flush=True)
    blob = read_blob(make_blob(str(tmp_path / "m"), vocab=200, hidden=hidden, layers=layers, inter=inter, seed=5,
                               random_norms=True, random_lb=True))
    ids = np.random.default_rng(2).integers(0, 200, 6)
    e = Engine(0)
    e.load_blob(blob, mode)
    assert_bitexact(e.forward(ids), oracle.model(blob).forward(ids, mode), "logits")
    e.close()


@pytest.mark.parametrize("hidden", [100, 250, 1027])
@pytest.mark.parametrize("mode", [FLOAT, FIXED, INT8])
def test_serve_odd_hidden(tmp_path, oracle, hidden, mode):
    """Serving steps whose recurrence runs inside the g_norm prologue at hidden sizes that are no
    multiple of 4 (rows at any 4-byte address, one to seven tail elements)."""
    from matmulfreellmcpu_amd import Engine, make_blob, read_blob
    print(f"serve hidden={hidden} mode={mode}", flush=True)
    blob = read_blob(make_blob(str(tmp_path / "m"), vocab=500, hidden=hidden, layers=2, inter=208, seed=hidden,
                               random_norms=True, random_lb=True))
    om = oracle.model(blob)
    rng = np.random.default_rng(hidden + mode)
    prompts = [rng.integers(0, 500, n) for n in (5, 9, 1, 20, 3)]
    want, wst = om.generate_serve(prompts, 4, mode, want_state=True)
    e = Engine(0)
    e.load_blob(blob, mode)
    e.reset(len(prompts))
    got = [list(p) + [int(t)] for p, t in zip(prompts, e.prefill_streams(prompts))]
    for _ in range(3):
        for g, t in zip(got, e.step([g[-1] for g in got])):
            g.append(int(t))
    for g, w in zip(got, want):
        np.testing.assert_array_equal(np.array(g), w)
    assert_bitexact(e.state(), wst, "states")
    e.close()


CHILD = """
import hashlib, sys
import numpy as np
sys.path[:0] = [{root!r}, {tests!r}]
from matmulfreellmcpu_amd import Engine
from test_gpu_parity import Dev
rng, e, h = np.random.default_rng(9), Engine(0), hashlib.md5()
for rows, K, N in ((20, 2048, 512), (3, 530, 70), (40, 1000, 3000)):
    x = rng.standard_normal((rows, K)).astype(np.float32)
    pid = e.register_proj(rng.integers(-1, 2, (N, K)).astype(np.int8), 30.0, np.ones(K, np.float32))
    dx, dout = Dev(e, x), Dev(e, shape=(rows, N))
    for mode in (0, 1, 2):
        e.bitlinear(pid, dx.ptr, dout.ptr, rows, mode=mode)
        e.sync()
        h.update(dout.get().tobytes())
print("RESULT", h.hexdigest(), e.workspace_bytes())
"""


def test_switches():
    """MMF_KW8_32=0 splits K at 8-32 rows (the partials are workspace), MMF_FLOAT_MFMA_MIN_ROWS moves
    the float line; the results stay the same bits."""
    here = os.path.dirname(os.path.abspath(__file__))
    code = CHILD.format(root=os.path.dirname(here), tests=here)

    def run(**env):
        print(f"switches {env}", flush=True)
        r = subprocess.run([sys.executable, "-c", code], env={**os.environ, **env}, capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-2000:]
        line = [ln for ln in r.stdout.splitlines() if ln.startswith("RESULT")][0].split()
        return line[1], int(line[2])

    plain, ws = run()
    split, ws_split = run(MMF_KW8_32="0")
    assert split == plain and ws_split > ws
    for n in ("0", "1", "30"):
        assert run(MMF_FLOAT_MFMA_MIN_ROWS=n) == (plain, ws)
