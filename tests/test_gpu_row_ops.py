"""Element-wise, norm and recurrent operators at sizes and addresses on both sides of their
vector forms, against the CPU restatement, bit for bit."""
import numpy as np
import pytest

from conftest import assert_bitexact
from test_gpu_parity import Dev, eng  # noqa: F401  (module fixture)

pytestmark = pytest.mark.gpu


def _at(eng, a, off):  # noqa: F811
    """Device copy of a, `off` floats past an aligned address: (keep-alive, pointer)."""
    d = Dev(eng, np.concatenate([np.zeros(off, np.float32), a.ravel()]))
    return d, d.ptr + 4 * off


# up to one, two and four groups of eight per thread, the general kernel, every K % 8
COLS = [1, 7, 8, 100, 1027, 2047, 2048, 2049, 4096, 4101, 8190, 8192, 8195, 9000]


@pytest.mark.parametrize("cols", COLS)
def test_norms(eng, oracle, cols):  # noqa: F811
    rng = np.random.default_rng(cols)
    for rows, off in ((1, 0), (5, 1), (9, 3)):
        print(f"norms rows={rows} cols={cols} off={off}", flush=True)
        x, o = (rng.standard_normal((rows, cols)).astype(np.float32) * s for s in (2.0, 3.0))
        x, o = x.astype(np.float32), o.astype(np.float32)
        w = (1 + 0.1 * rng.standard_normal(cols)).astype(np.float32)
        (kx, px), (ko, po), (kw, pw) = _at(eng, x, off), _at(eng, o, off), _at(eng, w, off)
        y = Dev(eng, shape=(rows * cols + off,))
        eng.rmsnorm(y.ptr + 4 * off, px, pw, rows, cols)
        eng.sync()
        assert_bitexact(y.get()[off:].reshape(rows, cols), oracle.rmsnorm(x, w, 1e-6), "rmsnorm")
        eng.rmsnorm_swishgate(y.ptr + 4 * off, px, po, pw, rows, cols)
        eng.sync()
        assert_bitexact(y.get()[off:].reshape(rows, cols), oracle.rmsnorm_swishgate(x, o, w, 1e-6), "swishgate")
        eng.rmsnorm(px, px, pw, rows, cols)  # in place
        eng.sync()
        assert_bitexact(kx.get()[off:].reshape(rows, cols), oracle.rmsnorm(x, w, 1e-6), "rmsnorm in place")


@pytest.mark.parametrize("cols", [7, 100, 2049, 9000])
def test_swishgate_without_gate(eng, oracle, cols):  # noqa: F811
    """A null gate is the plain norm, on the short-row kernel as on the long-row one."""
    print(f"swishgate without gate cols={cols}", flush=True)
    rng = np.random.default_rng(cols)
    x = rng.standard_normal((3, cols)).astype(np.float32)
    w = (1 + 0.1 * rng.standard_normal(cols)).astype(np.float32)
    dx, dw, y = Dev(eng, x), Dev(eng, w), Dev(eng, shape=(3, cols))
    eng.rmsnorm_swishgate(y.ptr, dx.ptr, None, dw.ptr, 3, cols)
    eng.sync()
    assert_bitexact(y.get(), oracle.rmsnorm(x, w, 1e-6), "norm")


@pytest.mark.parametrize("n", [1, 7, 8, 12, 1016, 1020, 1023, 1024, 1029, 100003])
def test_swiglu_sizes(eng, oracle, n):  # noqa: F811
    rng = np.random.default_rng(n)
    a, b = (rng.standard_normal(n).astype(np.float32) * 4 for _ in range(2))
    for off in (0, 1, 2):
        (ka, pa), (kb, pb) = _at(eng, a, off), _at(eng, b, off)
        out = Dev(eng, shape=(n + off,))
        eng.swiglu(out.ptr + 4 * off, pa, pb, n)
        eng.sync()
        assert_bitexact(out.get()[off:], oracle.swiglu(a, b), f"swiglu n={n}")


def test_swiglu_beyond_a_grid(eng, oracle):  # noqa: F811
    """More elements than 2^32 threads of four (64 GiB, in place): some at the start, past 2^32
    elements, past 2^30 (the largest grid's first sweep) and the tail."""
    n = (1 << 34) + 13
    print(f"swiglu n={n}", flush=True)
    big = Dev(eng, shape=(n,))
    rng = np.random.default_rng(5)
    at = {e: rng.standard_normal(13).astype(np.float32) * 4 for e in (0, (1 << 30) - 5, (1 << 32) + 7, (1 << 34) - 40, n - 13)}
    for e, v in at.items():
        eng._chk(eng.lib.mmf_upload(eng.h, big.ptr + 4 * e, v.ctypes.data, v.nbytes))
    eng.swiglu(big.ptr, big.ptr, big.ptr, n)
    eng.sync()
    for e, v in at.items():
        got = np.empty_like(v)
        eng._chk(eng.lib.mmf_download(eng.h, got.ctypes.data, big.ptr + 4 * e, got.nbytes))
        tail = 5 if e == n - 13 else 0  # n % 8 elements go by the tail rule
        pad = np.concatenate([v[:13 - tail], np.zeros(3 + tail, np.float32)])  # (a multiple of 8: no tail)
        want = oracle.swiglu(pad, pad)[:13 - tail]
        if tail:
            want = np.concatenate([want, oracle.swiglu(v[-tail:], v[-tail:])])
        assert_bitexact(got, want, f"swiglu at {e}")


# the plain loop of few steps and both sides of its lines (by the ring's column groups and transfers,
# and less than a tile); the ring scan (16-byte transfers at D % 8 == 0, aligned; else 4-byte ones)
# over less than, exactly and more than whole 128-step tiles, and partial column groups
@pytest.mark.parametrize("T,D,off", [(14, 256, 0), (15, 256, 0), (20, 257, 0), (21, 257, 0), (20, 64, 1), (21, 64, 1), (24, 2056, 0),
                                     (25, 2056, 0), (28, 2057, 0), (29, 2057, 0), (57, 4097, 0), (58, 4097, 0), (34, 5000, 0),
                                     (35, 5000, 0), (127, 20480, 0), (128, 20480, 0), (1, 16, 0), (5, 2048, 0), (127, 64, 0), (128, 64, 0), (129, 48, 0), (1000, 256, 0),
                                     (1, 1, 0), (63, 100, 0), (64, 17, 0), (65, 250, 0), (300, 129, 0), (200, 64, 1), (700, 2056, 0), (700, 2061, 0)])
def test_scan_sizes(eng, oracle, T, D, off):  # noqa: F811
    print(f"scan T={T} D={D} off={off}", flush=True)
    rng = np.random.default_rng(T * 7 + D)
    i = rng.standard_normal((T, D)).astype(np.float32)
    f = (1 / (1 + np.exp(-rng.standard_normal((T, D))))).astype(np.float32)
    s0 = rng.standard_normal(D).astype(np.float32)
    for state in (None, s0):
        want = oracle.hgrn_scan(i, f, None if state is None else state.copy())
        want, ws = want if isinstance(want, tuple) else (want, None)
        (ki, pi), (kf, pf) = _at(eng, i, off), _at(eng, f, off)
        out = Dev(eng, shape=(T * D + off,))
        st = None if state is None else Dev(eng, state)
        eng.hgrn_scan(out.ptr + 4 * off, pi, pf, T, D, None if st is None else st.ptr)
        eng.sync()
        assert_bitexact(out.get()[off:].reshape(T, D), want, "scan")
        if st is not None:
            assert_bitexact(st.get(), want[-1] if ws is None else ws, "state")
        eng.hgrn_scan(pi, pi, pf, T, D, None)  # in place
        eng.sync()
        if state is None:
            assert_bitexact(ki.get()[off:].reshape(T, D), want, "scan in place")
            kx, px = _at(eng, i, off)
            eng.hgrn_scan(pf, px, pf, T, D, None)  # over the gates
            eng.sync()
            assert_bitexact(kf.get()[off:].reshape(T, D), want, "scan in place of the gates")


@pytest.mark.parametrize("hidden", [100, 250, 1027])
@pytest.mark.parametrize("T", [2, 130, 300])
def test_prefill_odd_hidden(tmp_path, oracle, hidden, T):
    """Prefill whose gate math and time scan run on partial column groups, with SIMD tail elements
    at the end of all T x hidden elements: logits of every position."""
    from matmulfreellmcpu_amd import Engine, make_blob, read_blob
    print(f"prefill hidden={hidden} T={T}", flush=True)
    blob = read_blob(make_blob(str(tmp_path / "m"), vocab=300, hidden=hidden, layers=2, inter=208, seed=hidden,
                               random_norms=True, random_lb=True))
    ids = np.random.default_rng(T).integers(0, 300, T)
    for mode in (0, 1):
        e = Engine(0)
        e.load_blob(blob, mode)
        assert_bitexact(e.forward(ids), oracle.model(blob).forward(ids, mode), f"mode {mode} logits")
        e.close()
