"""The few-row float GEMM at the edges of its row and output blocks, its weight chunks and its hand
over to the matrix cores, against the CPU restatement, bit for bit."""
import numpy as np
import pytest

from conftest import assert_bitexact
from test_gpu_parity import Dev, eng  # noqa: F401  (module fixture)

pytestmark = pytest.mark.gpu

# (rows, K, N): one and several outputs per lane and rows per block, chains of less than, exactly
# and more than the 4- and 8-word weight chunks, every tail length, partial output sets, and both
# sides of the lines to the matrix cores (100000 outputs per round of tiles; fewer for short and long chains)
SHAPES = [(1, 7, 1), (1, 8, 9), (2, 129, 24), (3, 514, 31), (4, 523, 40), (5, 1036, 63), (7, 1029, 65), (9, 1150, 1000),
          (15, 1023, 2049), (16, 2048, 2560), (17, 700, 5290), (18, 64, 5001), (64, 1024, 1406), (64, 1024, 1564),
          (400, 100, 225), (3, 6912, 11000), (1, 9000, 70), (2, 18000, 20)]
# both sides of each line between the forms (rows per block and outputs per lane: 65536, 49152 and
# 20480 outputs per row group, a quarter or a sixth of the rows idle, two blocks' rows in LDS) and
# to the matrix cores over several rounds of tiles
FORMS = [(1, 33, 65521), (1, 33, 65537), (2, 33, 20465), (2, 33, 20481), (2, 33, 49157), (3, 40, 49157), (4, 40, 49141),
         (4, 40, 49157), (5, 40, 25000), (6, 41, 16400), (7, 40, 24600), (7, 520, 5130), (8, 40, 24570), (8, 40, 24580),
         (9, 40, 4100), (13, 600, 13000), (9, 600, 26000), (9, 600, 26003), (12, 521, 26000), (16, 520, 26000),
         (12, 5150, 4100), (4, 5200, 25000), (2, 10300, 24600), (1, 10300, 65540)]


@pytest.mark.parametrize("rows,K,N", SHAPES + FORMS)
def test_float_rows(eng, oracle, rows, K, N):  # noqa: F811
    print(f"float rows={rows} K={K} N={N}", flush=True)
    rng = np.random.default_rng(rows + K + N)
    x = (rng.standard_normal((rows, K)) * 2).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(K)).astype(np.float32)
    wq = rng.integers(-1, 2, (N, K)).astype(np.int8)
    sw = float(np.float32(1.0 / 0.0157))
    pid = eng.register_proj(wq, sw, nw)
    dx, dout = Dev(eng, x), Dev(eng, shape=(rows, N))
    eng.bitlinear(pid, dx.ptr, dout.ptr, rows, mode=0)
    eng.sync()
    assert_bitexact(dout.get(), oracle.bitlinear(x, nw, wq, sw, 1e-6, 0)["out"], "out")
    eng.proj_release(pid)


@pytest.mark.parametrize("name", ["odd", "small", "tall", "wide"])
@pytest.mark.parametrize("T", [1, 2, 9, 30, 90])
def test_float_prompts(blobs, oracle, name, T):
    """Short prompts through every GEMM kind (store, residual, swiglu pair): all logits."""
    from matmulfreellmcpu_amd import Engine, read_blob
    print(f"float prompt blob={name} T={T}", flush=True)
    blob = read_blob(blobs(name))
    ids = np.random.default_rng(T).integers(0, blob.config.vocab_size, T)
    e = Engine(0)
    e.load_blob(blob, 0)
    assert_bitexact(e.forward(ids), oracle.model(blob).forward(ids, 0), "logits")
    e.close()
