"""Serving steps on the fused decode kernels (a grid of output blocks by streams), on both sides
of the stream counts where the row path takes over, against the CPU restatement, bit for bit."""
import numpy as np
import pytest

from conftest import assert_bitexact

pytestmark = pytest.mark.gpu

FLOAT, FIXED, INT8 = 0, 1, 2

# (blob, streams): one stream (with SIMD tails on "odd"), the lm_head's switch to the row kernels
# (4 / 5; 2 / 3 for the integer modes beyond vocabulary 8192), and the last fused and first row step
# of each width and mode
CASES = [("odd", 1, FLOAT), ("odd", 1, FIXED), ("odd", 1, INT8), ("odd", 2, FLOAT),
         ("small", 1, FLOAT), ("small", 4, FIXED), ("small", 5, INT8), ("small", 49, FLOAT), ("small", 37, FIXED),
         ("wide", 12, FLOAT), ("wide", 13, FLOAT), ("wide", 9, FIXED), ("wide", 10, INT8),
         ("h2048", 1, FIXED), ("h2048", 2, INT8), ("h2048", 3, INT8), ("h2048", 3, FIXED), ("h2048", 4, FIXED), ("h2048", 3, FLOAT), ("h2048", 4, FLOAT),
         ("h2560", 2, FIXED), ("h2560", 3, INT8), ("h2560", 2, FLOAT), ("h2560", 1, INT8)]


@pytest.mark.parametrize("name,streams,mode", CASES)
def test_step_matches_oracle(blobs, oracle, name, streams, mode):
    """Ids of every stream, the last step's argmax against its logits, and the final states;
    then the same context again with one stream fewer (other strides in the kept buffers)."""
    from matmulfreellmcpu_amd import Engine, read_blob
    print(f"step blob={name} streams={streams} mode={mode}", flush=True)
    blob = read_blob(blobs(name))
    om = oracle.model(blob)
    rng = np.random.default_rng(streams + 100 * mode)
    new = 4
    e = Engine(0)
    e.load_blob(blob, mode)
    for B in (streams, streams - 1):
        if B == 0:
            break
        prompts = [rng.integers(0, blob.config.vocab_size, 1 + (3 * b) % 5) for b in range(B)]
        want, wst = om.generate_serve(prompts, new, mode, want_state=True)
        e.reset(B)
        got = [list(p) for p in prompts]
        first = e.prefill_streams(prompts)
        for b in range(B):
            got[b].append(int(first[b]))
        for k in range(new - 1):
            am, lg = e.step([g[-1] for g in got], want_logits=True)
            np.testing.assert_array_equal(am, lg.argmax(1))
            for b in range(B):
                got[b].append(int(am[b]))
        for b in range(B):
            np.testing.assert_array_equal(np.array(got[b]), want[b])
        assert_bitexact(e.state(), wst, f"states of {B} streams")
    e.close()
