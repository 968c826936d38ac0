"""The direct f16 kernels where a launch's matrices hold different counts: each matrix runs the body of its own token tiles, and
Q4_0 has a form of its own between the small and the large launches. Each form gives a token the bits it has alone (which
test_mm_direct_gpu.py holds to the oracle's order): no tolerance."""
import numpy as np
import pytest

from libosmos_amd import synth
from tests.test_mm_direct_gpu import TYPES, group
from tests.test_mm_gpu import mm_x16, run

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import torch  # noqa: F401
    from tests import gpu_util
    return gpu_util


@pytest.mark.parametrize("name,cols", [(n, c) for n in TYPES for c in (256, 2304)])
def test_counts(g, name, cols):
    t, rows, n = synth.ID[name], 48, 70
    w = synth.iq_blocks(t, rows, cols, 7) if name.startswith("IQ") else synth.random_blocks(t, rows, cols, 7)
    x = np.random.default_rng(8).normal(0, 1, (n, cols)).astype(np.float32)
    one = np.concatenate([run(g, name, w, rows, cols, mm_x16(g, x[i:i + 1])[0], 1) for i in range(n)])
    x16, _ = mm_x16(g, x)
    wd = g.dev(w)
    # (row tiles, most): Q4_0's middle form at one, two and four tiles, then large launches of two passes
    for tiles, most in [(330, 16), (801, 32), (450, 70), (900, 40), (900, 70)]:
        cnt, y = group(g, t, wd, rows, cols, x16, n, tiles, most, tiles + most)
        assert (g.bits(y) == g.bits(np.concatenate([one[:c] for c in cnt]))).all(), (tiles, most)


@pytest.mark.parametrize("name", TYPES)
def test_one_large_matrix(g, name):
    """one matrix of 800 row tiles (the same 16 rows again): the large form without a body by count, a last pass of 6"""
    t, cols, n = synth.ID[name], 256, 70
    w = synth.iq_blocks(t, 16, cols, 9) if name.startswith("IQ") else synth.random_blocks(t, 16, cols, 9)
    x16, _ = mm_x16(g, np.random.default_rng(10).normal(0, 1, (n, cols)).astype(np.float32))
    print("mm_run", name, flush=True)
    y = run(g, name, np.concatenate([w] * 800), 16 * 800, cols, x16, n)
    few = run(g, name, w, 16, cols, x16, n)
    assert (g.bits(y.reshape(n, 800, 16)) == g.bits(few)[:, None, :]).all()
