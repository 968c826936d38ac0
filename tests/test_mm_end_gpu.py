"""the staged f16 kernel on a matrix that ends where its memory does, at widths that leave its last round short: the bits are
those of the matrix in the middle of the buffer, a whole number of 2 MiB pages. What the threads past the staged words read is
never stored and shows in no bits: test_mm_stage.py checks that it lies inside the matrix."""
import numpy as np
import pytest

from libosmos_amd import synth
from tests.test_mm_gpu import mm_x16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import torch  # noqa: F401
    from tests import gpu_util
    return gpu_util


# rounds of 512 (Q2_K, IQ2_XS, IQ2_S), 1024 (Q6_K, Q8_0) and 256 values (Q4_0)
@pytest.mark.parametrize("name,cols", [("Q2_K", 768), ("IQ2_XS", 768), ("IQ2_S", 1792), ("Q6_K", 2304), ("Q8_0", 2176),
                                       ("Q4_0", 320)])
@pytest.mark.parametrize("n", [5, 40])
def test_last_row(g, name, cols, n):
    import torch
    t, rows, page = synth.ID[name], 80, 1 << 21
    w = synth.iq_blocks(t, rows, cols, 8) if name.startswith("IQ") else synth.random_blocks(t, rows, cols, 8)
    raw = torch.from_numpy(np.ascontiguousarray(w).reshape(-1).view(np.uint8)).cuda()
    x16, _ = mm_x16(g, np.random.default_rng(9).normal(0, 1, (n, cols)).astype(np.float32))
    buf = torch.zeros(16 * page, dtype=torch.uint8, device="cuda")
    out = []
    for at in (page, buf.numel() - raw.numel()):
        at -= at % 2
        buf[at:at + raw.numel()] = raw
        y = torch.full((n, rows), float("nan"), device="cuda")
        print("mm_run", name, cols, n, at, flush=True)
        g.call("mm_run", t, g.a(buf[at:]), rows, cols, g.a(x16), n, g.a(y), rows, None)
        out.append(g.host(y).copy())
    assert not np.isnan(out[0]).any() and (g.bits(out[0]) == g.bits(out[1])).all()
