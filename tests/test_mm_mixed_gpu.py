"""mm_group of IQ2_XS and IQ2_S in launches tall enough for four row tiles a wave, whose decode rounds its products by another
instruction than the small launches': the same bits as the matrix alone, at one and two token tiles and on both staging word
sizes (a row of whole 4-byte words or not), with zero, negative, subnormal and infinite block scales among the rows."""
import numpy as np
import pytest

from libosmos_amd import synth
from tests.test_mm_direct_gpu import group
from tests.test_mm_gpu import mm_x16, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["IQ2_XS", "IQ2_S"])
@pytest.mark.parametrize("cols", [512, 768])
def test_tall(name, cols):
    from tests import gpu_util as g
    t, rows, n = synth.ID[name], 64, 40
    w = synth.iq_blocks(t, rows, cols, 3)
    for r, d in enumerate((0x0000, 0x8000, 0xB123, 0x0001, 0x8001, 0x7BFF, 0x7C00, 0xFC00)):
        w[r, :2] = np.array([d], np.uint16).view(np.uint8)
    x16, _ = mm_x16(g, np.abs(np.random.default_rng(4).normal(0, 1, (n, cols))).astype(np.float32))
    one = run(g, name, w, rows, cols, x16, n)
    for tiles, most in [(4096, 16), (4096, 32), (4096, 40)]:
        cnt, y = group(g, t, g.dev(w), rows, cols, x16, n, tiles, most, tiles + most)
        want = np.concatenate([one[:c] for c in cnt])
        nan = np.isnan(want)
        assert (np.isnan(y) == nan).all() and (g.bits(y)[~nan] == g.bits(want)[~nan]).all(), (tiles, most)
