"""mm_run and mm_group on blocks whose f16 scale is infinite: a value is the decoder's (infinite for every sub-scale, 0 among
them), not 0 times infinity. Every value of a row is made the same sign and x positive, so that a row's exact sum is that
infinity whatever the order: no tolerance. quant_dequant gives the values that are expected."""
import numpy as np
import pytest

from libosmos_amd import synth
from oracle import orc

pytestmark = pytest.mark.gpu


def iq1_entry(name):
    """an IQ1 grid entry with no -1: by the decoder's values at a finite scale"""
    for i in range(2048):
        if (orc.dequant(synth.ID[name], block(name, 0x3C00, 0, i), 256) > 0).all():
            return i
    raise AssertionError("no entry of zeros and ones")


def block(name, d, s, entry=0):
    """a block of one grid entry, no signs (IQ1: a positive delta), the sub-scale s everywhere and the f16 bits d"""
    d2 = np.array([d], np.uint16).view(np.uint8)
    if name == "IQ2_XXS":
        b = np.concatenate([d2, np.tile(np.array([0, s << 28], np.uint32), 8).view(np.uint8)])
    elif name == "IQ3_XXS":
        b = np.concatenate([d2, np.zeros(64, np.uint8), np.full(8, s << 28, np.uint32).view(np.uint8)])
    elif name == "IQ1_S":
        qh = sum((entry >> 8) << (3 * i) for i in range(4)) | (s & 7) << 12
        b = np.concatenate([d2, np.full(32, entry & 255, np.uint8), np.full(8, qh, np.uint16).view(np.uint8)])
    else:  # IQ1_M: the scale's nibbles on top of the four scale words
        sc = sum((s & 7) << (3 * i) for i in range(4))
        words = np.array([sc | ((d >> (4 * i)) & 15) << 12 for i in range(4)], np.uint16)
        b = np.concatenate([np.full(32, entry & 255, np.uint8), np.full(16, (entry >> 8) * 17, np.uint8), words.view(np.uint8)])
    return b.reshape(1, -1)


@pytest.mark.parametrize("name", ["IQ2_XXS", "IQ3_XXS", "IQ1_S", "IQ1_M"])
@pytest.mark.parametrize("n", [1, 40])
def test_infinite_scale(name, n):
    from tests import gpu_util as g
    from tests.test_mm_gpu import mm_x16
    import torch
    t, rows, cols = synth.ID[name], 16, 512
    entry = iq1_entry(name) if name.startswith("IQ1") else 0
    # rows: both infinities and a finite scale, each at sub-scales 0 .. 4 (and the last row's second block finite)
    w = [np.concatenate([block(name, (0x7C00, 0xFC00, 0x2C00)[r % 3], r // 3, entry), block(name, 0x2C00, 1, entry)], 1)
         for r in range(rows)]
    w = np.concatenate(w)
    vals = np.stack([orc.dequant(t, w[r:r + 1], cols) for r in range(rows)])
    want = vals.astype(np.float64).sum(1)
    assert np.isposinf(want[0]) and np.isneginf(want[1]) and np.isfinite(want[2])
    wd, x16 = g.dev(w), mm_x16(g, np.ones((n, cols), np.float32))[0]
    y = [torch.full((n, rows), float("nan"), device="cuda") for _ in range(2)]
    print("infinite", name, n, flush=True)
    g.call("mm_run", t, g.a(wd), rows, cols, g.a(x16), n, g.a(y[0]), rows, None)
    g.call("mm_group", t, g.a(g.table([wd])), g.a(g.dev(np.array([n], np.int32))), 1, n, rows, cols, g.a(x16),
           g.a(g.dev(np.zeros(1, np.uint32))), cols, g.a(y[1]), g.a(g.dev(np.zeros(1, np.uint32))), rows, None)
    big = np.isinf(want)
    for out in y:
        h = g.host(out)
        assert (h[:, big] == want[big]).all()
        assert np.allclose(h[:, ~big], want[~big], rtol=2.0 ** -10)  # (f16 weights: half a unit in the last place)
