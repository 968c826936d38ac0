"""mmq_group at the edges of its tiles: the last tile's tokens at each count of live results (4, 5, 8, 9, 16), two-tile
passes with a short last tile, fewer blocks than K partitions, rows that leave waves of a workgroup without any, dx and sx
off 16-byte alignment. Bit for bit against the oracle: the contract fixes every sum's order, so the tolerance is zero."""
import numpy as np
import pytest

from libosmos_amd import synth
from oracle import orc
from tests.test_mmq_gpu import g, x8_dev  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("rows,cols,counts", [(80, 256, [4, 5, 0, 8, 9]), (16, 768, [16, 3]), (144, 1536, [17, 24, 31, 1]),
                                              (64, 512, [12, 7])])
def test_tiles(g, rows, cols, counts, off):  # noqa: F811
    import torch
    t = synth.ID["Q4_K"]
    rng = np.random.default_rng(rows + cols)
    ws = [synth.random_blocks(t, rows, cols, 90 + m) for m in range(len(counts))]
    pads = [max(16, (c + 15) // 16 * 16) for c in counts]
    soff = np.concatenate([[0], np.cumsum(pads)[:-1]]).astype(np.uint32)
    slots = int(sum(pads))
    x = rng.normal(0, 1, (slots, cols)).astype(np.float32)
    x8, dx, sx = x8_dev(g, x, np.arange(slots, dtype=np.int32), cols)
    o8, odx, osx = orc.mmq_x8_rows(x, np.arange(slots, dtype=np.int32), cols)
    dx, sx = (torch.cat([torch.zeros(off, device="cuda"), v])[off:] for v in (dx, sx))
    ys = rows + 3
    yoff = (soff * ys).astype(np.uint32)
    y = torch.full((slots * ys,), float("nan"), device="cuda")
    print("mmq_group", rows, cols, counts, off, flush=True)
    g.call("mmq_group", t, g.a(g.table([g.dev(w) for w in ws])), g.a(g.dev(np.array(counts, np.int32))), len(counts),
           max(counts), rows, cols, g.a(x8), g.a(dx), g.a(sx), g.a(g.dev(soff)), g.a(y), g.a(g.dev(yoff)), ys, None)
    yh = g.host(y).reshape(slots, ys)
    for m, c in enumerate(counts):
        for k in range(pads[m]):
            s = int(soff[m]) + k
            if k < c:
                assert (g.bits(yh[s, :rows]) == g.bits(orc.mmq_rows(ws[m], rows, cols, o8, odx, osx, s))).all(), (m, k)
                assert np.isnan(yh[s, rows:]).all()
            else:
                assert np.isnan(yh[s]).all()
