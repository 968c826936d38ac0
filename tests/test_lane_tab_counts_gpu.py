"""q8_gate_up and q8_group_tok over a routed step's table (more entries than four times their most tokens: the staged tiles'
side of the rule) with every count of 0 .. 8 among its entries, so that every pass size of the tiles (1 to 4 tokens at 16
lanes, 1 and 2 at 32) is a first and a last pass. The bits are those of the same entries launched one at a time (the per-row
kernels, which test_lane_gpu.py holds to the oracle): the contract fixes every sum's order, so the tolerance is zero."""
import math

import numpy as np
import pytest

from libosmos_amd import synth

pytestmark = pytest.mark.gpu
TYPES = ["IQ2_XXS", "IQ2_XS", "IQ1_M", "IQ1_S", "IQ2_S", "IQ3_XXS", "Q2_K", "Q4_0", "Q4_K", "Q3_K"]


@pytest.mark.parametrize("name", TYPES)
@pytest.mark.parametrize("cols", [512, 1024, 2048, 4096])
@pytest.mark.parametrize("most", [3, 8])
def test_counts(name, cols, most):
    import torch
    from tests import gpu_util as g
    t, n_mat = synth.ID[name], 4 * most + 4
    rng = np.random.default_rng(cols + most)
    cnt = (np.arange(n_mat) % (most + 1)).astype(np.int32)
    xrow = np.concatenate([[0], np.cumsum(cnt)[:-1]]).astype(np.int32)
    n = int(cnt.sum())
    x = g.dev(rng.normal(0, 1, (n, cols)).astype(np.float32))
    q, d = torch.zeros(n, cols, dtype=torch.int8, device="cuda"), torch.zeros(n, cols // 32, device="cuda")
    g.call("q8_round", g.a(x), n, cols, cols, g.a(q), g.a(d), None)
    scale, ct, xr = (g.dev(v) for v in (rng.uniform(0.1, 1, n).astype(np.float32), cnt, xrow))
    for gate_up, rows in ((True, 16), (False, 512)):
        mk = synth.iq_blocks if name.startswith("IQ") else synth.random_blocks
        mats = [[g.dev(mk(t, rows, cols, 10 * j + i)) for i in range(4)] * (n_mat // 4) for j in range(1 + gate_up)]
        out = []
        for sel in ([slice(0, n_mat)], [slice(i, i + 1) for i in range(n_mat)]):
            y = torch.full((n, rows), 7.0, device="cuda")
            for s in sel:
                tab = [g.table(m[s]) for m in mats]
                c, r, k = ct[s].contiguous(), xr[s].contiguous(), len(mats[0][s])
                print("counts", name, cols, most, gate_up, k, flush=True)
                if gate_up:
                    g.call("q8_gate_up", t, g.a(tab[0]), g.a(tab[1]), g.a(c), g.a(r), None, None, k, most, rows, cols, g.a(q),
                           g.a(d), g.a(scale), math.inf, g.a(y), rows, None)
                else:
                    g.call("q8_group_tok", t, g.a(tab[0]), g.a(c), g.a(r), None, k, most, rows, cols, g.a(q), g.a(d), g.a(y),
                           rows, None)
            out.append(g.bits(g.host(y)))
        assert (out[0] == out[1]).all()
