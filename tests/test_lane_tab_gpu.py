"""q8_gate_up and q8_group_tok over pointer tables of several matrices (the staged tiles) against the same entries launched one
at a time (the per-row kernels, which test_lane_gpu.py holds to the oracle): every lane type at the widths of both lane
counts, entries of 0 to 8 tokens through xin and win, one matrix at a 2-byte offset, and row counts that do and do not
fill whole workgroups."""
import math

import numpy as np
import pytest

from libosmos_amd import synth

pytestmark = pytest.mark.gpu
TYPES = ["IQ2_XXS", "IQ2_XS", "IQ1_M", "IQ1_S", "IQ2_S", "IQ3_XXS", "Q2_K", "Q4_0", "Q4_K", "Q3_K"]


@pytest.fixture(scope="module")
def g():
    import torch  # noqa: F401
    from tests import gpu_util
    return gpu_util


@pytest.mark.parametrize("name", TYPES)
@pytest.mark.parametrize("cols,rows", [(512, 64), (1024, 48), (2048, 32), (4096, 16), (768, 32)])
@pytest.mark.parametrize("most", [1, 3, 8])
def test_entries_agree(g, name, cols, rows, most):
    import torch
    t, n_mat = synth.ID[name], 6
    rng = np.random.default_rng(cols + most)
    mk = lambda s: (synth.iq_blocks if name.startswith("IQ") else synth.random_blocks)(t, rows, cols, s)  # noqa: E731
    mats = [[g.dev(mk(10 * j + i)) for i in range(n_mat)] for j in range(2)]
    for j in range(2):  # a matrix that is only 2-byte aligned
        w = mats[j][1].reshape(-1)
        mats[j][1] = torch.cat([torch.zeros(2, dtype=torch.uint8, device="cuda"), w])[2:]
    cnt = np.minimum([most, 1, 0, most, 2, 5], most).astype(np.int32)
    xrow = np.concatenate([[0], np.cumsum(cnt)[:-1]]).astype(np.int32)
    n, n_x = int(cnt.sum()), 5
    xin, win = rng.integers(0, n_x, n).astype(np.int32), rng.permutation(n).astype(np.int32)
    x = g.dev(rng.normal(0, 1, (n_x, cols)).astype(np.float32))
    q, d = torch.zeros(n_x, cols, dtype=torch.int8, device="cuda"), torch.zeros(n_x, cols // 32, device="cuda")
    g.call("q8_round", g.a(x), n_x, cols, cols, g.a(q), g.a(d), None)
    scale = g.dev(rng.uniform(0.1, 1, n).astype(np.float32))
    xi, wi, ct, xr = (g.dev(v) for v in (xin, win, cnt, xrow))
    print("tab", name, cols, rows, most, flush=True)

    def both(sel):
        out = [torch.full((n, rows), 7.0, device="cuda") for _ in range(2)]
        for s in sel:
            tab = [g.table(mats[j][s]) for j in range(2)]
            c, r, k = ct[s].contiguous(), xr[s].contiguous(), len(mats[0][s])
            g.call("q8_gate_up", t, g.a(tab[0]), g.a(tab[1]), g.a(c), g.a(r), g.a(xi), g.a(wi), k, most, rows, cols, g.a(q),
                   g.a(d), g.a(scale), math.inf, g.a(out[0]), rows, None)
            g.call("q8_group_tok", t, g.a(tab[0]), g.a(c), g.a(r), g.a(xi), k, most, rows, cols, g.a(q), g.a(d),
                   g.a(out[1]), rows, None)
        return [g.bits(g.host(o)) for o in out]
    alone = both([slice(i, i + 1) for i in range(n_mat)])
    for a, b in zip(both([slice(0, n_mat)]), alone):
        assert (a == b).all()
