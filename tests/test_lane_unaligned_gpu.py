"""q8_group_tok at one token on a matrix that is only 2-byte aligned: the last row's last bytes are its own (the aligned
copy's bits)."""
import numpy as np
import pytest

from libosmos_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["Q3_K", "IQ1_S", "IQ1_M", "Q4_0", "Q4_K"])
@pytest.mark.parametrize("cols", [1024, 2048, 4096])
def test_one_token_two_byte_offset(name, cols):
    import torch
    from tests import gpu_util as g
    t, rows = synth.ID[name], 24
    w = g.dev((synth.iq_blocks if name.startswith("IQ") else synth.random_blocks)(t, rows, cols, 3)).reshape(-1)
    x = g.dev(np.random.default_rng(4).normal(0, 1, (1, cols)).astype(np.float32))
    q, d = torch.zeros(1, cols, dtype=torch.int8, device="cuda"), torch.zeros(1, cols // 32, device="cuda")
    g.call("q8_round", g.a(x), 1, cols, cols, g.a(q), g.a(d), None)
    out = []
    for off in (0, 2, 6, 14):
        buf = torch.cat([torch.zeros(off, dtype=torch.uint8, device="cuda"), w, torch.zeros(64, dtype=torch.uint8, device="cuda")])
        y = torch.zeros(1, rows, device="cuda")
        g.call("q8_group_tok", t, g.a(g.table([buf[off:]])), g.a(g.dev(np.array([1], np.int32))),
               g.a(g.dev(np.zeros(1, np.int32))), None, 1, 1, rows, cols, g.a(q), g.a(d), g.a(y), rows, None)
        out.append(g.bits(g.host(y)))
    assert all((o == out[0]).all() for o in out[1:])
