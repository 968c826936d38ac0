"""The direct f16 kernels' forms (a launch's size and tokens choose one): each form gives a token the bits it has alone
and, on data where every matrix-core step is exact, the oracle's - at widths of fewer blocks than the K split has classes,
of a partial last round and of several rounds, at the edges of the token tiles, and with matrices of different counts
(none among them) in one launch. The alone bits are within the reference's bound of the float64 sum."""
import numpy as np
import pytest

from libosmos_amd import synth
from oracle import orc
from tests.test_mm_gpu import bound_check, mm_x16, run

pytestmark = pytest.mark.gpu
TYPES = ["Q4_0", "Q3_K", "Q4_K", "IQ2_XXS", "IQ3_XXS", "IQ1_S", "IQ1_M"]
# (row tiles a launch, its largest count): few and many at one, two and four token tiles a workgroup
FORMS = [(3, 16), (2112, 16), (3, 32), (912, 32), (3, 130), (780, 130)]


@pytest.fixture(scope="module")
def g():
    import torch  # noqa: F401
    from tests import gpu_util
    return gpu_util


def group(g, t, w, rows, cols, x16, n_x, tiles, most, seed):
    """the one matrix as tiles / (rows / 16) of one launch's, counts 0 .. most over the first tokens of the n_x: the counts
    and each one's outputs"""
    import torch
    n_mat = tiles * 16 // rows
    cnt = np.random.default_rng(seed).integers(0, most + 1, n_mat).astype(np.int32)
    cnt[:3] = [most, 0, 1][:n_mat]
    cnt = np.minimum(cnt, n_x)
    place = (np.concatenate([[0], np.cumsum(cnt)[:-1]]) * rows).astype(np.uint32)
    y = torch.full((int(cnt.sum()), rows), float("nan"), device="cuda")
    print("mm_group", t, cols, n_mat, most, flush=True)
    g.call("mm_group", t, g.a(g.table([w] * n_mat)), g.a(g.dev(cnt)), n_mat, most, rows, cols, g.a(x16),
           g.a(g.dev(np.zeros(n_mat, np.uint32))), cols, g.a(y), g.a(g.dev(place)), rows, None)
    return cnt, g.host(y)


@pytest.mark.parametrize("name,cols", [(n, c) for n in TYPES for c in (256, 768, 2304)])
def test_forms_agree(g, name, cols):
    t, rows, n = synth.ID[name], 48, 130
    w = synth.iq_blocks(t, rows, cols, 5) if name.startswith("IQ") else synth.random_blocks(t, rows, cols, 5)
    w[0, :2] = 0 if name != "IQ1_M" else w[0, :2]  # a zero scale
    x = np.random.default_rng(6).normal(0, 1, (n, cols)).astype(np.float32)
    one = np.stack([run(g, name, w, rows, cols, mm_x16(g, x[i:i + 1])[0], 1)[0] for i in range(n)])
    bound_check(name, w, rows, cols, x, one)
    x16, _ = mm_x16(g, x)
    for m in (15, 16, 17, 32, 33, 64, 65, 130):
        print("mm_run", name, cols, m, flush=True)
        assert (g.bits(run(g, name, w, rows, cols, x16, m)) == g.bits(one[:m])).all(), m
    wd = g.dev(w)
    for tiles, most in FORMS:
        cnt, y = group(g, t, wd, rows, cols, x16, n, tiles, most, tiles + most)
        assert (g.bits(y) == g.bits(np.concatenate([one[:c] for c in cnt]))).all(), (tiles, most)


@pytest.mark.parametrize("name", TYPES)
def test_forms_order(g, name):
    from tests import mmorder
    t, cols, group_ = synth.ID[name], {"IQ3_XXS": 2048, "Q4_0": 512}.get(name, 1024), True
    w, x, ordered, chain = mmorder.case(name, cols, group_, 11)
    want = orc.mm_rows(t, w, 16, cols, x, group_)
    x16, _ = mm_x16(g, x)
    for tiles, most in FORMS:
        cnt, y = group(g, t, g.dev(w), 16, cols, x16, x.shape[0], tiles, most, 3)
        assert (g.bits(y) == g.bits(np.concatenate([want[:c] for c in cnt]))).all(), (tiles, most)


def test_q4_0_odd_width(g):
    """a Q4_0 width of whole slabs but not whole 256s takes the staged kernel"""
    rows, cols = 32, 320
    w = synth.random_blocks(synth.ID["Q4_0"], rows, cols, 8)
    x = np.random.default_rng(9).normal(0, 1, (20, cols)).astype(np.float32)
    bound_check("Q4_0", w, rows, cols, x, run(g, "Q4_0", w, rows, cols, mm_x16(g, x)[0], 20))
