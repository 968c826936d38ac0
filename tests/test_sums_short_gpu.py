"""The MoE plumbing's short forms: sums of 1 to 9 rows (1, 2, 4 or 8 in flight), copies of short rows and one of more words
than a launch's threads, SwiGLU rows of up to two tiles and just past them. Bit for bit numpy's float32 steps in the contract's order; the
SwiGLU's bytes are those of the same rows among many, which test_plumbing_gpu.py holds to a bound."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import torch  # noqa: F401
    from tests import gpu_util
    return gpu_util


@pytest.mark.parametrize("k", range(1, 10))
@pytest.mark.parametrize("dim", [5, 260])
def test_sums(g, k, dim):
    import torch
    rng = np.random.default_rng(k)
    n_tok, rows = 3, 3 * k
    y, sh = (rng.normal(0, 1, s).astype(np.float32) for s in ((rows, dim), (n_tok, dim)))
    where, w = rng.permutation(rows).astype(np.int32), rng.uniform(0, 1, rows).astype(np.float32)
    yd, wh, shd = g.dev(y), g.dev(where), g.dev(sh)
    out = torch.full((n_tok, dim), float("nan"), device="cuda")
    print("sums", dim, k, flush=True)
    g.call("q4x_moe_sum", g.a(yd), g.a(wh), g.a(g.dev(w)), n_tok, k, dim, g.a(shd), g.a(g.dev(np.zeros(n_tok, np.float32))),
           g.a(out), None)
    want, plain = np.zeros((n_tok, dim), np.float32), np.zeros((n_tok, dim), np.float32)
    for j in range(k):
        r = where.reshape(n_tok, k)[:, j]
        want, plain = want + y[r] * w.reshape(n_tok, k)[:, j:j + 1], plain + y[r]
    assert (g.bits(g.host(out)) == g.bits(want + sh * np.float32(0.5))).all()  # (the gate at a zero logit: exactly 1/2)
    g.call("ops_gather_sum_add", g.a(out), g.a(yd), g.a(wh), k, n_tok, dim, g.a(shd), None)
    assert (g.bits(g.host(out)) == g.bits(plain + sh)).all()


@pytest.mark.parametrize("n,dim", [(1, 4), (300, 4), (257, 12), (33, 256), (5, 1020), (5, 1028)])
def test_rows(g, n, dim):
    import torch
    rng = np.random.default_rng(n)
    y, idx = rng.normal(0, 1, (40, dim)).astype(np.float32), rng.integers(0, 40, n).astype(np.int32)
    dst = torch.full((n, dim), float("nan"), device="cuda")
    print("rows", n, dim, flush=True)
    g.call("ops_gather_rows", g.a(dst), g.a(g.dev(y)), g.a(g.dev(idx)), n, dim, None)
    assert (g.bits(g.host(dst)) == g.bits(y[idx])).all()


def test_rows_by_strides(g):
    import torch
    n, dim = (1 << 22) + 3, 1024  # (2^30 + 768 words)
    if torch.cuda.mem_get_info()[0] < 20e9:
        pytest.skip("needs 17 GB of device memory")
    src = torch.randn(7, dim, device="cuda")
    idx = (torch.arange(n, device="cuda") % 7).to(torch.int32)
    dst = torch.empty(n, dim, device="cuda")
    at = torch.tensor([0, 1, (1 << 21) - 1, 1 << 21, (1 << 22) - 1, 1 << 22, n - 1], device="cuda")
    dst[at] = 0.0
    print("rows by strides", flush=True)
    g.call("ops_gather_rows", g.a(dst), g.a(src), g.a(idx), n, dim, None)
    assert torch.equal(dst[at], src[at % 7])
    del dst
    torch.cuda.empty_cache()


@pytest.mark.parametrize("n", [1, 3, 16, 17, 32, 33])
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("ff", [16, 528])
def test_swiglu_rows(g, n, off, ff):
    import torch
    rng = np.random.default_rng(n + ff)
    gg, uu = (rng.normal(0, 2, n * ff).astype(np.float32) for _ in range(2))
    gd, ud = (torch.from_numpy(np.concatenate([np.zeros(off, np.float32), a])).cuda()[off:] for a in (gg, uu))
    idx = rng.integers(-1, n, n).astype(np.int32)
    print("swiglu", n, off, ff, flush=True)

    def rows(ids):
        slots = (len(ids) + 15) // 16 * 16
        y = torch.full((slots * ff,), 7.0, dtype=torch.float16, device="cuda")
        ov = torch.zeros(1, dtype=torch.int32, device="cuda")
        g.call("q4x_swiglu_rows", g.a(gd), g.a(ud), ff, g.a(g.dev(ids)), len(ids), g.a(y), g.a(ov), None)
        return g.host(y).view(np.uint16).reshape(-1, ff // 16, 16, 16).transpose(0, 2, 1, 3).reshape(-1, ff)
    one, many = rows(idx), rows(np.concatenate([idx, np.zeros(64, np.int32)]))
    assert (one[:n] == many[:n]).all() and (one[n:] == np.float16(7.0).view(np.uint16)).all()
