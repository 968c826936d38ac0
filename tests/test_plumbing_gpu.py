"""The MoE plumbing's table and row kernels at the edges of their forms: osmos_lane_tables against a host restatement from
one pick to the most, and the sums and copies bit for bit against numpy's float32 steps in the contract's order, with rows
that take the 16-byte form and rows that do not (odd lengths, a 4-byte offset)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import torch  # noqa: F401
    from tests import gpu_util
    return gpu_util


@pytest.mark.parametrize("n_tok,k,n_exp", [(1, 1, 1), (1, 32, 1024), (4, 10, 512), (8, 9, 257), (64, 10, 512), (33, 7, 40),
                                           (300, 3, 4), (128, 32, 64), (4096, 1, 3)])
def test_lane_tables(g, n_tok, k, n_exp):
    import torch
    rng = np.random.default_rng(n_tok + k)
    ids = np.stack([rng.choice(n_exp, k, replace=False) for _ in range(n_tok)]).astype(np.int32)
    n = n_tok * k
    flat = ids.reshape(-1)
    base, size = [0x1000000, 0x2000000, 0x3000000], [4096, 512, 96]
    i32 = lambda: torch.full((n,), -7, dtype=torch.int32, device="cuda")  # noqa: E731
    tok, pair, cnt, xrow, order = i32(), i32(), i32(), i32(), i32()
    ptr = [torch.zeros(n, dtype=torch.int64, device="cuda") for _ in range(3)]
    print("lane_tables", n_tok, k, n_exp, flush=True)
    g.call("osmos_lane_tables", g.a(g.dev(flat)), n_tok, k, n_exp, (ctypes.c_void_p * 3)(*base), (ctypes.c_uint64 * 3)(*size),
           g.a(tok), g.a(pair), g.a(cnt), g.a(xrow), *[g.a(p) for p in ptr], g.a(order), None)
    by = np.argsort(flat, kind="stable")
    assert (g.host(pair) == by).all() and (g.host(tok) == by // k).all()
    row = np.empty(n, np.int64)
    row[by] = np.arange(n)
    assert (g.host(order).reshape(n_tok, k) == np.sort(row.reshape(n_tok, k), axis=1)).all()
    want = []
    first = 0
    for e in range(n_exp):
        c = int((flat == e).sum())
        want += [(min(8, c - p), first + p, e) for p in range(0, c, 8)]
        first += c
    gc, gx, gp = g.host(cnt), g.host(xrow), [g.host(p) for p in ptr]
    assert [(int(gc[i]), int(gx[i])) for i in range(len(want))] == [w[:2] for w in want]
    for j in range(3):
        assert (gp[j][:len(want)] == [base[j] + w[2] * size[j] for w in want]).all()
    assert (gc[len(want):] == 0).all()


@pytest.mark.parametrize("dim,off", [(256, 0), (1028, 0), (7168, 0), (1028, 1), (30, 0), (7, 0)])
@pytest.mark.parametrize("k", [1, 8, 13, 32])
def test_sums_and_rows(g, dim, off, k):
    import torch
    rng = np.random.default_rng(dim + k)
    n_tok, rows = 5, 5 * k
    buf = lambda a: torch.from_numpy(np.concatenate([np.zeros(off, np.float32), a.reshape(-1)])).cuda()[off:]  # noqa: E731
    y, sh = (rng.normal(0, 1, s).astype(np.float32) for s in ((rows, dim), (n_tok, dim)))
    where = rng.permutation(rows).astype(np.int32)
    w = rng.uniform(0, 1, rows).astype(np.float32)
    yd, shd, out = buf(y), buf(sh), buf(np.zeros((n_tok, dim), np.float32))
    print("sums", dim, off, k, flush=True)
    # the gate's exponential is the device's: at a zero logit it is exactly 1/2
    g.call("q4x_moe_sum", g.a(yd), g.a(g.dev(where)), g.a(g.dev(w)), n_tok, k, dim, g.a(shd),
           g.a(g.dev(np.zeros(n_tok, np.float32))), g.a(out), None)
    want, plain = np.zeros((n_tok, dim), np.float32), np.zeros((n_tok, dim), np.float32)
    for j in range(k):
        r = where.reshape(n_tok, k)[:, j]
        want = want + y[r] * w.reshape(n_tok, k)[:, j:j + 1]
        plain = plain + y[r]
    assert (g.bits(g.host(out).reshape(n_tok, dim)) == g.bits(want + sh * np.float32(0.5))).all()
    g.call("ops_gather_sum_add", g.a(out), g.a(yd), g.a(g.dev(where)), k, n_tok, dim, g.a(shd), None)
    assert (g.bits(g.host(out).reshape(n_tok, dim)) == g.bits(plain + sh)).all()
    dst = buf(np.zeros((rows, dim), np.float32))
    g.call("ops_gather_rows", g.a(dst), g.a(yd), g.a(g.dev(where)), rows, dim, None)
    assert (g.bits(g.host(dst).reshape(rows, dim)) == g.bits(y[where])).all()


@pytest.mark.parametrize("n,cols,xs,off", [(1, 16, 16, 0), (16, 48, 48, 0), (17, 256, 260, 0), (33, 48, 51, 0), (40, 96, 96, 1)])
def test_x16_forms(g, n, cols, xs, off):
    """mm_x16's bytes for aligned and unaligned rows, and q4x_swiglu_rows' aligned and unaligned forms the same bytes (the
    tail slots of the last tile untouched)"""
    import torch
    from tests.test_mm_gpu import x16_layout
    rng = np.random.default_rng(n + cols)
    x = rng.normal(0, 1, (n, xs)).astype(np.float32)
    flat = torch.from_numpy(np.concatenate([np.zeros(off, np.float32), x.reshape(-1)])).cuda()
    x16 = torch.full(((n + 15) // 16 * 16 * cols,), float("nan"), dtype=torch.float16, device="cuda")
    print("x16", n, cols, xs, off, flush=True)
    g.call("mm_x16", g.a(flat[off:]), xs, n, cols, g.a(x16), None, None)
    assert (g.host(x16).view(np.uint16) == x16_layout(np.ascontiguousarray(x[:, :cols])).view(np.uint16)).all()
    gg, uu = (rng.normal(0, 2, n * cols).astype(np.float32) for _ in range(2))
    idx = rng.integers(-1, n, n).astype(np.int32)
    out = []
    for o in (0, 1):
        gd, ud = (torch.from_numpy(np.concatenate([np.zeros(o, np.float32), a])).cuda()[o:] for a in (gg, uu))
        y = torch.full(((n + 15) // 16 * 16 * cols,), 7.0, dtype=torch.float16, device="cuda")
        ov = torch.zeros(1, dtype=torch.int32, device="cuda")
        g.call("q4x_swiglu_rows", g.a(gd), g.a(ud), cols, g.a(g.dev(idx)), n, g.a(y), g.a(ov), None)
        out.append(g.host(y).astype(np.float32).reshape(-1, cols // 16, 16, 16).transpose(0, 2, 1, 3).reshape(-1, cols))
    assert (out[0] == out[1]).all() and (out[0][n:] == 7.0).all()
    r = np.where(idx[:, None] >= 0, gg.reshape(n, cols)[idx].astype(np.float64), 0.0)
    want = r / (1 + np.exp(-r)) * uu.reshape(n, cols)[idx]
    assert np.allclose(out[0][:n], want, rtol=2.0 ** -10, atol=2.0 ** -24)
