"""The work that users of this library have it do, as cases to be timed: each a call sequence through the public C ABI
(libosmos_amd.capi) or libosmos_amd.layer on seeded synthetic inputs, over the library's range of sizes, batches and
GGUF types.

Families (a case's "kind"):
  mv      the decode's dense projections at 1 .. 8 tokens: mv_strided over a stack of layers' matrices, launched eagerly
  layer   routed MoE layers at decode batches: LaneLayer.forward (osmos_lane_layer), a stack of layers captured in a graph
          (the decode's launch pattern) or launched eagerly
  engine  the same layer by the engine's own sequence: osmos_lane_tables, q8_round, q8_gate_up, q8_round, q8_group_tok,
          ops_gather_sum_add
  mm      a prompt batch's dense projections: mm_x16 once, then mm_run for each matrix that reads the same input
  moe     a prompt batch's routed experts on the f16 units: q4x_route, q4x_expert_tiles, mm_x16_rows, mm_group (gate, up),
          q4x_swiglu_rows, mm_group (down), q4x_moe_sum
  mmq     the experts' down projection of a prompt batch on the int8 units: mmq_x8_rows, mmq_group
  group   the experts' gate projection of a prompt batch under the lane contract: ops_gather_rows, q8_round,
          osmos_lane_group
  dequant a matrix decoded to f32 or f16: quant_dequant, quant_dequant_f16

Weights are random GGUF blocks whose scales give values of about 0.02 rms (a trained matrix's), activations N(0, 1),
routing uniform at decode and Zipf(1.1)-loaded for prompts.
"""
import ctypes
import math
import os
import re

import numpy as np
import torch

from libosmos_amd import capi
from libosmos_amd.layer import LaneLayer

# name -> (type id, values a block, bytes a block, the rms of a value over the block's f16 scale)
TYPES = {"Q4_0": (2, 32, 18, 4.6), "Q3_K": (11, 256, 110, 42.0), "Q4_K": (12, 256, 144, 325.0),
         "IQ2_XXS": (16, 256, 66, 53.0), "IQ3_XXS": (18, 256, 98, 150.0), "IQ1_S": (19, 256, 50, 7.4),
         "IQ1_M": (29, 256, 56, 7.4)}
SCALE_AT = {"Q4_0": [0], "Q3_K": [108], "Q4_K": [0, 2], "IQ2_XXS": [0], "IQ3_XXS": [0], "IQ1_S": [0]}
LANE = ["IQ3_XXS", "IQ2_XXS", "IQ1_S", "IQ1_M"]  # the expert types of the routed layers
WRMS = 0.02


def row_bytes(name, cols):
    return cols // TYPES[name][1] * TYPES[name][2]


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # one token through a stack of 16 layers' projections, one eager call each: the smallest launches there are
        dict(name="mv q4_0 1 token", kind="mv", type="Q4_0", rows=8192, cols=2048, n=1, layers=16),
        # a small odd batch of decoding sequences through the same kind of stack
        dict(name="mv q3_k 7 tokens", kind="mv", type="Q3_K", rows=6144, cols=2048, n=7, layers=12),
        # the headline: one token through 512-expert layers, as a captured graph
        dict(name="layer iq3_xxs 1 token", kind="layer", type="IQ3_XXS", dim=2048, ff=512, experts=512, k=10, n=1,
             layers=6, graph=True),
        # a serving batch through the same layer
        dict(name="layer iq3_xxs 32 tokens", kind="layer", type="IQ3_XXS", dim=2048, ff=512, experts=512, k=10, n=32,
             layers=1, graph=False),
        # a few sequences through a wide layer of very small types, a shared expert always picked
        dict(name="layer iq1_s 3 tokens", kind="layer", type="IQ1_S", dim=7168, ff=2048, experts=257, k=9, n=3,
             layers=1, graph=False),
        # the engine's own sequence of calls for a decode step of four sequences, as a captured graph
        dict(name="engine iq3_xxs 4 tokens", kind="engine", type="IQ3_XXS", dim=2048, ff=512, experts=512, k=10, n=4,
             layers=2, graph=True),
        # a short prompt (or a large decode batch): three projections that read one input
        dict(name="mm q4_k 64 tokens", kind="mm", type="Q4_K", rows=6144, cols=2048, n=64, mats=3),
        # a long ragged prompt, near the most tokens of one call
        dict(name="mm q4_k 1999 tokens", kind="mm", type="Q4_K", rows=7168, cols=2048, n=1999, mats=1),
        # a prompt's whole routed layer on the f16 units, from the router's logits to the tokens' sums
        dict(name="moe iq2_xxs 512 tokens", kind="moe", type="IQ2_XXS", down="Q4_K", dim=7168, ff=2048, experts=256, k=8,
             n=512),
        # the same prompt's down projection on the int8 units
        dict(name="mmq q4_k 512 tokens", kind="mmq", type="Q4_K", rows=7168, cols=2048, experts=256, k=8, n=512),
        # the same prompt's gate projection with the bits of the decode's lane
        dict(name="group iq2_xxs 512 tokens", kind="group", type="IQ2_XXS", rows=2048, cols=7168, experts=256, k=8,
             n=512),
        # a matrix decoded for a library product or a conversion
        dict(name="dequant iq3_xxs f16", kind="dequant", type="IQ3_XXS", rows=7168, cols=2048, f16=True),
    ]


def _log(rng, lo, hi, step=1):
    """a multiple of `step` in [lo, hi], spread over the logarithm"""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi, max(lo, round(v / step) * step)))


def draw(rng):
    kind = rng.choice(["mv", "layer", "engine", "mm", "moe", "mmq", "group", "dequant"])
    if kind == "mv":
        return dict(kind=kind, type=rng.choice(["Q4_0", "Q4_K", "Q3_K", "IQ3_XXS", "IQ2_XXS"]),
                    rows=_log(rng, 512, 8192, 8), cols=_log(rng, 512, 8192, 256), n=rng.randint(1, 8), layers=8)
    if kind in ("layer", "engine"):
        most = 64 if kind == "layer" else 8
        if rng.random() < 0.5:
            return dict(kind=kind, type=rng.choice(LANE), dim=2048, ff=512, experts=512, k=10, n=_log(rng, 1, most),
                        layers=2, graph=rng.random() < 0.5)
        return dict(kind=kind, type=rng.choice(LANE), dim=7168, ff=2048, experts=257, k=9, n=_log(rng, 1, 8), layers=1,
                    graph=rng.random() < 0.5)
    if kind == "mm":
        return dict(kind=kind, type=rng.choice(list(TYPES)), rows=_log(rng, 512, 8192, 16), cols=_log(rng, 512, 7168, 256),
                    n=_log(rng, 9, 2048), mats=rng.randint(1, 3))
    if kind == "moe":
        t, d = rng.choice([("IQ2_XXS", "Q4_K"), ("IQ3_XXS", "IQ3_XXS"), ("Q4_K", "Q4_K"), ("IQ1_S", "IQ1_M")])
        return dict(kind=kind, type=t, down=d, dim=_log(rng, 1024, 4096, 256), ff=_log(rng, 512, 2048, 256),
                    experts=rng.choice([64, 128, 256]), k=rng.choice([4, 8]), n=_log(rng, 65, 1024))
    if kind == "mmq":
        return dict(kind=kind, type="Q4_K", rows=_log(rng, 1024, 7168, 16), cols=_log(rng, 512, 2048, 256),
                    experts=rng.choice([1, 16, 64, 256]), k=8, n=_log(rng, 17, 1024))
    if kind == "group":
        return dict(kind=kind, type=rng.choice(LANE), rows=_log(rng, 512, 2048, 16), cols=_log(rng, 512, 7168, 256),
                    experts=rng.choice([1, 16, 64, 256]), k=8, n=_log(rng, 17, 512))
    return dict(kind=kind, type=rng.choice(list(TYPES)), rows=_log(rng, 256, 8192, 16), cols=_log(rng, 512, 7168, 256),
                f16=rng.random() < 0.5)


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _blocks(gen, name, rows, cols, mats):
    """mats x (rows x cols) GGUF blocks: random codes, grid indices, signs and sub-scales, f16 scales |N(0, s)|"""
    _, v, b, gain = TYPES[name]
    n = mats * rows * (cols // v)
    raw = torch.randint(0, 256, (n, b), dtype=torch.uint8, device="cuda", generator=gen)
    for at in SCALE_AT.get(name, [None]):
        d = (torch.randn(n, device="cuda", generator=gen).abs_() * (WRMS / gain)).half().view(torch.int16).to(torch.int32)
        if at is None:  # IQ1_M: the f16's nibbles on top of the four scale words
            for k in range(4):
                raw[:, 49 + 2 * k] = (raw[:, 49 + 2 * k] & 15) | (((d >> (4 * k)) & 15) << 4).to(torch.uint8)
        else:
            raw[:, at] = (d & 255).to(torch.uint8)
            raw[:, at + 1] = ((d >> 8) & 255).to(torch.uint8)
    return raw.reshape(mats, -1)


def _picks(gen, n, experts, k):
    """k distinct experts a token, uniform (a trained router's load at decode batches); the last expert of a layer of
    257 is the shared one, which every token takes"""
    shared = experts == 257
    r = torch.rand(n, experts, device="cuda", generator=gen)
    if shared:
        r[:, -1] = 2.0
    return torch.topk(r, k, dim=1).indices.to(torch.int32).contiguous()


def _zipf_logits(gen, n, experts):
    """router logits whose top-k are picks without replacement at Zipf(1.1) odds, experts in a random order"""
    p = 1.0 / torch.arange(1, experts + 1, device="cuda", dtype=torch.float64) ** 1.1
    odds = torch.log(p / p.sum())[torch.randperm(experts, device="cuda", generator=gen)]
    u = torch.rand(n, experts, device="cuda", generator=gen, dtype=torch.float64).clamp_(1e-12, 1 - 1e-12)
    return (odds - torch.log(-torch.log(u))).float().contiguous()


def _grouped(case, gen):
    """a prompt's picks by expert: cnt per expert, the picks' tokens sorted by expert"""
    k = min(case["k"], case["experts"])
    ids = torch.topk(_zipf_logits(gen, case["n"], case["experts"]), k, dim=1).indices.reshape(-1)
    order = torch.argsort(ids, stable=True)
    cnt = torch.bincount(ids, minlength=case["experts"]).to(torch.int32)
    return cnt, (order // k).to(torch.int32), int(cnt.max())


def _table(w):
    return w.data_ptr() + torch.arange(w.shape[0], dtype=torch.int64, device="cuda") * w.shape[1]


class State:
    """the calls of one pass (function, arguments without the stream), what they read and write, and the graph if the
    program keeps one"""

    def __init__(self):
        self.calls, self.keep, self.out, self.data, self.graph = [], [], [], {}, None

    def a(self, t):
        self.keep.append(t)
        return capi.addr(t)

    def call(self, name, *args):
        self.calls.append((getattr(capi.lib(), name), args))

    def launch(self, stream):
        s = ctypes.c_void_p(stream)
        for f, args in self.calls:
            if not f(*args, s):
                raise RuntimeError("%s refused" % f.__name__)

    def capture(self):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            self.launch(side.cuda_stream)
            torch.cuda.synchronize()
            self.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(self.graph, stream=side):
                self.launch(side.cuda_stream)
        torch.cuda.synchronize()


def prepare(case, seed):
    gen, st = _gen(seed), State()
    globals()["_prepare_" + case["kind"]](case, gen, st)
    if case.get("graph"):
        st.capture()
    return st


def run(st):
    if st.graph is not None:
        st.graph.replay()
    else:
        st.launch(torch.cuda.current_stream().cuda_stream)
    return st.out


def _prepare_mv(c, gen, st):
    t, rows, cols, n = TYPES[c["type"]][0], c["rows"], c["cols"], c["n"]
    w = _blocks(gen, c["type"], rows, cols, c["layers"])
    x = torch.randn(n, cols, device="cuda", generator=gen)
    st.data = dict(w=w, x=x)
    for i in range(c["layers"]):
        y = torch.empty(n, rows, device="cuda")
        st.out.append(y)
        st.call("mv_strided", t, st.a(w[i]), rows, cols, st.a(x), cols, n, st.a(y), rows)


def _layer_inputs(c, gen, st):
    n, k, dim, ff, e = c["n"], c["k"], c["dim"], c["ff"], c["experts"]
    st.data["layers"] = []
    for _ in range(c["layers"]):
        st.data["layers"].append(dict(
            gate=_blocks(gen, c["type"], ff, dim, e), up=_blocks(gen, c["type"], ff, dim, e),
            down=_blocks(gen, c["type"], dim, ff, e), ids=_picks(gen, n, e, k),
            w=torch.softmax(torch.randn(n, k, device="cuda", generator=gen), dim=1),
            x=torch.randn(n, dim, device="cuda", generator=gen), add=torch.randn(n, dim, device="cuda", generator=gen)))
    return st.data["layers"]


class _Forward:
    """LaneLayer.forward as one of a State's calls"""
    __name__ = "LaneLayer.forward"

    def __init__(self, layer):
        self.layer = layer

    def __call__(self, *args):
        return self.layer.forward(*args) is not None


def _prepare_layer(c, gen, st):
    t = TYPES[c["type"]][0]
    for d in _layer_inputs(c, gen, st):
        lay = LaneLayer(t, t, c["dim"], c["ff"], c["experts"], c["k"], d["gate"], d["up"], d["down"])
        lay.workspace(c["n"])
        out = torch.empty(c["n"], c["dim"], device="cuda")
        st.out.append(out)
        st.calls.append((_Forward(lay), (d["x"], d["ids"], d["w"], d["add"], out)))


def _prepare_engine(c, gen, st):
    t, n, k, dim, ff, e = TYPES[c["type"]][0], c["n"], c["k"], c["dim"], c["ff"], c["experts"]
    p = n * k
    for d in _layer_inputs(c, gen, st):
        base = (ctypes.c_void_p * 3)(*[d[m].data_ptr() for m in ("gate", "up", "down")])
        size = (ctypes.c_uint64 * 3)(*[d[m].shape[1] for m in ("gate", "up", "down")])
        st.keep += [base, size]
        i32 = lambda: torch.zeros(p, dtype=torch.int32, device="cuda")  # noqa: E731
        tok, pair, cnt, xrow, order = i32(), i32(), i32(), i32(), i32()
        wg, wu, wd = (torch.zeros(p, dtype=torch.int64, device="cuda") for _ in range(3))
        xq, xd = torch.empty(n, dim, dtype=torch.int8, device="cuda"), torch.empty(n, dim // 32, device="cuda")
        h, y = torch.empty(p, ff, device="cuda"), torch.empty(p, dim, device="cuda")
        hq, hd = torch.empty(p, ff, dtype=torch.int8, device="cuda"), torch.empty(p, ff // 32, device="cuda")
        out = torch.empty(n, dim, device="cuda")
        most = min(n, 8)
        st.call("osmos_lane_tables", st.a(d["ids"]), n, k, e, base, size, st.a(tok), st.a(pair), st.a(cnt), st.a(xrow),
                st.a(wg), st.a(wu), st.a(wd), st.a(order))
        st.call("q8_round", st.a(d["x"]), n, dim, dim, st.a(xq), st.a(xd))
        st.call("q8_gate_up", t, st.a(wg), st.a(wu), st.a(cnt), st.a(xrow), st.a(tok), st.a(pair), p, most, ff, dim,
                st.a(xq), st.a(xd), st.a(d["w"]), math.inf, st.a(h), ff)
        st.call("q8_round", st.a(h), p, ff, ff, st.a(hq), st.a(hd))
        st.call("q8_group_tok", t, st.a(wd), st.a(cnt), st.a(xrow), None, p, most, dim, ff, st.a(hq), st.a(hd), st.a(y),
                dim)
        st.call("ops_gather_sum_add", st.a(out), st.a(y), st.a(order), k, n, dim, st.a(d["add"]))
        st.out.append(out)


def _prepare_mm(c, gen, st):
    t, rows, cols, n = TYPES[c["type"]][0], c["rows"], c["cols"], c["n"]
    w = _blocks(gen, c["type"], rows, cols, c["mats"])
    x = torch.randn(n, cols, device="cuda", generator=gen)
    x16 = torch.empty((n + 15) // 16 * 16 * cols, dtype=torch.float16, device="cuda")
    over = torch.zeros(1, dtype=torch.int32, device="cuda")
    st.data = dict(w=w, x=x)
    st.call("mm_x16", st.a(x), cols, n, cols, st.a(x16), st.a(over))
    for i in range(c["mats"]):
        y = torch.empty(n, rows, device="cuda")
        st.out.append(y)
        st.call("mm_run", t, st.a(w[i]), rows, cols, st.a(x16), n, st.a(y), rows)


def _prepare_moe(c, gen, st):
    n, k, dim, ff, e = c["n"], c["k"], c["dim"], c["ff"], c["experts"]
    tg, td, p = TYPES[c["type"]][0], TYPES[c["down"]][0], n * k
    gate, up = _blocks(gen, c["type"], ff, dim, e), _blocks(gen, c["type"], ff, dim, e)
    down = _blocks(gen, c["down"], dim, ff, e)
    logits = _zipf_logits(gen, n, e)
    x, shared = (torch.randn(n, dim, device="cuda", generator=gen) for _ in range(2))
    gatel = torch.randn(n, device="cuda", generator=gen)
    st.data = dict(gate=gate, up=up, down=down, logits=logits, x=x, shared=shared, shared_logit=gatel)
    bd = capi.Q4xExpertBounds()
    capi.lib().q4x_expert_bounds(p, e, ctypes.byref(bd))
    i32 = lambda m: torch.zeros(max(m, 1), dtype=torch.int32, device="cuda")  # noqa: E731
    ids, rows, w = i32(p), i32(p), torch.empty(p, device="cuda")
    tb = capi.Q4xExpertTiles()
    ptr = [torch.zeros(bd.entries, dtype=torch.int64, device="cuda") for _ in range(3)]
    for j, m in enumerate((gate, up, down)):
        tb.base[j], tb.bytes[j], tb.ptr[j], tb.tab[j] = m.data_ptr(), m.shape[1], ptr[j].data_ptr(), None
    f = {}
    for name, size in (("cnt", bd.entries), ("gidx", bd.slots), ("hidx", bd.slots), ("xg", bd.entries), ("yg", bd.entries),
                       ("xd", bd.entries), ("yd", bd.entries), ("where", p), ("off", 3 * e)):
        f[name] = i32(size)
        setattr(tb, name, f[name].data_ptr())
    st.keep += [tb, f]
    slots = (bd.slots + 15) // 16 * 16
    xg16 = torch.empty(slots * dim, dtype=torch.float16, device="cuda")
    xd16 = torch.empty(slots * ff, dtype=torch.float16, device="cuda")
    over = i32(1)
    yg, yu, yd = (torch.empty(p, m, device="cuda") for m in (ff, ff, dim))
    out = torch.empty(n, dim, device="cuda")
    st.call("q4x_route", st.a(logits), n, e, k, st.a(ids), st.a(w), st.a(rows))
    st.call("q4x_expert_tiles", st.a(ids), p, k, e, dim, ff, ctypes.byref(tb))
    st.call("mm_x16_rows", st.a(x), dim, st.a(f["gidx"]), bd.slots, dim, st.a(xg16), st.a(over))

    def group(t, j, rows_, cols, x16, xoff, y, yoff):  # one call a run: parts of 1, 2, 4 or 8 tiles of 16 tokens
        for r in range(4):
            if bd.count[r]:
                s = slice(bd.first[r], bd.first[r] + bd.count[r])
                st.call("mm_group", t, st.a(ptr[j][s]), st.a(f["cnt"][s]), bd.count[r], 16 << r, rows_, cols, st.a(x16),
                        st.a(f[xoff][s]), cols, st.a(y), st.a(f[yoff][s]), rows_)
    group(tg, 0, ff, dim, xg16, "xg", yg, "yg")
    group(tg, 1, ff, dim, xg16, "xg", yu, "yg")
    st.call("q4x_swiglu_rows", st.a(yg), st.a(yu), ff, st.a(f["hidx"]), bd.slots, st.a(xd16), st.a(over))
    group(td, 2, dim, ff, xd16, "xd", yd, "yd")
    st.call("q4x_moe_sum", st.a(yd), st.a(f["where"]), st.a(w), n, k, dim, st.a(shared), st.a(gatel), st.a(out))
    st.out = [out, w]


def _prepare_mmq(c, gen, st):
    rows, cols, e = c["rows"], c["cols"], c["experts"]
    w = _blocks(gen, "Q4_K", rows, cols, e)
    cnt, tok, most = _grouped(c, gen)
    p, host = tok.numel(), cnt.tolist()
    x = torch.randn(p, cols, device="cuda", generator=gen)  # each pick's own activations, sorted by expert
    idx, soff, row = [], [], 0
    for m in host:
        soff.append(len(idx))
        idx += list(range(row, row + m)) + [-1] * (-m % 16)
        row += m
    slots = len(idx)
    idx = torch.tensor(idx, dtype=torch.int32, device="cuda")
    yoff = ((torch.cumsum(cnt, 0) - cnt) * rows).to(torch.int32)
    x8 = torch.empty(slots * cols, dtype=torch.int8, device="cuda")
    dx, sx = (torch.empty(slots * cols // 32, device="cuda") for _ in range(2))
    y = torch.empty(p, rows, device="cuda")
    st.data = dict(w=w, x=x, cnt=host)
    st.out = [y]
    st.call("mmq_x8_rows", st.a(x), cols, st.a(idx), slots, cols, st.a(x8), st.a(dx), st.a(sx))
    st.call("mmq_group", 12, st.a(_table(w)), st.a(cnt), e, most, rows, cols, st.a(x8), st.a(dx), st.a(sx),
            st.a(torch.tensor(soff, dtype=torch.int32, device="cuda")), st.a(y), st.a(yoff), rows)


def _prepare_group(c, gen, st):
    rows, cols, e = c["rows"], c["cols"], c["experts"]
    w = _blocks(gen, c["type"], rows, cols, e)
    cnt, tok, most = _grouped(c, gen)
    p = tok.numel()
    x = torch.randn(c["n"], cols, device="cuda", generator=gen)
    xg = torch.empty(p, cols, device="cuda")
    q, d = torch.empty(p, cols, dtype=torch.int8, device="cuda"), torch.empty(p, cols // 32, device="cuda")
    y = torch.empty(p, rows, device="cuda")
    st.data = dict(w=w, x=x, tok=tok, cnt=cnt.tolist())
    st.out = [y]
    st.call("ops_gather_rows", st.a(xg), st.a(x), st.a(tok), p, cols)
    st.call("q8_round", st.a(xg), p, cols, cols, st.a(q), st.a(d))
    st.call("osmos_lane_group", TYPES[c["type"]][0], st.a(_table(w)), st.a(cnt),
            st.a((torch.cumsum(cnt, 0) - cnt).to(torch.int32)), e, most, rows, cols, st.a(q), st.a(d), st.a(y), rows)


def _prepare_dequant(c, gen, st):
    w = _blocks(gen, c["type"], c["rows"], c["cols"], 1)
    y = torch.empty(c["rows"], c["cols"], device="cuda", dtype=torch.float16 if c["f16"] else torch.float32)
    st.data = dict(w=w)
    st.out = [y]
    st.call("quant_dequant_f16" if c["f16"] else "quant_dequant", TYPES[c["type"]][0], st.a(w), c["rows"] * c["cols"],
            st.a(y))


# ---------------------------------------------------------------- the work of a pass

def _distinct(c):
    """the experts that n tokens' picks reach on average (decode: uniform, a layer of 257 with its shared one)"""
    n, k, e = c["n"], c["k"], c["experts"]
    if e == 257:
        return 1 + 256 * (1 - (1 - (k - 1) / 256) ** n)
    return e * (1 - (1 - k / e) ** n)


def _distinct_zipf(c):
    p = 1.0 / np.arange(1, c["experts"] + 1) ** 1.1
    p /= p.sum()
    k = min(c["k"], c["experts"])
    return float(np.sum(1 - (1 - np.minimum(p, 1)) ** (c["n"] * k)))


def work(c):
    kind, n = c["kind"], c.get("n", 0)
    if kind == "mv":
        r, k = c["rows"], c["cols"]
        return {"bytes": c["layers"] * (r * row_bytes(c["type"], k) + n * r * 4) + n * k * 4,
                "flops": 2.0 * c["layers"] * n * r * k}
    if kind in ("layer", "engine"):
        dim, ff = c["dim"], c["ff"]
        per = 2 * ff * row_bytes(c["type"], dim) + dim * row_bytes(c["type"], ff)
        return {"bytes": c["layers"] * (_distinct(c) * per + n * dim * 12 + n * c["k"] * 8),
                "flops": 6.0 * c["layers"] * n * c["k"] * dim * ff}
    if kind == "mm":
        r, k = c["rows"], c["cols"]
        return {"bytes": c["mats"] * (r * row_bytes(c["type"], k) + n * r * 4) + n * k * 4,
                "flops": 2.0 * c["mats"] * n * r * k}
    if kind == "moe":
        dim, ff = c["dim"], c["ff"]
        per = 2 * ff * row_bytes(c["type"], dim) + dim * row_bytes(c["down"], ff)
        return {"bytes": _distinct_zipf(c) * per + n * dim * 12 + n * c["experts"] * 4,
                "flops": 6.0 * n * min(c["k"], c["experts"]) * dim * ff}
    if kind in ("mmq", "group"):
        r, k, p = c["rows"], c["cols"], n * min(c["k"], c["experts"])
        return {"bytes": _distinct_zipf(c) * r * row_bytes(c["type"], k) + p * r * 4 + (p if kind == "mmq" else n) * k * 4,
                "flops": 2.0 * p * r * k}
    v = c["rows"] * c["cols"]
    return {"bytes": c["rows"] * row_bytes(c["type"], c["cols"]) + v * (2 if c["f16"] else 4), "flops": 0.0}


def tolerance(c):
    if c["kind"] == "mm":
        # f32 sums of f16 products: against 64-bit sums of the same f16 values the path is off by 1.1e-7 (2048 columns),
        # and by as much with its partial sums added in another order
        return {"rel": 5e-7, "max": 2e-5}
    if c["kind"] == "moe":
        # the same sums three times over, and the activations rounded to f16 between them, where a sum that lies near
        # the middle of two f16 values may round to the other one: 1.3e-5 from the 64-bit sums
        return {"rel": 5e-5, "max": 1e-3}
    return "exact"  # (the lane, matvec, int8 and decode contracts fix every bit)


# ---------------------------------------------------------------- the same in 64 bits

_GRIDS = {}


def _grid(name):
    """a codebook of the file format, [entries, values] (the format's packed index lists, expanded here)"""
    if name not in _GRIDS:
        here = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "libosmos_amd", "csrc")
        with open(os.path.join(here, "iq_grids.h")) as f:
            text = re.search(r"#define IQ_PACKED_%s((?:[^\n]*\\\n)*[^\n]*)" % name, f.read()).group(1)
        p = np.array([int(v, 16) for v in re.findall(r"0x[0-9a-fA-F]+", text)], np.int64)
        if name == "IQ3XXS":
            m, n, b = [4, 12, 20, 28, 36, 44, 52, 62], 4, 3
        else:
            m, n, b = ([-1, 0, 1, 0] if name == "IQ1S" else [8, 25, 43, 0]), 8, 2
        g = np.array(m)[(p[:, None] >> (b * np.arange(n))) & ((1 << b) - 1)]
        _GRIDS[name] = torch.tensor(g, dtype=torch.float64, device="cuda")
    return _GRIDS[name]


def _f16(b, at):
    return (b[:, at] | b[:, at + 1] << 8).to(torch.int16).view(torch.float16).double()


def _signs(i):
    """7-bit sign indices as 8 factors of +-1, the eighth the parity's"""
    bits = (i.unsqueeze(-1) >> torch.arange(7, device=i.device)) & 1
    return 1.0 - 2.0 * torch.cat([bits, bits.sum(-1, keepdim=True) & 1], -1).double()


def _u32(b):
    return b[..., 0] | b[..., 1] << 8 | b[..., 2] << 16 | b[..., 3] << 24


def decode(name, raw, rows, cols):
    """GGUF blocks' values in 64 bits, [rows, cols]"""
    b = raw.reshape(-1, TYPES[name][2]).long()
    n = b.shape[0]
    ar = lambda m: torch.arange(m, device=b.device)  # noqa: E731
    if name == "Q4_0":
        v = _f16(b, 0)[:, None] * (torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1) - 8)
    elif name == "Q4_K":
        s, g = b[:, 4:16], b[:, 16:].reshape(n, 4, 1, 32)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6) << 4], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6) << 4], 1)
        q = torch.cat([g & 15, g >> 4], 2).reshape(n, 8, 32)
        v = (_f16(b, 0)[:, None] * sc)[..., None] * q - (_f16(b, 2)[:, None] * mn)[..., None]
    elif name == "Q3_K":
        s = b[:, 96:108]
        lo = torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1)
        hi = ((s[:, 8:].reshape(n, 1, 4) >> (2 * ar(4)).reshape(1, 4, 1)) & 3).reshape(n, 16)
        q2 = (b[:, 32:96].reshape(n, 2, 1, 32) >> (2 * ar(4)).reshape(1, 1, 4, 1)) & 3
        hb = (b[:, None, None, :32] >> (4 * ar(2).reshape(1, 2, 1, 1) + ar(4).reshape(1, 1, 4, 1))) & 1
        v = (_f16(b, 108)[:, None] * ((lo | hi << 4) - 32))[..., None] * (q2 + 4 * hb - 4).reshape(n, 16, 16)
    elif name == "IQ2_XXS":
        g = b[:, 2:].reshape(n, 8, 8)
        aux = _u32(g[..., 4:])
        v = _grid("IQ2XXS")[g[..., :4]] * _signs((aux[..., None] >> (7 * ar(4))) & 127)
        v = v.reshape(n, 8, 32) * (_f16(b, 0)[:, None] * (0.5 + (aux >> 28)) / 4)[..., None]
    elif name == "IQ3_XXS":
        aux = _u32(b[:, 66:].reshape(n, 8, 4))
        v = _grid("IQ3XXS")[b[:, 2:66]].reshape(n, 8, 4, 8) * _signs((aux[..., None] >> (7 * ar(4))) & 127)
        v = v.reshape(n, 8, 32) * (_f16(b, 0)[:, None] * (0.5 + (aux >> 28)) / 2)[..., None]
    elif name == "IQ1_S":
        qh = b[:, 34:50:2] | b[:, 35:50:2] << 8
        i = b[:, 2:34].reshape(n, 8, 4) | ((qh[..., None] >> (3 * ar(4))) & 7) << 8
        v = _grid("IQ1S")[i].reshape(n, 8, 32) + (0.125 - 0.25 * (qh >> 15))[..., None]
        v = v * (_f16(b, 0)[:, None] * (2 * ((qh >> 12) & 7) + 1))[..., None]
    else:  # IQ1_M
        w = b[:, 48:56:2] | b[:, 49:56:2] << 8
        d = ((w >> 12) << (4 * ar(4))).sum(1).to(torch.int16).view(torch.float16).double()
        s = ((w[..., None] >> (3 * ar(4))) & 7).reshape(n, 16)
        nib = ((b[:, 32:48, None] >> (4 * ar(2))) & 15).reshape(n, 32)
        v = _grid("IQ1S")[b[:, :32] | (nib & 7) << 8] + (0.125 - 0.25 * (nib >> 3))[..., None]
        v = v.reshape(n, 16, 16) * (d[:, None] * (2 * s + 1))[..., None]
    return v.reshape(rows, cols)


def _round8(x):
    """the lane's rounded activations, as 64-bit values: 32-value blocks of int8 codes times their scale"""
    b = x.float().reshape(x.shape[0], -1, 32)
    a = b.abs().amax(-1, keepdim=True)
    q = torch.round(b * torch.where(a > 0, 127.0 / a, torch.zeros_like(a)))
    return (q.double() * (a / 127.0).double()).reshape(x.shape)


def _silu(x):
    return x / (1 + torch.exp(-x))


def _h16(x):
    return x.float().half().double()


def exact(case, seed):
    gen, st = _gen(seed), State()
    c = dict(case, graph=False)
    globals()["_prepare_" + c["kind"]](c, gen, st)
    d, kind = st.data, c["kind"]
    if kind == "mv":
        return [d["x"].double() @ decode(c["type"], w, c["rows"], c["cols"]).T for w in d["w"]]
    if kind == "mm":
        return [_h16(d["x"]) @ _h16(decode(c["type"], w, c["rows"], c["cols"])).T for w in d["w"]]
    if kind == "dequant":
        return [decode(c["type"], d["w"][0], c["rows"], c["cols"])]
    if kind in ("layer", "engine"):
        out = []
        for L in d["layers"]:
            x, y = _round8(L["x"]), L["add"].double()
            for e in torch.unique(L["ids"]).tolist():
                t, j = torch.nonzero(L["ids"] == e, as_tuple=True)
                g = x[t] @ decode(c["type"], L["gate"][e], c["ff"], c["dim"]).T
                u = x[t] @ decode(c["type"], L["up"][e], c["ff"], c["dim"]).T
                h = _round8(_silu(g) * u * L["w"][t, j][:, None].double())
                y[t] += h @ decode(c["type"], L["down"][e], c["dim"], c["ff"]).T
            out.append(y)
        return out
    if kind == "moe":
        p, x = torch.softmax(d["logits"].double(), 1), _h16(d["x"])
        w, ids = torch.topk(p, c["k"], dim=1)
        w = w / w.sum(1, keepdim=True).clamp_min(6.103515625e-5)
        y = d["shared"].double() * torch.sigmoid(d["shared_logit"].double())[:, None]
        for e in torch.unique(ids).tolist():
            t, j = torch.nonzero(ids == e, as_tuple=True)
            g = x[t] @ _h16(decode(c["type"], d["gate"][e], c["ff"], c["dim"])).T
            u = x[t] @ _h16(decode(c["type"], d["up"][e], c["ff"], c["dim"])).T
            y[t] += w[t, j][:, None] * (_h16(_silu(g) * u) @ _h16(decode(c["down"], d["down"][e], c["dim"], c["ff"])).T)
        return [y, w.reshape(-1)]
    y, row = [], 0
    x = d["x"] if kind == "mmq" else d["x"][d["tok"].long()]
    if kind == "mmq":
        b = x.reshape(x.shape[0], -1, 32)
        s = b.abs().amax(-1, keepdim=True) / 127.0
        x = (torch.round(b / s).clamp(-127, 127).double() * s.double()).reshape(x.shape)
    else:
        x = _round8(x)
    for e, m in enumerate(d["cnt"]):
        if m:
            y.append(x[row:row + m] @ decode(c["type"], d["w"][e], c["rows"], c["cols"]).T)
        row += m
    return [torch.cat(y)]
