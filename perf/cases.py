"""What a program that uses this library has it do, as cases that can be timed and checked: one DeepSeek-R1 MoE layer
(E 7168, H 2048, 256 routed + 1 shared expert) called the ways an engine calls it.

  layer     Context.moe_layer / moe_layer_normed on device rows: a decode step (1 .. 8 rows) or a prefill chunk
  narrow    the reference-named flow of the engine for up to 8 rows, host to host: fl_ffn_begin -> fl_fetch -> fl_moe
  wide      the reference-named flow of a prefill chunk: fl_ffn_begin / fl_fetch per 64 rows -> fl_wide_moe -> fl_wide_finish

Formats: iq2 = every matrix IQ2_XXS; q3 / q2 = the real shards' mix (routed gate/up IQ2_XXS, routed down Q3_K / Q2_K,
shared expert Q5_K, Q5_K, Q6_K). Weights are random bytes with the formats' scales, drawn in ggml's layout and packed
once, as a program that loads a model does. One context per set of options serves every layer, as in an engine."""
import ctypes
import math
import os

import numpy as np
import torch

import loki_amd
from loki_amd import FLW, FLOut, Context, MoeLayerWeights, lib

E, H, NE, TOPK = 7168, 2048, 256, 8
IQ2, Q6, Q5, Q2, Q3 = loki_amd.FL_IQ2, loki_amd.FL_Q6K, loki_amd.FL_Q5K, loki_amd.FL_Q2K, loki_amd.FL_Q3K
BLOCK = {IQ2: 66, Q2: 84, Q3: 110, Q5: 176, Q6: 210}                       # bytes per 256 weights
SCALES = {IQ2: (0,), Q2: (80, 82), Q3: (108,), Q5: (0, 2), Q6: (208,)}     # offsets of the fp16 d (and dmin)
FORMATS = {"iq2": (IQ2, IQ2, IQ2, IQ2), "q3": (Q3, Q5, Q5, Q6), "q2": (Q2, Q5, Q5, Q6)}   # routed down, shared gate, up, down
SHAPES = ((H, E), (H, E), (E, H))


def listed():
    return [
        # a token of a chat, one layer of the chain: the norm in front and the residual in the block
        {"name": "decode_1", "kind": "layer", "n": 1, "fmt": "iq2", "keep": 0, "share": False, "normed": True, "hot": 0},
        # the engine's default of two experts per token: the smallest call
        {"name": "decode_1_keep2", "kind": "layer", "n": 1, "fmt": "iq2", "keep": 2, "share": False, "normed": False, "hot": 0},
        # the chat client's setting (three experts, shared over the rows) on a short speculative batch
        {"name": "decode_3_keep3_share", "kind": "layer", "n": 3, "fmt": "iq2", "keep": 3, "share": True, "normed": False, "hot": 0},
        # eight users, or eight drafted tokens, at once
        {"name": "decode_8", "kind": "layer", "n": 8, "fmt": "iq2", "keep": 0, "share": False, "normed": False, "hot": 0},
        # the same with the formats of the real shards
        {"name": "real_decode_1", "kind": "layer", "n": 1, "fmt": "q3", "keep": 0, "share": False, "normed": False, "hot": 0},
        {"name": "real_decode_6", "kind": "layer", "n": 6, "fmt": "q2", "keep": 0, "share": False, "normed": False, "hot": 0},
        # a short question, an ordinary prompt chunk, a long one whose tokens favour 16 experts
        {"name": "prefill_37", "kind": "layer", "n": 37, "fmt": "iq2", "keep": 0, "share": False, "normed": False, "hot": 0},
        {"name": "prefill_512", "kind": "layer", "n": 512, "fmt": "iq2", "keep": 0, "share": False, "normed": False, "hot": 0},
        {"name": "prefill_2048_hot", "kind": "layer", "n": 2048, "fmt": "iq2", "keep": 0, "share": False, "normed": False, "hot": 16},
        # a prompt of the real shards' formats
        {"name": "real_prefill_201", "kind": "layer", "n": 201, "fmt": "q3", "keep": 0, "share": False, "normed": False, "hot": 0},
        # the engine's own calls, from host rows to host rows: a token, and a prompt
        {"name": "dropin_decode_1", "kind": "narrow", "n": 1, "fmt": "iq2", "keep": 0, "share": False, "normed": False, "hot": 0},
        {"name": "dropin_prefill_190", "kind": "wide", "n": 190, "fmt": "iq2", "keep": 0, "share": False, "normed": False, "hot": 0},
    ]


def draw(rng):
    c = {"kind": rng.choice(["layer"] * 6 + ["narrow", "wide"]), "fmt": rng.choice(["iq2", "iq2", "q3", "q2"]), "keep": 0,
         "share": False, "normed": False, "hot": 0}
    spread = lambda lo, hi: max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo - 0.49), math.log(hi + 0.49))))))  # noqa: E731
    if c["kind"] == "narrow":
        c["n"], c["fmt"] = rng.randint(1, 8), "iq2"
    elif c["kind"] == "wide":
        c["n"], c["fmt"] = spread(65, 512), "iq2"
    else:
        c["n"] = spread(1, 2000 if c["fmt"] == "iq2" else 500)
        c["normed"] = rng.random() < 0.4
        c["hot"] = 16 if c["n"] >= 256 and rng.random() < 0.4 else 0
        if rng.random() < 0.3:
            c["keep"] = rng.randint(2, 4)
            c["share"] = rng.random() < 0.5
    return c


# ------------------------------------------------------------------------------------------------ inputs
def random_matrices(fmt, count, g):
    """`count` expert matrices in ggml's layout: [count * R * K / 256, block bytes], uniform quants, fp16 scales."""
    nb = count * H * (E // 256)
    words = torch.randint(-(1 << 63), (1 << 63) - 1, ((nb * BLOCK[fmt] + 7) // 8,), dtype=torch.int64, device="cuda", generator=g)
    b = words.view(torch.uint8)[:nb * BLOCK[fmt]].view(nb, BLOCK[fmt])
    for at in SCALES[fmt]:
        if fmt == IQ2:
            d = (torch.randn(nb, device="cuda", generator=g) * 0.002).abs().half()
        else:
            d = (torch.rand(nb, device="cuda", generator=g) * 0.002 + 1e-4).half()
        b[:, at:at + 2] = d.view(torch.uint8).view(nb, 2)
    return b


def drawn_weights(case, seed):
    """The layer as a model file holds it: router, bias, norm weight, and [routed, shared] x [gate, up, down] bytes."""
    g = torch.Generator(device="cuda").manual_seed(seed * 1000003 + 17)
    down, sg, su, sd = FORMATS[case["fmt"]]
    w = {"router": torch.randn((NE, E), device="cuda", generator=g) * 0.02,
         "bias": torch.randn(NE, device="cuda", generator=g) * (0.05 if case["n"] > 8 else 0.01),
         "norm": 1 + 0.1 * torch.randn(E, device="cuda", generator=g)}
    if case["hot"]:
        w["bias"][torch.randperm(NE, device="cuda", generator=g)[:case["hot"]]] += 0.5
    w["routed"] = [random_matrices(f, NE, g) for f in (IQ2, IQ2, down)]
    w["shared"] = [random_matrices(f, 1, g) for f in (sg, su, sd)]
    return w


def drawn_rows(case, seed):
    """The rows that go in, and (for the engine's flow) the residual that is added back; host rows there."""
    g = torch.Generator(device="cuda").manual_seed(seed * 1000003 + 18)
    x = torch.randn((case["n"], E), device="cuda", generator=g)
    if case["kind"] == "layer":
        return x, None
    return x.cpu().numpy(), torch.randn((case["n"], E), device="cuda", generator=g).cpu().numpy()


_contexts = {}


def context(case):
    """The program's context for these options (one stream, torch's; every layer goes through it)."""
    key = (case["kind"], case["fmt"], case["keep"], case["share"])
    if key not in _contexts:
        c = Context()
        if case["kind"] == "layer":
            c.set_layer_formats(*FORMATS[case["fmt"]])
            c.set_keep(case["keep"], 2.5)
            c.set_share_experts(case["share"])
        _contexts[key] = c
    return _contexts[key]


class State:
    """One layer resident on the GPU, tiled, with a batch of rows. The engine's flow declares the matrices as tiled."""

    def __init__(self, case, seed):
        self.case, self.ctx = case, context(case)
        w = drawn_weights(case, seed)
        tiled = []
        for group, count in (("routed", NE), ("shared", 1)):
            fmts = (IQ2, IQ2, FORMATS[case["fmt"]][0]) if group == "routed" else FORMATS[case["fmt"]][1:]
            for k in range(3):
                m = w[group][k].view(-1)
                tiled.append(self.ctx.pack(m, *SHAPES[k], count) if fmts[k] == IQ2 else m)
                w[group][k] = None
        self.layer, self.norm = MoeLayerWeights(w["router"], w["bias"], *tiled), w["norm"]
        self.x, self.fi = drawn_rows(case, seed)
        self.declared = []
        if case["kind"] == "layer":
            self.y = torch.empty_like(self.x)
            return
        for m in tiled:
            self.ctx.register_tiled(m)
            self.declared.append(m)
        self.w = FLW()
        self.w.gate_inp, self.w.probs_b, self.w.gate_f16 = w["router"].data_ptr(), w["bias"].data_ptr(), 0
        self.w.sh_gate, self.w.sh_up, self.w.sh_down = (m.data_ptr() for m in tiled[3:])
        self.out = FLOut()
        if case["kind"] == "wide" and lib().fl_wide_init(self.ctx.ctx, case["n"], TOPK) != 1:
            raise RuntimeError("fl_wide_init failed")

    def __del__(self):
        for m in getattr(self, "declared", ()):
            self.ctx.unregister_tiled(m)


def prepare(case, seed):
    return State(case, seed)


# ------------------------------------------------------------------------------------------------ one pass
def host(p, shape, dtype):
    """The library's pinned mirror at `p` as an array (no copy)."""
    return np.frombuffer((ctypes.c_char * (4 * math.prod(shape))).from_address(ctypes.addressof(p.contents)), dtype).reshape(shape)


def ptr(a):
    return ctypes.c_void_p(a.ctypes.data)


def run(s):
    n = s.case["n"]
    if s.case["kind"] == "layer":
        if s.case["normed"]:
            return s.ctx.moe_layer_normed(s.layer, s.x, s.norm, 1e-6, s.y, residual=True)
        return s.ctx.moe_layer(s.layer, s.x, s.y)
    L, c, fl, out = s.layer, s.ctx.ctx, lib(), s.out
    if s.case["kind"] == "narrow":
        s.ctx.check(fl.fl_ffn_begin(c, ctypes.byref(s.w), n, ptr(s.x), ptr(s.fi), -1))
        fl.fl_fetch(c, n, 1, ctypes.byref(out))
        sel, wts = host(out.sel, (n, TOPK), np.int32).copy(), host(out.wts, (n, TOPK), np.float32).copy()
        fl.fl_moe(c, L.gate.data_ptr(), L.up.data_ptr(), L.down.data_ptr(), NE, IQ2, ptr(sel), ptr(wts), TOPK, n, ctypes.byref(out))
        return {"h": host(out.h, (n, E), np.float32), "moe": host(out.moe, (n, E), np.float32), "sel": sel, "wts": wts}
    sel, wts = np.empty((n, TOPK), np.int32), np.empty((n, TOPK), np.float32)
    for r in range(0, n, 64):
        m = min(64, n - r)
        s.ctx.check(fl.fl_ffn_begin(c, ctypes.byref(s.w), m, ptr(s.x[r:r + m]), ptr(s.fi[r:r + m]), r))
        fl.fl_fetch(c, m, 1, ctypes.byref(out))
        sel[r:r + m], wts[r:r + m] = host(out.sel, (m, TOPK), np.int32), host(out.wts, (m, TOPK), np.float32)
    # the engine's lists: every expert's (row, k) pairs in row order, eight to a slot
    order = np.argsort(sel.ravel(), kind="stable")
    es = sel.ravel()[order]
    count = np.bincount(es, minlength=NE)
    slots = (count + 7) // 8
    rank = np.arange(es.size) - (np.cumsum(count) - count)[es]
    at = ((np.cumsum(slots) - slots)[es] + rank // 8) * 8 + rank % 8
    ns = int(slots.sum())
    ids = np.repeat(np.arange(NE, dtype=np.int32), slots)
    rows, kidx, wk = np.full(ns * 8, -1, np.int32), np.zeros(ns * 8, np.int32), np.zeros(ns * 8, np.float32)
    rows[at], kidx[at], wk[at] = order // TOPK, order % TOPK, wts.ravel()[order]
    fl.fl_wide_moe(c, L.gate.data_ptr(), L.up.data_ptr(), L.down.data_ptr(), IQ2, NE, ptr(ids), ptr(rows), ptr(kidx), ptr(wk), ns, TOPK, 0)
    fl.fl_wide_finish(c, n, TOPK, ctypes.byref(out))
    return {"h": host(out.h, (n, E), np.float32), "moe": host(out.moe, (n, E), np.float32), "sel": sel, "wts": wts}


# ------------------------------------------------------------------------------------------------ what it cannot do without
def work(case):
    n, keep = case["n"], case["keep"] or TOPK
    used = NE * (1 - (1 - keep / NE) ** n)                  # distinct experts that n rows are expected to pick
    down, sg, su, sd = (BLOCK[f] for f in FORMATS[case["fmt"]])
    blocks = H * E // 256
    bytes_ = blocks * (used * (2 * BLOCK[IQ2] + down) + sg + su + sd) + NE * (E + 1) * 4
    bytes_ += n * E * 4 * (2 if case["kind"] == "layer" else 4)
    return {"bytes": bytes_, "flops": 2.0 * n * E * ((keep + 1) * 3 * H + NE)}


def tolerance(case):
    # Outputs are fp32 sums (2e-7 off 64 bits as long as every int8 rounding falls the same way: one token, mostly). Over
    # many rows a few of the 8-bit activations (Q8_K of x and of h) round the other way for a last-bit change in front
    # of them, and each moves its whole row by about 1e-3: 2e-4 .. 6e-4 in all, measured at 37 .. 2048 rows against
    # exact(). Four times that. Which experts are picked, and with which weight, does not move.
    return {"rel": 2.5e-3, "max": 4e-2}


# ------------------------------------------------------------------------------------------------ in 64 bits
def codebook():
    """ggml's iq2xxs codebook, the format's constant, as [256, 8], and the signs of the 7 stored bits as [128, 8]."""
    with open(os.path.join(os.path.dirname(loki_amd.__file__), "csrc", "iq2xxs_grid.inc")) as f:
        v = [int(t.strip().rstrip("uUlL"), 16) for t in f.read().replace("\n", ",").split(",") if t.strip().startswith("0x")]
    grid = torch.tensor([[(x >> (8 * k)) & 255 for k in range(8)] for x in v], dtype=torch.float64, device="cuda")
    bits = [[(i >> k) & 1 for k in range(7)] + [bin(i).count("1") & 1] for i in range(128)]
    return grid, 1 - 2 * torch.tensor(bits, dtype=torch.float64, device="cuda")


def f16(b, at):
    return b[:, at:at + 2].contiguous().view(torch.float16).double()


def dequantise(fmt, b, R, K, tables):
    """Blocks [R * K / 256, bytes] of ggml's format as a matrix of doubles."""
    n, ar = b.shape[0], lambda *v: torch.tensor(v, device="cuda")  # noqa: E731
    d = f16(b, SCALES[fmt][0])
    i = lambda lo, hi: b[:, lo:hi].to(torch.int32)  # noqa: E731
    if fmt == IQ2:
        w = b[:, 2:].contiguous().view(torch.int32).view(n, 8, 2)
        l = torch.arange(4, device="cuda", dtype=torch.int32)
        idx, sg = (w[:, :, :1] >> (8 * l)) & 255, (w[:, :, 1:] >> (7 * l)) & 127
        v = tables[0][idx.long()] * tables[1][sg.long()]
        return (v.view(n, 8, 32) * ((((w[:, :, 1:] >> 28) & 15) + 0.5) * 0.25 * d[:, :, None])).view(R, K)
    if fmt in (Q2, Q3):   # two halves of 128, four 2-bit planes of 32 columns each
        qs = i(16, 80) if fmt == Q2 else i(32, 96)
        q = (qs.view(n, 2, 1, 32) >> ar(0, 2, 4, 6).view(1, 1, 4, 1)) & 3
        if fmt == Q2:
            sc = i(0, 16)
            v = q.reshape(n, 16, 16) * (d * (sc & 15))[:, :, None] - (f16(b, 82) * (sc >> 4))[:, :, None]
            return v.view(R, K)
        hi = (i(0, 32).view(n, 1, 1, 32) >> ar(0, 1, 2, 3, 4, 5, 6, 7).view(1, 2, 4, 1)) & 1
        s = i(96, 108)
        low = torch.cat((s[:, :8] & 15, s[:, :8] >> 4), 1)
        top = (s[:, 8:].repeat(1, 4) >> ar(0, 2, 4, 6).repeat_interleave(4)) & 3
        return ((q - 4 * (1 - hi)).reshape(n, 16, 16) * (d * (low + 16 * top - 32))[:, :, None]).view(R, K)
    if fmt == Q5:
        s = i(4, 16)
        sc = torch.cat((s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)), 1)
        mn = torch.cat((s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)), 1)
        q = (i(48, 176).view(n, 4, 1, 32) >> ar(0, 4).view(1, 1, 2, 1)) & 15
        hi = (i(16, 48).view(n, 1, 32) >> torch.arange(8, device="cuda").view(1, 8, 1)) & 1
        return ((q.reshape(n, 8, 32) + 16 * hi) * (d * sc)[:, :, None] - (f16(b, 2) * mn)[:, :, None]).view(R, K)
    ql, qh = i(0, 128).view(n, 2, 2, 32), i(128, 192).view(n, 2, 1, 32)
    q = torch.cat((ql & 15, ql >> 4), 2) | (((qh >> ar(0, 2, 4, 6).view(1, 1, 4, 1)) & 3) << 4)
    sc = b[:, 192:208].contiguous().view(torch.int8).double()
    return ((q - 32).reshape(n, 16, 16) * (d * sc)[:, :, None]).view(R, K)


def q8k(x):
    """Rows through Q8_K (ggml's quantize_row_q8_K): the values that the products see."""
    v = x.double().view(x.shape[0], -1, 256)
    top = v.gather(2, v.abs().argmax(2, keepdim=True))      # the signed value of the largest magnitude
    inv = torch.where(top == 0, torch.zeros_like(top), -127 / top)
    q = torch.clamp(torch.round(inv * v), max=127)
    return torch.where(inv == 0, torch.zeros_like(v), q / inv).view(x.shape)


def route(case, x, w):
    """DeepSeek's rule: sigmoid scores, 8 groups by their two best, 4 kept, 8 picks, weights x 2.5; then the keep."""
    n = x.shape[0]
    p = torch.sigmoid((x.double() @ w["router"].double().t()).float().double()).float()
    c = p + w["bias"]
    groups = c.view(n, 8, 32).topk(2, 2).values.sum(2).topk(4, 1).indices
    allow = torch.zeros((n, 8), dtype=torch.bool, device="cuda").scatter_(1, groups, True)
    sel = c.masked_fill(~allow.repeat_interleave(32, 1), -math.inf).topk(TOPK, 1).indices
    wt = p.gather(1, sel).double()
    wt = wt / wt.sum(1, keepdim=True).clamp(min=6.103515625e-5) * 2.5
    if not case["keep"]:
        return sel, wt
    k, own = case["keep"], min(2, case["keep"])
    order = torch.sort(wt, dim=1, descending=True, stable=True).indices
    if case["share"] and n > 1:     # rows prefer, after their own two, experts that other rows already use
        so, rank = sel.gather(1, order).tolist(), []
        use = {e for r in so for e in r[:own]}
        for r in so:
            pick = list(range(own)) + [j for j in range(own, TOPK) if r[j] in use][:k - own]
            new = [j for j in range(own, TOPK) if j not in pick][:k - len(pick)]
            use |= {r[j] for j in new}
            rank.append(pick + new)
        order = order.gather(1, torch.tensor(rank, device="cuda"))
    else:
        order = order[:, :k]
    sel, wt = sel.gather(1, order), wt.gather(1, order)
    return sel, wt * (2.5 / wt.sum(1, keepdim=True))


def exact(case, seed):
    w, tables = drawn_weights(case, seed), codebook()
    x, fi = (None if v is None else torch.as_tensor(v, device="cuda") for v in drawn_rows(case, seed))
    rows = x
    if case["normed"]:
        v = x.double()
        rows = (v / torch.sqrt((v * v).mean(1, keepdim=True) + 1e-6) * w["norm"].double()).float()
    sel, wt = route(case, rows, w)
    a = q8k(rows)
    down, sg, su, sd = FORMATS[case["fmt"]]

    def expert(mats, fmts, e, v):
        nb = H * (E // 256)
        gate, up, dn = (dequantise(f, m[e * nb:(e + 1) * nb], *sh, tables) for f, m, sh in zip(fmts, mats, SHAPES))
        g = v @ gate.t()
        return q8k(g * torch.sigmoid(g) * (v @ up.t())) @ dn.t()

    moe = torch.zeros((case["n"], E), dtype=torch.float64, device="cuda")
    for e in sel.unique().tolist():
        t, k = (sel == e).nonzero(as_tuple=True)
        moe.index_add_(0, t, expert(w["routed"], (IQ2, IQ2, down), e, a[t]) * wt[t, k][:, None])
    full = moe + expert(w["shared"], (sg, su, sd), 0, a)
    if case["kind"] == "layer":
        return full + x.double() if case["normed"] else full
    return {"h": full + fi.double(), "moe": moe, "sel": None, "wts": wt}
