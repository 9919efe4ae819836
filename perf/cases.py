"""Timed cases of the training path, called through the C ABI of include/om.h the way a host tape calls it.

Each case is the work of one layer, block or step on tensors the caller already holds on the device: the small
MLP step (launch latency), Linear layers of ragged sizes, the feed-forward sub-block of a MiniLM-sized and of a
BERT-base-sized encoder, self-attention with and without a padding mask, attention between sequences of different odd
lengths, the 3x3 convolutions, a CRNN's conv stage and its CTC head, a whole pre-LN encoder block's training step, and
the clipped AdamW update of a BERT-sized parameter arena. `kind` selects the path; the other entries are its sizes.

Backward halves that depend on a forward decision (which activations a ReLU kept, which element a pool took) start
from saved tensors prepared here, so a rounding difference in the forward does not flip a whole gradient element.
"""
import ctypes as C
import importlib
import math

import torch

_PKG = importlib.import_module("onemodel-csharp_amd")
_CTX = None
DEV = "cuda"


def _ctx():
    """One library context (stream and scratch) for the process, as a training program keeps it."""
    global _CTX
    if _CTX is None:
        _CTX = _PKG.Context(0)
    return _CTX


# ------------------------------------------------------------------------------------------------------------- cases
def listed():
    return [
        # the MNIST-sized classifier's training step: the smallest launches, where latency is all there is
        {"name": "mlp_step", "kind": "mlp", "batch": 64, "din": 784, "hidden": 256, "dout": 10},
        # a Linear layer over a ragged batch with odd widths, forward and backward
        {"name": "linear_ragged", "kind": "linear", "rows": 1517, "din": 391, "dout": 1003, "bias": True},
        # the feed-forward sub-block of the MiniLM-sized encoder (32 sequences of 128)
        {"name": "ffn_minilm", "kind": "ffn", "rows": 4096, "d": 384, "f": 1536},
        # the same of the BERT-base-sized encoder at its largest batch (32 sequences of 512)
        {"name": "ffn_bert_large", "kind": "ffn", "rows": 16384, "d": 768, "f": 3072},
        # self-attention of the MiniLM-sized encoder with a padding mask
        {"name": "attn_minilm", "kind": "attn", "batch": 32, "heads": 12, "seq": 128, "dim": 32, "mask": True},
        # self-attention of the BERT-base-sized encoder, unpadded
        {"name": "attn_bert", "kind": "attn", "batch": 8, "heads": 12, "seq": 512, "dim": 64, "mask": False},
        # attention between sequences of different odd lengths with the weights kept (the per-op record)
        {"name": "attn_cross", "kind": "cross", "batch": 8, "heads": 8, "lq": 77, "lk": 131, "dim": 40, "mask": True},
        # a residual network's 3x3 convolution with its ReLU, forward and all three gradients
        {"name": "conv_56", "kind": "conv", "n": 32, "cin": 64, "h": 56, "w": 56, "cout": 64, "dx": True},
        # the CRNN's second stage: conv, ReLU and max pool, and their backward
        {"name": "crnn_stage", "kind": "stage", "n": 32, "cin": 32, "h": 16, "w": 64, "cout": 64, "pw": 2},
        # the CRNN's classifier over the time steps and the CTC loss, forward and backward
        {"name": "ctc_head", "kind": "ctc", "batch": 32, "time": 32, "classes": 37, "din": 256, "maxlen": 10},
        # one training step of the MiniLM-sized pre-LN block: forward, MSE, backward and AdamW
        {"name": "block_step", "kind": "block", "batch": 32, "seq": 128, "heads": 12, "dim": 32, "f": 1536},
        # global-norm clipping and AdamW over a four-layer BERT-base arena
        {"name": "adamw_bert", "kind": "adam", "params": 28358409, "segments": 66},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mlp", "linear", "linear", "ffn", "ffn", "attn", "attn", "cross", "conv", "stage", "ctc",
                       "block", "adam"])
    if kind == "mlp":
        return {"kind": kind, "batch": _log(rng, 16, 256), "din": _log(rng, 100, 1024), "hidden": 16 * rng.randint(4, 32),
                "dout": rng.randint(2, 32)}
    if kind == "linear":
        return {"kind": kind, "rows": _log(rng, 64, 8192), "din": _log(rng, 64, 2048), "dout": _log(rng, 64, 2048),
                "bias": rng.random() < 0.8}
    if kind == "ffn":
        d = rng.choice([256, 320, 384, 512, 640, 768])
        return {"kind": kind, "rows": rng.choice([1, 2, 4, 8, 16, 32]) * rng.choice([64, 96, 100, 128, 256, 512]), "d": d,
                "f": rng.choice([2 * d, 4 * d])}
    if kind == "attn":
        return {"kind": kind, "batch": _log(rng, 1, 32), "heads": rng.choice([4, 6, 8, 12]),
                "seq": 64 * rng.choice([1, 2, 2, 3, 4, 6, 8]), "dim": rng.choice([32, 64]), "mask": rng.random() < 0.5}
    if kind == "cross":
        return {"kind": kind, "batch": _log(rng, 1, 16), "heads": rng.choice([4, 8, 12]), "lq": rng.randint(16, 300),
                "lk": rng.randint(16, 300), "dim": 8 * rng.randint(2, 10), "mask": rng.random() < 0.5}
    if kind == "conv":
        hw = rng.randint(9, 64)
        return {"kind": kind, "n": _log(rng, 1, 32), "cin": rng.choice([16, 32, 48, 64, 128]), "h": hw,
                "w": max(5, hw + rng.randint(-4, 4)), "cout": rng.choice([32, 64, 96, 128]), "dx": rng.random() < 0.8}
    if kind == "stage":
        return {"kind": kind, "n": _log(rng, 4, 48), "cin": rng.choice([1, 32, 64, 128]), "h": 2 * rng.randint(2, 16),
                "w": 4 * rng.randint(8, 40), "cout": rng.choice([32, 64, 128, 256]), "pw": rng.choice([1, 2])}
    if kind == "ctc":
        t = rng.randint(24, 96)
        return {"kind": kind, "batch": _log(rng, 4, 64), "time": t, "classes": rng.randint(20, 64),
                "din": rng.choice([128, 256, 512]), "maxlen": max(4, t // 4)}
    if kind == "block":
        return {"kind": kind, "batch": _log(rng, 1, 32), "seq": 64 * rng.choice([1, 2, 3, 4]),
                "heads": rng.choice([4, 8, 12]), "dim": rng.choice([32, 64]), "f": rng.choice([768, 1024, 1536, 2048])}
    return {"kind": "adam", "params": _log(rng, 100000, 30000000), "segments": rng.randint(4, 100)}


# ------------------------------------------------------------------------------------------------------------ inputs
class _Rng:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed & ((1 << 63) - 1))

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device=DEV).mul_(std)

    def uniform(self, bound, *shape):
        return torch.rand(shape, generator=self.g, device=DEV).mul_(2 * bound).sub_(bound)

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.g, device=DEV, dtype=torch.int32)

    def linear(self, din, dout):
        b = 1.0 / math.sqrt(din)
        return self.uniform(b, dout, din), self.uniform(b, dout)


def _new(*shape, dtype=torch.float32):
    return torch.empty(shape, device=DEV, dtype=dtype)


def _key_mask(r, batch, lq, lk):
    """Additive [batch, lq, lk] padding mask: keys past each sequence's length (half to all of lk) are -inf."""
    n = r.ints(max(1, lk // 2), lk + 1, batch).long()
    m = torch.zeros(batch, lq, lk, device=DEV)
    return m.masked_fill_(torch.arange(lk, device=DEV)[None, None, :] >= n[:, None, None], -math.inf)


def _inputs(c, seed):
    r = _Rng(seed)
    k = c["kind"]
    s = {}
    if k == "mlp":
        s["x"] = r.normal(c["batch"], c["din"])
        s["w1"], s["b1"] = r.linear(c["din"], c["hidden"])
        s["w2"], s["b2"] = r.linear(c["hidden"], c["dout"])
        s["t"] = r.ints(0, c["dout"], c["batch"])
    elif k == "linear":
        s["x"] = r.normal(c["rows"], c["din"])
        s["w"], s["b"] = r.linear(c["din"], c["dout"])
        s["g"] = r.normal(c["rows"], c["dout"], std=1.0 / c["rows"])
    elif k == "ffn":
        s["x"], s["res"] = r.normal(c["rows"], c["d"]), r.normal(c["rows"], c["d"])
        s["w1"], s["b1"] = r.linear(c["d"], c["f"])
        s["w2"], s["b2"] = r.linear(c["f"], c["d"])
        s["g"] = r.normal(c["rows"], c["d"], std=2.0 / (c["rows"] * c["d"]))
    elif k == "attn":
        b, h, n, d = c["batch"], c["heads"], c["seq"], c["dim"]
        s["qkv"] = r.normal(b * n, 3 * h * d)
        s["mask"] = _key_mask(r, b, n, n) if c["mask"] else None
        s["g"] = r.normal(b * n, h * d, std=1.0 / (b * n))
    elif k == "cross":
        b, h, d = c["batch"], c["heads"], c["dim"]
        s["q"], s["k"], s["v"] = r.normal(b, c["lq"], h, d), r.normal(b, c["lk"], h, d), r.normal(b, c["lk"], h, d)
        s["mask"] = _key_mask(r, b, c["lq"], c["lk"]) if c["mask"] else None
        s["g"] = r.normal(b, c["lq"], h, d, std=1.0 / (b * c["lq"]))
    elif k in ("conv", "stage"):
        n, ci, co, h, w = c["n"], c["cin"], c["cout"], c["h"], c["w"]
        # images for a first layer, a previous stage's rectified activations after it
        s["x"] = r.normal(n, ci, h, w)
        s["x"] = s["x"].abs_().mul_(0.5) if ci == 1 else s["x"].clamp_(min=0)
        b = 1.0 / math.sqrt(9 * ci)
        s["w"], s["b"] = r.uniform(b, co, ci, 3, 3), r.uniform(b, co)
        if k == "conv":
            s["g"] = r.normal(n, co, h, w, std=1.0 / (n * h * w))
        else:
            act = r.normal(n, co, h, w).clamp_(min=0)
            oh, ow, pw = h // 2, w // c["pw"], c["pw"]
            win = act.view(n, co, oh, 2, ow, pw).permute(0, 1, 2, 4, 3, 5).reshape(n, co, oh, ow, 2 * pw)
            at = win.argmax(-1)
            row = torch.arange(oh, device=DEV)[:, None] * 2 + at // pw
            col = torch.arange(ow, device=DEV)[None, :] * pw + at % pw
            plane = torch.arange(n * co, device=DEV).view(n, co, 1, 1) * (h * w)
            s["act"], s["idx"] = act, (plane + row * w + col).to(torch.int32)
            s["g"] = r.normal(n, co, oh, ow, std=1.0 / (n * oh * ow))
    elif k == "ctc":
        b, t, cls = c["batch"], c["time"], c["classes"]
        s["x"] = r.normal(t * b, c["din"])
        s["w"], s["b"] = r.linear(c["din"], cls)
        s["tlen"] = r.ints(1, c["maxlen"] + 1, b)
        s["ilen"] = torch.full((b,), t, device=DEV, dtype=torch.int32)
        s["labels"] = r.ints(1, cls, int(s["tlen"].sum()))
    elif k == "block":
        b, n, d, f = c["batch"], c["seq"], c["heads"] * c["dim"], c["f"]
        s["x"], s["target"], s["mask"] = r.normal(b * n, d), r.normal(b * n, d), _key_mask(r, b, n, n)
        shapes = _block_shapes(d, f)
        total = sum(math.prod(v) for v in shapes.values())
        s["p"], off = _new(total), 0
        for name, shape in shapes.items():
            m = math.prod(shape)
            v = s["p"][off:off + m]
            if name in ("ga1", "ga2"):
                v.copy_(r.normal(m, std=0.02).add_(1.0))
            else:
                v.copy_(r.uniform(1.0 / math.sqrt(f if name in ("w2", "b2") else d), m))
            off += m
        scale = 2.0 / (b * n * d) * math.sqrt(b * n)  # moments of gradients of the loss's own size
        s["m"] = r.normal(total, std=0.1 * scale)
        s["v"] = r.normal(total).square_().add_(0.1).mul_(scale * scale)
    elif k == "adam":
        n = c["params"]
        s["p"], s["g"] = r.normal(n, std=0.05), r.normal(n, std=1e-3)
        s["m"] = r.normal(n, std=1e-4)
        s["v"] = r.normal(n, std=1e-3).square_().add_(1e-8)
    return s


def _block_shapes(d, f):
    return {"ga1": (d,), "be1": (d,), "wqkv": (3 * d, d), "bqkv": (3 * d,), "wo": (d, d), "bo": (d,), "ga2": (d,),
            "be2": (d,), "w1": (f, d), "b1": (f,), "w2": (d, f), "b2": (d,)}


def _views(flat, shapes):
    out, off = {}, 0
    for name, shape in shapes.items():
        m = math.prod(shape)
        out[name] = flat[off:off + m].view(shape)
        off += m
    return out


LR, B1, B2, EPS, WD, STEP = 1e-4, 0.9, 0.999, 1e-8, 0.01, 1000


# ----------------------------------------------------------------------------------------------------------- prepare
class _Calls:
    """The library calls of one pass with their arguments bound, and the outputs they leave."""

    def __init__(self):
        self.ctx = _ctx()
        self.calls, self.keep, self.out = [], [], {}

    def add(self, name, *args):
        conv = []
        for a in args:
            if isinstance(a, torch.Tensor):
                self.keep.append(a)
                conv.append(C.c_void_p(a.data_ptr()))
            else:
                conv.append(a)
        self.calls.append((getattr(self.ctx.L, name), name, (self.ctx.h, *conv)))


def _dw_items(items):
    arr = (_PKG.om_linear_dw * len(items))()
    for a, (g, x, dw, db) in zip(arr, items):
        a.g, a.x, a.dw, a.db = g.data_ptr(), x.data_ptr(), dw.data_ptr(), db.data_ptr() if db is not None else None
        a.in_, a.out, a.acc_dw, a.acc_db = x.shape[1], g.shape[1], 0, 0
    return arr


def _adam_scalars(ctx):
    ss, sq = C.c_float(), C.c_float()
    ctx.L.om_adam_scalars(LR, B1, B2, STEP, C.byref(ss), C.byref(sq))
    return ss.value, sq.value


def prepare(case, seed):
    c, s, q = case, _inputs(case, seed), _Calls()
    k, o = case["kind"], q.out
    if k == "mlp":
        b, di, h, do = c["batch"], c["din"], c["hidden"], c["dout"]
        a, dz, dh, lp, bad = _new(b, h), _new(b, do), _new(b, h), _new(b, do), _new(1, dtype=torch.int32)
        o.update(z=_new(b, do), loss=_new(1), dw1=_new(h, di), db1=_new(h), dw2=_new(do, h), db2=_new(do))
        q.add("om_linear_relu_fwd", s["x"], s["w1"], s["b1"], a, b, di, h)
        q.add("om_linear_fwd", a, s["w2"], s["b2"], o["z"], b, h, do)
        q.add("om_xent_fwd_unit", o["z"], s["t"], lp, o["loss"], bad, dz, b, do, -100, None)
        q.add("om_linear_bwd", dz, a, s["w2"], dh, o["dw2"], o["db2"], b, h, do, 0, 0, 0)
        q.add("om_linear_relu_bwd", dh, a, s["x"], s["w1"], None, o["dw1"], o["db1"], b, di, h, 0, 0, 0)
    elif k == "linear":
        r, di, do = c["rows"], c["din"], c["dout"]
        o.update(y=_new(r, do), dx=_new(r, di), dw=_new(do, di))
        if c["bias"]:
            o["db"] = _new(do)
        q.add("om_linear_fwd", s["x"], s["w"], s["b"] if c["bias"] else None, o["y"], r, di, do)
        q.add("om_linear_bwd", s["g"], s["x"], s["w"], o["dx"], o["dw"], o.get("db"), r, di, do, 0, 0, 0)
    elif k == "ffn":
        r, d, f = c["rows"], c["d"], c["f"]
        a, sl, dh = _new(r, f), _new(r, f), _new(r, f)
        o.update(y=_new(r, d), dx=_new(r, d), dw1=_new(f, d), db1=_new(f), dw2=_new(d, f), db2=_new(d))
        q.add("om_linear_gelu_fwd_slope", s["x"], s["w1"], s["b1"], a, sl, r, d, f)
        q.add("om_linear_fwd_resid", a, s["w2"], s["b2"], s["res"], o["y"], r, f, d)
        q.add("om_linear_bwd_dx_slope", s["g"], s["w2"], sl, dh, r, f, d)
        q.add("om_linear_bwd_dx_resid", dh, s["w1"], s["g"], o["dx"], r, d, f)
        q.add("om_linear_bwd_dw_group", 2, _dw_items([(s["g"], a, o["dw2"], o["db2"]), (dh, s["x"], o["dw1"], o["db1"])]), r)
        q.keep += [a, sl, dh, s]
    elif k == "attn":
        b, h, n, d = c["batch"], c["heads"], c["seq"], c["dim"]
        e, st = h * d, _new(2 * b * h * n)
        o.update(o=_new(b * n, e), dqkv=_new(b * n, 3 * e))
        x, y = s["qkv"], o["dqkv"]
        qkv, dq = [x[:, i * e:] for i in range(3)], [y[:, i * e:] for i in range(3)]
        sc = 1.0 / math.sqrt(d)
        q.add("om_attention_fwd_flash", *qkv, 3 * e, s["mask"], 1, o["o"], e, st, b, h, n, d, sc)
        q.add("om_attention_bwd_flash", *qkv, 3 * e, s["mask"], 1, o["o"], e, st, s["g"], e, *dq, 3 * e, b, h, n, d, sc, 0)
    elif k == "cross":
        b, h, lq, lk, d = c["batch"], c["heads"], c["lq"], c["lk"], c["dim"]
        o.update(o=_new(b, lq, h, d), dq=_new(b, lq, h, d), dk=_new(b, lk, h, d), dv=_new(b, lk, h, d))
        p, ds, sc = _new(b, h, lq, lk), _new(b, h, lq, lk), 1.0 / math.sqrt(d)
        q.add("om_attention_fwd", s["q"], s["k"], s["v"], s["mask"], 1, o["o"], p, b, h, lq, lk, d, sc)
        q.add("om_attention_bwd", s["q"], s["k"], s["v"], p, s["g"], o["dq"], o["dk"], o["dv"], ds, b, h, lq, lk, d, sc, 0)
    elif k == "conv":
        n, ci, co, h, w = c["n"], c["cin"], c["cout"], c["h"], c["w"]
        o.update(y=_new(n, co, h, w), dw=_new(co, ci, 3, 3), db=_new(co))
        if c["dx"]:
            o["dx"] = _new(n, ci, h, w)
        q.add("om_conv2d_relu_fwd", s["x"], s["w"], s["b"], o["y"], n, ci, h, w, co, 3, 3, 1, 1)
        q.add("om_conv2d_bwd", s["g"], s["x"], s["w"], o.get("dx"), o["dw"], o["db"], n, ci, h, w, co, 3, 3, 1, 1, 0, 0)
    elif k == "stage":
        n, ci, co, h, w, pw = c["n"], c["cin"], c["cout"], c["h"], c["w"], c["pw"]
        a, idx, da, oh, ow = _new(n, co, h, w), _new(n, co, h // 2, w // pw, dtype=torch.int32), _new(n, co, h, w), h // 2, w // pw
        o.update(y=_new(n, co, oh, ow), dw=_new(co, ci, 3, 3), db=_new(co))
        if ci > 1:
            o["dx"] = _new(n, ci, h, w)
        q.add("om_conv2d_relu_pool_fwd", s["x"], s["w"], s["b"], a, o["y"], idx, n, ci, h, w, co, 3, 3, 1, 1, 2, pw, 2, pw)
        q.add("om_maxpool_relu_bwd", s["g"], s["idx"], s["act"], da, n, co, h, w, oh, ow, 2, pw, 2, pw, 0, 0, 0)
        q.add("om_conv2d_bwd", da, s["x"], s["w"], o.get("dx"), o["dw"], o["db"], n, ci, h, w, co, 3, 3, 1, 1, 0, 0)
    elif k == "ctc":
        b, t, cls, di = c["batch"], c["time"], c["classes"], c["din"]
        host = [x.cpu().contiguous() for x in (s["ilen"], s["tlen"], s["labels"])]
        hp, nt, ml = [C.c_void_p(x.data_ptr()) for x in host], int(host[2].numel()), int(host[1].max())
        nb = q.ctx.L.om_ctc_tables_bytes(t, b, ml)
        tab, lp, z, dlp, one = _new((nb + 3) // 4 + 2), _new(t * b, cls), _new(t * b, cls), _new(t * b, cls), torch.ones(1, device=DEV)
        dz = _new(t * b, cls)
        o.update(lp=lp, loss=_new(1), dx=_new(t * b, di), dw=_new(cls, di), db=_new(cls))
        lens = (s["labels"], s["ilen"], s["tlen"])
        q.add("om_linear_fwd", s["x"], s["w"], s["b"], z, t * b, di, cls)
        q.add("om_logsoftmax_fwd", z, lp, t * b, cls)
        q.add("om_ctc_fwd_tables", lp, *lens, *hp, nt, t, b, cls, 0, 1, 0, o["loss"], tab, nb)
        q.add("om_ctc_bwd_tables", lp, *lens, *hp, nt, one, dlp, t, b, cls, 0, 1, 0, tab, nb)
        q.add("om_logsoftmax_bwd", dlp, lp, dz, t * b, cls, 0)
        q.add("om_linear_bwd", dz, s["x"], s["w"], o["dx"], o["dw"], o["db"], t * b, di, cls, 0, 0, 0)
        q.keep += host
    elif k == "block":
        _block_calls(c, s, q)
    elif k == "adam":
        n, seg = c["params"], c["segments"]
        cuts = [n * i // seg for i in range(seg + 1)]
        ptrs = (C.c_void_p * seg)(*[s["g"].data_ptr() + 4 * v for v in cuts[:-1]])
        lens = (C.c_int64 * seg)(*[b - a for a, b in zip(cuts, cuts[1:])])
        coef = _new(1)
        o.update(p=s["p"], m=s["m"], v=s["v"], norm=_new(1))
        q.add("om_clip_grad_norm", seg, ptrs, lens, 1.0, 0, 0, o["norm"], coef)
        q.add("om_adam_step_scaled", s["p"], s["g"], s["m"], s["v"], None, n, LR, B1, B2, EPS, WD, 1, *_adam_scalars(q.ctx), coef)
    torch.cuda.synchronize()  # the inputs come from torch's stream, the calls run on the context's
    return q


def _block_calls(c, s, q):
    b, n, hd, dim, f = c["batch"], c["seq"], c["heads"], c["dim"], c["f"]
    d, r = hd * dim, b * n
    p = _views(s["p"], _block_shapes(d, f))
    grads = torch.zeros_like(s["p"])
    gr = _views(grads, _block_shapes(d, f))
    ln1, ln2, x1, x1g, qkv, dqkv = _new(r, d), _new(r, d), _new(r, d), _new(r, d), _new(r, 3 * d), _new(r, 3 * d)
    st1, st2, stats, ao, dao = _new(2, r), _new(2, r), _new(2 * b * hd * n), _new(r, d), _new(r, d)
    a, sl, dh, dl, gy = _new(r, f), _new(r, f), _new(r, f), _new(r, d), _new(r, d)
    ch = q.ctx.L.om_layernorm_bwd_chunks(r, d)
    parts = [_new(ch, d, dtype=torch.float64) for _ in range(4)]
    o = q.out
    o.update(y=_new(r, d), loss=_new(1), dx=_new(r, d), grads=grads, p=s["p"], m=s["m"], v=s["v"])
    sc, e = 1.0 / math.sqrt(dim), d
    q3, d3 = [qkv[:, i * e:] for i in range(3)], [dqkv[:, i * e:] for i in range(3)]
    q.add("om_layernorm_fwd", s["x"], p["ga1"], p["be1"], ln1, st1[0], st1[1], r, d, 1e-5)
    q.add("om_linear_fwd", ln1, p["wqkv"], p["bqkv"], qkv, r, d, 3 * d)
    q.add("om_attention_fwd_flash", *q3, 3 * e, s["mask"], 1, ao, e, stats, b, hd, n, dim, sc)
    q.add("om_linear_fwd_resid", ao, p["wo"], p["bo"], s["x"], x1, r, d, d)
    q.add("om_layernorm_fwd", x1, p["ga2"], p["be2"], ln2, st2[0], st2[1], r, d, 1e-5)
    q.add("om_linear_gelu_fwd_slope", ln2, p["w1"], p["b1"], a, sl, r, d, f)
    q.add("om_linear_fwd_resid_mse", a, p["w2"], p["b2"], x1, s["target"], o["y"], gy, o["loss"], r, f, d, None)
    q.add("om_linear_bwd_dx_slope", gy, p["w2"], sl, dh, r, f, d)
    q.add("om_linear_bwd", dh, ln2, p["w1"], dl, None, None, r, d, f, 0, 0, 0)
    q.add("om_layernorm_bwd_partials", dl, x1, p["ga2"], st2[0], st2[1], gy, x1g, 0, parts[0], parts[1], r, d)
    q.add("om_linear_bwd", x1g, ao, p["wo"], dao, None, None, r, d, d, 0, 0, 0)
    q.add("om_attention_bwd_flash", *q3, 3 * e, s["mask"], 1, ao, e, stats, dao, e, *d3, 3 * e, b, hd, n, dim, sc, 0)
    q.add("om_linear_bwd", dqkv, ln1, p["wqkv"], dl, None, None, r, d, 3 * d, 0, 0, 0)
    q.add("om_layernorm_bwd_partials", dl, s["x"], p["ga1"], st1[0], st1[1], x1g, o["dx"], 0, parts[2], parts[3], r, d)
    dw = _dw_items([(gy, a, gr["w2"], gr["b2"]), (dh, ln2, gr["w1"], gr["b1"]), (x1g, ao, gr["wo"], gr["bo"]),
                    (dqkv, ln1, gr["wqkv"], gr["bqkv"])])
    cs = (_PKG.om_column_sum * 4)()
    for item, part, out in zip(cs, parts, ("ga2", "be2", "ga1", "be1")):
        item.part, item.out, item.chunks, item.cols, item.acc = part.data_ptr(), gr[out].data_ptr(), ch, d, 0
    q.add("om_param_grads_group", 4, dw, r, 4, cs)
    total = s["p"].numel()
    q.add("om_adam_step", s["p"], grads, s["m"], s["v"], None, total, LR, B1, B2, EPS, WD, 1, *_adam_scalars(q.ctx))
    q.keep += [s, ln1, ln2, x1, x1g, dqkv, ao, a, dh, gy, parts]


def run(state):
    for fn, name, args in state.calls:
        if fn(*args):
            raise RuntimeError("%s: %s" % (name, state.ctx.L.om_last_error(state.ctx.h).decode()))
    return state.out


# -------------------------------------------------------------------------------------------------------------- work
def work(case):
    c, k = case, case["kind"]
    if k == "mlp":
        b, di, h, do = c["batch"], c["din"], c["hidden"], c["dout"]
        return {"bytes": 4 * (b * di + 2 * (di * h + h * do) + b * do), "flops": 2 * b * (2 * di * h + 3 * h * do)}
    if k == "linear":
        r, di, do = c["rows"], c["din"], c["dout"]
        return {"bytes": 4 * (2 * r * (di + do) + 2 * di * do), "flops": 6 * r * di * do}
    if k == "ffn":
        r, d, f = c["rows"], c["d"], c["f"]
        return {"bytes": 4 * (5 * r * d + 4 * d * f), "flops": 12 * r * d * f}
    if k == "attn":
        b, h, n, d = c["batch"], c["heads"], c["seq"], c["dim"]
        return {"bytes": 4 * (b * n * h * d * 8 + (b * n * n if c["mask"] else 0)), "flops": 14 * b * h * n * n * d}
    if k == "cross":
        b, h, lq, lk, d = c["batch"], c["heads"], c["lq"], c["lk"], c["dim"]
        return {"bytes": 4 * (b * h * d * (4 * lq + 4 * lk) + (b * lq * lk if c["mask"] else 0)),
                "flops": 12 * b * h * lq * lk * d}
    if k in ("conv", "stage"):
        n, ci, co, hw = c["n"], c["cin"], c["cout"], c["h"] * c["w"]
        dx = c["dx"] if k == "conv" else ci > 1
        by = 4 * (n * hw * (ci * (2 if dx else 1) + 2 * co) + 18 * ci * co)
        return {"bytes": by, "flops": 18 * n * hw * ci * co * (3 if dx else 2)}
    if k == "ctc":
        r, di, cls = c["batch"] * c["time"], c["din"], c["classes"]
        return {"bytes": 4 * (2 * r * di + r * cls + 2 * di * cls), "flops": 6 * r * di * cls}
    if k == "block":
        b, n, d, f = c["batch"], c["seq"], c["heads"] * c["dim"], c["f"]
        r, par = b * n, sum(math.prod(v) for v in _block_shapes(d, f).values())
        return {"bytes": 4 * (4 * r * d + b * n * n + 7 * par), "flops": 3 * 2 * r * (4 * d * d + 2 * d * f) + 14 * r * n * d}
    return {"bytes": 28 * c["params"], "flops": 12 * c["params"]}


def tolerance(case):
    # 32-bit sums in another order. Against 64 bits the Linear weight gradients over 16384 rows were 1.7e-6 off, over
    # 4096 rows 6e-7, everything else at most 5e-7: about four times that.
    rel = {"ffn": 8e-6, "linear": 5e-6, "block": 5e-6}.get(case["kind"], 3e-6)
    return {"rel": rel, "max": 40 * rel}


# ------------------------------------------------------------------------------------------------------------- exact
def _gelu(x):
    return 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))


def _attend(q, k, v, mask, scale):
    """q, k, v [B, H, L, D] in 64 bits; mask [B, Lq, Lk] or None."""
    x = torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale
    if mask is not None:
        x = x + mask[:, None]
    return torch.matmul(torch.softmax(x, -1), v)


def _heads(x, b, n, h, d):
    return x.reshape(b, n, h, d).permute(0, 2, 1, 3).contiguous()


def _merge(x):
    b, h, n, d = x.shape
    return x.permute(0, 2, 1, 3).reshape(b * n, h * d)


def _conv(x, w, flip=False):
    """3x3, stride 1, padding 1 as nine products; flip: the input gradient's transposed convolution."""
    n, ci, h, wd = x.shape
    xp = torch.nn.functional.pad(x, (1, 1, 1, 1))
    co = w.shape[1] if flip else w.shape[0]
    y = torch.zeros(n, co, h * wd, device=x.device, dtype=x.dtype)
    for i in range(3):
        for j in range(3):
            tap = w[:, :, 2 - i, 2 - j].t() if flip else w[:, :, i, j]
            y += torch.matmul(tap.contiguous(), xp[:, :, i:i + h, j:j + wd].reshape(n, ci, h * wd))
    return y.view(n, co, h, wd)


def _conv_dw(g, x):
    n, ci, h, w = x.shape
    co = g.shape[1]
    xp = torch.nn.functional.pad(x, (1, 1, 1, 1))
    gm = g.permute(1, 0, 2, 3).reshape(co, -1)
    dw = torch.empty(co, ci, 3, 3, device=x.device, dtype=x.dtype)
    for i in range(3):
        for j in range(3):
            dw[:, :, i, j] = gm @ xp[:, :, i:i + h, j:j + w].permute(0, 2, 3, 1).reshape(-1, ci)
    return dw


def _ctc_loss(lp, labels, tlen):
    """Mean over the batch of -log p / target length (blank 0), lp [T, B, C] in 64 bits."""
    t, b, _ = lp.shape
    off, total = 0, 0.0
    for i in range(b):
        n = int(tlen[i])
        ext = torch.zeros(2 * n + 1, dtype=torch.long, device=lp.device)
        ext[1::2] = labels[off:off + n].long()
        off += n
        e = lp[:, i, ext]
        skip = torch.zeros(2 * n + 1, dtype=torch.bool, device=lp.device)
        skip[2:] = (ext[2:] != 0) & (ext[2:] != ext[:-2])
        low = torch.full((2,), -1e300, device=lp.device, dtype=lp.dtype)
        al = torch.cat([e[0, :2], torch.full((2 * n - 1,), -1e300, device=lp.device, dtype=lp.dtype)])
        for k in range(1, t):
            s2 = torch.where(skip, torch.cat([low, al[:-2]]), torch.full_like(al, -1e300))
            al = torch.logsumexp(torch.stack([al, torch.cat([low[:1], al[:-1]]), s2]), 0) + e[k]
        total = total - torch.logsumexp(al[-2:], 0) / n
    return total / b


def _adam64(p, g, m, v):
    m = B1 * m + (1 - B1) * g
    v = B2 * v + (1 - B2) * g * g
    upd = LR / (1 - B1 ** STEP) * m / (v.sqrt() / math.sqrt(1 - B2 ** STEP) + EPS)
    return p * (1 - LR * WD) - upd, m, v


def exact(case, seed):
    c, k = case, case["kind"]
    s = {n: v.double() if isinstance(v, torch.Tensor) and v.dtype == torch.float32 else v
         for n, v in _inputs(case, seed).items()}
    if k == "mlp":
        w = {n: s[n].requires_grad_() for n in ("w1", "b1", "w2", "b2")}
        z = torch.relu(s["x"] @ w["w1"].t() + w["b1"]) @ w["w2"].t() + w["b2"]
        loss = torch.nn.functional.cross_entropy(z, s["t"].long())
        g = torch.autograd.grad(loss, [w["w1"], w["b1"], w["w2"], w["b2"]])
        return {"z": z.detach(), "loss": loss.detach().view(1), "dw1": g[0], "db1": g[1], "dw2": g[2], "db2": g[3]}
    if k == "linear":
        y = s["x"] @ s["w"].t()
        out = {"y": y + s["b"] if c["bias"] else y, "dx": s["g"] @ s["w"], "dw": s["g"].t() @ s["x"]}
        if c["bias"]:
            out["db"] = s["g"].sum(0)
        return out
    if k == "ffn":
        h = s["x"] @ s["w1"].t() + s["b1"]
        a = _gelu(h)
        slope = 0.5 * (1 + torch.erf(h / math.sqrt(2.0))) + h * torch.exp(-0.5 * h * h) / math.sqrt(2 * math.pi)
        dh = (s["g"] @ s["w2"]) * slope
        return {"y": a @ s["w2"].t() + s["b2"] + s["res"], "dx": dh @ s["w1"] + s["g"], "dw1": dh.t() @ s["x"],
                "db1": dh.sum(0), "dw2": s["g"].t() @ a, "db2": s["g"].sum(0)}
    if k == "attn":
        b, h, n, d = c["batch"], c["heads"], c["seq"], c["dim"]
        x = s["qkv"].requires_grad_()
        e = h * d
        y = _merge(_attend(*[_heads(x[:, i * e:(i + 1) * e], b, n, h, d) for i in range(3)], s["mask"], 1 / math.sqrt(d)))
        return {"o": y.detach(), "dqkv": torch.autograd.grad(y, x, s["g"])[0]}
    if k == "cross":
        qkv = [s[n].requires_grad_() for n in ("q", "k", "v")]
        y = _attend(*[t.permute(0, 2, 1, 3).contiguous() for t in qkv], s["mask"], 1 / math.sqrt(c["dim"]))
        y = y.permute(0, 2, 1, 3)
        g = torch.autograd.grad(y, qkv, s["g"])
        return {"o": y.detach().contiguous(), "dq": g[0], "dk": g[1], "dv": g[2]}
    if k in ("conv", "stage"):
        y = torch.relu(_conv(s["x"], s["w"]) + s["b"][None, :, None, None])
        g = s["g"]
        if k == "stage":
            y = torch.nn.functional.max_pool2d(y, (2, c["pw"]), (2, c["pw"]))
            full = torch.zeros(s["act"].numel(), device=DEV, dtype=torch.float64)
            full[s["idx"].long().view(-1)] = g.reshape(-1)
            g = full.view(s["act"].shape) * (s["act"] > 0)
        out = {"y": y, "dw": _conv_dw(g, s["x"]), "db": g.sum((0, 2, 3))}
        if c["dx"] if k == "conv" else c["cin"] > 1:
            out["dx"] = _conv(g, s["w"], True)
        return out
    if k == "ctc":
        b, t, cls = c["batch"], c["time"], c["classes"]
        if b * t > 1100:
            return None  # the recursion above is a loop over sequences and time steps
        w = {n: s[n].requires_grad_() for n in ("x", "w", "b")}
        lp = torch.log_softmax(w["x"] @ w["w"].t() + w["b"], -1)
        loss = _ctc_loss(lp.view(t, b, cls), s["labels"], s["tlen"])
        g = torch.autograd.grad(loss, [w["x"], w["w"], w["b"]])
        return {"lp": lp.detach(), "loss": loss.detach().view(1), "dx": g[0], "dw": g[1], "db": g[2]}
    if k == "block":
        b, n, hd, dim, f = c["batch"], c["seq"], c["heads"], c["dim"], c["f"]
        d = hd * dim
        flat, x = s["p"].requires_grad_(), s["x"].requires_grad_()
        p = _views(flat, _block_shapes(d, f))
        ln = torch.nn.functional.layer_norm
        qkv = ln(x, (d,), p["ga1"], p["be1"], 1e-5) @ p["wqkv"].t() + p["bqkv"]
        ao = _merge(_attend(*[_heads(qkv[:, i * d:(i + 1) * d], b, n, hd, dim) for i in range(3)], s["mask"],
                            1 / math.sqrt(dim)))
        x1 = ao @ p["wo"].t() + p["bo"] + x
        y = _gelu(ln(x1, (d,), p["ga2"], p["be2"], 1e-5) @ p["w1"].t() + p["b1"]) @ p["w2"].t() + p["b2"] + x1
        loss = (y - s["target"]).square().mean()
        g, dx = torch.autograd.grad(loss, [flat, x])
        np_, m, v = _adam64(flat.detach(), g, s["m"], s["v"])
        return {"y": y.detach(), "loss": loss.detach().view(1), "dx": dx, "grads": g, "p": np_, "m": m, "v": v}
    norm = s["g"].norm()
    g = s["g"] * min(1.0, 1.0 / (float(norm) + 1e-6))
    p, m, v = _adam64(s["p"], g, s["m"], s["v"])
    return {"p": p, "m": m, "v": v, "norm": norm.view(1)}
