"""The work whose speed is kept in view: what midge's engine and a serving loop
ask of the library, each through the entry point that they call.

    apply      expert_apply with the routing given (mh_stack_apply_dev)
    decode     embedding rows, then the MoE layers of a decode step for one or
               several sequences (mh_dequant_dev, mh_stack_decode)
    prefill    embedding rows of a prompt chunk, then one layer's MoE for the
               whole chunk (mh_dequant_dev, mh_moe_prefill_dev)
    matvec     trunk and head matrices on 1..64 tokens (mh_matvec_dev)
    attention  one layer's attention over the tokens of a chunk, one by one,
               as the batched prefill calls it (mh_attention_dev)
    sample     the next token from the logits (mh_sample_dev)
    token      a whole decode token and its sampling (mh_forward_dev,
               mh_sample_dev)

The listed sizes are gpt-oss's (hidden = ffn = 2880, top-4, 32 experts a layer
or 128); `draw` spreads over batch and chunk sizes, other widths, dtypes,
context lengths and vocabularies. Weights and activations are random with the
spreads of real layers: 4-bit codes uniform, block scales powers of two,
int8 weights uniform under a row scale, router logits of a few units.
"""
import ctypes as C
import math

import torch

import midge_amd
from midge_amd import DT_F32, DT_MXFP4, DT_Q4G32, DT_Q8R, DevBuf, _lib
from midge_amd.kern import WT, dequant_dev, matvec_dev
from midge_amd.layout import blob_sizes
from midge_amd.moe import MoELayer, Stack, moe_prefill_dev, sample_dev
from midge_amd.synth import MoEShape

DTS = {"f32": DT_F32, "q8r": DT_Q8R, "q4g32": DT_Q4G32, "mxfp4": DT_MXFP4}
HEADS, KV_HEADS, HEAD_DIM = 64, 8, 64
EPS = 1e-5


# ------------------------------------------------------------------ cases

def _moe(kind, name=None, hidden=2880, ffn=2880, experts=128, top_k=4, dt="mxfp4", layers=1, tokens=1):
    c = dict(kind=kind, hidden=hidden, ffn=ffn, experts=experts, top_k=top_k, dt=dt, layers=layers, tokens=tokens)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one token's four experts with the routing made elsewhere: the smallest MoE call
        _moe("apply", "apply_one_token", experts=32),
        # a decode step of one sequence: the launch that a chat spends its time in
        _moe("decode", "decode_b1", layers=8),
        # decode steps of a small and of a larger serving batch
        _moe("decode", "decode_b16", layers=2, tokens=16),
        _moe("decode", "decode_b40", layers=1, tokens=40),
        # the engine's own prompt chunk (64 tokens) on a 128-expert layer
        _moe("prefill", "prefill_64", tokens=64),
        # longer prompts on a 32-expert layer: the batched prefill, and the largest call
        _moe("prefill", "prefill_512", experts=32, tokens=512),
        _moe("prefill", "prefill_2000", experts=32, tokens=2000),
        # a trunk projection for one token: latency
        dict(name="qkv_b1", kind="matvec", dt="q8r", rows=5120, cols=2880, batch=1),
        # a long 4-bit matrix for one token: streaming
        dict(name="mxfp4_b1", kind="matvec", dt="mxfp4", rows=524288, cols=2880, batch=1),
        # the output head for a serving batch
        dict(name="lm_head_b32", kind="matvec", dt="q8r", rows=201088, cols=2880, batch=32),
        # one token's attention in a full layer at a usual context
        dict(name="attention_1044", kind="attention", tokens=1, pos=1043, window=0),
        # a whole token of a two-layer slice (one sliding layer, one full), head and sampling included
        dict(name="token_2_layers", kind="token", layers=2, pos=266, vocab=201088, temp=0.8, topp=0.9),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# other widths than gpt-oss's: a smaller model's, and one of odd multiples of 32
_WIDTHS = [(2880, 2880)] * 4 + [(2048, 1536), (1024, 768), (1504, 1056)]


def draw(rng):
    kind = rng.choice(["apply", "decode", "decode", "decode", "prefill", "prefill", "prefill", "matvec", "matvec",
                       "attention", "sample", "token"])
    if kind in ("apply", "decode", "prefill"):
        hidden, ffn = rng.choice(_WIDTHS)
        dt = rng.choice(["mxfp4", "mxfp4", "mxfp4", "q4g32"])
        c = dict(hidden=hidden, ffn=ffn, experts=rng.choice([32, 64, 128]), top_k=rng.choice([2, 4, 4, 4, 8]), dt=dt)
        if kind == "apply":
            return _moe(kind, **c)
        if kind == "decode":
            tokens = _log(rng, 1, 64)
            return _moe(kind, tokens=tokens, layers=rng.randint(1, 8) if tokens == 1 else rng.randint(1, 2), **c)
        return _moe(kind, tokens=_log(rng, 16, 2000 if dt == "mxfp4" and c["top_k"] <= 4 else 64), **c)
    if kind == "matvec":
        dt = rng.choice(["q8r", "q8r", "q8r", "mxfp4", "q4g32", "f32"])
        cols = rng.choice([2880, 2880, 4096, 2048, 1504, 640])
        batch = rng.choice([1, 1, _log(rng, 2, 64)])
        # a batch multiplies the reads of the types that have no batched kernel: those stay trunk-sized
        return dict(kind=kind, dt=dt, rows=_log(rng, 128, 201088 if dt == "q8r" or batch == 1 else 5760), cols=cols,
                    batch=batch)
    if kind == "attention":
        tokens = _log(rng, 1, 16)
        return dict(kind=kind, tokens=tokens, pos=_log(rng, 1, 4000), window=rng.choice([0, 128]))
    if kind == "sample":
        return dict(kind=kind, vocab=_log(rng, 20000, 201088), spread=rng.choice([3.0, 6.0, 12.0]),
                    temp=rng.choice([0.0, 0.7, 1.0]), topp=rng.choice([0.9, 0.95]))
    return dict(kind=kind, layers=rng.randint(1, 3), pos=_log(rng, 1, 2000), vocab=_log(rng, 20000, 201088),
                temp=rng.choice([0.0, 0.8]), topp=0.9)


# ----------------------------------------------------------- device memory

class Mem(DevBuf):
    """A library allocation that torch can look into, freed with its last view."""

    @property
    def __cuda_array_interface__(self):
        return {"shape": (self.nbytes,), "typestr": "|u1", "data": (self.ptr, False), "version": 2}

    def __del__(self):
        if self.ptr:
            self.free()


def alloc(nbytes, dtype=torch.uint8, shape=None):
    """(device pointer, view of it as a tensor, which keeps it alive)."""
    m = Mem(nbytes)
    t = torch.as_tensor(m, device="cuda").view(dtype)
    return m.ptr, t if shape is None else t.view(shape)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & (2**63 - 1))


class Tensor:
    """A random weight matrix in one of the four storage types, on the device."""

    def __init__(self, dt, rows, cols, g, lo, hi):
        self.dt, self.rows, self.cols = dt, rows, cols
        db, sb = blob_sizes(dt, rows, cols)
        ptr, data = alloc(db)
        sptr, self.scales = 0, None
        if dt == DT_F32:
            self.data = data.view(torch.float32).view(rows, cols)
            self.data.normal_(0, lo, generator=g)
        elif dt == DT_Q8R:
            self.data = data.view(torch.int8).view(rows, cols)
            self.data.random_(-127, 128, generator=g)
            sptr, self.scales = alloc(sb, torch.float32)
            self.scales.uniform_(lo, hi, generator=g)
        else:
            self.data = data.view(rows, cols // 2)
            self.data.random_(0, 256, generator=g)
            sptr, self.scales = alloc(sb, torch.float16, (rows, cols // 32))
            _scales_(self.scales, dt, g)
        self.wt = WT(dt, rows, cols, ptr, sptr or None)

    def exact(self, r0=0, r1=None):
        """Rows r0..r1 in 64 bits."""
        d = self.data[r0:r1]
        if self.dt == DT_F32:
            return d.double()
        if self.dt == DT_Q8R:
            return d.double() * self.scales[r0:r1, None].double()
        return _dequant4(self.dt, d, self.scales[r0:r1])


def _scales_(s, dt, g):
    """Block scales: powers of two for MXFP4 (its e8m0 scales), any f16 for q4g32."""
    if dt == DT_MXFP4:
        s.copy_(torch.exp2(torch.randint(-8, -3, s.shape, device="cuda", generator=g).float()))
    else:
        s.copy_(torch.rand(s.shape, device="cuda", generator=g) * 0.03 + 0.002)


def _dequant4(dt, codes, scales):
    if dt == DT_MXFP4:
        table = [0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6]
    else:
        table = [i - 8 for i in range(16)]
    table = torch.tensor(table, dtype=torch.float64, device="cuda")
    v = torch.stack((table[(codes & 15).long()], table[(codes >> 4).long()]), -1)   # low nibble = even column
    rows = codes.shape[0]
    return (v.view(rows, -1, 32) * scales.double()[:, :, None]).view(rows, -1)


def _vector(n, g, mean, spread):
    ptr, t = alloc(4 * n, torch.float32)
    t.normal_(mean, spread, generator=g)
    return ptr, t


# -------------------------------------------------------------- MoE layers

class Layer:
    """One MoE layer: expert table at the container's offsets, int8 router, norm."""

    def __init__(self, c, g):
        self.shape = MoEShape(hidden=c["hidden"], ffn=c["ffn"], n_experts=c["experts"], top_k=c["top_k"],
                              expert_dt=DTS[c["dt"]])
        s, lay = self.shape, self.shape.layout
        ptr, table = alloc(lay.layer_stride)
        self.table = table.view(s.n_experts, lay.expert_stride)
        for m in range(3):
            self.blob(m, 0).random_(0, 256, generator=g)
            _scales_(self.blob(m, 1), s.expert_dt, g)
            self.blob(m, 2).normal_(0, 0.02, generator=g)
        # logits of a few units: sums of `hidden` products of a normal and a uniform int8
        top = 4.0 / (73.6 * math.sqrt(s.hidden))
        self.router = Tensor(DT_Q8R, s.n_experts, s.hidden, g, top / 4, top)
        bptr, self.bias = _vector(s.n_experts, g, 0.0, 0.2)
        nptr, self.norm = _vector(s.hidden, g, 1.0, 0.1)
        self.layer = MoELayer(s, ptr, self.router.wt, bptr, nptr)

    def blob(self, m, part):
        """Every expert's data, scales or bias of gate, up or down (a strided view)."""
        lay = self.shape.layout
        db, sb = blob_sizes(lay.dt, lay.rows[m], lay.cols[m])
        off, n = lay.off[3 * m + part], (db, sb, 4 * lay.rows[m])[part]
        v = self.table[:, off:off + n]
        return v if part == 0 else v.view(torch.float16 if part == 1 else torch.float32)

    def weight(self, e, m):
        lay = self.shape.layout
        return _dequant4(lay.dt, self.blob(m, 0)[e].reshape(lay.rows[m], -1),
                         self.blob(m, 1)[e].reshape(lay.rows[m], -1))

    def route(self, x):
        s = self.shape
        xb = x / torch.sqrt((x * x).mean(-1, keepdim=True) + s.norm_eps) * self.norm.double()
        logits = xb @ self.router.exact().T + self.bias.double()
        val, sel = torch.topk(logits, s.top_k, dim=-1)
        return xb, sel, torch.softmax(val, -1)

    def experts(self, xb, sel, w):
        """sum_i w_i expert_{sel_i}(xb) per token, in 64 bits."""
        s, out = self.shape, torch.zeros_like(xb)
        for e in torch.unique(sel).tolist():
            t, i = torch.nonzero(sel == e, as_tuple=True)
            g = xb[t] @ self.weight(e, 0).T + self.blob(0, 2)[e].double()
            u = xb[t] @ self.weight(e, 1).T + self.blob(1, 2)[e].double()
            g, u = g.clamp(max=s.limit), u.clamp(-s.limit, s.limit)
            y = (g * torch.sigmoid(s.alpha * g) * (u + 1)) @ self.weight(e, 2).T + self.blob(2, 2)[e].double()
            out.index_add_(0, t, y * w[t, i][:, None])
        return out

    def exact(self, x):
        xb, sel, w = self.route(x)
        return x + self.experts(xb, sel, w), sel.int(), w


class Decode:
    """The MoE half of the layer loop of a decode step."""

    def __init__(self, c, g):
        n, h, k = c["tokens"], c["hidden"], c["top_k"]
        self.n = n
        self.embed = Tensor(DT_F32, n, h, g, 1.0, 0.0)
        self.layers = [Layer(c, g) for _ in range(c["layers"])]
        self.xp, self.x = alloc(4 * n * h, torch.float32, (n, h))
        self.sp, self.sel = alloc(4 * len(self.layers) * n * k, torch.int32, (len(self.layers), n, k))
        self.wp, self.w = alloc(4 * len(self.layers) * n * k, torch.float32, (len(self.layers), n, k))
        torch.cuda.synchronize()
        self.stack = Stack([layer.layer for layer in self.layers], n)

    def run(self):
        dequant_dev(self.embed.wt, 0, self.n, self.xp)
        self.stack.decode(self.xp, self.n, self.sp, self.wp)
        return {"x": self.x, "sel": self.sel, "w": self.w}

    def exact(self):
        x, sel, w = self.embed.exact(), [], []
        for layer in self.layers:
            x, s, v = layer.exact(x)
            sel.append(s)
            w.append(v)
        return {"x": x, "sel": torch.stack(sel), "w": torch.stack(w)}

    def __del__(self):
        if hasattr(self, "stack"):
            self.stack.destroy()


class Apply:
    """One token through its experts, the routing given: x += sum_i w_i expert_i(xb)."""

    def __init__(self, c, g):
        h, k, e = c["hidden"], c["top_k"], c["experts"]
        self.layer = Layer(c, g)
        self.xbp, self.xb = _vector(h, g, 0.0, 1.0)
        self.embed = Tensor(DT_F32, 1, h, g, 1.0, 0.0)
        self.xp, self.x = alloc(4 * h, torch.float32)
        self.sp, self.sel = alloc(4 * k, torch.int32)
        self.sel.copy_(torch.randperm(e, device="cuda", generator=g)[:k])
        self.wp, self.w = alloc(4 * k, torch.float32)
        self.w.copy_(torch.softmax(torch.randn(k, device="cuda", generator=g), 0))
        torch.cuda.synchronize()
        self.stack = Stack([self.layer.layer], 1)

    def run(self):
        dequant_dev(self.embed.wt, 0, 1, self.xp)
        self.stack.apply(0, self.xbp, self.sp, self.wp, self.xp)
        return {"x": self.x}

    def exact(self):
        y = self.layer.experts(self.xb.double()[None], self.sel.long()[None], self.w.double()[None])
        return {"x": self.embed.exact()[0] + y[0]}

    def __del__(self):
        if hasattr(self, "stack"):
            self.stack.destroy()


class Prefill:
    """The MoE half of one layer of the batched prefill, on a chunk's embedding rows."""

    def __init__(self, c, g):
        n, h, k = c["tokens"], c["hidden"], c["top_k"]
        self.n = n
        self.embed = Tensor(DT_F32, n, h, g, 1.0, 0.0)
        self.layer = Layer(c, g)
        self.xp, self.x = alloc(4 * n * h, torch.float32, (n, h))
        self.sp, self.sel = alloc(4 * n * k, torch.int32, (n, k))
        self.wp, self.w = alloc(4 * n * k, torch.float32, (n, k))

    def run(self):
        dequant_dev(self.embed.wt, 0, self.n, self.xp)
        moe_prefill_dev(self.layer.layer, self.xp, self.n, self.sp, self.wp)
        return {"x": self.x, "sel": self.sel, "w": self.w}

    def exact(self):
        x, sel, w = self.layer.exact(self.embed.exact())
        return {"x": x, "sel": sel, "w": w}


# -------------------------------------------------------- trunk and head

class Matvec:
    def __init__(self, c, g):
        self.batch = c["batch"]
        self.t = Tensor(DTS[c["dt"]], c["rows"], c["cols"], g, 1e-3, 1e-2)
        self.xp, self.x = _vector(self.batch * c["cols"], g, 0.0, 1.0)
        self.yp, self.y = alloc(4 * self.batch * c["rows"], torch.float32, (self.batch, c["rows"]))

    def run(self):
        matvec_dev(self.t.wt, self.xp, self.yp, self.batch)
        return self.y

    def exact(self):
        return _times(self.x.double().view(self.batch, -1), self.t)


def _times(x, t):
    """x W^T in 64 bits, some rows of W at a time."""
    step = max(1, (1 << 27) // t.cols)
    return torch.cat([x @ t.exact(r, r + step).T for r in range(0, t.rows, step)], -1)


class Attention:
    """One attention layer with its f16 k/v cache filled up to `pos`."""

    def __init__(self, c, g, hidden=2880):
        self.tokens, self.pos, self.hidden = c["tokens"], c["pos"], hidden
        ctx = self.pos + self.tokens
        self.cap = c["window"] if 0 < c["window"] < ctx else ctx
        qd, kvd = HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM
        self.wq = Tensor(DT_Q8R, qd, hidden, g, 1e-4, 4e-4)
        self.wk = Tensor(DT_Q8R, kvd, hidden, g, 1e-4, 4e-4)
        self.wv = Tensor(DT_Q8R, kvd, hidden, g, 1e-4, 4e-4)
        self.wo = Tensor(DT_Q8R, hidden, qd, g, 1e-4, 4e-4)
        d = self.desc = _lib.MhAttnLayer()
        d.hidden, d.n_heads, d.n_kv_heads, d.head_dim = hidden, HEADS, KV_HEADS, HEAD_DIM
        d.ctx, d.window, d.qk_norm, d.sinks = ctx, c["window"], 0, 1
        d.norm_eps, d.attn_scale = EPS, HEAD_DIM ** -0.5
        d.wq, d.wk, d.wv, d.wo = (t.wt.c() for t in (self.wq, self.wk, self.wv, self.wo))
        self.bias = {}
        for name, n in (("bq", qd), ("bk", kvd), ("bv", kvd), ("bo", hidden), ("sink", HEADS)):
            ptr, self.bias[name] = _vector(n, g, 0.0, 0.1)
            setattr(d, name, ptr)
        d.attn_norm, self.norm = _vector(hidden, g, 1.0, 0.1)
        half = HEAD_DIM // 2
        angle = torch.arange(ctx, device="cuda").double()[:, None] * 150000.0 ** (
            -torch.arange(half, device="cuda").double() / half)
        d.rope_cos, self.cos = alloc(4 * ctx * half, torch.float32, (ctx, half))
        d.rope_sin, self.sin = alloc(4 * ctx * half, torch.float32, (ctx, half))
        self.cos.copy_(torch.cos(angle))
        self.sin.copy_(torch.sin(angle))
        d.kc, self.k = alloc(2 * self.cap * kvd, torch.float16, (self.cap, kvd))
        d.vc, self.v = alloc(2 * self.cap * kvd, torch.float16, (self.cap, kvd))
        self.k.normal_(0, 1, generator=g)
        self.v.normal_(0, 1, generator=g)

    def call(self, xp):
        for i in range(self.tokens):
            _lib.call("mh_attention_dev", C.byref(self.desc), xp + 4 * self.hidden * i, self.pos + i)

    def exact(self, x):
        """The residual rows after attention, and the cache with the new rows (f16, as the layer keeps it)."""
        k, v, out = self.k.double(), self.v.double(), []
        b = {n: t.double() for n, t in self.bias.items()}
        wq, wk, wv, wo = (t.exact() for t in (self.wq, self.wk, self.wv, self.wo))
        for i in range(self.tokens):
            p, r = self.pos + i, x[i]
            xb = r / torch.sqrt((r * r).mean() + EPS) * self.norm.double()
            q = self._turn(wq @ xb + b["bq"], p).view(KV_HEADS, HEADS // KV_HEADS, HEAD_DIM)
            k[p % self.cap] = self._turn(wk @ xb + b["bk"], p).half().double()
            v[p % self.cap] = (wv @ xb + b["bv"]).half().double()
            n = min(p + 1, self.cap)
            kk, vv = (t[:n].view(n, KV_HEADS, HEAD_DIM).permute(1, 0, 2) for t in (k, v))
            s = q @ kk.transpose(1, 2).contiguous() * HEAD_DIM ** -0.5
            sink = b["sink"].view(KV_HEADS, -1, 1)
            a = torch.softmax(torch.cat((s, sink), -1), -1)[..., :n] @ vv.contiguous()
            out.append(r + wo @ a.reshape(-1) + b["bo"])
        return torch.stack(out), k.half(), v.half()

    def _turn(self, u, p):
        u = u.view(-1, 2, HEAD_DIM // 2)
        c, s = self.cos[p].double(), self.sin[p].double()
        return torch.stack((u[:, 0] * c - u[:, 1] * s, u[:, 1] * c + u[:, 0] * s), 1).reshape(-1)


class AttentionChunk:
    """The attention half of one layer of the batched prefill: embedding rows, then token by token."""

    def __init__(self, c, g):
        self.n = c["tokens"]
        self.layer = Attention(c, g)
        # a residual that does not hide the layer's own output (~0.05) from a comparison
        self.embed = Tensor(DT_F32, self.n, self.layer.hidden, g, 0.02, 0.0)
        self.xp, self.x = alloc(4 * self.n * self.layer.hidden, torch.float32, (self.n, self.layer.hidden))

    def run(self):
        dequant_dev(self.embed.wt, 0, self.n, self.xp)
        self.layer.call(self.xp)
        return {"x": self.x, "k": self.layer.k, "v": self.layer.v}

    def exact(self):
        x, k, v = self.layer.exact(self.embed.exact())
        return {"x": x, "k": k.double(), "v": v.double()}


class Sample:
    def __init__(self, c, g):
        self.c = c
        self.lp, self.logits = _vector(c["vocab"], g, 0.0, c["spread"])
        self.u = float(torch.rand(1, device="cuda", generator=g))
        self.op, self.out = alloc(4, torch.int32)

    def run(self):
        sample_dev(self.lp, self.c["vocab"], self.c["temp"], self.c["topp"], self.u, self.op)
        return self.out

    def exact(self):
        return None


class Token:
    """A decode token of a few layers, as the engine's forward() and sample() run it."""

    def __init__(self, c, g):
        self.c, n, h = c, c["layers"], 2880
        moe = dict(hidden=h, ffn=2880, experts=32, top_k=4, dt="mxfp4")
        self.attn = [Attention(dict(tokens=1, pos=c["pos"], window=128 if i % 2 == 0 else 0), g, h) for i in range(n)]
        self.moe = [Layer(moe, g) for _ in range(n)]
        self.embed = Tensor(DT_Q8R, c["vocab"], h, g, 2e-4, 2e-3)
        self.head = Tensor(DT_Q8R, c["vocab"], h, g, 2e-4, 8e-4)
        nptr, self.norm = _vector(h, g, 1.0, 0.1)
        self.token = int(torch.randint(0, c["vocab"], (1,), device="cuda", generator=g))
        self.u = float(torch.rand(1, device="cuda", generator=g))
        self.xp, self.x = alloc(4 * h, torch.float32)
        self.lp, self.logits = alloc(4 * c["vocab"], torch.float32)
        self.sp, self.sel = alloc(4 * 4 * n, torch.int32, (n, 4))
        self.op, self.out = alloc(4, torch.int32)
        torch.cuda.synchronize()
        d = _lib.MhModelDesc()
        d.hidden, d.vocab, d.n_layers, d.norm_eps = h, c["vocab"], n, EPS
        d.embed, d.lm_head, d.final_norm = self.embed.wt.c(), self.head.wt.c(), nptr
        d.attn = (_lib.MhAttnLayer * n)(*[a.desc for a in self.attn])
        d.moe = (_lib.MhMoeLayer * n)(*[m.layer.c() for m in self.moe])
        p = C.c_void_p()
        _lib.call("mh_model_create", C.byref(d), C.byref(p))
        self.model = p

    def run(self):
        _lib.call("mh_forward_dev", self.model, self.token, self.c["pos"], self.xp, self.lp, self.sp, None)
        sample_dev(self.lp, self.c["vocab"], self.c["temp"], self.c["topp"], self.u, self.op)
        return {"x": self.x, "logits": self.logits, "sel": self.sel, "token": self.out,
                "k": [a.k for a in self.attn], "v": [a.v for a in self.attn]}

    def exact(self):
        x, sel, ks, vs = self.embed.exact(self.token, self.token + 1), [], [], []
        for a, m in zip(self.attn, self.moe):
            x, k, v = a.exact(x)
            x, s, _ = m.exact(x)
            sel.append(s[0])
            ks.append(k.double())
            vs.append(v.double())
        xb = x / torch.sqrt((x * x).mean() + EPS) * self.norm.double()
        return {"x": x[0], "logits": _times(xb, self.head)[0], "sel": torch.stack(sel), "token": None, "k": ks, "v": vs}

    def __del__(self):
        if hasattr(self, "model"):
            _lib.call("mh_model_destroy", self.model)


_KINDS = {"apply": Apply, "decode": Decode, "prefill": Prefill, "matvec": Matvec, "attention": AttentionChunk,
          "sample": Sample, "token": Token}


def prepare(case, seed):
    midge_amd.init(0)
    state = _KINDS[case["kind"]](case, _gen(seed))
    torch.cuda.synchronize()
    return state


def run(state):
    return state.run()


def exact(case, seed):
    if case["kind"] == "sample":
        return None
    return prepare(case, seed).exact()


# ------------------------------------------------------------------- work

def _matrix(dt, rows, cols):
    return sum(blob_sizes(dt, rows, cols))


def _moe_work(c, tokens, layers):
    """Every expert that some token is routed to is read once, each product is made once."""
    h, f, e, k, dt = c["hidden"], c["ffn"], c["experts"], c["top_k"], DTS[c["dt"]]
    expert = 2 * _matrix(dt, f, h) + _matrix(dt, h, f) + 4 * (2 * f + h)
    read = e * (1 - (1 - k / e) ** tokens) * expert
    router = _matrix(DT_Q8R, e, h) + 4 * e + 4 * h
    return {"bytes": layers * (read + router) + 8 * tokens * h,
            "flops": layers * tokens * (6 * h * f * k + 2 * e * h)}


def _attention_work(tokens, pos, window, h=2880):
    qd, kvd = HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM
    n = min(pos + 1, window or pos + 1)
    weights = _matrix(DT_Q8R, qd + 2 * kvd, h) + _matrix(DT_Q8R, h, qd) + 4 * (qd + 2 * kvd + 2 * h)
    return {"bytes": tokens * (weights + 4 * n * kvd + 8 * h),
            "flops": tokens * (2 * h * (2 * qd + 2 * kvd) + 4 * n * qd)}


def work(case):
    c, kind = case, case["kind"]
    if kind == "apply":
        w = _moe_work(dict(c, experts=c["top_k"]), 1, 1)
        return {"bytes": w["bytes"], "flops": 6 * c["hidden"] * c["ffn"] * c["top_k"]}
    if kind in ("decode", "prefill"):
        return _moe_work(c, c["tokens"], c["layers"])
    if kind == "matvec":
        return {"bytes": _matrix(DTS[c["dt"]], c["rows"], c["cols"]) + 4 * c["batch"] * (c["rows"] + c["cols"]),
                "flops": 2 * c["batch"] * c["rows"] * c["cols"]}
    if kind == "attention":
        return _attention_work(c["tokens"], c["pos"], c["window"])
    if kind == "sample":
        return {"bytes": 4 * c["vocab"], "flops": 4 * c["vocab"]}
    moe = _moe_work(dict(hidden=2880, ffn=2880, experts=32, top_k=4, dt="mxfp4"), 1, c["layers"])
    attn = [_attention_work(1, c["pos"], 128 if i % 2 == 0 else 0) for i in range(c["layers"])]
    head = _matrix(DT_Q8R, c["vocab"], 2880) + 8 * c["vocab"]
    return {"bytes": moe["bytes"] + sum(a["bytes"] for a in attn) + head,
            "flops": moe["flops"] + sum(a["flops"] for a in attn) + 2 * 2880 * c["vocab"]}


def tolerance(case):
    """About four times the errors against 64 bits that these ranges show."""
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind == "matvec":
        return {"rel": 2e-6}      # 32-bit sums; batched int8 rounds x to 2^-22 of its largest (3.5e-7 seen)
    if kind in ("attention", "token"):
        return {"rel": 1e-4}      # a k or v at a rounding boundary moves by 2^-11 in the f16 cache (1e-5 seen)
    if kind == "prefill" and case["dt"] == "mxfp4" and case["tokens"] * case["top_k"] >= 8 * case["experts"]:
        return {"rel": 1.6e-4, "differ": 1e-3}   # the scaled matrix instruction's sums (4e-5 seen)
    # 32-bit sums, the router's softmax amplifying a layer's differences in the next ones (2.8e-6 seen at 8 layers)
    return {"rel": 2e-5, "differ": 1e-3}
