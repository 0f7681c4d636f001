"""The work that programs have this library do, as measured cases.

Every case goes through a public entry point of the Python binding of include/z2h.h
(zonos2_amd.z2h): one MoE layer on device tensors, a decode step of a batch of requests, a prompt
prefill, a mixed pass of prompt chunks and decode columns, and frame sampling. The models are cut to a
few layers of the 24-layer configuration (d_model 2048, 16 / 4 heads, head_dim 128, SwiGLU 1536, 32
experts top-4) or of the released topology (16 experts top-1, a dense first layer); each layer has its
full size, and the experts that a step touches are more than the caches hold.

Weights are made on the device from the seed, as GGUF block bytes whose values are about N(0, 0.02).
The router's output rows and second layer have zero row sums, so that its activations' common mean
favours no expert: routing spreads over the experts as a trained, load-balanced router's does.

`exact` restates each path in 64 bits on the decoded weights. What the formats define stays as defined:
activations go through the weight type's activation encoding (Q8_K, Q8_0 or f16), cached keys and
values and decode queries are f16; everything else, sums included, is float64.
"""
import math
import zlib
from pathlib import Path
import sys

import numpy as np
import torch

_PKG = str(Path("zonos2.cpp_amd").resolve())
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
from zonos2_amd import configs                                      # noqa: E402
from zonos2_amd.synth import Tensor                                  # noqa: E402
from zonos2_amd.z2h import Context, Model                            # noqa: E402

DEV = "cuda"
D, NH, NKV, HD, FF, RD = 2048, 16, 4, 128, 1536, 128
TYPES = {"q4_k": configs.Q4_K, "q8_0": configs.Q8_0, "q6_k": configs.Q6_K, "f16": configs.F16}
SAMPLER = dict(temperature=0.9, top_k=100, top_p=0.95, min_p=0.02, rep_penalty=1.1, rep_codebooks=4, greedy=0)


def listed():
    return [
        # one request of the released model, host buffers in and out: what a reader waiting for speech has
        dict(name="single_q8_0", kind="step", weights="q8_0", experts=16, top_k=1, dense=1, layers=4, requests=1,
             kv_low=700, kv_high=700, host=True, zipf=0.0),
        # the serving batch: 16 ragged requests, device-resident inputs
        dict(name="step16_q4_k", kind="step", weights="q4_k", experts=32, top_k=4, dense=0, layers=4, requests=16,
             kv_low=32, kv_high=2048, host=False, zipf=0.0),
        # a full server: 64 requests of very different lengths, a few popular experts
        dict(name="step64_q8_0", kind="step", weights="q8_0", experts=32, top_k=4, dense=0, layers=2, requests=64,
             kv_low=16, kv_high=4096, host=False, zipf=1.2),
        # an odd number of requests on the other K-quant, host buffers (the C++ API's step)
        dict(name="step37_q6_k", kind="step", weights="q6_k", experts=32, top_k=4, dense=0, layers=2, requests=37,
             kv_low=16, kv_high=2048, host=True, zipf=0.0),
        # one MoE layer under a caller's own loop: a decode batch
        dict(name="moe16_q4_k", kind="moe", weights="q4_k", experts=32, top_k=4, rows=16),
        # ... and a large prompt batch of an odd size
        dict(name="moe1500_q8_0", kind="moe", weights="q8_0", experts=32, top_k=4, rows=1500),
        # a voice prompt of ordinary length on the 24-layer configuration
        dict(name="prefill1024_q4_k", kind="prefill", weights="q4_k", experts=32, top_k=4, dense=0, layers=2, rows=1024),
        # a shorter one of an odd length on the released topology and its published weight type
        dict(name="prefill333_q8_0", kind="prefill", weights="q8_0", experts=16, top_k=1, dense=1, layers=4, rows=333),
        # a short odd prompt just past the width where the tiled matmuls begin
        dict(name="prefill77_q6_k", kind="prefill", weights="q6_k", experts=32, top_k=4, dense=0, layers=2, rows=77),
        # continuous batching's mixed pass, prompt chunks beside decode columns
        dict(name="mixed2088_q4_k", kind="mixed", weights="q4_k", experts=32, top_k=4, dense=0, layers=2, chunks=8,
             chunk=256, requests=32),
        dict(name="mixed2088_f16", kind="mixed", weights="f16", experts=32, top_k=4, dense=0, layers=2, chunks=8,
             chunk=256, requests=32),
        # the frame sampler between two steps of the serving batch
        dict(name="sample16", kind="sample", requests=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "moe", "moe", "prefill", "prefill", "mixed", "sample"])
    w = rng.choice(list(TYPES))
    topo = dict(experts=32, top_k=4) if rng.random() < 0.7 else dict(experts=16, top_k=rng.choice([1, 2]))
    dense = rng.choice([0, 1])
    if kind == "sample":
        return dict(kind=kind, requests=_log(rng, 1, 64))
    if kind == "moe":
        return dict(kind=kind, weights=w, rows=_log(rng, 1, 1500), **topo)
    if kind == "prefill":
        return dict(kind=kind, weights=w, dense=dense, layers=2, rows=_log(rng, 5, 1024), **topo)
    if kind == "mixed":
        return dict(kind=kind, weights=w, dense=dense, layers=2, chunks=rng.randint(1, 7), chunk=_log(rng, 16, 256),
                    requests=rng.randint(1, 32), **topo)
    return dict(kind=kind, weights=w, dense=dense, layers=2, requests=_log(rng, 1, 64), kv_low=rng.randint(1, 64),
                kv_high=_log(rng, 100, 3000), host=rng.random() < 0.5, zipf=rng.choice([0.0, 1.2]), **topo)


# ---------------------------------------------------------------- weights
def _gen(seed, name):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed << 20) ^ zlib.crc32(name.encode()))
    return g


def _randn(seed, name, shape):
    return torch.randn(shape, generator=_gen(seed, name), device=DEV, dtype=torch.float32)


class Blocks:
    """A quantized matrix [..., K]: GGUF bytes for upload, float64 values for `exact`."""

    def __init__(self, typ, shape, seed, name):
        self.typ, self.shape = typ, shape
        g = _gen(seed, name)
        K = shape[-1]
        rows = int(np.prod(shape[:-1]))
        def unit(n):
            return torch.randn((rows, K // n, n), generator=g, device=DEV, dtype=torch.float32)
        def uni(*s):
            return torch.rand(s, generator=g, device=DEV, dtype=torch.float32)
        if typ == configs.F32:
            self.x = unit(K).mul_(0.02)
        elif typ == configs.F16:
            self.x = unit(K).mul_(0.02).half()
        elif typ == configs.Q8_0:
            self.q = unit(32).mul_(40).round_().clamp_(-127, 127).to(torch.int8)
            self.d = (0.0005 * (0.8 + 0.4 * uni(rows, K // 32, 1))).half()
        elif typ == configs.Q6_K:
            self.q = unit(256).mul_(10).round_().clamp_(-32, 31).to(torch.int8)
            self.sc = (50 + 60 * uni(rows, K // 256, 16)).round_().to(torch.int8)
            self.d = (2.5e-5 * (0.8 + 0.4 * uni(rows, K // 256, 1))).half()
        else:
            self.q = unit(256).mul_(3).add_(7.5).round_().clamp_(0, 15).to(torch.uint8)
            self.sc = (22 + 41 * uni(rows, K // 256, 8)).round_().to(torch.uint8)
            self.mn = (self.sc.float() + 6 * uni(rows, K // 256, 8) - 3).round_().clamp_(0, 63).to(torch.uint8)
            self.d = (1.6e-4 * (0.8 + 0.4 * uni(rows, K // 256, 1))).half()
            self.dmin = (7.5 * self.d.float()).half()

    def bytes(self):
        h8 = lambda t: t.contiguous().view(torch.uint8)
        if self.typ in (configs.F32, configs.F16):
            b = h8(self.x.reshape(self.x.shape[0], -1))
        elif self.typ == configs.Q8_0:
            b = torch.cat([h8(self.d), h8(self.q)], -1)
        elif self.typ == configs.Q6_K:
            v = (self.q.view(*self.q.shape[:2], 2, 4, 32).short() + 32).to(torch.uint8)   # 128-halves, quarters
            ql = torch.cat([(v[..., 0, :] & 15) | ((v[..., 2, :] & 15) << 4), (v[..., 1, :] & 15) | ((v[..., 3, :] & 15) << 4)], -1)
            h = v >> 4
            qh = h[..., 0, :] | (h[..., 1, :] << 2) | (h[..., 2, :] << 4) | (h[..., 3, :] << 6)
            b = torch.cat([ql.flatten(2), qh.flatten(2), h8(self.sc), h8(self.d)], -1)
        else:
            p = self.q.view(*self.q.shape[:2], 4, 2, 32)
            qs = (p[..., 0, :] | (p[..., 1, :] << 4)).flatten(2)
            s, m = self.sc, self.mn
            sc = torch.cat([s[..., :4] | ((s[..., 4:] >> 4) << 6), m[..., :4] | ((m[..., 4:] >> 4) << 6),
                            (s[..., 4:] & 15) | ((m[..., 4:] & 15) << 4)], -1)
            b = torch.cat([h8(self.d), h8(self.dmin), sc, qs], -1)
        return b.reshape(-1).cpu().numpy()

    def values(self, r0=0, r1=None):
        """float64 rows [r0, r1) of the flattened [rows, K] matrix"""
        s = slice(r0, r1)
        K = self.shape[-1]
        if self.typ in (configs.F32, configs.F16):
            return self.x[s].double().reshape(-1, K)
        if self.typ == configs.Q8_0:
            return (self.q[s].double() * self.d[s].double()).reshape(-1, K)
        if self.typ == configs.Q6_K:
            sc = self.sc[s].double().repeat_interleave(16, -1)
            return (self.q[s].double() * sc * self.d[s].double()).reshape(-1, K)
        sc, mn = (t[s].double().repeat_interleave(32, -1) for t in (self.sc, self.mn))
        return (self.d[s].double() * sc * self.q[s].double() - self.dmin[s].double() * mn).reshape(-1, K)


def _vector(name, shape, seed):
    """The fp32 tensors: norms near one, |N(0,1)| head temperatures, the router's matrices and biases."""
    x = _randn(seed, name, shape)
    if name.endswith("norm.weight"):
        return 1.0 + 0.05 * x
    if name.endswith("attn_temp"):
        return 0.5 + 0.5 * x.abs()
    if name.endswith(("router_mlp0.weight", "router_mlp2.weight")):
        x = x * RD ** -0.5
    elif name.endswith("router_mlp4.weight"):
        x = x * 0.3
    elif name.endswith("router_bias"):
        return 1e-3 * x
    else:
        return 0.02 * x
    if name.endswith(("router_mlp2.weight", "router_mlp4.weight")):
        x = x - x.mean(-1, keepdim=True)
    return x


def _config(case):
    layers = case.get("layers", 1)
    dense = case.get("dense", 0)
    return configs.ModelConfig("cut", n_layer=layers, n_embd=D, n_head=NH, n_head_kv=NKV, head_dim=HD,
                               n_expert=case["experts"], top_k=case["top_k"], n_ff=FF, bulk=TYPES[case["weights"]],
                               expert_used=[0] * dense + [case["top_k"]] * (layers - dense))


class Weights:
    """Every tensor of a configuration, made when asked for."""

    def __init__(self, cfg, seed):
        self.cfg, self.seed = cfg, seed
        self.spec = {n: (t, tuple(reversed(ne))) for n, t, ne, _ in cfg.tensors()}

    def vec(self, name):
        return _vector(name, self.spec[name][1], self.seed)

    def mat(self, name):
        t, shape = self.spec[name]
        return Blocks(t, shape, self.seed, name)

    def upload(self):
        out = {}
        for n, (t, shape) in self.spec.items():
            if t == configs.F32:
                b = self.vec(n).contiguous().view(torch.uint8).reshape(-1).cpu().numpy()
            else:
                b = self.mat(n).bytes()
            out[n] = Tensor(n, t, tuple(reversed(shape)), b)
        return out


# ---------------------------------------------------------------- inputs
def _rng(seed, what):
    return np.random.default_rng([seed, zlib.crc32(what.encode())])


def _ids(cfg, n, seed):
    r = _rng(seed, "ids")
    return np.concatenate([r.integers(0, cfg.audio_vocab, (n, cfg.n_codebooks)),
                           r.integers(0, cfg.text_vocab + 1, (n, 1))], axis=1).astype(np.int32)


def _lens(case):
    """Rows in the cache per request: a property of the case, so that every seed costs the same."""
    if case["kv_low"] >= case["kv_high"]:
        return [case["kv_low"]] * case["requests"]
    r = np.random.default_rng(1000 + case["requests"])
    return [int(x) for x in np.exp(r.uniform(math.log(case["kv_low"]), math.log(case["kv_high"]), case["requests"]))]


def _layout(case):
    """(chunk starts, decode lengths) of a mixed pass."""
    r = np.random.default_rng(2000 + case["chunks"])
    starts = [int(x) * 256 for x in r.integers(0, 4, case["chunks"])]
    return starts, [int(x) for x in r.integers(32, 1201, case["requests"])]


def _mixed_rows(case):
    """slot, position, speaker row (-1: token ids) of every row, and the rows whose logits are read"""
    starts, lens = _layout(case)
    slot, pos, emap, out = [], [], [], []
    for i, s in enumerate(starts):
        for j in range(case["chunk"] + 1):
            slot.append(i); pos.append(s + j); emap.append(i if j == 0 else -1)
        out.append(len(slot) - 1)
    for i, n in enumerate(lens):
        slot.append(len(starts) + i); pos.append(n); emap.append(-1); out.append(len(slot) - 1)
    return [np.array(x, np.int32) for x in (slot, pos, emap, out)]


def _kv(seed, layer, slot, n):
    """f16 key and value rows [n][NKV][HD] already in a slot's cache"""
    x = _randn(seed, f"kv.{layer}.{slot}", (2, n, NKV, HD)).half()
    return x[0], x[1]


def _fill(ctx, seed, layers, rows):
    for L in range(layers):
        for s, n in rows:
            if n:
                k, v = (t.cpu().numpy().view(np.uint16) for t in _kv(seed, L, s, n))
                ctx.kv_write(L, s, 0, k, v)


def _bias(case):
    """log-popularity of the experts (Zipf), 0 where none is asked for"""
    E, s = case["experts"], case.get("zipf", 0.0)
    r = np.random.default_rng(99).permutation(E) + 1
    p = 1.0 / r.astype(np.float64) ** s
    return np.log(p / p.sum()).astype(np.float32)


_streams = []


def _stream():
    """the stream that the program gives its device calls"""
    if not _streams:
        _streams.append(torch.cuda.Stream())
    return _streams[0].cuda_stream


# ---------------------------------------------------------------- prepare / run
def prepare(case, seed):
    kind = case["kind"]
    if kind == "sample":
        # the sampler needs a context of the right vocabulary, not its weights: the smallest model
        cfg = configs.ModelConfig("frames", n_layer=1, n_embd=256, n_head=4, n_head_kv=2, head_dim=64, n_expert=0, top_k=0,
                                  n_ff=256, bulk=configs.F16, audio_vocab=1026)
        ctx = Context(None, case["requests"], 256, model=Model(cfg.hparams(), Weights(cfg, seed).upload()))
        n, ncb = case["requests"], cfg.n_codebooks
        r = _rng(seed, "sample")
        return dict(kind=kind, ctx=ctx, logits=3.0 * _randn(seed, "logits", (n, ncb, cfg.audio_vocab)), u=r.random((n, ncb)),
                    hist=r.integers(0, 1024, (n, ncb, 64)).astype(np.int32), len=np.full((n, ncb), 64, np.int32), sp=[SAMPLER] * n)
    cfg = _config(case)
    mdl = Model(cfg.hparams(), Weights(cfg, seed).upload())
    if kind == "moe":
        T = case["rows"]
        ctx = Context(None, 1, 256, model=mdl, max_rows=T)
        return dict(kind=kind, ctx=ctx, T=T, x=_randn(seed, "x", (T, D)), out=torch.empty((T, D), device=DEV))
    if kind == "prefill":
        T = case["rows"]
        return dict(kind=kind, ctx=Context(None, 1, T + 1, model=mdl, max_rows=T), ids=_ids(cfg, T, seed))
    if kind == "mixed":
        starts, lens = _layout(case)
        slot, pos, emap, rows = _mixed_rows(case)
        cap = max([s + case["chunk"] + 1 for s in starts] + [n + 1 for n in lens])
        ctx = Context(None, len(starts) + len(lens), cap, model=mdl, max_rows=len(slot))
        _fill(ctx, seed, case["layers"], list(enumerate(starts + lens)))
        return dict(kind=kind, ctx=ctx, slot=slot, pos=pos, emap=emap, rows=rows, ids=_ids(cfg, len(slot), seed),
                    emb=_randn(seed, "speaker", (len(starts), D)).cpu().numpy())
    lens = _lens(case)
    T = len(lens)
    ctx = Context(None, T, max(lens) + 1, model=mdl)
    _fill(ctx, seed, case["layers"], list(enumerate(lens)))
    if case["zipf"]:
        for L in range(case["dense"], case["layers"]):
            ctx.set_logit_bias(L, _bias(case))
    ids = _ids(cfg, T, seed)
    slot, past = np.arange(T, dtype=np.int32), np.array(lens, np.int32)
    st = dict(kind=kind, ctx=ctx, T=T, host=case["host"], slot=slot, past=past, ids=ids)
    if not case["host"]:
        st.update(d=[torch.from_numpy(a).to(DEV) for a in (slot, past, ids)],
                  out=torch.empty((T, cfg.n_codebooks * cfg.audio_vocab), device=DEV))
    return st


def run(st):
    ctx, kind = st["ctx"], st["kind"]
    if kind == "sample":
        return ctx.sample(st["sp"], st["u"], st["hist"], st["len"], d_logits=st["logits"].data_ptr())
    if kind == "moe":
        ctx.moe_forward_device(0, st["T"], st["x"].data_ptr(), 0, st["out"].data_ptr(), stream=_stream())
        return st["out"]
    if kind == "prefill":
        return ctx.prefill(0, st["ids"])
    if kind == "mixed":
        return ctx.step_mixed(st["slot"], st["pos"], st["ids"], st["rows"], emb_map=st["emap"], emb=st["emb"])
    if st["host"]:
        return ctx.step(st["slot"], st["past"], ids=st["ids"])
    slot, past, ids = st["d"]
    ctx.step_device(st["T"], slot.data_ptr(), past.data_ptr(), st["past"], ids.data_ptr(), 0, st["out"].data_ptr(), stream=_stream())
    return st["out"]


# ---------------------------------------------------------------- what a pass cannot do without
def _nbytes(typ, *shape):
    return int(np.prod(shape[:-1])) * configs.row_bytes(typ, shape[-1])


def _touched(case, rows):
    p = np.exp(_bias(case).astype(np.float64))
    return float((1.0 - (1.0 - np.minimum(1.0, case["top_k"] * p)) ** rows).sum())


def work(case):
    kind = case["kind"]
    if kind == "sample":
        n = case["requests"] * 9 * 1026
        return {"bytes": 4 * n + case["requests"] * 9 * (64 * 4 + 8 + 4 + 4), "flops": 10 * n}
    t = TYPES[case["weights"]]
    E, k = case["experts"], case["top_k"]
    ffn_w = 3 * _nbytes(t, FF, D)

    def moe(rows):
        router = 4 * (D * RD + 2 * RD * RD + RD * E)
        return (_touched(case, rows) * ffn_w + router, rows * (2 * k * 3 * FF * D + 2 * (D * RD + 2 * RD * RD + RD * E)))
    if kind == "moe":
        b, f = moe(case["rows"])
        return {"bytes": int(b + 8 * case["rows"] * D), "flops": int(f)}
    cfg = _config(case)
    nout, hi = cfg.n_codebooks * cfg.audio_vocab, cfg.high_tier()
    if kind == "prefill":
        rows, heads = case["rows"], 1
        keys, cached = rows * (rows + 1) // 2, 0
    elif kind == "mixed":
        starts, lens = _layout(case)
        _, pos, _, out = _mixed_rows(case)
        rows, heads = len(pos), len(out)
        keys, cached = int((pos.astype(np.int64) + 1).sum()), sum(starts) + sum(lens)
    else:
        lens = _lens(case)
        rows = heads = len(lens)
        keys, cached = sum(lens) + rows, sum(lens)
    R = (NH + 2 * NKV) * HD + NH
    attn_w = _nbytes(t, R, D) + _nbytes(t, D, NH * HD)
    b = rows * _nbytes(hi, 10, D) + _nbytes(hi, nout, D) + 4 * heads * nout
    f = 2 * heads * nout * D
    for L in range(case["layers"]):
        mb, mf = moe(rows) if L >= case["dense"] else (ffn_w, rows * 2 * 3 * FF * D)
        b += attn_w + mb + (cached + rows) * 2 * NKV * HD * 2
        f += rows * 2 * (R * D + D * NH * HD) + 4 * keys * NH * HD + mf
    return {"bytes": int(b), "flops": int(f)}


# ---------------------------------------------------------------- the same in 64 bits
def _encode(x, typ):
    """The weight type's activation encoding of fp32 rows, as float64 values."""
    x = x.float()
    if typ == configs.F32:
        return x.double()
    if typ == configs.F16:
        return x.half().double()
    n = 32 if typ == configs.Q8_0 else 256
    b = x.reshape(x.shape[0], -1, n)
    a = b.abs()
    if typ == configs.Q8_0:
        amax = a.amax(-1, keepdim=True)
        inv = torch.where(amax > 0, 127.0 / amax, torch.zeros_like(amax))
        return ((b * inv).round().double() * (amax / 127.0).half().double()).reshape(x.shape)
    top = b.gather(-1, a.argmax(-1, keepdim=True))
    s = -127.0 / top
    q = (b * s).round().clamp(max=127.0).double() * (1.0 / s).double()
    return torch.where(top != 0, q, torch.zeros_like(q)).reshape(x.shape)


def _mm(x, w, r0=0, r1=None):
    return _encode(x, w.typ) @ w.values(r0, r1).T


def _rms(x, w=None, eps=1e-5):
    y = x / ((x * x).mean(-1, keepdim=True) + eps).sqrt()
    return y if w is None else y * w


def _silu(x):
    return x / (1.0 + torch.exp(-x))


def _gelu(x):
    return 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))


def _moe64(W, L, x, state, bias):
    """One MoE layer: (output, router state)."""
    b = f"blk.{L}."
    v = lambda n: W.vec(b + n).double()
    x = x.float().double()                                           # the layer's input is an fp32 row
    s = x @ v("router_down.weight").T + v("router_down.bias")
    if state is not None and b + "router_eda_scale" in W.spec:
        s = s + state * v("router_eda_scale")
    h = _gelu(_rms(s, v("router_norm.weight")) @ v("router_mlp0.weight").T + v("router_mlp0.bias"))
    h = _gelu(h @ v("router_mlp2.weight").T + v("router_mlp2.bias"))
    p = torch.softmax(h @ v("router_mlp4.weight").T + bias, -1)
    sel = (p + v("router_bias")).topk(W.cfg.expert_used[L], -1).indices
    G, U, Dn = (W.mat(b + f"ffn_{n}_exps.weight") for n in ("gate", "up", "down"))
    out = torch.zeros_like(x)
    xe = _encode(x, G.typ)
    for e in range(W.cfg.n_exp(L)):
        t, j = (sel == e).nonzero(as_tuple=True)
        if len(t):
            y = (xe[t] @ U.values(e * FF, (e + 1) * FF).T) * _silu(xe[t] @ G.values(e * FF, (e + 1) * FF).T)
            out.index_add_(0, t, _mm(y, Dn, e * D, (e + 1) * D) * p[t, sel[t, j]][:, None])
    return out, s


def _rope(x, pos, base):
    th = pos.double()[:, None] * base ** (-2.0 * torch.arange(HD // 2, device=DEV, dtype=torch.float64) / HD)
    c, s = th.cos()[:, None], th.sin()[:, None]
    y = torch.empty_like(x)
    y[..., 0::2] = x[..., 0::2] * c - x[..., 1::2] * s
    y[..., 1::2] = x[..., 0::2] * s + x[..., 1::2] * c
    return y


def _model64(case, seed, slot, pos, ids, emap, emb, cached, out_rows, f16_rows):
    """Logits of `out_rows` after one pass over rows (slot, pos); cached: (slot, rows already there).
    f16_rows: keys, values and queries are f16 (the cache); else the rows of one prompt, unrounded."""
    cfg = _config(case)
    W = Weights(cfg, seed)
    T = len(slot)
    idt = torch.from_numpy(ids.astype(np.int64)).to(DEV)
    x = torch.zeros((T, D), device=DEV, dtype=torch.float64)
    for c in range(cfg.n_codebooks + 1):
        tab = W.mat(f"audio_embd.{c}.weight" if c < cfg.n_codebooks else "text_embd.weight").values()
        x = x + tab[idt[:, c]]
    if emap is not None:
        m = torch.from_numpy(emap.astype(np.int64)).to(DEV)
        e = torch.from_numpy(emb).to(DEV).double()
        x = torch.where((m >= 0)[:, None], e[m.clamp(min=0)], x)
    res = _rms(x)
    post = torch.from_numpy(pos.astype(np.int64)).to(DEV)
    rnd = (lambda t: t.half().double()) if f16_rows else (lambda t: t)
    zb = torch.from_numpy(_bias(case)).to(DEV).double() if case.get("zipf") else 0.0
    state = None
    for L in range(cfg.n_layer):
        b = f"blk.{L}."
        h = _rms(res, W.vec(b + "attn_norm.weight").double())
        q, k, v, g = (_mm(h, W.mat(b + f"attn_{n}.weight")) for n in ("q", "k", "v", "gate"))
        q = _rms(q.view(T, NH, HD), eps=1e-6) * W.vec(b + "attn_temp").double()[:, None]
        q = rnd(_rope(q, post, cfg.rope_freq_base))
        k = rnd(_rope(_rms(k.view(T, NKV, HD), eps=1e-6), post, cfg.rope_freq_base))
        v = rnd(v.view(T, NKV, HD))
        o = torch.zeros((T, NH, HD), device=DEV, dtype=torch.float64)
        for s, n in cached:
            r = torch.from_numpy(np.nonzero(slot == s)[0]).to(DEV)
            if not len(r):
                continue
            ks, vs = (torch.cat([c.double(), t[r]]) for c, t in zip(_kv(seed, L, s, n), (k, v)))
            at = torch.cat([torch.arange(n, device=DEV), post[r]])
            for hh in range(NH):
                sc = (q[r, hh] @ ks[:, hh // (NH // NKV)].T) / math.sqrt(HD)
                sc = sc.masked_fill(at[None, :] > post[r][:, None], -math.inf)
                o[r, hh] = torch.softmax(sc, -1) @ vs[:, hh // (NH // NKV)]
        o = o * torch.sigmoid(g)[..., None]
        res = res + _mm(o.reshape(T, NH * HD), W.mat(b + "attn_output.weight"))
        h = _rms(res, W.vec(b + "ffn_norm.weight").double())
        if cfg.expert_used[L]:
            y, state = _moe64(W, L, h, state, zb)
        else:
            y = _mm(_mm(h, W.mat(b + "ffn_up.weight")) * _silu(_mm(h, W.mat(b + "ffn_gate.weight"))), W.mat(b + "ffn_down.weight"))
        res = res + y
    h = _rms(res[torch.from_numpy(out_rows.astype(np.int64)).to(DEV)], W.vec("output_norm.weight").double())
    return cfg.logit_softcap * torch.tanh(_mm(h, W.mat("output.weight")) / cfg.logit_softcap)


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None
    cfg = _config(case)
    if kind == "moe":
        return _moe64(Weights(cfg, seed), 0, _randn(seed, "x", (case["rows"], D)), None, 0.0)[0]
    if kind == "prefill":
        T = case["rows"]
        pos = np.arange(T)
        return _model64(case, seed, np.zeros(T, int), pos, _ids(cfg, T, seed), None, None, [(0, 0)], pos[-1:], False)[0].cpu().numpy()
    if kind == "mixed":
        starts, lens = _layout(case)
        slot, pos, emap, out = _mixed_rows(case)
        emb = _randn(seed, "speaker", (len(starts), D)).cpu().numpy()
        y = _model64(case, seed, slot, pos, _ids(cfg, len(slot), seed), emap, emb, list(enumerate(starts + lens)), out, True)
        return y.cpu().numpy()
    lens = _lens(case)
    T = len(lens)
    y = _model64(case, seed, np.arange(T), np.array(lens), _ids(cfg, T, seed), None, None, list(enumerate(lens)), np.arange(T), True)
    return y.cpu().numpy() if case["host"] else y


def tolerance(case):
    """About four times the distance from `exact`. One MoE layer: 2.7e-7 where no value of the SwiGLU rows'
    encoding falls on the other side of a rounding, 1.2e-4 where some do. A whole model: such values in
    every layer's four encodings change the next layers' inputs, by a 6-8e-3 share for the 256-value blocks
    of the K-quants, 1-3e-3 for Q8_0's 32, 1-2e-4 for f16 activations."""
    if case["kind"] == "sample":
        return "exact"
    if case["kind"] == "moe":
        return {"rel": 5e-4}
    return {"rel": {"q8_0": 1e-2, "f16": 1e-3}.get(case["weights"], 3e-2)}
