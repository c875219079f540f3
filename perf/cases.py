"""The workloads this library is timed on, through its C ABI (include/cmol_hip.h).

Four kinds of case, each a dict of plain values:

- gemm: one projection, `cmolhip_gemm` on device vectors: a decode token (n = 1), a
  lock-step batch (n up to 32) or a prompt (more), with or without the RMSNorm in front.
- attn: one layer's decode attention, `cmolhip_attn_decode`, for n sessions of ragged
  lengths over fp32 or fp16 caches.
- decode / batch: a decode step of a model for one session (`cmolhip_decode`) or for many
  in lock-step (`cmolhip_decode_batch`), with the logits back on the host as a sampler
  needs them.
- prefill: a prompt of n tokens behind pos0 cached positions (`cmolhip_prefill`).

Shapes are those of the SmolLM2 / SmolLM3 presets (libcmol_amd/synth.py).  A model case
names its layer count: the whole model, or a stack of its blocks with a small vocabulary,
so that the layers themselves are what is timed.
"""
import ctypes as C
import math

import numpy as np
import torch

from libcmol_amd import native

Q4_0, Q5_0, Q8_0, Q4_K, Q6_K = 2, 6, 8, 12, 14
BLOCK = {Q4_0: (32, 18), Q5_0: (32, 22), Q8_0: (32, 34), Q4_K: (256, 144), Q6_K: (256, 210)}

# d_model, heads, kv heads, d_ffn, rope base, rms eps, NoPE interval
SHAPES = {
    "135m": (576, 9, 3, 1536, 1e4, 1e-5, 0),
    "360m": (960, 15, 5, 2560, 1e4, 1e-5, 0),
    "small": (512, 8, 2, 1536, 1e4, 1e-5, 0),
    "3b": (2048, 16, 4, 11008, 5e6, 1e-6, 4),
}


def listed():
    return [
        # one decode token through the widest projection of the 3B shape: the call whose
        # bandwidth the project quotes
        {"name": "matvec_q4_1", "kind": "gemm", "dtype": Q4_0, "rows": 11008, "cols": 2048, "n": 1, "norm": True},
        # the same projection of a Q4_K_M file for 20 sessions in lock-step
        {"name": "gemm_q4k_20", "kind": "gemm", "dtype": Q4_K, "rows": 11008, "cols": 2048, "n": 20, "norm": True},
        # the tied Q8_0 head of the 3B shape for 32 sessions
        {"name": "head_q8_32", "kind": "gemm", "dtype": Q8_0, "rows": 128256, "cols": 2048, "n": 32, "norm": True},
        # decode attention of 8 chats over the default (fp32) caches
        {"name": "attn_f32_8", "kind": "attn", "n": 8, "heads": 16, "kv": 4, "dh": 128, "max_ctx": 4096,
         "lo": 64, "hi": 4096, "f16": False},
        # the same for 32 sessions over fp16 caches, long uneven contexts
        {"name": "attn_f16_32", "kind": "attn", "n": 32, "heads": 16, "kv": 4, "dh": 128, "max_ctx": 16384,
         "lo": 512, "hi": 16384, "f16": True},
        # single-chat decode of the smallest model, early in a conversation (launches and latency)
        {"name": "decode_135m_q8", "kind": "decode", "shape": "135m", "dtype": Q8_0, "head": Q8_0, "layers": 30,
         "vocab": 49152, "max_ctx": 2048, "pos": 96, "f16": False},
        # single-chat decode of the 3B model behind a 2048-token prompt (the headline)
        {"name": "decode_3b_q4", "kind": "decode", "shape": "3b", "dtype": Q4_0, "head": Q8_0, "layers": 36,
         "vocab": 128256, "max_ctx": 4096, "pos": 2048, "f16": False},
        # 16 chats in lock-step on the 360M shape: eight blocks, contexts 64..1024
        {"name": "batch_360m_16", "kind": "batch", "shape": "360m", "dtype": Q5_0, "head": Q5_0, "layers": 8,
         "vocab": 4096, "max_ctx": 1088, "n": 16, "lo": 64, "hi": 1024, "f16": False},
        # 32 chats in lock-step on the 3B shape, fp16 caches: four blocks, contexts 512..4096
        {"name": "batch_3b_32", "kind": "batch", "shape": "3b", "dtype": Q4_0, "head": Q8_0, "layers": 4,
         "vocab": 4096, "max_ctx": 8192, "n": 32, "lo": 512, "hi": 4096, "f16": True},
        # a long prompt in one pass on the 3B shape: four blocks
        {"name": "prefill_3b_2048", "kind": "prefill", "shape": "3b", "dtype": Q4_0, "head": Q8_0, "layers": 4,
         "vocab": 4096, "max_ctx": 2304, "pos": 0, "n": 2048, "chunk": 2048, "f16": False},
        # a further turn of a served chat: 700 tokens behind 1300 cached ones, fp16 caches,
        # the library's default chunk
        {"name": "prefill_turn_f16", "kind": "prefill", "shape": "3b", "dtype": Q4_0, "head": Q8_0, "layers": 4,
         "vocab": 4096, "max_ctx": 4096, "pos": 1300, "n": 700, "chunk": 512, "f16": True},
        # a one-line question: 45 tokens into an empty cache
        {"name": "prefill_short", "kind": "prefill", "shape": "3b", "dtype": Q4_0, "head": Q8_0, "layers": 4,
         "vocab": 4096, "max_ctx": 4096, "pos": 0, "n": 45, "chunk": 512, "f16": False},
    ]


def _logu(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "attn", "attn", "decode", "batch", "batch", "prefill", "prefill"])
    if kind == "gemm":
        dt = rng.choice([Q4_0, Q4_0, Q5_0, Q8_0, Q4_K, Q6_K])
        bv = BLOCK[dt][0]
        return {"kind": kind, "dtype": dt, "rows": _logu(rng, 192, 22016), "cols": bv * max(1, _logu(rng, 512, 11008) // bv),
                "n": _logu(rng, 1, 1500), "norm": rng.random() < 0.5}
    if kind == "attn":
        heads, kv, dh = rng.choice([(16, 4, 128), (9, 3, 64), (15, 5, 64)])
        ctx = _logu(rng, 256, 8192)
        return {"kind": kind, "n": _logu(rng, 1, 32), "heads": heads, "kv": kv, "dh": dh, "max_ctx": ctx,
                "lo": max(1, ctx // 8), "hi": ctx, "f16": rng.random() < 0.5}
    shape = rng.choice(["135m", "360m", "3b", "small"])
    dt = rng.choice([Q4_0, Q5_0, Q8_0] if SHAPES[shape][0] % 256 else [Q4_0, Q5_0, Q8_0, Q4_K, Q6_K])
    c = {"kind": kind, "shape": shape, "dtype": dt, "head": Q8_0, "layers": rng.randint(2, 4), "vocab": 4096,
         "f16": rng.random() < 0.5}
    if kind == "decode":
        pos = _logu(rng, 16, 4000)
        return dict(c, pos=pos, max_ctx=pos + rng.choice([64, 1024, 4096]))
    if kind == "batch":
        hi = _logu(rng, 128, 4000)
        return dict(c, n=rng.randint(2, 32), lo=max(16, hi // 8), hi=hi, max_ctx=hi + rng.choice([64, 1024]))
    # (prompts of up to eight tokens are a lock-step decode step of as many vectors)
    n, pos = _logu(rng, 9, 1800), rng.choice([0, 0, _logu(rng, 16, 2000)])
    return dict(c, n=n, pos=pos, chunk=rng.choice([512, 512, 2048]), max_ctx=pos + n + 256)


# ---- inputs -----------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _quant_rows(dt, rows, cols, g):
    """Raw GGUF rows [rows][row bytes] (uint8, on the GPU) of weights ~ N(0, 0.02): the 32-value
    formats by GGML's quantisers, the K-quants as super-blocks of that spread."""
    dev = "cuda"
    bv, bb = BLOCK[dt]
    nb = rows * cols // bv
    out = torch.empty(nb, bb, dtype=torch.uint8, device=dev)
    if dt in (Q4_K, Q6_K):
        out.copy_(torch.randint(0, 256, (nb, bb), generator=g, device=dev, dtype=torch.uint8))
        spread = 1.0 + torch.rand(nb, 1, generator=g, device=dev)
        if dt == Q4_K:
            out[:, 0:2] = (spread * 9e-5).half().view(torch.uint8)
            out[:, 2:4] = (spread * 6.7e-4).half().view(torch.uint8)
        else:
            out[:, 192:208] = torch.randint(8, 41, (nb, 16), generator=g, device=dev, dtype=torch.uint8)
            out[:, 208:210] = (spread * 3e-5).half().view(torch.uint8)
        return out.view(rows, cols // bv * bb)
    step = max(1, (1 << 22) // 32)
    for b0 in range(0, nb, step):
        x = torch.randn(min(step, nb - b0), 32, generator=g, device=dev) * 0.02
        o = out[b0:b0 + x.shape[0]]
        big = x.gather(1, x.abs().argmax(1, keepdim=True))
        d = big.abs() / 127 if dt == Q8_0 else big / (-8.0 if dt == Q4_0 else -16.0)
        o[:, 0:2] = d.half().view(torch.uint8)
        if dt == Q8_0:
            o[:, 2:] = (x / d).round().to(torch.int8).view(torch.uint8)
            continue
        mid = 8 if dt == Q4_0 else 16
        q = (x / d + mid + 0.5).floor().clamp(0, 2 * mid - 1).to(torch.int32)
        n0 = o.shape[1] - 16
        o[:, n0:] = ((q[:, :16] & 15) | ((q[:, 16:] & 15) << 4)).to(torch.uint8)
        if dt == Q5_0:
            bit = (q >> 4).view(-1, 4, 8) << torch.arange(8, device=dev, dtype=torch.int32)
            o[:, 2:6] = bit.sum(2).to(torch.uint8)
    return out.view(rows, cols // bv * bb)


def _dequant(dt, raw, rows, cols):
    """float64 values [rows][cols] of raw GGUF rows."""
    bv, bb = BLOCK[dt]
    b = raw.reshape(-1, bb)

    def f16(lo):
        return b[:, lo:lo + 2].contiguous().view(torch.float16).double()

    if dt == Q8_0:
        v = f16(0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif dt in (Q4_0, Q5_0):
        qs = b[:, bb - 16:].to(torch.int32)
        q = torch.cat([qs & 15, qs >> 4], 1)
        if dt == Q5_0:
            h = (b[:, 2:6].to(torch.int32).unsqueeze(2) >> torch.arange(8, device=b.device, dtype=torch.int32)) & 1
            q = q | (h.reshape(-1, 32) << 4)
        v = f16(0) * (q - (8 if dt == Q4_0 else 16)).double()
    elif dt == Q4_K:
        s, qs = b[:, 4:16].to(torch.int32), b[:, 16:].to(torch.int32).view(-1, 4, 32)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = torch.stack([qs & 15, qs >> 4], 2).view(-1, 8, 32).double()
        v = (f16(0) * sc).unsqueeze(2) * q - (f16(2) * mn).unsqueeze(2)
    else:
        ql, qh = b[:, :128].to(torch.int32).view(-1, 2, 2, 32), b[:, 128:192].to(torch.int32).view(-1, 2, 32)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        lo, hi = ql & 15, ql >> 4
        q = torch.stack([lo[:, :, 0] | ((qh & 3) << 4), lo[:, :, 1] | (((qh >> 2) & 3) << 4),
                         hi[:, :, 0] | (((qh >> 4) & 3) << 4), hi[:, :, 1] | (((qh >> 6) & 3) << 4)], 2)
        v = f16(208).unsqueeze(2) * sc.unsqueeze(2) * (q.reshape(-1, 16, 16) - 32).double()
    return v.reshape(rows, cols)


def _host(t):
    return np.ascontiguousarray(t.cpu().numpy())


def _lens(c, g):
    """Context lengths of n sessions, log-uniform in lo..hi, the longest at hi."""
    u = torch.rand(c["n"], generator=g, device="cuda").cpu().numpy()
    n = np.floor(np.exp(math.log(c["lo"]) + u * (math.log(c["hi"] + 1) - math.log(c["lo"]))))
    n[0] = c["hi"]
    return n.clip(c["lo"], c["hi"]).astype(np.int64)


def _gemm_inputs(c, seed):
    g = _gen(seed)
    raw = _quant_rows(c["dtype"], c["rows"], c["cols"], g)
    x = torch.randn(c["n"], c["cols"], generator=g, device="cuda")
    nw = 1 + 0.1 * torch.randn(c["cols"], generator=g, device="cuda") if c["norm"] else None
    return raw, x, nw


def _attn_inputs(c, seed):
    g = _gen(seed)
    lens = _lens(c, g)
    q = torch.randn(c["n"], c["heads"] * c["dh"], generator=g, device="cuda")
    kv = []
    for _ in range(2):
        t = torch.empty(c["n"], c["kv"], c["max_ctx"], c["dh"], device="cuda",
                        dtype=torch.float16 if c["f16"] else torch.float32)
        for i in range(c["n"]):
            t[i] = torch.randn(t.shape[1:], generator=g, device="cuda")
        kv.append(t)
    return lens, q, kv[0], kv[1]


class _Inputs:
    """Weights, tokens and cached K/V rows of a model case.  Two distinct layers' weights, the
    model's layers taking them in turn (each has its own copy on the device)."""

    def __init__(self, c, seed):
        g = _gen(seed)
        d, self.heads, self.kv, f, base, self.eps, self.nope = SHAPES[c["shape"]]
        self.d, self.f, self.dh = d, f, d // self.heads
        self.kvd = kvd = self.kv * self.dh
        self.mats = {"q": (d, d), "k": (kvd, d), "v": (kvd, d), "o": (d, d), "gate": (f, d), "up": (f, d), "down": (d, f)}
        self.sets = []
        for _ in range(min(2, c["layers"])):
            w = {m: _quant_rows(c["dtype"], r, k, g) for m, (r, k) in self.mats.items()}
            w["norms"] = 1 + 0.1 * torch.randn(2, d, generator=g, device="cuda")
            self.sets.append(w)
        self.embd = _quant_rows(c["head"], c["vocab"], d, g)
        self.out_norm = 1 + 0.1 * torch.randn(d, generator=g, device="cuda")
        i = np.arange(self.dh // 2)
        ang = np.arange(c["max_ctx"])[:, None] / base ** (2.0 * i / self.dh)
        self.rope = np.ascontiguousarray(np.stack([np.cos(ang), np.sin(ang)], 2).astype(np.float32))
        n = c.get("n", 1)
        self.tokens = torch.randint(0, c["vocab"], (n,), generator=g, device="cuda").cpu().numpy().astype(np.int32)
        self.lens = _lens(c, g) if c["kind"] == "batch" else np.array([c["pos"]])
        # [session][layer] -> (k, v), each [len][kv heads * d_head], the spread of real keys and values
        self.past = [[tuple(torch.randn(int(m), kvd, generator=g, device="cuda") for _ in range(2))
                      for _ in range(c["layers"])] for m in self.lens]


class _Model:
    """A device model and the buffers of one call."""

    def __init__(self, c, seed):
        t = _Inputs(c, seed)
        lib = native.lib()
        keep = []

        def ten(x, dt, rows, cols):
            a = _host(x)
            keep.append(a)
            return native.HostTensor(C.c_void_p(a.ctypes.data), dt, rows, cols)

        sets = []
        for w in t.sets:
            s = {m: ten(w[m], c["dtype"], r, k) for m, (r, k) in t.mats.items()}
            s["attn_norm"], s["ffn_norm"] = (ten(w["norms"][j], 0, 1, t.d) for j in range(2))
            sets.append(s)
        layers = (native.LayerTensors * c["layers"])()
        for i, L in enumerate(layers):
            for k, v in sets[i % len(sets)].items():
                setattr(L, k, v)
        sessions = c["n"] if c["kind"] == "batch" else 1
        desc = native.ModelDesc()
        desc.hp = native.HParams(c["layers"], t.heads, t.kv, t.d, t.dh, t.f, c["vocab"], c["max_ctx"], sessions,
                                 t.nope, int(c["f16"]), c.get("chunk", 512), SHAPES[c["shape"]][4], t.eps)
        desc.embd = ten(t.embd, c["head"], c["vocab"], t.d)
        desc.out_norm = ten(t.out_norm, 0, 1, t.d)
        desc.layers = layers
        desc.rope_table = C.c_void_p(t.rope.ctypes.data)
        self.h = C.c_void_p()
        native.check(lib.cmolhip_model_create(C.byref(desc), 0, C.byref(self.h)), "model_create")
        for s, per in enumerate(t.past):
            for l, (k, v) in enumerate(per):
                if len(k):
                    a, b = _host(k), _host(v)
                    native.check(lib.cmolhip_kv_upload(self.h, s, l, len(a), native.ptr(a), native.ptr(b)), "kv_upload")
        self.n = sessions
        self.tokens = t.tokens
        self.pos = t.lens.astype(np.int32)
        self.slots = np.arange(sessions, dtype=np.int32)
        self.logits = torch.empty(sessions, c["vocab"], pin_memory=True)
        self.ids = np.zeros(sessions, np.int32)

    def __del__(self):
        if getattr(self, "h", None):
            native.lib().cmolhip_model_destroy(self.h)
            self.h = None


_ctx = None


def _calls():
    """The context a program makes its kernel calls on: one stream, scratch for any of them."""
    global _ctx
    if _ctx is None:
        _ctx = native.Ctx(512 << 20)
    return _ctx


def prepare(case, seed):
    c, lib = case, native.lib()
    s = {"case": c}
    if c["kind"] == "gemm":
        raw, x, nw = _gemm_inputs(c, seed)
        n, rows, cols = c["n"], c["rows"], c["cols"]
        fold = lib.cmolhip_pick_fold(rows, cols, 1 if n == 1 else 32)
        s["weights"] = native.Ctx(lib.cmolhip_qtensor_bytes(c["dtype"], rows, cols, fold) + raw.numel() + (1 << 20))
        h = _host(raw)
        w = s["weights"].qtensor([h.reshape(-1)], c["dtype"], cols, [rows], fold=fold)
        y = torch.empty(n, rows, device="cuda")
        s.update(w=w, x=x, nw=nw, y=y)
        s["args"] = (_calls().h, C.byref(w), C.c_void_p(x.data_ptr()), C.c_void_p(y.data_ptr()), n,
                     C.c_void_p(nw.data_ptr()) if nw is not None else None, C.c_float(1e-5))
    elif c["kind"] == "attn":
        lens, q, k, v = _attn_inputs(c, seed)
        dl = torch.tensor(lens, dtype=torch.int32, device="cuda")
        out = torch.empty_like(q)
        s.update(q=q, k=k, v=v, dl=dl, out=out)
        s["args"] = (_calls().h, c["n"], *(C.c_void_p(t.data_ptr()) for t in (q, k, v, dl)), c["heads"], c["kv"],
                     c["dh"], c["max_ctx"], int(c["f16"]), 0, C.c_void_p(out.data_ptr()))
    else:
        m = s["model"] = _Model(c, seed)
        lg, ids = C.c_void_p(m.logits.data_ptr()), native.ptr(m.ids)
        if c["kind"] == "decode":
            s["args"] = (m.h, 0, int(m.tokens[0]), int(m.pos[0]), lg, ids)
        elif c["kind"] == "batch":
            s["args"] = (m.h, m.n, native.ptr(m.slots), native.ptr(m.tokens), native.ptr(m.pos), lg, ids)
        else:
            s["args"] = (m.h, 0, native.ptr(m.tokens), c["n"], c["pos"], lg, ids)
    name = {"gemm": "cmolhip_gemm", "attn": "cmolhip_attn_decode", "decode": "cmolhip_decode",
            "batch": "cmolhip_decode_batch", "prefill": "cmolhip_prefill"}[c["kind"]]
    s["call"], s["what"] = getattr(lib, name), name
    torch.cuda.synchronize()   # the inputs are complete before the library's own stream reads them
    return s


def run(state):
    rc = state["call"](*state["args"])
    if rc:
        native.check(rc, state["what"])
    if "y" in state:
        return state["y"]
    if "out" in state:
        return state["out"]
    return state["model"].logits


# ---- what a pass cannot do without ------------------------------------------------------

def _wbytes(dt, rows, cols):
    bv, bb = BLOCK[dt]
    return rows * cols // bv * bb


def work(case):
    c = case
    if c["kind"] == "gemm":
        n, r, k = c["n"], c["rows"], c["cols"]
        return {"bytes": _wbytes(c["dtype"], r, k) + 4 * n * (r + k), "flops": 2 * n * r * k}
    if c["kind"] == "attn":
        mean = (c["hi"] - c["lo"]) / max(1e-9, math.log((c["hi"] + 1) / c["lo"]))
        pos = c["n"] * min(c["hi"], max(c["lo"], mean))
        return {"bytes": pos * c["kv"] * c["dh"] * 2 * (2 if c["f16"] else 4) + 8 * c["n"] * c["heads"] * c["dh"],
                "flops": 4 * pos * c["heads"] * c["dh"]}
    d, h, kv, f, *_ = SHAPES[c["shape"]]
    dh = d // h
    kvd, es = kv * dh, 2 if c["f16"] else 4
    par = d * (2 * d + 2 * kvd) + 3 * d * f
    wb = c["layers"] * _wbytes(c["dtype"], 1, 1 << 8) * par / 256 + _wbytes(c["head"], c["vocab"], d)
    if c["kind"] == "prefill":
        n, p = c["n"], c["pos"]
        att = n * p + n * (n + 1) / 2
        return {"bytes": wb + c["layers"] * (p + n) * kvd * 2 * es + 4 * c["vocab"],
                "flops": c["layers"] * (2 * n * par + 4 * att * d) + 2 * c["vocab"] * d}
    if c["kind"] == "decode":
        n, pos = 1, c["pos"] + 1
    else:
        mean = (c["hi"] - c["lo"]) / max(1e-9, math.log((c["hi"] + 1) / c["lo"]))
        n, pos = c["n"], c["n"] * min(c["hi"], max(c["lo"], mean))
    return {"bytes": wb + c["layers"] * pos * kvd * 2 * es + 4 * n * c["vocab"],
            "flops": c["layers"] * (2 * n * par + 4 * pos * d) + 2 * n * c["vocab"] * d}


def tolerance(case):
    """About four times what float32 sums in one order and 64 bits differ by here: 1e-7..3e-7 for a
    product or an attention, up to 2e-6 for a model, 1e-5 where new K/V rows are rounded to fp16
    (a value next to a rounding boundary may fall to either side)."""
    if case["kind"] in ("gemm", "attn"):
        return {"rel": 1e-6}
    return {"rel": 4e-5 if case["f16"] else 1e-5}


# ---- the same in 64 bits ----------------------------------------------------------------

def _rms(x, w, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w.double()


def _attend(q, k, v, first):
    """Causal attention of q [n][heads][dh] at positions first.. over k, v [T][kv][dh]."""
    n, h, dh = q.shape
    g = h // k.shape[1]
    out = torch.empty_like(q)
    t = torch.arange(k.shape[0], device=q.device)
    for i in range(0, n, 512):
        m = min(512, n - i)
        seen = t[None, :] <= first + i + torch.arange(m, device=q.device)[:, None]
        for j in range(h):
            s = (q[i:i + m, j] @ k[:, j // g].T / math.sqrt(dh)).masked_fill(~seen, -math.inf)
            out[i:i + m, j] = s.softmax(1) @ v[:, j // g]
    return out


def exact(case, seed):
    c = case
    if c["kind"] == "gemm":
        raw, x, nw = _gemm_inputs(c, seed)
        x = x.double() if nw is None else _rms(x.double(), nw, 1e-5)
        return x @ _dequant(c["dtype"], raw, c["rows"], c["cols"]).T
    if c["kind"] == "attn":
        lens, q, k, v = _attn_inputs(c, seed)
        return torch.stack([_attend(q[i].double().view(1, c["heads"], c["dh"]),
                                    k[i, :, :n].double().transpose(0, 1), v[i, :, :n].double().transpose(0, 1),
                                    int(n)).view(-1) for i, n in enumerate(lens)])
    t = _Inputs(c, seed)
    tok = torch.tensor(t.tokens, device="cuda", dtype=torch.int64)
    embd = _dequant(c["head"], t.embd, c["vocab"], t.d)
    x = embd[tok]
    sets = [dict({m: _dequant(c["dtype"], w[m], *t.mats[m]) for m in t.mats}, norms=w["norms"]) for w in t.sets]
    rope = torch.tensor(t.rope, device="cuda").double()
    n = len(x)
    pos = (torch.tensor(t.lens, device="cuda") if c["kind"] == "batch" else c["pos"] + torch.arange(n, device="cuda"))

    def rotate(y, heads):
        y = y.view(n, heads, t.dh // 2, 2)
        cs, sn = rope[pos][:, None, :, 0], rope[pos][:, None, :, 1]
        return torch.stack([y[..., 0] * cs - y[..., 1] * sn, y[..., 0] * sn + y[..., 1] * cs], 3).reshape(n, heads, t.dh)

    def cached(y):
        return (y.half() if c["f16"] else y.float()).double()

    for l in range(c["layers"]):
        w = sets[l % len(sets)]
        h = _rms(x, w["norms"][0], t.eps)
        q, k, v = (h @ w[m].T for m in "qkv")
        if t.nope and (l + 1) % t.nope == 0:
            q, k = q.view(n, t.heads, t.dh), k.view(n, t.kv, t.dh)
        else:
            q, k = rotate(q, t.heads), rotate(k, t.kv)
        k, v = cached(k), cached(v.view(n, t.kv, t.dh))
        outs = []
        for i in range(n if c["kind"] == "batch" else 1):
            pk, pv = (cached(a.double()).view(-1, t.kv, t.dh) for a in t.past[i][l])
            own = slice(i, i + 1) if c["kind"] == "batch" else slice(None)
            outs.append(_attend(q[own], torch.cat([pk, k[own]]), torch.cat([pv, v[own]]), len(pk)))
        x = x + torch.cat(outs).view(n, -1) @ w["o"].T
        h = _rms(x, w["norms"][1], t.eps)
        gate = h @ w["gate"].T
        x = x + (gate * torch.sigmoid(gate) * (h @ w["up"].T)) @ w["down"].T
    if c["kind"] == "prefill":
        x = x[-1:]
    return _rms(x, t.out_norm, t.eps) @ embd.T
