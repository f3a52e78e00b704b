"""What a user of this library has it do, as cases that can be timed and compared.

A case is one call a serving program makes:

- ``layer``: ``Attention.forward`` of one layer, projections included, on a KV cache;
- ``qkv``: ``Attention.forward_qkv`` (per-head norms, RoPE, cache write, attention), where
  the program runs its own projections;
- ``prefill``: ``attn_prefill`` and its two opt-in precision modes on q, k and v;
- ``step``: ``attn_decode_step``, one token against a long cache;
- ``head``: the LM head and the greedy choice of the next token.

``rows`` tokens start at position ``pos``: one row is a decode step, several at position 0
a prompt, several further on a prompt's next chunk. The shapes are this repository's three
model shapes (Qwen3-0.6B, Mistral-7B, Gemma-4 global and local layers) over f32, IEEE-half
and E4M3 caches.
"""
import math

import torch

import eyebrowse_amd as eb

MODELS = {
    # h query heads, hkv KV heads, head dim, model width, scores' scale, q/k/v norms, rotated
    # pairs, RoPE base. Without a width there are no projections (kind "qkv").
    "qwen": dict(h=16, hkv=8, hd=128, hidden=1024, scale=128 ** -0.5, norms="qk", angles=64,
                 theta=1e6),
    "mistral": dict(h=32, hkv=8, hd=128, hidden=4096, scale=128 ** -0.5, norms="", angles=64,
                    theta=1e6),
    "gemma": dict(h=16, hkv=8, hd=256, hidden=0, scale=1.0, norms="qkv", angles=32, theta=1e6),
}
EPS = 1e-6
CACHE = {"f32": (eb.DType.F32, torch.float32, 4), "f16": (eb.DType.F16, torch.float16, 2),
         "f8": (eb.DType.F8E4M3, torch.float8_e4m3fn, 1)}


# ------------------------------------------------------------------------------ the cases

def _attend(kind, model, rows, pos, cache="f32", window=0, max_seq=0):
    return dict(kind=kind, model=model, rows=rows, pos=pos, cache=cache, window=window,
                max_seq=max_seq or max(256, 1 << (pos + rows - 1).bit_length()))


def listed():
    return [
        # A chat's first answer tokens: everything is small, latency and launches count.
        dict(name="qwen layer, token 100", **_attend("layer", "qwen", 1, 100)),
        # A token of a 7B model in the middle of a document, half cache.
        dict(name="mistral layer, token 6000, half", **_attend("layer", "mistral", 1, 6000, "f16")),
        # The longest context of the 7B shape: the whole cache is read for one token.
        dict(name="mistral step, 32768 keys", kind="step", model="mistral", keys=32768, cache="f32",
             window=0, max_seq=32768),
        # A global layer's token over a long narrow cache.
        dict(name="gemma qkv, token 12000, e4m3", **_attend("qkv", "gemma", 1, 12000, "f8")),
        # A short question.
        dict(name="qwen layer, prompt 64", **_attend("layer", "qwen", 64, 0)),
        # An ordinary prompt that the program keeps in a half cache.
        dict(name="qwen layer, prompt 1000, half", **_attend("layer", "qwen", 1000, 0, "f16")),
        # A long prompt of the 7B shape: the largest case.
        dict(name="mistral layer, prompt 4096", **_attend("layer", "mistral", 4096, 0)),
        # Norms, partial rotary and head_dim 256 of a global layer's prompt.
        dict(name="gemma qkv, prompt 2000", **_attend("qkv", "gemma", 2000, 0)),
        # A long prompt's next chunk (or the second turn of a chat) over an E4M3 cache.
        dict(name="mistral qkv, 256 rows at 8192, e4m3", **_attend("qkv", "mistral", 256, 8192, "f8")),
        # A local layer: a chunk with a sliding window.
        dict(name="gemma qkv, 500 rows at 3000, window 1024",
             **_attend("qkv", "gemma", 500, 3000, "f32", 1024)),
        # A prompt in the f16 mode, where a program can do with its tolerance.
        dict(name="mistral prefill f16 mode, 3001", kind="prefill", model="mistral", mode="f16", rows=3001),
        # The end of every token: the LM head and the argmax.
        dict(name="qwen head", kind="head", rows=1, vocab=151936, hidden=1024),
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, even over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    what = rng.choice(("token", "prompt", "prompt", "chunk", "prefill", "step", "head"))
    model = rng.choice(sorted(MODELS))
    cache = rng.choice(sorted(CACHE))
    # E4M3 rows come through forward_qkv: behind a projection, whose last bits are free, a
    # few of their three-bit fractions would round either way.
    kind = "layer" if MODELS[model]["hidden"] and cache != "f8" else "qkv"
    window = rng.choice((0, 0, 1024)) if model == "gemma" else 0
    if what == "token":
        return _attend(kind, model, 1, _spread(rng, 16, 16000), cache, window)
    if what == "prompt":
        return _attend(kind, model, _spread(rng, 9, 4096), 0, cache, window)
    if what == "chunk":
        return _attend(kind, model, _spread(rng, 9, 700), _spread(rng, 64, 8192), cache, window)
    if what == "prefill":
        mode = rng.choice(("f32", "f16", "pv16") if model != "gemma" else ("f32", "pv16"))
        return dict(kind="prefill", model=model, mode=mode, rows=_spread(rng, 32, 4096))
    if what == "step":
        keys = _spread(rng, 256, 32768)
        return dict(kind="step", model=model, keys=keys, cache=cache, window=window,
                    max_seq=keys + rng.randrange(512))
    # Heads from the Mistral size (32768 x 4096) to the Qwen one (151936 x 1024).
    hidden = 128 * rng.randint(8, 32)
    return dict(kind="head", rows=rng.choice((1, 1, 2, 3)), hidden=hidden,
                vocab=_spread(rng, 30000, 155000000 // hidden))


# ---------------------------------------------------------------------------- the inputs

def _inputs(case, seed):
    """The case's inputs as torch tensors, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    kind = case["kind"]
    if kind == "head":
        vocab, hidden = case["vocab"], case["hidden"]
        return {"x": normal(case["rows"], hidden),
                "w": (normal(vocab, hidden) / math.sqrt(hidden)).half()}
    m = MODELS[case["model"]]
    h, hkv, hd, hidden = m["h"], m["hkv"], m["hd"], m["hidden"]
    if kind == "prefill":
        n = case["rows"]
        return {"q": normal(n, h, hd), "k": normal(n, hkv, hd), "v": normal(n, hkv, hd)}
    t = CACHE[case["cache"]][1]
    d = {"kc": normal(case["max_seq"], hkv, hd).to(t), "vc": normal(case["max_seq"], hkv, hd).to(t)}
    if kind == "step":
        d.update(q=normal(h, hd), k=normal(1, hkv, hd), v=normal(1, hkv, hd))
        return d
    for n in m["norms"]:
        # Gemma's V norm has no learned gain.
        d[n + "_norm"] = (torch.ones(hd, device="cuda") if n == "v" else 1 + 0.1 * normal(hd))
    if kind == "layer":
        d["x"] = normal(case["rows"], hidden)
        for n, o, i in (("q", h * hd, hidden), ("k", hkv * hd, hidden), ("v", hkv * hd, hidden),
                        ("o", hidden, h * hd)):
            d["w" + n] = (normal(o, i) / math.sqrt(i)).half()
    else:
        d.update(q=normal(case["rows"], h * hd), k=normal(case["rows"], hkv * hd),
                 v=normal(case["rows"], hkv * hd))
    return d


# ------------------------------------------------------------------- the library's tensors

class _Memory:
    """A library tensor's memory as torch reads it. It does not own it: the state does."""
    TYPES = {eb.DType.F32: "<f4", eb.DType.F16: "<f2", eb.DType.U32: "<i4", eb.DType.F8E4M3: "|u1"}

    def __init__(self, ptr, shape, dtype):
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=shape, strides=None,
                                             typestr=self.TYPES[dtype], version=2)


_devices = []


def _device():
    if not _devices:
        _devices.append(eb.Device.new(0))
    return _devices[0]


def _view(t):
    return torch.as_tensor(_Memory(t.data_ptr, t.shape, t.dtype), device="cuda")


def _tensor(x, dtype=eb.DType.F32):
    """x (a torch tensor) in a library tensor."""
    t = eb.Tensor.empty(_device(), tuple(x.shape), dtype)
    _view(t).copy_(x.view(torch.uint8) if dtype == eb.DType.F8E4M3 else x)
    return t


# ------------------------------------------------------------------------ prepare and run

def prepare(case, seed):
    dev = _device()
    dev.synchronize()  # pooled buffers may still be read by an earlier call
    d = _inputs(case, seed)
    kind = case["kind"]
    s = {"case": case, "dev": dev, "views": {}}
    if kind == "head":
        s.update(x=_tensor(d["x"]), w=_tensor(d["w"], eb.DType.F16),
                 logits=eb.Tensor.empty(dev, (case["rows"], case["vocab"])),
                 token=eb.Tensor.empty(dev, (1,), eb.DType.U32))
        s["result"] = {"logits": _view(s["logits"]), "token": _view(s["token"])}
        torch.cuda.synchronize()
        return s
    m = MODELS[case["model"]]
    h, hkv, hd = m["h"], m["hkv"], m["hd"]
    if kind == "prefill":
        s.update(q=_tensor(d["q"]), k=_tensor(d["k"]), v=_tensor(d["v"]),
                 o=eb.Tensor.empty(dev, (case["rows"], h, hd)))
        s["result"] = {"out": _view(s["o"])}
        torch.cuda.synchronize()
        return s
    dt = CACHE[case["cache"]][0]
    kv = eb.KvCache.new(dev, 1, case["max_seq"], hkv, hd, dt)
    s["kv"] = kv
    s["result"] = {}
    for n, t in (("k", kv.k[0]), ("v", kv.v[0])):
        view = _view(t)
        x = d[n + "c"]
        view.copy_(x.view(torch.uint8) if dt == eb.DType.F8E4M3 else x)
        s["result"][n + "_cache"] = view
    if kind == "step":
        s.update(q=_tensor(d["q"]), k=_tensor(d["k"]), v=_tensor(d["v"]),
                 o=eb.Tensor.empty(dev, (h, hd)))
        s["result"]["out"] = _view(s["o"])
        torch.cuda.synchronize()
        return s
    s["rope"] = eb.Rope.build_partial(dev, case["max_seq"], hd, m["angles"], m["theta"])
    s["weights"] = {n: _tensor(d[n]) for n in ("q_norm", "k_norm", "v_norm") if n in d}
    if kind == "layer":
        s["weights"].update({n + "_proj": _tensor(d["w" + n], eb.DType.F16) for n in "qkvo"})
        s["x"] = _tensor(d["x"])
    else:
        s.update(q=_tensor(d["q"]), k=_tensor(d["k"]), v=_tensor(d["v"]))
    s["attn"] = eb.Attention(h, hkv, hd, m["scale"], norm_eps=EPS, window=case["window"],
                             hidden=m["hidden"], **s["weights"])
    torch.cuda.synchronize()
    return s


def run(s):
    case, dev = s["case"], s["dev"]
    kind = case["kind"]
    rec = eb.Recorder(dev)
    if kind == "head":
        rows, vocab, hidden = case["rows"], case["vocab"], case["hidden"]
        eb.linear_f16w(rec, s["x"], s["w"], s["logits"], rows, hidden, vocab)
        eb.argmax(rec, s["logits"], s["token"], vocab)  # the first row's token
        rec.submit()
        return s["result"]
    m = MODELS[case["model"]]
    h, hkv, hd = m["h"], m["hkv"], m["hd"]
    if kind == "prefill":
        f = {"f32": eb.attn_prefill, "f16": eb.attn_prefill_fast, "pv16": eb.attn_prefill_pv16}
        f[case["mode"]](rec, s["q"], s["k"], s["v"], s["o"], h, hkv, case["rows"], hd, m["scale"])
        rec.submit()
        return s["result"]
    if kind == "step":
        kc, vc = s["kv"].k[0], s["kv"].v[0]
        eb.attn_decode_step_window(rec, s["q"], s["k"], s["v"], kc, vc, s["o"], h, hkv,
                                   case["keys"] - 1, hd, case["max_seq"], m["scale"],
                                   case["window"])
        rec.submit()
        return s["result"]
    if kind == "layer":
        out = s["attn"].forward(rec, s["x"], s["rope"], s["kv"], 0, case["rows"], case["pos"])
    else:
        out = s["attn"].forward_qkv(rec, s["q"], s["k"], s["v"], s["rope"], s["kv"], 0,
                                    case["rows"], case["pos"])
    rec.submit()
    # The output's memory comes from the device's pool: the state keeps it until its next
    # pass, and a view of memory seen before is made once.
    s["out"] = out
    ptr = out.data_ptr
    view = s["views"].get(ptr)
    if view is None:
        view = s["views"][ptr] = _view(out)
    return {"out": view, **s["result"]}


# -------------------------------------------------------------------- what a pass has to do

def _span(case):
    """(first key any row reads, visible query-key pairs) of an attention case."""
    rows, pos, window = case["rows"], case["pos"], case["window"]
    w = window or pos + rows
    first = max(0, pos - w + 1)
    pairs = sum(min(w, p + 1) for p in range(pos, pos + rows))
    return first, pairs


def work(case):
    kind = case["kind"]
    if kind == "head":
        rows, vocab, hidden = case["rows"], case["vocab"], case["hidden"]
        return {"bytes": 2 * vocab * hidden + 4 * rows * (vocab + hidden), "flops": 2 * rows * vocab * hidden}
    m = MODELS[case["model"]]
    h, hkv, hd, hidden = m["h"], m["hkv"], m["hd"], m["hidden"]
    if kind == "prefill":
        n = case["rows"]
        return {"bytes": 4 * n * hd * 2 * (h + hkv), "flops": 2 * h * hd * n * (n + 1)}
    size = CACHE[case["cache"]][2]
    if kind == "step":
        keys = min(case["keys"], case["window"] or case["keys"])
        return {"bytes": 2 * keys * hkv * hd * size + 8 * h * hd + 8 * hkv * hd,
                "flops": 4 * h * hd * keys}
    rows, pos = case["rows"], case["pos"]
    first, pairs = _span(case)
    cache = 2 * hkv * hd * size * (pos - first + rows)  # older keys read, new rows written
    flops = 4 * h * hd * pairs
    if kind == "qkv":
        return {"bytes": cache + 4 * rows * hd * 2 * (h + hkv), "flops": flops}
    weights = hidden * hd * 2 * (h + hkv)
    return {"bytes": cache + 2 * weights + 8 * rows * hidden, "flops": flops + 2 * rows * weights}


def tolerance(case):
    # About four times the distance from the 64-bit results, measured over many draws.
    kind = case["kind"]
    if kind == "prefill" and case["mode"] == "f16":
        return {"rel": 1.5e-3}  # 3.7e-4
    if kind == "prefill" and case["mode"] == "pv16":
        return {"rel": 1e-3}  # 2.7e-4
    if kind == "layer" and case["cache"] == "f16":
        # 2.2e-5: new rows whose last bits come from a projection round to one of two halves.
        return {"rel": 1e-4}
    if kind in ("layer", "qkv") and case["cache"] == "f8":
        # 3.5e-5: normed rows may round to a neighbouring E4M3 value here and there.
        return {"rel": 1.5e-4, "differ": 1e-4}
    return {"rel": 1e-5}  # 2e-7 to 2.5e-6


# ------------------------------------------------------------------------- 64-bit results

def _rounded(x, cache):
    """x as the cache holds it."""
    return x if cache == "f32" else x.float().to(CACHE[cache][1]).double()


def _attention(q, k, v, pos, scale, window):
    """Rows of q [rows, h, hd] at pos.. over keys k, v [keys, hkv, hd], in 64 bits."""
    rows, h, hd = q.shape
    g = h // k.shape[1]
    out = torch.empty_like(q)
    for head in range(h):
        kh, vh = k[:, head // g], v[:, head // g].contiguous()
        for r0 in range(0, rows, 1024):
            r1 = min(rows, r0 + 1024)
            lo = max(0, pos + r0 - window + 1) if window else 0
            hi = pos + r1
            s = (q[r0:r1, head] * scale) @ kh[lo:hi].t().contiguous()
            at = torch.arange(pos + r0, pos + r1, device=q.device)[:, None]
            key = torch.arange(lo, hi, device=q.device)[None]
            seen = key <= at
            if window:
                seen &= key > at - window
            out[r0:r1, head] = torch.softmax(s.masked_fill(~seen, -math.inf), 1) @ vh[lo:hi]
    return out


def _norm(x, gain):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gain.double()


def _rotate(x, pos, angles, theta):
    """RoPE of x [rows, heads, hd] at pos..: pair (p, p + hd/2), the first `angles` turned."""
    rows, _, hd = x.shape
    p = torch.arange(hd // 2, device=x.device, dtype=torch.float64)
    a = torch.arange(pos, pos + rows, device=x.device, dtype=torch.float64)[:, None] * theta ** (-2 * p / hd)
    a = torch.where(p < angles, a, torch.zeros_like(a))
    c, s = a.cos().float().double()[:, None], a.sin().float().double()[:, None]
    x1, x2 = x[..., : hd // 2], x[..., hd // 2:]
    return torch.cat((x1 * c - x2 * s, x2 * c + x1 * s), -1)


def exact(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "head":
        out = torch.cat([d["x"].double() @ w.double().t().contiguous() for w in d["w"].split(16384)], 1)
        return {"logits": out, "token": None}
    m = MODELS[case["model"]]
    h, hkv, hd = m["h"], m["hkv"], m["hd"]
    if kind == "prefill":
        return {"out": _attention(d["q"].double(), d["k"].double(), d["v"].double(), 0, m["scale"], 0)}
    cache = case["cache"]
    kc, vc = d["kc"].double(), d["vc"].double()
    if kind == "step":
        rows, pos = 1, case["keys"] - 1
        q, k, v = (d[n].double().view(1, -1, hd) for n in "qkv")
    else:
        rows, pos = case["rows"], case["pos"]
        if kind == "layer":
            x = d["x"].double()
            q, k, v = (x @ d["w" + n].double().t().contiguous() for n in "qkv")
        else:
            q, k, v = (d[n].double() for n in "qkv")
        q, k, v = q.view(rows, h, hd), k.view(rows, hkv, hd), v.view(rows, hkv, hd)
        if "q_norm" in d:
            q, k = _norm(q, d["q_norm"]), _norm(k, d["k_norm"])
        if "v_norm" in d:
            v = _norm(v, d["v_norm"])
        q, k = (_rotate(t, pos, m["angles"], m["theta"]) for t in (q, k))
    kc[pos:pos + rows], vc[pos:pos + rows] = _rounded(k, cache), _rounded(v, cache)
    out = _attention(q, kc[:pos + rows], vc[:pos + rows], pos, m["scale"], case["window"])
    if kind == "step":
        out = out.view(h, hd)
    else:
        out = out.reshape(rows, h * hd)
    if kind == "layer":
        out = out @ d["wo"].double().t().contiguous()
    caches = {} if cache == "f8" else {"k_cache": kc, "v_cache": vc}
    return {"out": out, "k_cache": None, "v_cache": None, **caches}
