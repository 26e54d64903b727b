"""What a program that uses popcorn_amd has it do, as cases that can be timed.

Every case goes through the public entry points (`Kernels.*` descriptors made
once and encoded on one stream, or the `Decoder`). Five kinds of work:

* ``decode_ops``: one token through a layer's decode operations, encoded one
  after the other (KV-cache write, split-KV attention, gated MLP).
* ``decoder``: one greedy token through a whole Gemma-shaped decoder, with
  bf16 or 4-bit weights, with or without the per-head norms and RoPE.
* ``attention``: one ``FlashAttention`` call: a token against its cache (one
  sequence or a batch), a few tokens at once (a verified draft, the tail of a
  chunked prompt), a prompt from nothing, a chunk of a prompt behind a cache.
* ``matmul``: one projection of 1 to 4096 rows: f16, bf16, f32 and 4-bit.
* ``layer``: a prompt's rows through one whole decoder layer, operation by
  operation, as a program without a fused step runs it.

Sizes are those of the repository's own decoder and prefill configurations
(the Gemma-2-2B and Gemma-7B shapes), or generic.
"""
import math

import torch

import popcorn_amd as pa
from popcorn_amd.decoder import Decoder, DecoderConfig

TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}
EPS = 1e-6
_ENV = []


def _env():
    """The library, stream and encoder that a program makes once."""
    if not _ENV:
        lib, stream = pa.KernelLibrary(), pa.Stream()
        _ENV.extend((lib, stream, pa.KernelCommandEncoder(lib, stream)))
    return _ENV


def _t(x, dtype=None):
    """The framework's view of a torch tensor."""
    if dtype is None:
        dtype = {torch.float32: "f32", torch.float16: "f16", torch.bfloat16: "bf16", torch.int32: "i32"}[x.dtype]
    return pa.Tensor(x.data_ptr(), tuple(x.shape), dtype, owner=[x])


class _DeviceView:
    def __init__(self, t):
        self.tensor = t  # keeps the memory's owner
        kind = {"f32": "<f4", "bf16": "<i2", "u32": "<i4", "i32": "<i4"}[t.dtype]
        self.__cuda_array_interface__ = {"shape": t.shape, "typestr": kind, "data": (t.ptr, False), "version": 3}


def _torch(t):
    """A torch view of a framework tensor's memory."""
    x = torch.as_tensor(_DeviceView(t), device="cuda")
    return x.view(torch.bfloat16) if t.dtype == "bf16" else x


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, shape, dtype, std=1.0, mean=0.0):
    return torch.randn(shape, device="cuda", generator=g).mul_(std).add_(mean).to(TORCH[dtype])


def _norm_weight(g, n):
    return _normal(g, (n,), "f32", 0.1, 1.0)


def _quantized(g, n, k):
    """4-bit values, group 64, bf16 scale and bias: about N(0, 0.02) weights."""
    packed = torch.randint(-2**31, 2**31, (n, k // 8), device="cuda", generator=g).to(torch.int32)
    scales = (0.002 + 0.005 * torch.rand((n, k // 64), device="cuda", generator=g)).to(torch.bfloat16)
    biases = (scales.float() * (-7.5 + torch.randn((n, k // 64), device="cuda", generator=g))).to(torch.bfloat16)
    return packed, scales, biases


def _weight(g, n, k, kind, std=0.02):
    return _quantized(g, n, k) if kind == "q4" else _normal(g, (n, k), kind, std)


def _tw(w, n, k):
    if not isinstance(w, tuple):
        return _t(w)
    p, s, b = w
    return pa.AffineQuantizedTensor(_t(p, "u32"), _t(s), _t(b), [n, k])


def _dense64(w):
    """A weight's values in 64 bits."""
    if not isinstance(w, tuple):
        return w.double()
    p, s, b = w
    q = (p.unsqueeze(-1) >> torch.arange(0, 32, 4, device=p.device, dtype=torch.int32)) & 15
    q = q.reshape(s.shape[0], s.shape[1], 64).double()
    return (q * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).reshape(s.shape[0], -1)


def _rms64(x, w=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w.double()


def _gelu64(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _rope64(x, cos, sin):
    a, b = x.chunk(2, -1)
    return torch.cat((a * cos - b * sin, a * sin + b * cos), -1)


def _attention64(q, k, v, scale, mask="causal", window=0):
    """q [Nq, Sq, Hd] against k, v [Nkv, Sk, Hd], in 64 bits."""
    nq, sq, hd = q.shape
    nkv, sk, _ = k.shape
    out = torch.empty(nq, sq, hd, dtype=torch.float64, device=q.device)
    i = torch.arange(sq, device=q.device).unsqueeze(1) + sk - sq
    j = torch.arange(sk, device=q.device).unsqueeze(0)
    seen = torch.ones(sq, sk, dtype=torch.bool, device=q.device) if mask == "all" else j <= i
    if mask == "window":
        seen = seen & (j > i - window)
    per = nq // nkv
    for h in range(nkv):
        kt, vd = k[h].double().t().contiguous(), v[h].double()
        for a in range(h * per, (h + 1) * per):
            s = (q[a].double() @ kt) * scale
            out[a] = torch.softmax(s.masked_fill_(~seen, -math.inf), -1) @ vd
    return out


# ---- decode_ops ------------------------------------------------------------------


def _decode_ops_inputs(c, seed):
    g, t = _gen(seed), c["dtype"]
    nq, nkv, hd, cap, h, f = c["nq"], c["nkv"], c["hd"], c["cap"], c["nq"] * c["hd"], c["ffn"]
    return {
        "k_new": _normal(g, (1, nkv, 1, hd), t), "v_new": _normal(g, (1, nkv, 1, hd), t),
        "q": _normal(g, (1, nq, 1, hd), t), "k": _normal(g, (1, nkv, cap, hd), t), "v": _normal(g, (1, nkv, cap, hd), t),
        "norm": _norm_weight(g, h), "gate": _normal(g, (f, h), t, 0.02), "up": _normal(g, (f, h), t, 0.02),
        "down": _normal(g, (h, f), t, 0.02)}


def _decode_ops_prepare(c, seed):
    lib, stream, enc = _env()
    x = _decode_ops_inputs(c, seed)
    nq, nkv, hd, cap, pos = c["nq"], c["nkv"], c["hd"], c["cap"], c["pos"]
    attn = torch.empty(1, nq, 1, hd, device="cuda", dtype=TORCH[c["dtype"]])
    out = torch.empty(nq * hd, device="cuda", dtype=TORCH[c["dtype"]])
    d = {n: _t(v) for n, v in x.items()}
    kernels = [
        pa.Kernels.KVCacheWrite(d["k_new"], d["k"], pos), pa.Kernels.KVCacheWrite(d["v_new"], d["v"], pos),
        pa.Kernels.FlashAttention(d["q"], d["k"], d["v"], out=_t(attn), scale=hd ** -0.5, batch=1, query_heads=nq,
                                  kv_heads=nkv, query_len=1, key_len=pos + 1, head_dim=hd, key_capacity=cap),
        pa.Kernels.GatedMLP(_t(attn).view([nq * hd]), d["norm"], d["gate"], d["up"], d["down"], _t(out), eps=EPS)]
    return {"enc": enc, "kernels": kernels, "keep": x, "out": (attn, out, x["k"], x["v"])}


def _decode_ops_exact(c, seed):
    x, pos = _decode_ops_inputs(c, seed), c["pos"]
    k, v = x["k"].double(), x["v"].double()
    k[:, :, pos], v[:, :, pos] = x["k_new"][:, :, 0].double(), x["v_new"][:, :, 0].double()
    attn = _attention64(x["q"][0], k[0, :, :pos + 1], v[0, :, :pos + 1], c["hd"] ** -0.5).unsqueeze(0)
    n = _rms64(attn.reshape(1, -1), x["norm"])
    h = _gelu64(n @ x["gate"].double().t()) * (n @ x["up"].double().t())
    return attn, (h @ x["down"].double().t()).reshape(-1), k, v


# ---- decoder -----------------------------------------------------------------------


def _decoder_config(c):
    return DecoderConfig(layers=c["layers"], hidden=c["hidden"], query_heads=c["nq"], kv_heads=c["nkv"],
                         head_dim=c["hd"], ffn=c["ffn"], vocab=c["vocab"], max_seq=c["cap"], eps=EPS,
                         attn_scale=c["hd"] ** -0.5, history_len=c["cap"], graph_steps=1,
                         attention_block=int(c["block"]), weight_bits=4 if c["weights"] == "q4" else 16)


def _decoder_weights(c, seed):
    """(name, layer, tensor or 4-bit triple) of every input the decoder keeps."""
    g = _gen(seed)
    h, qw, kw, hd, f = c["hidden"], c["nq"] * c["hd"], c["nkv"] * c["hd"], c["hd"], c["ffn"]
    kind = c["weights"]
    yield "embedding", 0, _weight(g, c["vocab"], h, kind)
    yield "final_norm", 0, _norm_weight(g, h)
    for l in range(c["layers"]):
        yield "w_qkv", l, _weight(g, qw + 2 * kw, h, kind)
        yield "w_o", l, _weight(g, h, qw, kind)
        yield "w_gate", l, _weight(g, f, h, kind)
        yield "w_up", l, _weight(g, f, h, kind)
        yield "w_down", l, _weight(g, h, f, kind)
        for n in ("norm_in", "norm_post_attn", "norm_pre_ffn", "norm_post_ffn"):
            yield n, l, _norm_weight(g, h)
        if c["block"]:
            yield "q_norm", l, _norm_weight(g, hd)
            yield "k_norm", l, _norm_weight(g, hd)
        yield "k_cache", l, _normal(g, (1, c["nkv"], c["cap"], hd), "bf16")
        yield "v_cache", l, _normal(g, (1, c["nkv"], c["cap"], hd), "bf16")


def _token(c, seed):
    return (seed * 7919 + 123) % c["vocab"]


def _decoder_prepare(c, seed):
    lib, stream, _ = _env()
    dec = Decoder(lib, stream, _decoder_config(c))
    dec.randomize(seed)
    stream.synchronize()
    for name, l, w in _decoder_weights(c, seed):
        if isinstance(w, tuple):
            for part, v in zip(("", ".scales", ".biases"), w):
                _torch(dec.tensor(name + part, l)).copy_(v)
        else:
            _torch(dec.tensor(name, l)).copy_(w.reshape(dec.tensor(name, l).shape))
    torch.cuda.synchronize()
    last = c["layers"] - 1
    # the graph is recorded when the decoder is set up, as a serving program does
    dec.reset(_token(c, seed), c["pos"])
    dec.step(1)
    dec.read()
    return {"dec": dec, "token": _token(c, seed), "pos": c["pos"],
            "out": tuple(_torch(dec.tensor(n, last)) for n in ("logits", "k_cache", "v_cache"))}


def _decoder_exact(c, seed):
    h, nq, nkv, hd, pos = c["hidden"], c["nq"], c["nkv"], c["hd"], c["pos"]
    w, shared = {}, {}
    x = None
    if c["block"]:
        inv = torch.tensor([10000.0 ** (-2.0 * i / hd) for i in range(hd // 2)], device="cuda").float().double()
        cos, sin = torch.cos(pos * inv), torch.sin(pos * inv)
    for name, l, v in _decoder_weights(c, seed):
        if name in ("embedding", "final_norm"):
            shared[name] = v
            continue
        w[name] = v
        if name != "v_cache":
            continue
        if x is None:
            e = shared["embedding"]
            t = _token(c, seed)
            x = _dense64(tuple(p[t:t + 1] for p in e) if isinstance(e, tuple) else e[t:t + 1]) * math.sqrt(h)
        n = _rms64(x, w["norm_in"])
        qkv = (n @ _dense64(w["w_qkv"]).t()).reshape(-1, hd)
        q, k, v = qkv[:nq], qkv[nq:nq + nkv], qkv[nq + nkv:]
        if c["block"]:
            q, k, v = _rope64(_rms64(q, w["q_norm"]), cos, sin), _rope64(_rms64(k, w["k_norm"]), cos, sin), _rms64(v)
        kc, vc = w["k_cache"].double(), w["v_cache"].double()
        kc[0, :, pos], vc[0, :, pos] = k, v
        a = _attention64(q.unsqueeze(1), kc[0, :, :pos + 1], vc[0, :, :pos + 1], hd ** -0.5).reshape(1, -1)
        x = x + _rms64(a @ _dense64(w["w_o"]).t(), w["norm_post_attn"])
        n = _rms64(x, w["norm_pre_ffn"])
        m = (_gelu64(n @ _dense64(w["w_gate"]).t()) * (n @ _dense64(w["w_up"]).t())) @ _dense64(w["w_down"]).t()
        x = x + _rms64(m, w["norm_post_ffn"])
        w.clear()
    n = _rms64(x, shared["final_norm"])
    e, logits = shared["embedding"], []
    for i in range(0, c["vocab"], 32768):
        part = tuple(p[i:i + 32768] for p in e) if isinstance(e, tuple) else e[i:i + 32768]
        logits.append(n @ _dense64(part).t())
    return torch.cat(logits, 1), kc, vc


# ---- attention ---------------------------------------------------------------------


def _attention_inputs(c, seed):
    g, t = _gen(seed), c["dtype"]
    return (_normal(g, (c["batch"], c["nq"], c["sq"], c["hd"]), t),
            _normal(g, (c["batch"], c["nkv"], c["cap"], c["hd"]), t),
            _normal(g, (c["batch"], c["nkv"], c["cap"], c["hd"]), t))


def _mask(c):
    if c["mask"] == "window":
        return pa.AttentionMask.causal_sliding_window(c["window"])
    return pa.AttentionMask.bidirectional if c["mask"] == "all" else pa.AttentionMask.causal


def _attention_prepare(c, seed):
    lib, stream, enc = _env()
    q, k, v = _attention_inputs(c, seed)
    out = torch.empty_like(q)
    kernel = pa.Kernels.FlashAttention(_t(q), _t(k), _t(v), out=_t(out), scale=c["hd"] ** -0.5, mask=_mask(c),
                                       batch=c["batch"], query_heads=c["nq"], kv_heads=c["nkv"], query_len=c["sq"],
                                       key_len=c["sk"], head_dim=c["hd"], key_capacity=c["cap"])
    return {"enc": enc, "kernels": [kernel], "keep": (q, k, v), "out": out}


def _attention_exact(c, seed):
    q, k, v = _attention_inputs(c, seed)
    return torch.stack([_attention64(q[b], k[b, :, :c["sk"]], v[b, :, :c["sk"]], c["hd"] ** -0.5, c["mask"], c["window"])
                        for b in range(c["batch"])])


def _pairs_seen(c):
    """Query-key pairs that the mask lets through, of one head."""
    total, past = 0, c["sk"] - c["sq"]
    for i in range(c["sq"]):
        n = c["sk"] if c["mask"] == "all" else past + i + 1
        total += min(n, c["window"]) if c["mask"] == "window" else n
    return total


def _keys_seen(c):
    """Keys that some query of the call sees."""
    if c["mask"] == "window":
        return min(c["sk"], c["window"] + c["sq"] - 1)
    return c["sk"]


# ---- matmul ------------------------------------------------------------------------


def _act(kind):
    return "bf16" if kind == "q4" else kind


def _matmul_inputs(c, seed):
    g = _gen(seed)
    return _normal(g, (c["m"], c["k"]), _act(c["kind"])), _weight(g, c["n"], c["k"], c["kind"])


def _matmul_prepare(c, seed):
    lib, stream, enc = _env()
    a, w = _matmul_inputs(c, seed)
    out = torch.empty(c["m"], c["n"], device="cuda", dtype=a.dtype)
    tw = _tw(w, c["n"], c["k"])
    kernel = pa.Kernels.Matmul(_t(a), tw, _t(out)) if c["kind"] == "q4" else pa.Kernels.Matmul(_t(a), tw, _t(out), True)
    return {"enc": enc, "kernels": [kernel], "keep": (a, w), "out": out}


def _matmul_exact(c, seed):
    a, w = _matmul_inputs(c, seed)
    return a.double() @ _dense64(w).t()


def _weight_bytes(kind, n, k):
    return n * k // 2 + n * (k // 64) * 4 if kind == "q4" else n * k * SIZE[kind]


# ---- layer -------------------------------------------------------------------------


def _layer_inputs(c, seed):
    g, kind = _gen(seed), c["weights"]
    m, h, nq, nkv, hd, f = c["m"], c["hidden"], c["nq"], c["nkv"], c["hd"], c["ffn"]
    x = {"x": _normal(g, (m, h), "bf16")}
    for n, rows, cols in (("wq", nq * hd, h), ("wk", nkv * hd, h), ("wv", nkv * hd, h), ("wo", h, nq * hd),
                          ("wg", f, h), ("wu", f, h), ("wd", h, f)):
        x[n] = _weight(g, rows, cols, kind)
    for n in ("n_in", "n_post_attn", "n_pre_ffn", "n_post_ffn"):
        x[n] = _norm_weight(g, h)
    x["n_q"], x["n_k"] = _norm_weight(g, hd), _norm_weight(g, hd)
    x["k"], x["v"] = (_normal(g, (1, nkv, c["cap"], hd), "bf16") for _ in range(2))
    x["inv_freq"] = torch.tensor([10000.0 ** (-2.0 * i / hd) for i in range(hd // 2)], device="cuda").float()
    x["positions"] = torch.arange(c["past"], c["past"] + m, device="cuda", dtype=torch.int32)
    return x


def _layer_prepare(c, seed):
    lib, stream, enc = _env()
    K = pa.Kernels
    x = _layer_inputs(c, seed)
    m, h, nq, nkv, hd, f, past = c["m"], c["hidden"], c["nq"], c["nkv"], c["hd"], c["ffn"], c["past"]
    keep, ks = [x], []

    def new(*shape, dtype="bf16"):
        y = torch.empty(shape, device="cuda", dtype=TORCH[dtype])
        keep.append(y)
        return _t(y)

    def matmul(a, name, rows, cols):
        y, w = new(m, rows), _tw(x[name], rows, cols)
        ks.append(K.Matmul(a, w, y) if isinstance(x[name], tuple) else K.Matmul(a, w, y, True))
        return y

    def norm(a, name=None, shape=None):
        y = new(*a.shape)
        src, dst = (a, y) if shape is None else (a.view(shape), y.view(shape))
        ks.append(K.RMSNorm(src, _t(x[name]) if name else None, dst, eps=EPS))
        return y

    def heads(a, n, name, rotate):
        shape = [1, m, n, hd]
        y = norm(a, name, shape)
        if rotate:
            r = new(1, m, n, hd)
            ks.append(K.RopeApply(y.view(shape), cos, sin, r))
            y = r
        z = new(1, n, m, hd)
        ks.append(K.Transpose12(y.view(shape), z))
        return z

    cos, sin = new(m, hd // 2, dtype="f32"), new(m, hd // 2, dtype="f32")
    ks.append(K.RopeBuildCosSin(_t(x["positions"]), _t(x["inv_freq"]), cos, sin))
    tx, kc, vc = _t(x["x"]), _t(x["k"]), _t(x["v"])
    n = norm(tx, "n_in")
    q, k, v = matmul(n, "wq", nq * hd, h), matmul(n, "wk", nkv * hd, h), matmul(n, "wv", nkv * hd, h)
    q, k, v = heads(q, nq, "n_q", True), heads(k, nkv, "n_k", True), heads(v, nkv, None, False)
    ks += [K.KVCacheWrite(k, kc, past), K.KVCacheWrite(v, vc, past)]
    a, at = new(1, nq, m, hd), new(1, m, nq, hd)
    ks += [K.FlashAttention(q, kc, vc, out=a, scale=hd ** -0.5, batch=1, query_heads=nq, kv_heads=nkv, query_len=m,
                            key_len=past + m, head_dim=hd, key_capacity=c["cap"]),
           K.Transpose12(a, at)]
    o = norm(matmul(at.view([m, nq * hd]), "wo", h, nq * hd), "n_post_attn")
    x2 = new(m, h)
    ks.append(K.Add(tx, o, x2))
    n = norm(x2, "n_pre_ffn")
    gate, up = matmul(n, "wg", f, h), matmul(n, "wu", f, h)
    act, hid = new(m, f), new(m, f)
    ks += [K.GeluTanh(gate, act), K.Mul(act, up, hid)]
    d = norm(matmul(hid, "wd", h, f), "n_post_ffn")
    out = new(m, h)
    ks.append(K.Add(x2, d, out))
    return {"enc": enc, "kernels": ks, "keep": keep, "out": (out.owner[0], x["k"], x["v"])}


def _layer_exact(c, seed):
    x = _layer_inputs(c, seed)
    m, nq, nkv, hd, past = c["m"], c["nq"], c["nkv"], c["hd"], c["past"]
    angle = x["positions"].double().unsqueeze(1) * x["inv_freq"].double()
    cos, sin = torch.cos(angle), torch.sin(angle)
    w = {n: _dense64(x[n]).t() for n in ("wq", "wk", "wv", "wo", "wg", "wu", "wd")}
    x0 = x["x"].double()
    n = _rms64(x0, x["n_in"])

    def heads(name, count):
        return (n @ w[name]).reshape(m, count, hd).transpose(0, 1).contiguous()

    q, k = _rope64(_rms64(heads("wq", nq), x["n_q"]), cos, sin), _rope64(_rms64(heads("wk", nkv), x["n_k"]), cos, sin)
    kc, vc = x["k"].double(), x["v"].double()
    kc[0, :, past:past + m], vc[0, :, past:past + m] = k, _rms64(heads("wv", nkv))
    a = _attention64(q, kc[0, :, :past + m], vc[0, :, :past + m], hd ** -0.5)
    x2 = x0 + _rms64(a.transpose(0, 1).reshape(m, -1) @ w["wo"], x["n_post_attn"])
    n = _rms64(x2, x["n_pre_ffn"])
    return x2 + _rms64((_gelu64(n @ w["wg"]) * (n @ w["wu"])) @ w["wd"], x["n_post_ffn"]), kc, vc


# ---- the cases ---------------------------------------------------------------------


def _case(work_kind, name=None, **sizes):
    return dict(({"name": name} if name else {}), work=work_kind, **sizes)


def listed():
    a = dict(batch=1, nq=8, nkv=4, hd=256, mask="causal", window=0)
    gemma2 = dict(hidden=2304, nq=8, nkv=4, hd=256, ffn=9216)
    return [
        # the smallest calls: a toy model's token in f32, all latency and launches
        _case("decode_ops", "decode_ops_tiny_f32", dtype="f32", nq=4, nkv=1, hd=64, cap=160, pos=128, ffn=1024),
        # one stream of chat at 4096 tokens of context
        _case("decoder", "decode_step_bf16", layers=26, vocab=256000, cap=4352, pos=4096, block=False, weights="bf16",
              **gemma2),
        # the same model quantized, early in a conversation, with the full attention block
        _case("decoder", "decode_step_q4", layers=26, vocab=256000, cap=2048, pos=1001, block=True, weights="q4",
              **gemma2),
        # a server's batch of 32 sequences, one token each
        _case("attention", "attention_decode_b32", dtype="f16", sq=1, sk=8192, cap=8192, **dict(a, batch=32)),
        # eight tokens at once behind a cache: a verified draft
        _case("attention", "attention_few_tokens", dtype="bf16", sq=8, sk=4104, cap=4352, **a),
        # a whole prompt from nothing
        _case("attention", "attention_prompt", dtype="f16", sq=2048, sk=2048, cap=2048, **dict(a, nq=16, nkv=16)),
        # a chunk of a long prompt behind its cache, with a ragged length
        _case("attention", "attention_chunk", dtype="bf16", sq=500, sk=8692, cap=9000, **a),
        # a long prompt's largest projection
        _case("matmul", "matmul_prompt_f16", kind="f16", m=2048, k=3072, n=24576),
        # a short prompt's down projection, with a ragged length
        _case("matmul", "matmul_short_bf16", kind="bf16", m=137, k=9216, n=2304),
        # eight sequences' rows through a quantized projection
        _case("matmul", "matmul_batch_q4", kind="q4", m=8, k=2304, n=9216),
        # a prompt through a quantized projection, with a ragged length
        _case("matmul", "matmul_prompt_q4", kind="q4", m=777, k=2304, n=9216),
        # a prompt's rows through a whole layer, operation by operation
        _case("layer", "layer_prompt", m=1000, past=0, cap=1024, weights="bf16", **gemma2),
    ]


PROJECTIONS = [(2304, 9216), (9216, 2304), (2304, 4096), (2048, 2304), (3072, 9216), (3072, 24576), (24576, 3072),
               (4096, 14336), (14336, 4096), (4096, 4096)]
HEADS = [(8, 4, 256), (16, 16, 256), (8, 1, 256), (32, 8, 128), (8, 2, 128), (4, 2, 64), (8, 2, 512)]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode_ops", "decoder", "attention", "attention", "attention", "matmul", "matmul", "matmul",
                       "layer"])
    if kind == "decode_ops":
        nq, nkv, hd = rng.choice([(4, 1, 64), (8, 2, 128), (8, 4, 256), (16, 4, 128)])
        cap = _log(rng, 32, 8192)
        return _case(kind, dtype=rng.choice(["f32", "bf16", "f16"]), nq=nq, nkv=nkv, hd=hd, cap=cap,
                     pos=rng.randrange(cap), ffn=rng.randrange(256, 9217, 8))
    if kind == "decoder":
        nq, nkv, hd = rng.choice([(8, 4, 256), (8, 1, 256), (16, 4, 128)])
        cap = _log(rng, 128, 16384)
        return _case(kind, layers=rng.randint(2, 12), hidden=128 * rng.randint(8, 28), nq=nq, nkv=nkv, hd=hd,
                     ffn=128 * rng.randint(16, 96), vocab=rng.randrange(8000, 256001, 4), cap=cap,
                     pos=rng.randrange(cap), block=rng.random() < 0.5, weights=rng.choice(["bf16", "q4"]))
    if kind == "attention":
        nq, nkv, hd = rng.choice(HEADS)
        phase = rng.choice(["decode", "few", "prompt", "chunk"])
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f16", "f32"])
        batch = 1
        if phase == "decode":
            sq, sk, batch = 1, _log(rng, 64, 32768), _log(rng, 1, 32)
            batch = max(1, min(batch, 1000000000 // (2 * nkv * sk * hd * SIZE[dtype])))
        elif phase == "few":
            sq, batch = rng.randint(2, 31), rng.choice([1, 1, 2, 4])
            sk = sq + _log(rng, 1, 16384)
        else:
            sq, batch = _log(rng, 32, 2048), rng.choice([1, 1, 1, 2])
            sk = sq + (_log(rng, 1, 16384) if phase == "chunk" else 0)
            most = 8e9 if dtype == "f32" else 60e9
            sq = max(32, min(sq, int(most / (4.0 * batch * nq * hd * sk))))
        mask = rng.choice(["causal", "causal", "causal", "window", "all"])
        return _case(kind, dtype=dtype, batch=batch, nq=nq, nkv=nkv, hd=hd, sq=sq, sk=sk,
                     cap=sk + rng.choice([0, rng.randint(1, 512)]), mask=mask,
                     window=_log(rng, 64, 4096) if mask == "window" else 0)
    if kind == "matmul":
        k, n = rng.choice(PROJECTIONS)
        form = rng.choice(["bf16", "bf16", "f16", "q4", "q4", "f32"])
        if rng.random() < 0.25:
            k, n = 128 * rng.randint(2, 64) if form == "q4" else 8 * rng.randint(32, 1024), rng.randint(256, 16384)
        m = _log(rng, 1, 4096)
        if k > 16384:
            m = max(m, 2)
        most = 20e9 if form == "f32" else 300e9
        return _case(kind, kind=form, m=max(2 if k > 16384 else 1, min(m, int(most / (2.0 * k * n)))), k=k, n=n)
    nq, nkv, hd = rng.choice([(8, 4, 256), (16, 16, 256), (16, 4, 128)])
    m, past = _log(rng, 2, 1500), rng.choice([0, _log(rng, 1, 8192)])
    return _case(kind, m=m, past=past, cap=m + past + rng.randint(0, 256), weights=rng.choice(["bf16", "bf16", "q4"]),
                 hidden=128 * rng.randint(8, 24), nq=nq, nkv=nkv, hd=hd, ffn=128 * rng.randint(16, 96))


def prepare(case, seed):
    state = {"decode_ops": _decode_ops_prepare, "decoder": _decoder_prepare, "attention": _attention_prepare,
             "matmul": _matmul_prepare, "layer": _layer_prepare}[case["work"]](case, seed)
    torch.cuda.synchronize()  # the inputs were made on torch's stream
    return state


def run(state):
    if "dec" in state:
        state["dec"].reset(state["token"], state["pos"])
        state["dec"].step(1)
    else:
        state["enc"].encode(state["kernels"])
    return state["out"]


def work(case):
    c = case
    if c["work"] == "decode_ops":
        e, h, kv = SIZE[c["dtype"]], c["nq"] * c["hd"], c["nkv"] * c["hd"]
        return {"bytes": e * (3 * h * c["ffn"] + 2 * kv * (c["pos"] + 3) + 4 * h),
                "flops": 6.0 * h * c["ffn"] + 4.0 * h * (c["pos"] + 1)}
    if c["work"] == "decoder":
        h, qw, kw = c["hidden"], c["nq"] * c["hd"], c["nkv"] * c["hd"]
        mats = [(qw + 2 * kw, h), (h, qw), (c["ffn"], h), (c["ffn"], h), (h, c["ffn"])]
        weights = c["layers"] * sum(_weight_bytes(c["weights"], n, k) for n, k in mats)
        weights += _weight_bytes(c["weights"], c["vocab"], h)
        params = c["layers"] * sum(n * k for n, k in mats) + c["vocab"] * h
        return {"bytes": weights + c["layers"] * 4 * kw * (c["pos"] + 2) + 4 * c["vocab"],
                "flops": 2.0 * params + 4.0 * c["layers"] * qw * (c["pos"] + 1)}
    if c["work"] == "attention":
        e = SIZE[c["dtype"]]
        return {"bytes": e * c["batch"] * c["hd"] * (2 * c["nq"] * c["sq"] + 2 * c["nkv"] * _keys_seen(c)),
                "flops": 4.0 * c["batch"] * c["nq"] * c["hd"] * _pairs_seen(c)}
    if c["work"] == "matmul":
        return {"bytes": SIZE[_act(c["kind"])] * c["m"] * (c["k"] + c["n"]) + _weight_bytes(c["kind"], c["n"], c["k"]),
                "flops": 2.0 * c["m"] * c["n"] * c["k"]}
    h, qw, kw, f, m = c["hidden"], c["nq"] * c["hd"], c["nkv"] * c["hd"], c["ffn"], c["m"]
    mats = [(qw, h), (kw, h), (kw, h), (h, qw), (f, h), (f, h), (h, f)]
    pairs = m * c["past"] + m * (m + 1) // 2
    return {"bytes": sum(_weight_bytes(c["weights"], n, k) for n, k in mats) + 4 * m * h + 4 * kw * (c["past"] + 2 * m),
            "flops": 2.0 * m * sum(n * k for n, k in mats) + 4.0 * qw * pairs}


def tolerance(case):
    c = case
    if c["work"] in ("decoder", "layer"):
        # a chain of 16-bit roundings: 26 layers of them, or one layer's
        return {"rel": 0.03 if c["work"] == "decoder" else 0.02, "max": 0.3}
    form = c.get("dtype") or c["kind"]
    if form == "f32":
        return {"rel": 1e-5, "max": 1e-4}
    if c["work"] == "decode_ops":  # four roundings on the way: 0.006 of the result in bf16
        return {"rel": 0.02, "max": 0.1} if form == "bf16" else {"rel": 0.0025, "max": 0.0125}
    # one rounding to 16 bits at the end: about 0.0017 of the result in bf16
    # and 0.00021 in f16; a value that rounds the other way is one unit in the
    # last place off
    return {"rel": 0.007, "max": 0.03} if form in ("bf16", "q4") else {"rel": 0.001, "max": 0.004}


def exact(case, seed):
    return {"decode_ops": _decode_ops_exact, "decoder": _decoder_exact, "attention": _attention_exact,
            "matmul": _matmul_exact, "layer": _layer_exact}[case["work"]](case, seed)
