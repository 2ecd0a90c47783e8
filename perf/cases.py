"""Performance cases of the compressed-KV GroupQueryAttention path.

Each case is one pass that a serving program makes through the package's
public entry points for one attention layer (or a short stack of layers):

* ``decode``: one generated token per sequence over the paged int8 or int4
  cache (``KvCache.decode_with_cache``: RoPE, quantise and append the token,
  attend over the whole context);
* ``prefill``: a chunk of new tokens per sequence, appended and then attended
  causally over the cached past (``KvCache.append`` + ``KvCache.prefill``): a
  whole prompt (past 0), a chunk of a long one, or the few tokens of a
  speculative verification over a long past;
* ``tq_decode``: one generated token per sequence over the TurboQuant cache
  (``TqCache.write_attend``);
* ``tq_prompt``: a prompt chunk into the TurboQuant cache: rotate its keys
  (``Runtime.rotary_embedding``), encode and store its rows
  (``TqCache.write``), and attend with the last position's query
  (``TqCache.attend``).

No pass advances the cache: the next pass writes the same slots, so that a
case's work stays the same however often it runs.
"""
import math

import numpy as np
import torch

import smallaios_amd as S

PAGE = S.PAGE_TOKENS
_runtime = None


def _rt():
    """The program's one runtime."""
    global _runtime
    if _runtime is None:
        _runtime = S.Runtime(0)
    return _runtime


# ---------------------------------------------------------------- the cases --
def _decode(name, batch, hq, hkv, d, lo, hi, quant="int8", dtype="bf16", out="f32",
            permuted=False, layers=1, window=0, theta=500000.0, outliers=False,
            interleaved=False):
    """lo..hi: tokens of a sequence's context, the step's own included."""
    return dict(name=name, path="decode", batch=batch, hq=hq, hkv=hkv, d=d, lo=lo, hi=hi,
                quant=quant, dtype=dtype, out=out, permuted=permuted, layers=layers,
                window=window, theta=theta, outliers=outliers, interleaved=interleaved)


def _prefill(name, batch, new, past, hq, hkv, d, quant="int8", dtype="bf16", out="f32",
             permuted=False, window=0, theta=500000.0, outliers=False, interleaved=False):
    return dict(name=name, path="prefill", batch=batch, new=new, past=past, hq=hq, hkv=hkv, d=d,
                quant=quant, dtype=dtype, out=out, permuted=permuted, window=window, theta=theta,
                outliers=outliers, interleaved=interleaved)


def _tq(name, path, batch, new, past, hq, hkv, d, bits=4, qjl=True, dtype="bf16"):
    return dict(name=name, path=path, batch=batch, new=new, past=past, hq=hq, hkv=hkv, d=d,
                bits=bits, qjl=qjl, dtype=dtype, theta=500000.0)


def listed():
    return [
        # an interactive session of a small model on f32 activations: one short
        # sequence, where the launch and the call are the cost
        _decode("decode_one_short", 1, 8, 2, 64, 512, 512, dtype="f32", theta=10000.0),
        # a few chats of ordinary length, bf16 out for the o_proj that follows
        _decode("decode_chats", 7, 32, 8, 128, 200, 1900, out="bf16", permuted=True),
        # a Llama-3-8B layer at batch 16 and 8k context
        _decode("decode_16x8k", 16, 32, 8, 128, 8192, 8192),
        # continuous batching of many unequal sequences, pages scattered
        _decode("decode_ragged_64", 64, 32, 8, 128, 128, 16384, permuted=True),
        # few sequences of long documents, keys with outlier channels
        _decode("decode_int4_32k", 4, 32, 8, 128, 32768, 32768, quant="int4", outliers=True),
        # a Gemma 3 4B stack: five sliding-window layers and one global layer
        _decode("decode_gemma_layers", 8, 8, 4, 256, 4001, 4001, out="bf16", layers=6,
                window=1024, theta=1000000.0),
        # a whole prompt into an empty cache
        _prefill("prefill_prompt", 1, 1000, 0, 32, 8, 128, out="bf16"),
        # a chunk of two long prompts
        _prefill("prefill_chunk", 2, 2048, 6144, 32, 8, 128),
        # a long prompt's chunk over the int4 cache
        _prefill("prefill_int4", 1, 1024, 3000, 32, 8, 128, quant="int4", outliers=True),
        # verification of a few drafted tokens per sequence over a long past
        _prefill("prefill_verify", 8, 5, 4000, 32, 8, 128, out="bf16", permuted=True),
        # the TurboQuant cache: a decode step, and a prompt going in
        _tq("tq_decode_16x8k", "tq_decode", 16, 1, 8191, 32, 8, 128),
        _tq("tq_prompt", "tq_prompt", 2, 1024, 0, 32, 8, 128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choices(["decode", "prefill", "tq_decode", "tq_prompt"], [5, 4, 2, 2])[0]
    hkv = rng.choice([1, 2, 4, 8, 8])
    d = rng.choice([64, 128, 128, 128, 256])
    group = rng.choice([1, 2, 4, 4, 8])
    if path.startswith("tq"):
        bits, qjl = rng.choice([3, 4, 4, 8]), rng.random() < 0.7
        hq = hkv * min(group, 4 if d == 256 else 8)
        dtype = rng.choice(["bf16", "f32"])
        if path == "tq_decode":
            batch, past = _log(rng, 1, 32), _log(rng, 63, 16383)
            while batch * past > 16 * 8191:
                batch = max(1, batch // 2)
            return _unnamed(_tq("", path, batch, 1, past, hq, hkv, d, bits, qjl, dtype))
        batch, new = _log(rng, 1, 8), _log(rng, 16, 2048)
        past = 0 if rng.random() < 0.5 else _log(rng, 16, 4096)
        return _unnamed(_tq("", path, batch, new, past, hq, hkv, d, bits, qjl, dtype))
    quant = rng.choice(["int8", "int8", "int4"])
    if quant == "int8" and rng.random() < 0.15:
        d = 168  # Gemma 4 31B's rows
    if quant == "int4" and d == 256:
        group = min(group, 4)
    more = dict(quant=quant, dtype=rng.choice(["bf16", "bf16", "f32"]),
                out=rng.choice(["bf16", "f32"]), permuted=rng.random() < 0.5,
                window=_log(rng, 64, 4096) if rng.random() < 0.2 else 0,
                outliers=rng.random() < 0.4, interleaved=rng.random() < 0.15)
    if path == "decode":
        batch, hi = _log(rng, 1, 64), _log(rng, 16, 32768)
        while batch * hi * hkv * d > 64 * 8192 * 8 * 128:
            batch = max(1, batch // 2)
        lo = hi if rng.random() < 0.4 else max(1, hi // rng.choice([2, 8, 100]))
        return _unnamed(_decode("", batch, hkv * group, hkv, d, lo, hi, **more))
    batch, new = _log(rng, 1, 16), _log(rng, 2, 2048)
    past = 0 if rng.random() < 0.35 else _log(rng, 16, 8192)
    c = _prefill("", batch, new, past, hkv * group, hkv, d, **more)
    while c["batch"] > 1 and work(c)["flops"] > 2.4e11:
        c["batch"] //= 2
    while work(c)["flops"] > 2.4e11:
        c["new"] = c["new"] // 2
    return _unnamed(c)


def _unnamed(c):
    return {k: v for k, v in c.items() if k != "name"}


def _lens(c):
    """Context lengths of a decode case (the step's token included)."""
    r = np.random.default_rng([c["batch"], c["lo"], c["hi"]])
    return r.integers(c["lo"], c["hi"] + 1, size=c["batch"]).astype(np.int64)


# ------------------------------------------------------------------- inputs --
_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def _gen(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 16 + stream)
    return g


def _randn(g, shape, dtype):
    return torch.randn(shape, generator=g, device="cuda").to(_DTYPES[dtype])


def _keys(g, c, n, dtype):
    """[batch, n, hkv*d] keys: N(0, 1), or Student t (3 degrees of freedom)
    with a few x20 channels, the outliers that keys of trained models show."""
    b, hkv, d = c["batch"], c["hkv"], c["d"]
    k = torch.randn((b, n, hkv, d), generator=g, device="cuda")
    if c.get("outliers"):
        chi = sum(torch.randn(k.shape, generator=g, device="cuda").square_() for _ in range(3))
        k = k / torch.sqrt(chi / 3)
        k[..., [7, d // 4 - 1, d // 2, d - 28]] *= 20.0
    return k.reshape(b, n, hkv * d).to(_DTYPES[dtype])


def _past_chunks(c, seed, layer, past):
    """The cached rows, as the chunks that earlier passes appended (bf16)."""
    g = _gen(seed, 3 + layer)
    step = max(1024, (131072 // (c["batch"] * c["hkv"])) // PAGE * PAGE)
    for t in range(0, past, step):
        n = min(step, past - t)
        yield _keys(g, c, n, "bf16"), _randn(g, (c["batch"], n, c["hkv"] * c["d"]), "bf16")


def _step_inputs(c, seed, layer, new):
    """(q, k, v) of the pass itself."""
    g = _gen(seed * 64 + layer, 1)
    q = _randn(g, (c["batch"], new, c["hq"] * c["d"]), c["dtype"])
    k = _keys(g, c, new, c["dtype"])
    v = _randn(g, (c["batch"], new, c["hkv"] * c["d"]), c["dtype"])
    return q, k, v


def _tables(c, rows):
    cos, sin = S.rope_tables(rows, c["d"], c["theta"])
    return torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda()


class _Pool:
    """A layer's pages as a tensor (the documented block layout); keeps the
    cache that owns the memory."""

    def __init__(self, cache, layer):
        self.cache = cache
        ptr, nbytes, _ = cache.pool(layer)
        self.__cuda_array_interface__ = dict(shape=(nbytes,), typestr="|u1", data=(ptr, False),
                                             version=2)

    def tensor(self):
        t = torch.as_tensor(self, device="cuda")
        t.owner = self  # an output outlives its state: the memory has to as well
        return t


def _layer_windows(c):
    """A stack's layers are sliding-window ones but for the last."""
    n = c.get("layers", 1)
    return [c["window"] if (n == 1 or i < n - 1) else 0 for i in range(n)]


def prepare(case, seed):
    if case["path"].startswith("tq"):
        return _prepare_tq(case, seed)
    c, rt = case, _rt()
    decode = c["path"] == "decode"
    b, new, layers = c["batch"], 1 if decode else c["new"], c.get("layers", 1)
    past = _lens(c) - 1 if decode else np.full(b, c["past"], dtype=np.int64)
    cap = int(past.max()) + new
    pages = (cap + PAGE - 1) // PAGE
    quant = S.KV_INT4 if c["quant"] == "int4" else S.KV_INT8
    cache = S.KvCache(rt, layers, c["hkv"], c["d"], b * pages, b, pages, quant)
    table = S.identity_page_table(b, pages)
    if c["permuted"]:
        table = np.random.default_rng(seed).permutation(table.ravel()).reshape(b, pages)
    cache.set_page_table(table.astype(np.int32))
    cos, sin = _tables(c, cap)
    windows = _layer_windows(c)
    feeds = [_past_chunks(c, seed, i, int(past.max())) for i in range(layers)]
    for rows in zip(*feeds):
        for i, (k, v) in enumerate(rows):
            cache.append(i, k, v, b, k.shape[1], cos, sin, cap, interleaved=c["interleaved"])
        cache.advance()
    cache.set_seq_lens(past.astype(np.int32))
    for i, w in enumerate(windows):
        cache.set_layer_window(i, w)
    inputs = [_step_inputs(c, seed, i, new) for i in range(layers)]
    outs = [torch.empty((b, new, c["hq"] * c["d"]), dtype=_DTYPES[c["out"]], device="cuda")
            for _ in range(layers)]
    pools = [_Pool(cache, i).tensor() for i in range(layers)]
    torch.cuda.synchronize()
    return dict(case=c, cache=cache, cos=cos, sin=sin, rows=cap, inputs=inputs, outs=outs,
                pools=pools)


def run(state):
    c = state["case"]
    if c["path"].startswith("tq"):
        return _run_tq(state)
    cache, cos, sin, rows = state["cache"], state["cos"], state["sin"], state["rows"]
    b, hq, il = c["batch"], c["hq"], c["interleaved"]
    for i, ((q, k, v), out) in enumerate(zip(state["inputs"], state["outs"])):
        if c["path"] == "decode":
            cache.decode_with_cache(i, q, k, v, out, b, hq, cos, sin, rows, interleaved=il)
        else:
            cache.append(i, k, v, b, c["new"], cos, sin, rows, interleaved=il)
            cache.prefill(i, q, out, b, c["new"], hq, cos, sin, rows, interleaved=il)
    return {"out": state["outs"], "cache": state["pools"]}


# --------------------------------------------------------------- TurboQuant --
_TQ_SEED = 42


def _prepare_tq(c, seed):
    rt = _rt()
    b, new, past = c["batch"], c["new"], c["past"]
    cache = S.TqCache(rt, 1, c["hkv"], c["d"], c["bits"], c["qjl"], b, past + new, _TQ_SEED)
    for k, v in _past_chunks(c, seed, 0, past):
        cache.write(0, k, v, b, k.shape[1])
        cache.advance()
    q, k, v = _step_inputs(c, seed, 0, new)
    cos, sin = _tables(c, past + new)
    out = torch.empty((b, 1, c["hq"] * c["d"]), device="cuda")
    q = q[:, -1:].contiguous()
    torch.cuda.synchronize()
    return dict(case=c, cache=cache, q=q, k=k, v=v, cos=cos, sin=sin, out=out,
                q_rot=torch.empty_like(q), k_rot=torch.empty_like(k))


def _run_tq(s):
    c, rt, cache = s["case"], _rt(), s["cache"]
    b, hq, hkv, d, new, past = c["batch"], c["hq"], c["hkv"], c["d"], c["new"], c["past"]
    if c["path"] == "tq_decode":
        # the step's q and k come rotated (this cache's entry points take no tables)
        cache.write_attend(0, s["q"], s["k"], s["v"], s["out"], b, hq)
        return {"out": s["out"]}
    rt.rotary_embedding(s["k"], s["k_rot"], b, hkv, new, d, s["cos"], s["sin"],
                        start_position=past, layout=S.ROPE_BSHD)
    rt.rotary_embedding(s["q"], s["q_rot"], b, hq, 1, d, s["cos"], s["sin"],
                        start_position=past + new - 1, layout=S.ROPE_BSHD)
    cache.write(0, s["k_rot"], s["v"], b, new)
    cache.attend(0, s["q_rot"], s["out"], b, hq)
    return {"out": s["out"], "k": s["k_rot"]}


# --------------------------------------------------------------------- work --
def _stored(d):
    return 192 if d == 168 else d


def _row_bytes(c):
    """Stored bytes of one (token, kv head): K and V."""
    d = _stored(c["d"])
    return d + d // 4 if c["quant"] == "int4" else 2 * d + 8


def _tq_bytes(c, read):
    """Bytes of a (row, kv head) of the TurboQuant cache: all that is stored,
    or what attention reads (V's residual and K's mean are not)."""
    d, q = c["d"], c["qjl"]
    n = 2 * d * c["bits"] // 8 + 16 + (d // 8 + 4 if q else 0)
    return n if read else n + (d // 8 + 4 if q else 0)


def work(case):
    c = case
    size = {"f32": 4, "bf16": 2}
    b, hq, hkv, d, e = c["batch"], c["hq"], c["hkv"], c["d"], size[c["dtype"]]
    if c["path"].startswith("tq"):
        new, past = c["new"], c["past"]
        io = b * hq * d * (e + 4) + b * new * hkv * d * 2 * e
        if c["path"] == "tq_prompt":
            io += 2 * b * hq * d * e + 2 * b * new * hkv * d * e + new * d * 4
        rows = b * hkv * (past + new)
        return {"bytes": float(io + rows * _tq_bytes(c, True) + b * new * hkv * _tq_bytes(c, False)),
                "flops": 4.0 * d * hq * b * (past + new)}
    new = 1 if c["path"] == "decode" else c["new"]
    pasts = _lens(c) - 1 if c["path"] == "decode" else np.full(b, c["past"], dtype=np.int64)
    byts = flops = 0.0
    for w in _layer_windows(c):
        for p in pasts:
            seen = np.arange(p + 1, p + new + 1, dtype=np.int64)
            first = 0
            if w:
                first = max(0, int(p) + 1 - w)
                seen = np.minimum(seen, w)
            flops += 4.0 * d * hq * float(seen.sum())
            byts += float(int(p) + new - first) * hkv * _row_bytes(c)
        byts += b * new * (hq * d * (e + size[c["out"]]) + hkv * (2 * d * e + _row_bytes(c)))
        byts += new * d * 4
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    """About four times the distance from exact() measured on an MI355X:
    bf16 outputs 1.7e-3; f32 outputs of decode up to 6.6e-5 (softmax weights
    of ~16 bits) and of prefill and the TurboQuant cache 2.1e-4 (binary16
    weights). The cache's bytes are the formats' own: the same."""
    if case.get("out") == "bf16":
        return {"rel": 7e-3, "max": 0.06}
    return {"rel": 3e-4 if case["path"] == "decode" else 1e-3, "max": 0.04}


# -------------------------------------------------------------------- exact --
def _rope(x, cos, sin, pos, interleaved):
    """x [.., n, h, d] rotated at positions pos [n] (products rounded one by
    one in x's own type)."""
    d = x.shape[-1]
    c, s = cos[pos].to(x.dtype)[:, None, :], sin[pos].to(x.dtype)[:, None, :]
    x0, x1 = (x[..., 0::2], x[..., 1::2]) if interleaved else (x[..., : d // 2], x[..., d // 2:])
    y0, y1 = c * x0 - s * x1, s * x0 + c * x1
    if interleaved:
        return torch.stack([y0, y1], dim=-1).reshape(x.shape)
    return torch.cat([y0, y1], dim=-1)


def _quantised(x, quant):
    """The cache's values of f32 rows x [.., d], dequantised, in 64 bits."""
    if quant == "int8":
        s = (x.abs().amax(-1, keepdim=True).double() / 127.0).float()
        s = torch.where(s == 0, torch.ones_like(s), s)
        q = torch.round((x.double() / s.double()).float()).clamp(-128, 127)
        return q.double() * s.double()
    g = x.reshape(*x.shape[:-1], x.shape[-1] // 32, 32)
    lo, hi = g.amin(-1, keepdim=True), g.amax(-1, keepdim=True)
    r = hi - lo
    s = torch.where(r > 0, (r.double() / 15.0).float(), torch.ones_like(r)).half().float()
    z = lo.half().float()
    t = ((g - z).double() / s.double()).float()
    q = torch.floor(t.double() + 0.5).clamp(0, 15)
    return (q.double() * s.double() + z.double()).reshape(x.shape)


def exact(case, seed):
    """The pass in 64 bits over the values that the cache stores (quantised by
    the formats' own 32-bit rules)."""
    c = case
    if c["path"].startswith("tq"):
        return _exact_tq(c, seed)
    b, hq, hkv, d, il = c["batch"], c["hq"], c["hkv"], c["d"], c["interleaved"]
    decode = c["path"] == "decode"
    new, layers = 1 if decode else c["new"], c.get("layers", 1)
    past = _lens(c) - 1 if decode else np.full(b, c["past"], dtype=np.int64)
    most = int(past.max())
    inv = (c["theta"] ** (-(2.0 * np.arange(d // 2, dtype=np.float64)) / d))[None, :]
    ang = np.arange(most + new, dtype=np.float64)[:, None] * inv
    cos = torch.from_numpy(np.cos(ang).astype(np.float32)).cuda()
    sin = torch.from_numpy(np.sin(ang).astype(np.float32)).cuda()
    outs = []
    for i, w in enumerate(_layer_windows(c)):
        ks, vs, t = [], [], 0
        for k, v in _past_chunks(c, seed, i, most):
            n = k.shape[1]
            pos = torch.arange(t, t + n, device="cuda")
            ks.append(_rope(k.float().view(b, n, hkv, d), cos, sin, pos, il))
            vs.append(v.float().view(b, n, hkv, d))
            t += n
        q, k, v = _step_inputs(c, seed, i, new)
        out = torch.empty((b, new, hq, d), dtype=torch.float64, device="cuda")
        k, v = k.float().view(b, new, hkv, d), v.float().view(b, new, hkv, d)
        q = q.double().view(b, new, hq, d)
        pk = torch.cat(ks, 1) if ks else k[:, :0]
        pv = torch.cat(vs, 1) if vs else v[:, :0]
        del ks, vs
        for bi in range(b):
            p = int(past[bi])
            pos = torch.arange(p, p + new, device="cuda")
            kk = _quantised(torch.cat([pk[bi, :p], _rope(k[bi], cos, sin, pos, il)]), c["quant"])
            vv = _quantised(torch.cat([pv[bi, :p], v[bi]]), c["quant"])
            qq = _rope(q[bi], cos, sin, pos, il) / math.sqrt(d)
            at = torch.arange(p + new, device="cuda")
            hide = at[None, :] > pos[:, None]
            if w:
                hide |= at[None, :] <= pos[:, None] - w
            for h in range(hq):
                kh = h // (hq // hkv)
                s = (qq[:, h] @ kk[:, kh].t()).masked_fill_(hide, -math.inf)
                out[bi, :, h] = torch.softmax(s, -1) @ vv[:, kh]
        outs.append(out.view(b, new, hq * d))
    return {"out": outs, "cache": [None] * layers}


def _tq_signs(c):
    """The rotation signs of each kv head of layer 0 (xorshift64)."""
    mask = (1 << 64) - 1
    rows = []
    for h in range(c["hkv"]):
        x = (_TQ_SEED * 0x9E3779B97F4A7C15 + h) & mask or 0x5EEDDEADBEEFCAFE
        row = []
        for _ in range(c["d"]):
            x ^= (x << 13) & mask
            x ^= x >> 7
            x ^= (x << 17) & mask
            row.append(1.0 if x & 1 == 0 else -1.0)
        rows.append(row)
    return torch.tensor(rows, device="cuda")


def _hadamard(x):
    """Normalised Walsh-Hadamard transform along the last axis, in x's type."""
    shape, n, h = x.shape, x.shape[-1], 1
    while h < n:
        y = x.reshape(-1, n // (2 * h), 2, h)
        x = torch.stack([y[:, :, 0] + y[:, :, 1], y[:, :, 0] - y[:, :, 1]], dim=2)
        h *= 2
    return (x * torch.tensor(1.0 / math.sqrt(n), dtype=x.dtype, device="cuda")).reshape(shape)


def _tq_rows(x, signs, bits, qjl):
    """(rotated values, residual signs, residual mean) of f32 rows x."""
    y = _hadamard(x * signs)
    lo, levels = y.amin(-1, keepdim=True), 2 ** bits - 1
    r = y.amax(-1, keepdim=True) - lo
    s = torch.where(r > 0, (r.double() / levels).float(), torch.ones_like(r))
    q = torch.floor(((y - lo).double() / s.double()).float().double() + 0.5).clamp(0, levels)
    rot = q.double() * s.double() + lo.double()
    if not qjl:
        return rot, None, None
    res = x - _hadamard(rot.float()) * signs
    return rot, torch.where(res >= 0, 1.0, -1.0).double(), res.double().abs().mean(-1)


def _exact_tq(c, seed):
    b, hq, hkv, d, past, new = c["batch"], c["hq"], c["hkv"], c["d"], c["past"], c["new"]
    rows = list(_past_chunks(c, seed, 0, past))
    q, k, v = _step_inputs(c, seed, 0, new)
    q = q[:, -1:].contiguous()
    got = {}
    if c["path"] == "tq_prompt":
        inv = (c["theta"] ** (-(2.0 * np.arange(d // 2, dtype=np.float64)) / d))[None, :]
        ang = np.arange(past + new, dtype=np.float64)[:, None] * inv
        cos = torch.from_numpy(np.cos(ang).astype(np.float32)).cuda()
        sin = torch.from_numpy(np.sin(ang).astype(np.float32)).cuda()
        pos = torch.arange(past, past + new, device="cuda")
        got["k"] = _rope(k.double().view(b, new, hkv, d), cos, sin, pos, False).view(k.shape)
        k = _rope(k.float().view(b, new, hkv, d), cos, sin, pos, False).view(k.shape).to(k.dtype)
        q = _rope(q.float().view(b, 1, hq, d), cos, sin, pos[-1:], False).view(q.shape).to(q.dtype)
    kk = torch.cat([r[0].float() for r in rows] + [k.float()], 1).view(b, past + new, hkv, d)
    vv = torch.cat([r[1].float() for r in rows] + [v.float()], 1).view(b, past + new, hkv, d)
    signs, g = _tq_signs(c), hq // hkv
    qq = q.float().view(b, hkv, g, d)
    out = torch.empty((b, hkv, g, d), dtype=torch.float64, device="cuda")
    for bi in range(b):
        for h in range(hkv):
            kr, ks, kc = _tq_rows(kk[bi, :, h], signs[h], c["bits"], c["qjl"])
            vr, _, _ = _tq_rows(vv[bi, :, h], signs[h], c["bits"], False)
            qr, qs, qc = _tq_rows(qq[bi, h], signs[h], c["bits"], c["qjl"])
            logit = qr @ kr.t()
            if c["qjl"]:
                logit += qc[:, None] * kc[None, :] * (qs @ ks.t()) / d
            p = torch.softmax(logit / math.sqrt(d), -1)
            out[bi, h] = _hadamard(p @ vr) * signs[h].double()
    got["out"] = out.view(b, 1, hq * d)
    return got
