"""The work whose speed is measured: calls of KV-cache attention as an engine
makes them, through the package's public entry points.

A case is one of six kinds:

  decode  one token of one or several sequences over resident caches
          (``Attention.prepare``'s call: ``janas_attn_run_dev``)
  block   a speculative verify or a block of up to 64 tokens; ``dropin``: through
          ``janas_attn_run`` (synchronous, an int8 cache in device memory)
  prompt  a prompt, or a chunk of a longer one (``janas_attn_run_dev``)
  layer   one attention layer of a prompt chunk from its projections on: query
          preparation, cache write, attention, Q8_K output for the next product
  step    the same for one token through several layers, captured once into a
          graph and replayed, as a serving loop does
  shift   a context shift of one layer's cache

Head shapes, cache types and lengths are the ones of the repository's benchmark
and tests (32 / 8 / 128, 16 / 2 / 256, 16 / 2 / 512 ...). All calls go to one
stream, as an engine's do: a layer's attention waits for the one before it.
"""
import math

import torch

import janas_amd as jm
from janas_amd import attention as at

DEV = "cuda:0"
KV = {"i8": jm.KV_I8, "i16": jm.KV_I16, "f16": jm.KV_F16, "f32": jm.KV_F32}
DTYPE = {"i8": torch.int8, "i16": torch.int16, "f16": torch.float16,
         "f32": torch.float32}
BYTES = {"i8": 1, "i16": 2, "f16": 2, "f32": 4}
TOP = {"i8": 127.0, "i16": 32767.0}
# head shapes (query heads, KV heads, head size)
HEADS = ((32, 8, 128), (32, 4, 128), (12, 4, 64), (16, 2, 256), (16, 4, 256))
WIDE = (16, 2, 512)
# products of the float-accurate kernels against the f16 kernel's: bounds the
# cost of a drawn case
PRODUCTS = {"f16": 1, "i8": 2, "i16": 4}
MOST_FLOPS = 5.5e11
MOST_BYTES = 1.2e9


def _case(kind, h, n_kv, hd, kv, **more):
    c = dict(kind=kind, h=h, n_kv=n_kv, hd=hd, kv=kv, scores="float", window=0,
             gate=False, seqs=1, layers=1, n=1, pos0=0, q8k=False,
             dropin=False, drop=0, keep=0, even=True)
    c.update(more)
    return c


def listed():
    return [
        # the smallest call: one token at 1k positions over an f32 cache, two
        # short launches
        _case("decode", 32, 8, 128, "f32", pos0=1023, name="decode-1k-f32"),
        # a long-context decode of a gated layer with large heads
        _case("decode", 16, 2, 256, "f16", pos0=32767, gate=True,
              name="decode-32k-gated-f16"),
        # a serving step: 8 users at unlike lengths in one call
        _case("decode", 32, 8, 128, "f16", pos0=8191, seqs=8, even=False,
              name="decode-ragged8-f16"),
        # the widest heads (512) over a 16-bit integer cache
        _case("decode", *WIDE, "i16", pos0=32767, name="decode-32k-hd512-i16"),
        # speculative decoding: 8 drafts checked at 8k
        _case("block", 32, 8, 128, "f16", n=8, pos0=8192, name="verify8-8k-f16"),
        # the engine's own prefill: blocks of 64 through the drop-in call
        _case("block", 32, 8, 128, "i8", n=64, pos0=4096, dropin=True,
              name="block64-4k-i8-dropin"),
        # a short prompt at once
        _case("prompt", 32, 8, 128, "f16", n=1024, name="prompt-1k-f16"),
        # a long prompt at once: the largest
        _case("prompt", 32, 8, 128, "f16", n=8192, name="prompt-8k-f16"),
        # a sliding-window layer's prompt over a 16-bit integer cache, ragged
        _case("prompt", 16, 2, 256, "i16", n=3001, window=1024,
              name="prompt-3k-window-i16"),
        # one layer of a chunked prefill over the engine's int8 cache
        _case("layer", 32, 8, 128, "i8", n=512, pos0=3584, q8k=True,
              name="layer-512-at-3k5-i8"),
        # a decode step's attention layers in a graph, 20k context, the INT16
        # way that the engine takes past 16384 positions
        _case("step", 32, 8, 128, "i8", pos0=20000, layers=4, scores="int16",
              q8k=True, name="step-20k-i8-int16"),
        # the context is full: half of it is dropped, the rest moves down
        _case("shift", 32, 8, 128, "i8", pos0=32768, keep=64, drop=16352,
              name="shift-32k-i8"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        if w["bytes"] <= MOST_BYTES and \
                w["flops"] * PRODUCTS.get(c["kv"], 1) <= MOST_FLOPS:
            return c


def _draw(rng):
    kind = rng.choice(("decode", "decode", "block", "block", "prompt", "prompt",
                       "layer", "step", "shift"))
    h, n_kv, hd = rng.choice(HEADS)
    if kind == "decode":
        kv = rng.choice(("f16", "f16", "i8", "i16", "f32"))
        if kv in ("f16", "i16", "i8") and rng.random() < 0.2:
            h, n_kv, hd = WIDE
        if kv == "f32" and hd > 128:
            kv = "f16"
        return _case("decode", h, n_kv, hd, kv, pos0=_log(rng, 40, 65000),
                     seqs=rng.choice((1, 1, 2, 3, 8)), even=rng.random() < 0.3,
                     gate=rng.random() < 0.4,
                     scores=rng.choice(("float", "int16")) if kv == "i8" else "float",
                     window=rng.choice((0, 0, 0, 1024)))
    if kind == "block":
        kv = rng.choice(("f16", "i8", "i8", "i16"))
        return _case("block", h, n_kv, hd, kv, n=rng.randint(2, 64),
                     pos0=_log(rng, 10, 16000), dropin=kv == "i8",
                     scores=rng.choice(("float", "int16")) if kv == "i8" else "float")
    if kind == "prompt":
        kv = rng.choice(("f16", "f16", "i8", "i16"))
        return _case("prompt", h, n_kv, hd, kv, n=_log(rng, 65, 8192),
                     pos0=rng.choice((0, 0, 256, _log(rng, 100, 8192))),
                     window=rng.choice((0, 0, 0, 1024)), gate=rng.random() < 0.3)
    if kind == "layer":
        return _case("layer", h, n_kv, hd, rng.choice(("i8", "i8", "i16", "f16")),
                     n=_log(rng, 70, 2048),
                     pos0=rng.choice((0, 512, _log(rng, 100, 8192))), q8k=True)
    if kind == "step":
        kv = rng.choice(("i8", "i8", "i16", "f16"))
        return _case("step", h, n_kv, hd, kv, pos0=_log(rng, 100, 30000),
                     layers=rng.randint(2, 4), q8k=True,
                     scores=rng.choice(("float", "int16")) if kv == "i8" else "float")
    n_pos = _log(rng, 1000, 40000)
    keep = rng.choice((0, 4, 64))
    return _case("shift", h, n_kv, hd, rng.choice(("i8", "i8", "i16")),
                 pos0=n_pos, keep=keep, drop=(n_pos - keep) // rng.choice((2, 2, 4)))


def _lengths(c):
    """Positions before the call of each sequence (seqs of them)."""
    if c["even"] or c["seqs"] == 1:
        return [c["pos0"]] * c["seqs"]
    # spread over [1/16, 1] of the longest, in no order
    p = c["pos0"]
    return [max(1, p // 16 + (p - p // 16) * ((i * 5 + 7) % 8) // 7)
            for i in range(c["seqs"])]


def _pairs(c, pos0):
    """Visible (token, position) pairs of a sequence, and the positions that
    any of its tokens sees."""
    n, w = c["n"], c["window"]
    if not w:
        return n * pos0 + n * (n + 1) // 2, pos0 + n
    lo = max(0, pos0 + 1 - w)
    pairs = sum(min(w, pos0 + j + 1) for j in range(n))
    return pairs, pos0 + n - lo


def work(c):
    h, n_kv, hd, n = c["h"], c["n_kv"], c["hd"], c["n"]
    eb, sc = BYTES[c["kv"]], 4 if c["kv"] in TOP else 0
    row = 2 * n_kv * (hd * eb + sc)          # a position's keys and values
    if c["kind"] == "shift":
        moved = c["pos0"] - c["keep"] - c["drop"]
        return {"bytes": 2.0 * moved * row, "flops": 6.0 * moved * n_kv * hd}
    total, flops = 0.0, 0.0
    for p in _lengths(c):
        pairs, seen = _pairs(c, p)
        flops += 4.0 * hd * h * pairs
        total += seen * row + 2 * 4 * n * h * hd
        if c["gate"]:
            total += 4 * n * h * hd
        if c["q8k"]:
            total += n * h * hd // 256 * at.Q8K_BYTES
        if c["kind"] in ("layer", "step"):
            # the projections read, the prepared query written, the new rows
            # written
            total += 2 * 4 * n * h * hd + 2 * 4 * n * n_kv * hd + n * row
    return {"bytes": total * c["layers"], "flops": flops * c["layers"]}


def tolerance(c):
    if c["kind"] == "shift":
        # the moved rows' bits are the engine's arithmetic
        return "exact"
    if c["scores"] == "int16":
        # quantized scores and weights: ties of their rounding
        return {"rel": 2e-5, "max": 2e-3, "differ": 5e-3}
    if c["kind"] in ("prompt", "layer") and (c["kv"] == "f16" or c["hd"] > 256):
        # f16 query and weights
        return {"rel": 2e-3, "max": 5e-2, "differ": 1e-2}
    # float-accurate; whole values: Q8_K numbers at a tie
    return {"rel": 5e-6, "max": 2e-4, "differ": 5e-3}


# ---- inputs ---------------------------------------------------------------

_streams = []


def _stream():
    """The program's stream."""
    if not _streams:
        _streams.append(torch.cuda.Stream())
    return _streams[0]


def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFF)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _quant(x, kv):
    """Rows at 8 or 16 bits with a scale each, as the cache write makes them."""
    top = TOP[kv]
    mx = x.abs().amax(-1)
    inv = torch.where(mx > 0, top / mx, torch.zeros_like(mx))
    return torch.round(x * inv[..., None]).to(DTYPE[kv]), mx / top


def _cache(c, seed, salt, cap):
    """A resident cache of cap rows: k, v (n_kv, cap, hd), ks, vs or None."""
    res = []
    for i in range(2):
        x = _randn(_gen(seed, salt + i), c["n_kv"], cap, c["hd"])
        if c["kv"] in TOP:
            res += list(_quant(x, c["kv"]))
        else:
            res += [x.to(DTYPE[c["kv"]]), None]
        del x
    return dict(k=res[0], ks=res[1], v=res[2], vs=res[3])


def _query(c, seed, salt):
    """Query rows, some heads sharper than others."""
    h = c["h"]
    sharp = 1.0 + torch.arange(h, device=DEV) % 4 * 0.5
    return _randn(_gen(seed, salt), c["n"], h, c["hd"]) * sharp[None, :, None]


def _tables(c, first, n):
    """The rotation of positions first .. first + n - 1, as the engine makes
    them (base 1e6)."""
    half = c["hd"] // 2
    f = 1e6 ** (-torch.arange(half, dtype=torch.float64, device=DEV) / half)
    a = torch.arange(first, first + n, dtype=torch.float64, device=DEV)[:, None] * f
    return a.cos().float().contiguous(), a.sin().float().contiguous()


def _projections(c, seed, salt):
    """What a layer's q, k, v products leave, and the norms' weights."""
    n, h, n_kv, hd = c["n"], c["h"], c["n_kv"], c["hd"]
    x = lambda i, *shape: _randn(_gen(seed, salt + i), *shape)
    return dict(q=2.0 * x(0, n, h, hd), k=1.5 * x(1, n, n_kv, hd),
                v=x(2, n, n_kv, hd), qn=1.0 + 0.2 * x(3, hd),
                kn=1.0 + 0.2 * x(4, hd))


def _q8k(c):
    return torch.zeros(c["n"], c["h"] * c["hd"] // 256, at.Q8K_BYTES,
                       dtype=torch.uint8, device=DEV)


def _q8k_fields(b):
    """The blocks' fields (struct janas_attn_q8k), as views."""
    f = lambda lo, hi, t: b[..., lo:hi].view(t)
    return [f(0, 4, torch.float32), f(4, 260, torch.int8),
            f(260, 292, torch.int16), f(292, 324, torch.float32),
            f(324, 580, torch.int8), f(580, 612, torch.int16),
            f(612, 628, torch.int16)]


def _instance(c, cap):
    a = jm.Attention(c["h"], c["n_kv"], c["hd"], cap, 1,
                     jm.INT16 if c["scores"] == "int16" else jm.FLOAT)
    if c["window"]:
        a.set_window(c["window"])
    return a


def _layer(c, seed, salt):
    """One layer's buffers, from its projections to its Q8_K output."""
    s = dict(cache=_cache(c, seed, salt, c["pos0"] + c["n"]),
             **_projections(c, seed, salt + 2))
    s["qr"], s["out"] = torch.empty_like(s["q"]), torch.empty_like(s["q"])
    s["q8k"] = _q8k(c)
    s["cs"], s["sn"] = _tables(c, c["pos0"], c["n"])
    return s


def _layer_calls(c, a, s, stream, path):
    """The layer's calls on a stream, as a function."""
    kc = s["cache"]
    n, hd = c["n"], c["hd"]
    cache = at.cache(kc["k"], kc["v"], kc["ks"], kc["vs"], kv_type=KV[c["kv"]])
    attend = a.prepare(KV[c["kv"]], [dict(
        kc, q=s["qr"], out=s["out"], out_q8k=s["q8k"], cap=c["pos0"] + n, n=n,
        pos0=c["pos0"])], stream=stream, path=path)

    def calls():
        # (the product that would leave the query in its buffer)
        torch.mul(s["q"], 1.0, out=s["qr"])
        at.q_prep(s["qr"], cs=s["cs"], sn=s["sn"], n_rot=hd, q_norm=s["qn"],
                  stream=stream)
        at.cache_write(cache, s["k"], s["v"], cs=s["cs"], sn=s["sn"], n_rot=hd,
                       pos0=c["pos0"], k_norm=s["kn"], stream=stream)
        attend()
    return calls


def _layer_outputs(s):
    kc = s["cache"]
    return [s["qr"], s["out"], _q8k_fields(s["q8k"])] + \
        [kc[x] for x in ("k", "v", "ks", "vs") if kc[x] is not None]


def _visible(c):
    """A decode's or prompt's sequences: (positions before, salt)."""
    return [(p, 100 + 10 * i) for i, p in enumerate(_lengths(c))]


def prepare(case, seed):
    c = case
    if c["kind"] == "shift":
        kc = _cache(c, seed, 1, c["pos0"])
        half = c["hd"] // 2
        f = 1e6 ** (-torch.arange(half, dtype=torch.float64, device=DEV) / half)
        ang = c["drop"] * f
        return dict(case=c, kc=kc, cs=ang.cos().float(), sn=ang.sin().float(),
                    cache=at.cache(kc["k"], kc["v"], kc["ks"], kc["vs"],
                                   kv_type=KV[c["kv"]]))
    if c["kind"] in ("layer", "step"):
        layers = [_layer(c, seed, 100 * (i + 1)) for i in range(c["layers"])]
        a = _instance(c, c["pos0"] + c["n"])
        st = dict(case=c, a=a, layers=layers, outputs=[_layer_outputs(s) for s in layers])
        torch.cuda.synchronize()
        if c["kind"] == "layer":
            st["calls"] = [_layer_calls(c, a, s, _stream().cuda_stream, "auto")
                           for s in layers]
            return st
        # the step's launches recorded once; capture needs the entry point
        # that allocates nothing
        with torch.cuda.stream(_stream()):
            _layer_calls(c, a, layers[0], _stream().cuda_stream, "noalloc")()
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            stream = torch.cuda.current_stream().cuda_stream
            for s in layers:
                _layer_calls(c, a, s, stream, "noalloc")()
        return st
    seqs = []
    for p, salt in _visible(c):
        q = _query(c, seed, salt + 2)
        gate = _randn(_gen(seed, salt + 3), *q.shape) if c["gate"] else None
        seqs.append(dict(_cache(c, seed, salt, p + c["n"]), q=q,
                         out=torch.empty_like(q), gate=gate, cap=p + c["n"],
                         n=c["n"], pos0=p))
    a = _instance(c, max(s["cap"] for s in seqs))
    st = dict(case=c, a=a, seqs=seqs, outputs=[s["out"] for s in seqs])
    if not c["dropin"]:
        st["call"] = a.prepare(KV[c["kv"]], seqs,
                               jm.GATE_ELEM if c["gate"] else jm.GATE_NONE,
                               stream=_stream().cuda_stream)
    torch.cuda.synchronize()
    return st


def run(state):
    c = state["case"]
    if c["kind"] == "shift":
        at.cache_shift(state["cache"], keep=c["keep"], drop=c["drop"],
                       n_pos=c["pos0"], cs=state["cs"], sn=state["sn"],
                       n_rot=c["hd"])
        kc = state["kc"]
        return [kc["k"], kc["v"], kc["ks"], kc["vs"]]
    if c["kind"] == "step":
        with torch.cuda.stream(_stream()):
            state["graph"].replay()
    elif c["kind"] == "layer":
        with torch.cuda.stream(_stream()):
            for calls in state["calls"]:
                calls()
    elif c["dropin"]:
        s = state["seqs"][0]
        state["a"].run(s["q"], s["k"], s["ks"], s["v"], s["vs"], s["n"],
                       s["pos0"], s["out"])
    else:
        state["call"]()
    return state["outputs"]


# ---- the same in 64 bits --------------------------------------------------

def _rows(kc, which, scale):
    x = kc[which].double()
    return x if kc[scale] is None else x * kc[scale].double()[..., None]


def _attend(c, q, k, v, pos0):
    """Attention of the rows of q (n, h, hd) over k, v (n_kv, cap, hd)."""
    n, h, hd = q.shape
    g, out = h // c["n_kv"], torch.empty_like(q)
    p = torch.arange(pos0 + n, device=DEV)
    last = torch.arange(pos0, pos0 + n, device=DEV)[:, None]
    unseen = p[None] > last
    if c["window"]:
        unseen |= p[None] + c["window"] <= last
    scale = float(torch.tensor(hd, dtype=torch.float32).rsqrt())
    for i in range(h):
        s = q[:, i].contiguous() @ k[i // g, :pos0 + n].t().contiguous()
        s.mul_(scale).masked_fill_(unseen, -math.inf)
        out[:, i] = torch.softmax(s, -1) @ v[i // g, :pos0 + n]
        del s
    return out


def _turn(x, cs, sn):
    half = x.shape[-1] // 2
    a, b = x[..., :half], x[..., half:]
    cs, sn = cs.double()[:, None], sn.double()[:, None]
    return torch.cat((a * cs - b * sn, a * sn + b * cs), -1)


def _norm(x, w):
    x = x.double()
    return x / (x.square().mean(-1, keepdim=True) + 1e-6).sqrt() * w.double()


def _exact_layer(c, s):
    kc, n = s["cache"], c["n"]
    q = _turn(_norm(s["q"], s["qn"]), s["cs"], s["sn"])
    new = (_turn(_norm(s["k"], s["kn"]), s["cs"], s["sn"]), s["v"].double())
    for x, name, z in zip(new, ("k", "v"), ("ks", "vs")):
        x = x.transpose(0, 1)
        if c["kv"] in TOP:
            x, kc[z][:, c["pos0"]:] = _quant(x.float(), c["kv"])
        kc[name][:, c["pos0"]:] = x.to(DTYPE[c["kv"]])
    out = _attend(c, q, _rows(kc, "k", "ks"), _rows(kc, "v", "vs"), c["pos0"])
    # the Q8_K scales follow the output; the cache's scales are compared too
    b = out.reshape(n, -1, 256)
    d = b.abs().amax(-1, keepdim=True) / 127
    d32 = b.reshape(n, -1, 8, 32).abs().amax(-1) / 127
    scales = [kc[x].double() for x in ("ks", "vs") if kc[x] is not None]
    return [q, out, [d, None, None, d32, None, None, None], None, None] + scales


def exact(case, seed):
    c = case
    if c["kind"] == "shift":
        kc = _cache(c, seed, 1, c["pos0"])
        return [None, None, None, _shifted(c, kc["vs"])]
    if c["kind"] in ("layer", "step"):
        return [_exact_layer(c, _layer(c, seed, 100 * (i + 1)))
                for i in range(c["layers"])]
    res = []
    for p, salt in _visible(c):
        kc = _cache(c, seed, salt, p + c["n"])
        o = _attend(c, _query(c, seed, salt + 2).double(), _rows(kc, "k", "ks"),
                    _rows(kc, "v", "vs"), p)
        if c["gate"]:
            o *= torch.sigmoid(_randn(_gen(seed, salt + 3), *o.shape).double())
        res.append(o)
    return res


def _shifted(c, rows):
    """Rows of a cache after the shift, where they move as they are."""
    x = rows.double().clone()
    x[:, c["keep"]:c["pos0"] - c["drop"]] = rows[:, c["keep"] + c["drop"]:].double()
    return x
