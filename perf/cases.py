"""Workloads of the decode path, as a program that uses the framework calls them.

Every case is a dict of plain values.  ``prepare`` makes what such a program holds (context, weights, pages, prompts),
``run`` is one pass through the public entry points, ``exact`` the same outputs in plain 64-bit torch.

Kinds and what they stand for:

* ``step``    one decode step of a resident decoder over cached contexts, one token per sequence: a chat of one user
              (batch 1) up to a full serving batch.  ``llama`` is the W8A8 stack, ``zoferax`` a bf16 layered decoder with
              sparse experts.  The pass takes the step back first (``rewind``), as speculative decoding does.
* ``prompt``  ingestion of prompts into a decoder: one short request, several that join together (ragged lengths), long ones.
* ``turn``    a short dialogue turn on a decoder with recurrent states (``nugelix``): a prompt, then token by token.
* ``linear``  a linear by itself, in each quantized arithmetic: int8 weights with bf16 activations, int8 x int8 with activations
              quantized per token and a bias, e4m3.
* ``attend``  paged decode attention by itself, block tables on the host.

The sizes are those of the repository's own benchmark stacks: "large" is width 4096 with 32 / 8 heads, "small" 2048 with 16 / 4.
"""
import math

import numpy as np
import torch

import fandhe_ai_amd as fa

PAGE = 16
VOCAB = 32000
DIM = 128                                                   # per head
SIZES = {"large": dict(d=4096, heads=32, kv=8, ff=14336, q_rank=1536, window=2048),
         "small": dict(d=2048, heads=16, kv=4, ff=8192, q_rank=768, window=1024)}
EXPERTS, TOP = 16, 4
EXPERT_SIZES = {"large": dict(ff=5376, vdim=128), "small": dict(ff=3072, vdim=64)}
EPS, THETA, SOFTCAP = 1e-5, 500000.0, 30.0
# the W8A8 stacks are the first layers of a model of 32: projections into the residual stream are scaled by its 64 sublayers.
# (Without that, int8 codes that fall either way make two correct implementations drift apart by a tenth.)
INTO_RESIDUAL = 0.02 / 64
KV_RANK, ROT, ROT_BASE, CONV, GLU_LIMIT, GLU_ALPHA = 512, 64, 1e6, 4, 7.0, 1.702


def listed():
    return [
        # one user's chat on the W8A8 stack: the weights of one token, launches and their gaps
        dict(name="step_one", kind="step", model="llama", size="large", layers=8, batch=1, low=700, high=700),
        # a serving batch with long contexts: the repository's headline workload, at a quarter of its depth
        dict(name="step_batch", kind="step", model="llama", size="large", layers=8, batch=32, low=1024, high=8192),
        # one request's prompt, of an ordinary odd length
        dict(name="prompt_one", kind="prompt", model="llama", size="large", layers=8, batch=1, low=300, high=300, cached=0),
        # long prompts together: the largest case
        dict(name="prompt_long", kind="prompt", model="llama", size="large", layers=8, batch=4, low=2048, high=2048, cached=0),
        # requests that join a running batch: lengths differ
        dict(name="prompt_ragged", kind="prompt", model="llama", size="small", layers=8, batch=5, low=64, high=509, cached=0),
        # a few users' dialogue turns on a decoder with recurrent states
        dict(name="turn_nugelix", kind="turn", model="nugelix", size="small", layers=8, batch=4, prompt=48, steps=16),
        # a document into the recurrent and latent-attention layers
        dict(name="prompt_nugelix", kind="prompt", model="nugelix", size="large", layers=4, batch=1, low=2048, high=2048, cached=0),
        # a serving batch on sparse experts
        dict(name="step_zoferax", kind="step", model="zoferax", size="small", layers=4, batch=32, low=500, high=2000),
        # prompts through sparse experts
        dict(name="prompt_zoferax", kind="prompt", model="zoferax", size="small", layers=4, batch=3, low=700, high=700, cached=0),
        # the attention operator of a serving batch, scattered pages
        dict(name="attend_batch", kind="attend", heads=32, kv=8, batch=64, low=128, high=4096, pages=40000),
        # the smallest call: one row through one projection
        dict(name="linear_row", kind="linear", op="w8a16", m=1, k=4096, n=4096),
        # the fp8 GEMM of a prompt's feed-forward
        dict(name="linear_prompt", kind="linear", op="e4m3", m=2048, k=4096, n=14336),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _lens_drawn(rng, batch, low, high, total):
    """Bounds of the sequences' lengths, both log-uniform, with about `total` tokens at most."""
    a, b = sorted((_log(rng, low, high), _log(rng, low, high)))
    b = max(low, min(b, 2 * total // batch - a)) if (a + b) * batch > 2 * total else b
    return min(a, b), max(low, b)


def draw(rng):
    kind = rng.choice(["step", "step", "prompt", "prompt", "turn", "linear", "attend"])
    size = rng.choice(["large", "small"])
    if kind == "step":
        model = rng.choice(["llama", "llama", "zoferax"])
        if model == "zoferax":
            size = "small"
        batch = _log(rng, 1, 64 if model == "llama" else 32)
        low, high = _lens_drawn(rng, batch, 100, 8192 if model == "llama" else 2500, 150000 if model == "llama" else 40000)
        return dict(kind=kind, model=model, size=size, layers=rng.randint(2, 8 if model == "llama" else 4), batch=batch, low=low, high=high)
    if kind == "prompt":
        model = rng.choice(["llama", "llama", "nugelix", "zoferax"])
        if model == "zoferax":
            size = "small"
        batch = _log(rng, 1, 8)
        most = 8192 // batch if model == "llama" else 4096 // batch
        if model == "llama" and rng.random() < 0.4:                # ragged: at most 4096 rows with their padding
            low, high = sorted((_log(rng, 16, 4096 // batch), _log(rng, 16, 4096 // batch)))
        else:
            low = high = _log(rng, 33, min(most, 2048))
        cached = rng.choice([0, 0, _log(rng, 50, 4000)]) if model == "llama" else 0
        return dict(kind=kind, model=model, size=size, layers={"llama": rng.randint(2, 8), "nugelix": 4, "zoferax": rng.randint(2, 4)}[model],
                    batch=batch, low=low, high=high, cached=cached)
    if kind == "turn":
        return dict(kind=kind, model="nugelix", size=size, layers=4 if size == "large" else rng.choice([4, 8]), batch=_log(rng, 1, 32),
                    prompt=_log(rng, 8, 256), steps=rng.randint(4, 16))
    if kind == "linear":
        op = rng.choice(["w8a16", "w8a8", "e4m3"])
        m = _log(rng, 1, 32) if op == "w8a16" else _log(rng, 1, 2048) if op == "w8a8" else _log(rng, 65, 2048)
        return dict(kind=kind, op=op, m=m, k=128 * _log(rng, 8, 112), n=_log(rng, 1024, 28672))
    heads, kv = rng.choice([(32, 8), (16, 4), (40, 8), (16, 16)])
    batch = _log(rng, 1, 64)
    low, high = _lens_drawn(rng, batch, 17, 8192, 140000)
    return dict(kind=kind, heads=heads, kv=kv, batch=batch, low=low, high=high, pages=sum(-(-n // PAGE) for n in _spread(batch, low, high)) + rng.randint(1, 9000))


# ------------------------------------------------------------------------------------------------ shared pieces

def _spread(batch, low, high):
    """Lengths of the sequences: evenly from low to high, in a fixed mixed order."""
    n = [low + (high - low) * i // max(1, batch - 1) for i in range(batch)]
    return [n[i] for i in np.random.RandomState(batch).permutation(batch)]


def _gen(seed, part):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1009 + part)
    return g


def _randn(g, *shape, std=1.0, mean=0.0, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(mean, std, generator=g)


_TYPES = {fa.capi.F32: ("<f4", torch.float32), fa.capi.BF16: ("<i2", torch.bfloat16), fa.capi.I8: ("<i1", torch.int8),
          fa.capi.E4M3: ("|u1", torch.uint8), fa.capi.I32: ("<i4", torch.int32), fa.capi.U32: ("<i4", torch.int32)}


class _Span:
    """A framework buffer as torch sees device memory; keeps the owner alive."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (ptr, False), "version": 2}


def _tensor(owner, shape=None, handle=None, dtype=None):
    """The torch tensor over a framework buffer (or over the raw handle of one that `owner` keeps); no copy."""
    typestr, kind = _TYPES[owner.dtype if dtype is None else dtype]
    ptr = fa.capi.lib.fa_buffer_device_ptr(owner._h if handle is None else handle)
    t = torch.as_tensor(_Span(owner, ptr, owner.shape if shape is None else shape, typestr), device="cuda")
    return t.view(kind) if t.dtype != kind else t


_ops = None


def _backend():
    global _ops
    if _ops is None:
        torch.zeros(1, device="cuda")
        _ops = fa.tape_for(fa.Device.Rocm(0))
    return _ops


def _buffer(be, t):
    """A torch tensor's values in a buffer of the framework."""
    kind = {torch.float32: fa.capi.F32, torch.bfloat16: fa.capi.BF16}[t.dtype]
    b = be.alloc_uninit(tuple(t.shape), kind)
    _tensor(b).copy_(t)
    torch.cuda.synchronize()
    return b


class _State:
    """What a pass works on."""

    def __init__(self, **more):
        self.__dict__.update(more)


class _Held:
    """Closes a decoder with the last thing that refers to it: the state, or an output that lies in the decoder's memory."""

    def __init__(self, dec):
        self.dec = dec

    def __del__(self):
        self.dec.close()


def _tables(seed, need, columns):
    """Block tables of sequences that need so many pages each, from a shuffled pool, and the pool's size."""
    total = sum(need)
    perm = np.random.RandomState(seed % (1 << 31)).permutation(total + 8).astype(np.uint32)
    t, p = np.full((len(need), columns), 0xFFFFFFFF, dtype=np.uint32), 0
    for b, n in enumerate(need):
        t[b, :n] = perm[p:p + n]
        p += n
    return t, total + 8


def _tokens(case, seed):
    """Context (where it is computed and not made up) and new tokens of every sequence."""
    rng = np.random.RandomState((seed * 7 + 3) % (1 << 31))
    if case["kind"] == "turn":
        return [rng.randint(0, VOCAB, case["prompt"] + case["steps"]).astype(np.int32) for _ in range(case["batch"])]
    more = 1 if case["kind"] == "step" and case["model"] != "llama" else 0
    if case["kind"] == "step" and case["model"] == "llama":
        return [rng.randint(0, VOCAB, 1).astype(np.int32) for _ in range(case["batch"])]
    return [rng.randint(0, VOCAB, n + more).astype(np.int32) for n in _spread(case["batch"], case["low"], case["high"])]


def _cached(case):
    """Tokens of every sequence that are cached before a pass."""
    if case["kind"] == "step":
        return _spread(case["batch"], case["low"], case["high"])
    return [case.get("cached", 0)] * case["batch"]


def _new(case):
    """Tokens of every sequence that a pass adds."""
    if case["kind"] == "step":
        return [1] * case["batch"]
    if case["kind"] == "turn":
        return [case["prompt"] + case["steps"]] * case["batch"]
    return _spread(case["batch"], case["low"], case["high"])


def _pages(case, seed):
    room = max(_new(case))                                  # a padded pass needs its places in the table's row
    need = [-(-(c + n) // PAGE) for c, n in zip(_cached(case), _new(case))]
    columns = -(-(max(_cached(case)) + room) // PAGE)
    t, total = _tables(seed, need, columns)
    return t, columns, total


# ------------------------------------------------------------------------------------------------ the W8A8 stack

def _llama_head(case, seed):
    s, g = SIZES[case["size"]], _gen(seed, 0)
    return dict(embed=_randn(g, VOCAB, s["d"]), norm=_randn(g, s["d"], std=0.1, mean=1.0), head=_randn(g, s["d"], VOCAB, std=0.02))


def _llama_layer(case, seed, i):
    s, g = SIZES[case["size"]], _gen(seed, 1 + i)
    eq, ekv = s["heads"] * DIM, s["kv"] * DIM
    return dict(attn_norm=_randn(g, s["d"], std=0.1, mean=1.0), ffn_norm=_randn(g, s["d"], std=0.1, mean=1.0),
                qkv=_randn(g, s["d"], eq + 2 * ekv, std=0.02), o=_randn(g, eq, s["d"], std=INTO_RESIDUAL),
                gu=_randn(g, s["d"], 2 * s["ff"], std=0.02), down=_randn(g, s["ff"], s["d"], std=INTO_RESIDUAL))


def _llama_pools(case, seed, i, blocks):
    g = _gen(seed, 500 + i)
    return [_randn(g, blocks, PAGE, SIZES[case["size"]]["kv"] * DIM, dtype=torch.bfloat16) for _ in range(2)]


def _llama(be, case, seed):
    s = SIZES[case["size"]]
    tables, columns, blocks = _pages(case, seed)
    dec = fa.Decoder(be, case["layers"], s["d"], s["heads"], s["kv"], s["ff"], VOCAB, columns, blocks, case["batch"],
                     head_dim=DIM, block_size=PAGE, rms_eps=EPS, rope_theta=THETA)
    held = _Held(dec)
    be.synchronize_device()                                 # the pools are cleared on the framework's stream, filled on torch's
    scratch = be.alloc_uninit((s["d"] * max(2 * s["ff"], VOCAB),))

    def quantized(w):
        _tensor(scratch)[:w.numel()].copy_(w.reshape(-1))
        torch.cuda.synchronize()
        q = be.quantize_weight(fa.DeviceBufferView(scratch, 0, tuple(w.shape)))
        be.synchronize_device()
        return q

    outputs = []
    for i in range(case["layers"]):
        w = _llama_layer(case, seed, i)
        dec.set_layer(i, _buffer(be, w["attn_norm"]), _buffer(be, w["ffn_norm"]), *[quantized(w[n]) for n in ("qkv", "o", "gu", "down")])
        kp, vp = fa.capi.buf_p(), fa.capi.buf_p()
        fa.check(fa.capi.lib.fa_decoder_kv_pools(dec._h, i, kp, vp))
        for h, values in zip((kp, vp), _llama_pools(case, seed, i, blocks)):
            t = _tensor(held, values.shape, handle=h, dtype=fa.capi.BF16)
            t.copy_(values)
            outputs.append(t)
    w = _llama_head(case, seed)
    dec.set_head(_buffer(be, w["embed"]), _buffer(be, w["norm"]), quantized(w["head"]))
    torch.cuda.synchronize()
    scratch.free()
    # padding of ragged prompts leaves rows behind that mean nothing: the pools are outputs where there is none
    return held, tables, outputs if len(set(_new(case))) == 1 else []


def _codes(x, dim, top=127.0):
    scale = x.abs().amax(dim, keepdim=True) / top
    return torch.round(x / torch.where(scale > 0, scale, 1.0)), scale


def _w8a8(x, w):
    xq, sx = _codes(x, -1)
    wq, sw = _codes(w.double(), 0)
    return (xq @ wq) * sx * sw


def _rms(x, w, eps=EPS):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _angles(positions, dims, base):
    f = torch.tensor(float(base), dtype=torch.float64, device="cuda") ** (-torch.arange(0, dims, 2, dtype=torch.float64, device="cuda") / dims)
    return positions.double()[:, None] * f


def _rotate(x, a):
    """Rotate-half of x [T, heads, dims] by the angles a [T, dims / 2]."""
    h = x.shape[-1] // 2
    u, v, c, s = x[..., :h], x[..., h:], torch.cos(a)[:, None], torch.sin(a)[:, None]
    return torch.cat([u * c - v * s, v * c + u * s], -1)


def _attention(q, k, v, scale, first, window=None):
    """q [T, H, d] at positions first .., k [S, G, d], v [S, G, dv] from position 0 on; one head group after another."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    out = torch.empty(T, H, v.shape[2], dtype=torch.float64, device="cuda")
    at, of = torch.arange(first, first + T, device="cuda")[:, None], torch.arange(k.shape[0], device="cuda")[None]
    seen = (of <= at) if window is None else (of <= at) & (at - of < window)
    for h in range(H):
        s = (q[:, h] @ k[:, h // (H // G)].T.contiguous()) * scale
        out[:, h] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ v[:, h // (H // G)]
    return out


def _llama_exact(case, seed):
    s = SIZES[case["size"]]
    H, G = s["heads"], s["kv"]
    tables, _, blocks = _pages(case, seed)
    new, cached, tokens = _new(case), _cached(case), _tokens(case, seed)
    w = _llama_head(case, seed)
    x = w["embed"].double()[torch.from_numpy(np.concatenate(tokens)).long().cuda()]
    starts = np.concatenate([[0], np.cumsum(new)])
    places = [torch.from_numpy(tables[b].astype(np.int64)).cuda() for b in range(len(new))]
    pools = []
    for i in range(case["layers"]):
        l = _llama_layer(case, seed, i)
        kp, vp = (p.double().reshape(blocks * PAGE, G, DIM) for p in _llama_pools(case, seed, i, blocks))
        y = _w8a8(_rms(x, l["attn_norm"].double()), l["qkv"])
        q, k, v = (y[:, a:b].reshape(len(x), -1, DIM) for a, b in ((0, H * DIM), (H * DIM, (H + G) * DIM), ((H + G) * DIM, (H + 2 * G) * DIM)))
        o = torch.empty(len(x), H, DIM, dtype=torch.float64, device="cuda")
        for b, (c, n) in enumerate(zip(cached, new)):
            rows = slice(starts[b], starts[b] + n)
            p = torch.arange(c + n, device="cuda")
            a = _angles(p[c:], DIM, THETA)
            slots = places[b][p // PAGE] * PAGE + p % PAGE
            kp[slots[c:]], vp[slots[c:]] = _rotate(k[rows], a), v[rows]
            o[rows] = _attention(_rotate(q[rows], a), kp[slots], vp[slots], DIM ** -0.5, c)
        x = x + _w8a8(o.reshape(len(x), -1), l["o"])
        gate, up = _w8a8(_rms(x, l["ffn_norm"].double()), l["gu"]).split(s["ff"], -1)
        x = x + _w8a8(gate * torch.sigmoid(gate) * up, l["down"])
        if len(set(new)) == 1:
            pools += [p.reshape(blocks, PAGE, G * DIM) for p in (kp, vp)]
    last = torch.from_numpy(starts[1:] - 1).cuda()
    return [_w8a8(_rms(x[last], w["norm"].double()), w["head"])] + pools


# ------------------------------------------------------------------------------------------------ layered decoders

def _config(case):
    s, n = SIZES[case["size"]], case["layers"]
    if case["model"] == "nugelix":
        latent = {"type": "latent_attention", "mlp": {"kind": "dense", "ff": s["ff"], "limit": GLU_LIMIT},
                  "mixer": {"heads": s["heads"], "dim": DIM, "rot_dim": ROT, "vdim": DIM, "q_rank": s["q_rank"], "kv_rank": KV_RANK,
                            "mask": {"size": s["window"]}, "rot": {"base": ROT_BASE, "dims": ROT}, "scale": (DIM + ROT) ** -0.5}}
        delta = {"type": "delta", "mlp": None, "mixer": {"heads": s["heads"], "kv_heads": s["heads"] // 2, "dim": DIM, "vdim": DIM, "conv": CONV}}
        return {"architecture": "Nugelix", "width": s["d"], "vocab": VOCAB, "norm": {"eps": EPS}, "logit_softcap": SOFTCAP,
                "layers": ([latent, delta, delta, delta] * -(-n // 4))[:n]}
    e = EXPERT_SIZES[case["size"]]
    layer = {"type": "attention", "mixer": {"heads": s["heads"], "kv_heads": s["kv"], "dim": DIM, "vdim": e["vdim"], "scale": DIM ** -0.5},
             "mlp": {"kind": "moe", "expert": {"ff": e["ff"]}, "router": {"experts": EXPERTS, "top": TOP}}}
    return {"architecture": "Zoferax", "width": s["d"], "vocab": VOCAB, "norm": {"eps": EPS}, "embedding": {"scale": s["d"] ** 0.5}, "layers": [layer] * n}


def _shapes(config):
    """Names and shapes of a checkpoint's tensors."""
    D = config["width"]
    out = {"embed": (VOCAB, D), "head": (VOCAB, D), "final.norm": (D,)}
    for i, l in enumerate(config["layers"]):
        p, m, x = "l%d." % i, "l%d.mix." % i, l["mixer"]
        H, wide = x["heads"], x["heads"] * x["vdim"]
        out.update({p + "norm1": (D,), m + "o": (D, wide)})
        if l["type"] == "attention":
            q, k, v = H * DIM, x["kv_heads"] * DIM, x["kv_heads"] * x["vdim"]
            out.update({m + "q": (q, D), m + "q.b": (q,), m + "q.norm": (q,), m + "k": (k, D), m + "k.b": (k,), m + "k.norm": (k,), m + "v": (v, D), m + "v.b": (v,)})
        elif l["type"] == "delta":
            nq = x["kv_heads"] * DIM
            out.update({p + "ls1": (D,), m + "g": (wide, D), m + "b": (H, D), m + "a": (H, D), m + "A_log": (H,), m + "dt_bias": (H,), m + "norm": (DIM,)})
            for n, rows in (("q", nq), ("k", nq), ("v", wide)):
                out.update({m + n: (rows, D), m + n + ".conv": (rows, CONV)})
        else:
            out.update({p + "ls1": (D,), m + "g": (H, D), m + "dq": (x["q_rank"], D), m + "dq.norm": (x["q_rank"],), m + "uq": (H * (DIM + ROT), x["q_rank"]),
                        m + "dkv": (KV_RANK + ROT, D), m + "dkv.norm": (KV_RANK,), m + "uk": (H * DIM, KV_RANK), m + "uv": (wide, KV_RANK)})
        f = p + "mlp."
        if l["mlp"] and l["mlp"]["kind"] == "moe":
            ff = l["mlp"]["expert"]["ff"]
            out.update({p + "norm2": (D,), f + "router": (EXPERTS, D)})
            out.update({f + "e%d.%s" % (e, n): s for e in range(EXPERTS) for n, s in (("up", (ff, D)), ("down", (D, ff)))})
        elif l["mlp"]:
            ff = l["mlp"]["ff"]
            out.update({p + "norm2": (D,), p + "ls2": (D,), f + "gate": (ff, D), f + "up": (ff, D), f + "down": (D, ff)})
    return out


def _weights(config, seed):
    """(name, bf16 tensor) of a checkpoint, in a fixed order."""
    g = _gen(seed, 0)
    for name, shape in sorted(_shapes(config).items()):
        leaf = name.split(".")[-1]
        if leaf in ("A_log", "dt_bias"):
            yield name, _randn(g, *shape, std=0.5, mean=-1.0).bfloat16()
        elif "norm" in leaf or leaf in ("ls1", "ls2"):
            yield name, _randn(g, *shape, std=0.1, mean=1.0).bfloat16()
        else:
            yield name, _randn(g, *shape, std=1.0 if leaf == "embed" else 0.1 if len(shape) == 1 else shape[1] ** -0.5).bfloat16()


def _layered(be, case, seed):
    config = _config(case)
    tables, columns, blocks = _pages(case, seed)
    dec = fa.models.build_layered(be, config, "bfloat16", fa.models.Capacity(blocks * PAGE, case["batch"]))
    for name, t in _weights(config, seed):
        dec.set_tensor(name, t.view(torch.int16).cpu().numpy().view(np.uint16), bf16=True)
    held = _Held(dec)
    full = np.full((case["batch"], dec.cfg.max_blocks_per_seq), 0xFFFFFFFF, dtype=np.uint32)
    full[:, :columns] = tables
    return held, full


def _zoferax_row(config, w, tokens):
    """Logits after the last of one sequence's tokens."""
    D, T = config["width"], len(tokens)
    f = torch.arange(D, device="cuda", dtype=torch.float64)
    a = torch.arange(T, device="cuda", dtype=torch.float64)[:, None] * 10000.0 ** (-(f - f % 2) / D)
    x = w["embed"][torch.from_numpy(tokens).long().cuda()].double() * config["embedding"]["scale"] + torch.where(f % 2 == 1, torch.cos(a), torch.sin(a))
    for i, l in enumerate(config["layers"]):
        p, m, mx, last = "l%d." % i, "l%d.mix." % i, l["mixer"], i == len(config["layers"]) - 1
        k, v = (x @ w[m + n].double().T + w[m + n + ".b"].double() for n in "kv")
        k = _rms(k, w[m + "k.norm"].double())
        x = x[-1:] if last else x                           # the last layer is read at one token only
        q = _rms(x @ w[m + "q"].double().T + w[m + "q.b"].double(), w[m + "q.norm"].double())
        o = _attention(q.reshape(len(x), -1, DIM), k.reshape(T, -1, DIM), v.reshape(T, -1, mx["vdim"]), mx["scale"], T - len(x))
        x = x + _rms(o.reshape(len(x), -1) @ w[m + "o"].double().T, w[p + "norm1"].double())
        best, at = torch.topk(x @ w[p + "mlp.router"].double().T, TOP, -1)
        share, y = torch.softmax(best, -1), torch.zeros_like(x)
        for e in range(EXPERTS):
            rows, place = torch.nonzero(at == e, as_tuple=True)
            if len(rows):
                h = torch.relu(x[rows] @ w[p + "mlp.e%d.up" % e].double().T) ** 2
                y[rows] += share[rows, place, None] * (h @ w[p + "mlp.e%d.down" % e].double().T)
        x = x + _rms(y, w[p + "norm2"].double())
    return _rms(x[-1], w["final.norm"].double()) @ w["head"].double().T


def _layer_norm(x, w):
    c = x - x.mean(-1, keepdim=True)
    return c / torch.sqrt((c * c).mean(-1, keepdim=True) + EPS) * w.double()


def _delta(h, w, m, mx):
    """The gated delta rule over h [B, T, D]: the state decays, takes the write, is read."""
    B, T, H, G = h.shape[0], h.shape[1], mx["heads"], mx["kv_heads"]

    def taps(n):
        y = h @ w[m + n].double().T
        y = torch.cat([torch.zeros(B, CONV - 1, y.shape[2], dtype=y.dtype, device="cuda"), y], 1)
        return torch.nn.functional.silu(sum(y[:, i:i + T] * w[m + n + ".conv"][:, i].double() for i in range(CONV))).reshape(B, T, -1, DIM)

    q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (taps("q"), taps("k")))
    q, k = q.repeat_interleave(H // G, 2) * DIM ** -0.5, k.repeat_interleave(H // G, 2)
    v, beta = taps("v"), torch.sigmoid(h @ w[m + "b"].double().T)
    decay = torch.exp(-torch.exp(w[m + "A_log"].double()) * torch.nn.functional.softplus(h @ w[m + "a"].double().T + w[m + "dt_bias"].double()))
    S, out = torch.zeros(B, H, DIM, DIM, dtype=torch.float64, device="cuda"), torch.empty_like(v)
    for t in range(T):
        S = S * decay[:, t, :, None, None]
        u = beta[:, t, :, None] * (v[:, t] - (S * k[:, t, :, :, None]).sum(2))
        S = S + k[:, t, :, :, None] * u[:, :, None]
        out[:, t] = (S * q[:, t, :, :, None]).sum(2)
    o = _rms(out, w[m + "norm"].double()) * torch.nn.functional.silu(h @ w[m + "g"].double().T).reshape(out.shape)
    return o.reshape(B, T, -1) @ w[m + "o"].double().T


def _latent(h, w, m, mx):
    """Latent attention over h [B, T, D]."""
    B, T, H = h.shape[0], h.shape[1], mx["heads"]
    a = _angles(torch.arange(T, device="cuda"), ROT, ROT_BASE)
    q = (_rms(h @ w[m + "dq"].double().T, w[m + "dq.norm"].double()) @ w[m + "uq"].double().T).reshape(B, T, H, DIM + ROT)
    y = h @ w[m + "dkv"].double().T
    c = _rms(y[..., :KV_RANK], w[m + "dkv.norm"].double())
    k, v = ((c @ w[m + n].double().T).reshape(B, T, H, -1) for n in ("uk", "uv"))
    o = []
    for b in range(B):
        shared = _rotate(y[b, :, None, KV_RANK:], a).expand(T, H, ROT)
        turned = torch.cat([q[b, ..., :DIM], _rotate(q[b, ..., DIM:], a)], -1)
        o.append(_attention(turned, torch.cat([k[b], shared], -1), v[b], mx["scale"], 0, mx["mask"]["size"]))
    o = torch.stack(o) * torch.sigmoid(h @ w[m + "g"].double().T)[..., None]
    return o.reshape(B, T, -1) @ w[m + "o"].double().T


def _nugelix_rows(config, w, tokens):
    """Logits [B, T, vocab] are large: those of the places asked for are formed by the caller from the normed rows."""
    x = w["embed"][torch.from_numpy(tokens).long().cuda()].double()
    for i, l in enumerate(config["layers"]):
        p, m = "l%d." % i, "l%d.mix." % i
        y = (_delta if l["type"] == "delta" else _latent)(_layer_norm(x, w[p + "norm1"]), w, m, l["mixer"])
        x = x + y * w[p + "ls1"].double()
        if l["mlp"]:
            h, f = _layer_norm(x, w[p + "norm2"]), p + "mlp."
            g = (h @ w[f + "gate"].double().T).clamp(max=GLU_LIMIT)
            u = (h @ w[f + "up"].double().T).clamp(-GLU_LIMIT, GLU_LIMIT)
            x = x + ((g * torch.sigmoid(GLU_ALPHA * g) * (u + 1.0)) @ w[f + "down"].double().T) * w[p + "ls2"].double()
    return _layer_norm(x, w["final.norm"])


def _layered_exact(case, seed):
    config, tokens = _config(case), _tokens(case, seed)
    w = dict(_weights(config, seed))
    if case["model"] == "zoferax":
        return [torch.stack([_zoferax_row(config, w, t) for t in tokens])]
    rows = _nugelix_rows(config, w, np.stack(tokens))
    return [SOFTCAP * torch.tanh(rows[:, -1] @ w["head"].double().T / SOFTCAP)]


# ------------------------------------------------------------------------------------------------ operators

def _linear_parts(case, seed):
    g = _gen(seed, 1)
    m, k, n = case["m"], case["k"], case["n"]
    return (_randn(g, m, k, dtype=torch.bfloat16 if case["op"] == "w8a16" else torch.float32), _randn(g, k, n, std=0.02), _randn(g, n, std=0.1))


def _e4m3(x):
    scale = x.abs().max() / 448.0
    return (x / scale).to(torch.float8_e4m3fn).double(), scale.double()


def _linear_exact(case, seed):
    x, w, bias = _linear_parts(case, seed)
    if case["op"] == "w8a8":
        return _w8a8(x.double(), w) + bias.double()
    if case["op"] == "w8a16":
        wq, sw = _codes(w.double(), 0)
        return (x.double() @ wq) * sw
    (xq, sx), (wq, sw) = _e4m3(x), _e4m3(w)
    return (xq @ wq) * (sx * sw)


def _attend_parts(case, seed):
    g = _gen(seed, 1)
    lens = _spread(case["batch"], case["low"], case["high"])
    need = [-(-n // PAGE) for n in lens]
    perm = np.random.RandomState(seed % (1 << 31)).permutation(case["pages"]).astype(np.uint32)
    tables, p = np.full((len(lens), max(need)), 0xFFFFFFFF, dtype=np.uint32), 0
    for b, n in enumerate(need):
        tables[b, :n] = perm[p:p + n]
        p += n
    q = _randn(g, case["batch"], 1, case["heads"] * DIM, dtype=torch.bfloat16)
    pools = [_randn(g, case["pages"], PAGE, case["kv"] * DIM, dtype=torch.bfloat16) for _ in range(2)]
    return q, pools, tables, np.array(lens, dtype=np.uint32)


def _attend_exact(case, seed):
    q, pools, tables, lens = _attend_parts(case, seed)
    out = []
    for b, n in enumerate(lens):
        p = torch.arange(int(n), device="cuda")
        slots = torch.from_numpy(tables[b].astype(np.int64)).cuda()[p // PAGE] * PAGE + p % PAGE
        k, v = (t.reshape(-1, case["kv"], DIM)[slots].double() for t in pools)
        out.append(_attention(q[b].double().reshape(1, case["heads"], DIM), k, v, fa.default_scale(DIM), int(n) - 1).reshape(1, -1))
    return torch.stack(out)


# ------------------------------------------------------------------------------------------------ the entry points

def prepare(case, seed):
    be = _backend()
    if case["kind"] == "linear":
        x, w, bias = _linear_parts(case, seed)
        dw = _buffer(be, w)
        kind = fa.capi.QW_E4M3_TENSOR if case["op"] == "e4m3" else fa.capi.QW_INT8_CHANNEL
        qw = be.quantize_weight(fa.DeviceBufferView(dw, 0, (case["k"], case["n"])), kind)
        x = _buffer(be, x)
        state = _State(case=case, be=be, x=be.quantize_tensor_e4m3(x) if case["op"] == "e4m3" else x, qw=qw,
                       bias=fa.DeviceBufferView(_buffer(be, bias), 0, (case["n"],)))
        be.synchronize_device()
        return state
    if case["kind"] == "attend":
        q, pools, tables, lens = _attend_parts(case, seed)
        layout = fa.PagedKvLayout.new(case["pages"], PAGE, case["kv"] * DIM)
        args = fa.PagedAttentionArgs(layout, case["batch"], 1, case["heads"], tables.shape[1], fa.default_scale(DIM), case["kv"])
        return _State(case=case, be=be, q=_buffer(be, q), pools=[_buffer(be, p) for p in pools], tables=tables, lens=lens, args=args)
    tokens, cached = _tokens(case, seed), np.array(_cached(case), dtype=np.uint32)
    pools = []
    if case["model"] == "llama":
        held, tables, pools = _llama(be, case, seed)
    else:
        held, tables = _layered(be, case, seed)
    dec = held.dec
    state = _State(case=case, be=be, held=held, tables=tables, cached=cached, outputs=pools)
    state.logits = _tensor(held, (case["batch"], VOCAB), handle=dec.logits_buffer(), dtype=fa.capi.F32)
    if case["kind"] == "step":
        state.tokens = np.array([t[-1] for t in tokens], dtype=np.int32)
        if case["model"] == "llama":
            dec.set_sequences(tables, cached)
        else:                                               # contexts of the decoder's own making
            dec.set_sequences(tables, np.zeros_like(cached))
            for at in range(0, int(cached.max()), 128):
                dec.forward([t[at:min(at + 128, c)].tolist() for t, c in zip(tokens, cached.tolist())])
    elif case["kind"] == "turn":
        state.prompt = np.stack([t[:case["prompt"]] for t in tokens])
        state.tokens = np.stack([t[case["prompt"]:] for t in tokens], 1)
    elif case["low"] == case["high"]:
        state.prompt = np.stack(tokens)
    else:
        state.prompt = tokens
    be.synchronize_device()
    return state


def run(state):
    case, be = state.case, state.be
    if case["kind"] == "linear":
        if case["op"] == "w8a8":
            return _tensor(be.linear_w8a8(state.x, state.qw, state.bias))
        if case["op"] == "w8a16":
            return _tensor(be.linear_w8a16(state.x, state.qw))
        return _tensor(be.gemm_e4m3(state.x[0], state.x[1], state.qw))
    if case["kind"] == "attend":
        return _tensor(be.paged_attention_forward(state.q, state.pools[0], state.pools[1], state.tables, state.lens, state.args))
    dec = state.held.dec
    if case["kind"] == "step":
        dec.rewind(state.cached)
        dec.set_tokens(state.tokens)
        dec.step()
    else:
        dec.set_sequences(state.tables, state.cached)
        if case["kind"] == "turn":
            dec.prefill(state.prompt)
            for t in state.tokens:                          # the user's program chooses each token
                dec.set_tokens(t)
                dec.step()
        elif case["low"] == case["high"]:
            dec.prefill(state.prompt)
        else:
            dec.prefill_padded(state.prompt)
    return [state.logits] + state.outputs


def exact(case, seed):
    if case["kind"] == "linear":
        return _linear_exact(case, seed)
    if case["kind"] == "attend":
        return _attend_exact(case, seed)
    return _llama_exact(case, seed) if case["model"] == "llama" else _layered_exact(case, seed)


def work(case):
    if case["kind"] == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        x = {"w8a8": 4, "w8a16": 2, "e4m3": 1}[case["op"]]
        return {"bytes": k * n + x * m * k + (4 if case["op"] == "w8a8" else 2) * m * n, "flops": 2 * m * n * k}
    if case["kind"] == "attend":
        seen = sum(_spread(case["batch"], case["low"], case["high"]))
        return {"bytes": seen * 2 * case["kv"] * DIM * 2 + 4 * case["batch"] * case["heads"] * DIM, "flops": 4 * seen * case["heads"] * DIM}
    s, new, cached = SIZES[case["size"]], _new(case), _cached(case)
    rows = sum(new)
    # scores: every new token sees what is cached, the new ones before it and itself
    pairs = sum(n * c + n * (n + 1) // 2 for c, n in zip(cached, new))
    if case["model"] == "llama":
        layer = s["d"] * (2 * s["heads"] + 2 * s["kv"]) * DIM + 3 * s["d"] * s["ff"]
        kv = (sum(new) + sum(cached)) * 2 * s["kv"] * DIM * 2
        return {"bytes": case["layers"] * (layer + kv) + s["d"] * VOCAB + 4 * case["batch"] * VOCAB,
                "flops": case["layers"] * (2 * layer * rows + 4 * pairs * s["heads"] * DIM) + 2 * case["batch"] * s["d"] * VOCAB}
    config = _config(case)
    sizes = {n: int(np.prod(z)) for n, z in _shapes(config).items() if n != "embed"}
    passes = 1 + case["steps"] if case["kind"] == "turn" else 1            # tokens that follow one another read the weights again
    head, body = sizes["head"], sum(sizes.values()) - sizes["head"]
    flops = 2 * head * case["batch"] * passes
    if case["model"] == "zoferax":
        e = EXPERT_SIZES[case["size"]]
        experts = sum(v for n, v in sizes.items() if ".mlp.e" in n)
        read = min(1.0, rows * TOP / EXPERTS)                              # of the experts, at the least
        kv = case["layers"] * (sum(new) + sum(cached)) * s["kv"] * (DIM + e["vdim"]) * 2
        return {"bytes": 2 * (body - experts + read * experts + head) + kv + 4 * case["batch"] * VOCAB,
                "flops": flops + 2 * rows * (body - experts + experts * TOP / EXPERTS) + 2 * case["layers"] * pairs * s["heads"] * (DIM + e["vdim"])}
    latents = sum(l["type"] != "delta" for l in config["layers"])
    state = case["batch"] * s["heads"] * DIM * DIM * 4 * (case["layers"] - latents)
    return {"bytes": passes * (2 * (body + head) + 2 * state) + 4 * case["batch"] * VOCAB,
            "flops": flops + 2 * rows * body + 2 * latents * min(pairs, rows * s["window"]) * s["heads"] * (2 * DIM + ROT)
            + (case["layers"] - latents) * rows * s["heads"] * 8 * DIM * DIM}


def tolerance(case):
    """About four times what another order of the f32 sums gives (measured with the other forms of the attention kernels)."""
    if case["kind"] == "linear" and case["op"] == "w8a8":
        return {"rel": 1e-5}                                # int32 sums; the scales are applied in f32
    if case["kind"] in ("linear", "attend"):
        return {"rel": 0.004, "max": 0.08}                  # one rounding to bf16
    # logits of 0.0017 .. 0.007 (W8A8: activations near a rounding edge get another code), 0.0045 and 0.002 of their r.m.s.
    return {"llama": {"rel": 0.028, "max": 0.19}, "nugelix": {"rel": 0.018, "max": 0.08}, "zoferax": {"rel": 0.008, "max": 0.05}}[case["model"]]
