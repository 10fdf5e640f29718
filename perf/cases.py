"""The work that a program has this library do, as timed cases over the C ABI.

Seven kinds, each through the entry points that a serving program calls:

  product   y = x W^T over a Q8_0 matrix: the repacked form that the model streams, or the
            model file's own layout (aotx_q8r_gemv / aotx_q8_gemv, fp32 or fp16 out)
  attend    paged attention over the page table: decode rows and prompt pieces
  pick      one token per row of logits, greedy or sampled
  experts   a routed feed-forward block: the router, then the grouped expert products
  model     whole passes of a decoder: a prompt chunk and / or decode steps over a seated cache
  text      the tokenizer: text to ids, or ids back to text

Matrix sizes are those of the 8B shape (4096 wide, 32 / 8 heads x 128, FFN 14336, vocabulary
128256), of the routed 8-expert shape and of the 4-layer test shape, with ragged sizes drawn
around them. Inputs come from the seed alone: Q8_0 weights of N(0, 0.02), activations, keys and
values of N(0, 1) in fp16. The library holds one page pool, one open model and one vocabulary
at a time; `_world` keeps the one that the current case needs, as a program does between calls,
and the states of a case share it.
"""
import ctypes
import math
import random
import zlib

import numpy as np
import torch

import aotx_amd as A
from aotx_amd.model import LLAMA_8B, TINY, Runtime, Shape, build_device, layout_pages
from aotx_amd.text import Tokenizer

# head norms and split rotary pairs: the layer kind that runs rotary turns in a kernel of its own
QK_NORM = Shape(layers=8, hidden=2048, ffn=6144, heads=16, kv_heads=8, head_dim=128, vocab=32000,
                qk_norm=True, pairs=A.AOTX_ROPE_PAIRS_SPLIT, theta=1e6)
SHAPES = {"8b": LLAMA_8B, "tiny": TINY, "qk_norm": QK_NORM}
EXPERTS = {"mixtral": (4096, 14336, 8, 2), "fine": (2048, 1024, 32, 4), "small": (1024, 2048, 16, 2)}
HEADS = {"8b": (32, 8, 128), "tiny": (4, 4, 64), "mqa": (16, 2, 64)}
KV_LAYERS = 6            # layers of the attention cases' pages: each state fills one of its own


def listed():
    return [
        # one token of one agent through a square attention matrix: launch and latency
        {"name": "product_1x4096x4096", "kind": "product", "m": 1, "n": 4096, "k": 4096, "file": False, "half": False},
        # all 64 slots of the runtime in one step through a gate or up matrix
        {"name": "product_64x14336x4096", "kind": "product", "m": 64, "n": 14336, "k": 4096, "file": False, "half": True},
        # a whole prompt chunk through a gate or up matrix
        {"name": "product_512x14336x4096", "kind": "product", "m": 512, "n": 14336, "k": 4096, "file": False, "half": False},
        # eight agents' down product over weights left as the model file has them
        {"name": "product_file_8x4096x14336", "kind": "product", "m": 8, "n": 4096, "k": 14336, "file": True, "half": False},
        # 32 agents whose conversations differ in length, one new token each
        {"name": "attend_ragged_32", "kind": "attend", "heads": "8b", "seqs": 32, "lo": 512, "hi": 8192, "piece": 1},
        # one agent far into a long conversation
        {"name": "attend_one_8000", "kind": "attend", "heads": "8b", "seqs": 1, "lo": 8000, "hi": 8000, "piece": 1},
        # a chunk of a long prompt: 512 new tokens after 2000 cached ones
        {"name": "attend_prompt_512", "kind": "attend", "heads": "8b", "seqs": 1, "lo": 2512, "hi": 2512, "piece": 512},
        # sampled tokens of 32 agents: top-k 40, top-p 0.9, temperature 0.8
        {"name": "pick_sampled_32", "kind": "pick", "rows": 32, "vocab": 128256, "top_k": 40, "top_p": 0.9, "temperature": 0.8},
        # one routed layer of the 8-expert shape, a token from each slot
        {"name": "experts_64", "kind": "experts", "shape": "mixtral", "tokens": 64},
        # decode steps of 32 agents at 2048 cached tokens each, the whole 8B model
        {"name": "decode_32x2048", "kind": "model", "shape": "8b", "slots": 32, "context": 2048, "prompt": 0, "steps": 4},
        # one agent's request to the whole 8B model: a 500-token prompt, then eight tokens
        {"name": "chat_500", "kind": "model", "shape": "8b", "slots": 1, "context": 0, "prompt": 500, "steps": 8},
        # the prompts of 64 agents as text
        {"name": "encode_64x4000", "kind": "text", "way": "encode", "texts": 64, "bytes": 4000},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(["product", "attend", "pick", "experts", "model", "text"], [7, 5, 2, 2, 2, 2])[0]
    if kind == "product":
        n, k = rng.choice([(4096, 4096), (6144, 4096), (14336, 4096), (4096, 14336), (1024, 4096),
                           (_log(rng, 40, 20000), 32 * _log(rng, 2, 448)),
                           (_log(rng, 40, 20000), 32 * _log(rng, 2, 448)), (128256, 4096)])
        file = rng.random() < 0.3
        m = _log(rng, 1, 64 if file or n > 20000 else 512)
        return {"kind": kind, "m": m, "n": n, "k": k, "file": file, "half": rng.random() < 0.5}
    if kind == "attend":
        heads = rng.choice(["8b", "8b", "8b", "tiny", "mqa"])
        piece = 1 if rng.random() < 0.7 else _log(rng, 4, 512)
        seqs = _log(rng, 1, 64) if piece == 1 else rng.randint(1, max(1, min(4, 512 // piece)))
        lo, hi = sorted(max(piece, _log(rng, 16, 8192)) for _ in range(2))
        return {"kind": kind, "heads": heads, "seqs": seqs, "lo": lo, "hi": hi, "piece": piece}
    if kind == "pick":
        greedy = rng.random() < 0.4
        return {"kind": kind, "rows": _log(rng, 1, 64), "vocab": rng.choice([4096, 32000, 128256, _log(rng, 1000, 152000)]),
                "top_k": 0 if greedy else rng.choice([0, 20, 40, 64]), "top_p": 1.0 if greedy else rng.choice([0.8, 0.9, 0.95, 1.0]),
                "temperature": 0.0 if greedy else rng.choice([0.6, 0.8, 1.0])}
    if kind == "experts":
        return {"kind": kind, "shape": rng.choice(list(EXPERTS)), "tokens": _log(rng, 1, 128)}
    if kind == "model":
        shape = rng.choice(["8b", "8b", "tiny", "qk_norm"])
        slots = _log(rng, 1, 32)
        prompt = 0 if rng.random() < 0.5 else _log(rng, 8, 512 // slots)
        return {"kind": kind, "shape": shape, "slots": slots, "context": _log(rng, 16, 2048) if not prompt or rng.random() < 0.3 else 0,
                "prompt": prompt, "steps": rng.randint(1, 4)}
    texts = _log(rng, 1, 1024)
    return {"kind": "text", "way": rng.choice(["encode", "decode"]), "texts": texts, "bytes": _log(rng, 40, min(8000, 1000000 // texts))}


# ---- what a program keeps between calls -------------------------------------------------

_kept = {"key": None, "world": None, "close": None}


def _world(key, make):
    """The pool, model or vocabulary of the case at hand; the last one is closed first."""
    if _kept["key"] != key:
        if _kept["close"] is not None:
            torch.cuda.synchronize()
            _kept["close"]()
        _kept.update(key=None, world=None, close=None)
        torch.cuda.empty_cache()
        world, close = make()
        _kept.update(key=key, world=world, close=close)
    return _kept["world"]


def _gen(*seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(zlib.crc32(repr(seed).encode()))
    return g


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


# ---- Q8_0 tensors in plain torch ----------------------------------------------------------

def _q8(rows, k, g):
    """N(0, 0.02) quantised to Q8_0 blocks: bytes [rows][k / 32][34]."""
    out = torch.empty(rows, k // 32, 34, dtype=torch.uint8, device="cuda")
    step = max(1, (64 << 20) // k)
    for r in range(0, rows, step):
        w = torch.randn(min(step, rows - r), k // 32, 32, device="cuda", generator=g) * 0.02
        d = w.abs().amax(dim=2) / 127.0
        q = torch.round(w / torch.where(d == 0, torch.ones_like(d), d)[..., None]).clamp(-127, 127).to(torch.int8)
        out[r:r + step, :, :2] = d.half().view(torch.uint8).view(*d.shape, 2)
        out[r:r + step, :, 2:] = q.view(torch.uint8)
    return out


def _values(q):
    """The weights of Q8_0 bytes [rows][blocks][34] as the reader gives them, half(q * scale), in 64 bits."""
    d = q[:, :, :2].contiguous().view(torch.half).float()
    return (q[:, :, 2:].view(torch.int8).float() * d).half().double().view(q.shape[0], -1)


def _product64(x, q):
    """x [m][k] (64 bits) times the rows of Q8_0 bytes, in pieces of rows."""
    step = max(1, (128 << 20) // (q.shape[1] * 32))
    return torch.cat([x @ _values(q[r:r + step]).t() for r in range(0, q.shape[0], step)], dim=1)


# ---- product ------------------------------------------------------------------------------

def _product_inputs(c, seed):
    g = _gen("product", seed, c["m"], c["n"], c["k"])
    return _q8(c["n"], c["k"], g), torch.randn(c["m"], c["k"], device="cuda", generator=g).half()


def _product_prepare(c, seed):
    L = A.lib()
    w, x = _product_inputs(c, seed)
    if not c["file"]:
        wr = torch.empty(L.aotx_q8r_size(c["n"], c["k"]), dtype=torch.uint8, device="cuda")
        A.check(L.aotx_q8_repack(A.ptr(w), c["n"], c["k"], A.ptr(wr), _stream()), "aotx_q8_repack")
        torch.cuda.synchronize()
        w = wr
    y = torch.zeros(c["m"], c["n"], dtype=torch.half if c["half"] else torch.float32, device="cuda")
    call = {(False, False): L.aotx_q8r_gemv, (False, True): L.aotx_q8r_gemv_f16,
            (True, False): L.aotx_q8_gemv, (True, True): L.aotx_q8_gemv_f16}[(c["file"], c["half"])]
    return {"case": c, "w": w, "x": x, "y": y, "call": call, "args": (A.ptr(w), c["n"], c["k"], A.ptr(x), c["m"], A.ptr(y))}


def _product_run(s):
    A.check(s["call"](*s["args"], _stream()), "the product")
    return s["y"]


def _product_work(c):
    n, k, m = c["n"], c["k"], c["m"]
    return {"bytes": n * k * 34 // 32 + m * k * 2 + m * n * (2 if c["half"] else 4), "flops": 2.0 * m * n * k}


def _product_exact(c, seed):
    w, x = _product_inputs(c, seed)
    return _product64(x.double(), w)


# ---- attend -------------------------------------------------------------------------------

class _Layer:
    """One layer of the pool's pages, given back when its state goes."""

    def __init__(self, world):
        self.free, self.at = world["free"], world["free"].pop()

    def __del__(self):
        self.free.append(self.at)


def _contexts(c):
    r = random.Random("%d %d %d" % (c["seqs"], c["lo"], c["hi"]))
    return [r.randint(c["lo"], c["hi"]) for _ in range(c["seqs"])]


def _attend_world(c):
    heads, kvh, d = HEADS[c["heads"]]
    ctx = _contexts(c)

    def make():
        L, kvm = A.lib(), A.KvMap()
        need = [layout_pages(n, KV_LAYERS, kvh, d) for n in ctx]
        kvm.limit = sum(need) + 8
        A.check(L.aotx_kv_open(ctypes.byref(kvm)), "aotx_kv_open")
        # pages come one at a time, in the order in which the conversations grew
        order = [i for i, n in enumerate(need) for _ in range(n)]
        random.Random(3).shuffle(order)
        for i, slot in enumerate(order):
            if L.aotx_kv_request(slot, 1) != 1:
                raise RuntimeError("page request refused")
            if i % 64 == 63:
                L.aotx_kv_serve(ctypes.byref(kvm), None)
        L.aotx_kv_serve(ctypes.byref(kvm), None)
        return {"free": list(range(KV_LAYERS)), "map": kvm}, lambda: L.aotx_kv_close(ctypes.byref(kvm))

    return _world(("attend", c["heads"], tuple(ctx)), make)


def _attend_inputs(c, seed):
    heads, kvh, d = HEADS[c["heads"]]
    ctx = _contexts(c)
    g = _gen("attend", seed, c["seqs"], c["hi"], c["piece"])
    n = sum(ctx)
    k = torch.randn(n, kvh, d, device="cuda", generator=g).half()
    v = torch.randn(n, kvh, d, device="cuda", generator=g).half()
    q = torch.randn(c["seqs"] * c["piece"], heads, d, device="cuda", generator=g).half()
    return ctx, q, k, v


def _attend_prepare(c, seed):
    heads, kvh, d = HEADS[c["heads"]]
    L, world = A.lib(), _attend_world(c)
    ctx, q, k, v = _attend_inputs(c, seed)
    layer = _Layer(world)
    at = torch.cat([torch.arange(n, dtype=torch.int32) for n in ctx]).cuda()
    slot = torch.repeat_interleave(torch.arange(len(ctx), dtype=torch.int32), torch.tensor(ctx)).cuda()
    A.check(L.aotx_kv_write(A.ptr(k), A.ptr(v), A.ptr(at), A.ptr(slot), sum(ctx), kvh, d, layer.at, KV_LAYERS, _stream()), "aotx_kv_write")
    torch.cuda.synchronize()
    p = c["piece"]
    pos = torch.cat([torch.arange(n - p, n, dtype=torch.int32) for n in ctx]).cuda()
    agent = torch.arange(len(ctx), dtype=torch.int32).repeat_interleave(p).cuda()
    out = torch.zeros_like(q)
    return {"case": c, "layer": layer, "q": q, "pos": pos, "agent": agent, "out": out,
            "args": (A.ptr(q), A.ptr(pos), A.ptr(agent), q.shape[0], heads, kvh, d, layer.at, KV_LAYERS, A.ptr(out))}


def _attend_run(s):
    A.check(A.lib().aotx_attend_paged(*s["args"], _stream()), "aotx_attend_paged")
    return s["out"]


def _attend_work(c):
    heads, kvh, d = HEADS[c["heads"]]
    ctx, p = _contexts(c), c["piece"]
    attended = sum(p * n - p * (p - 1) // 2 for n in ctx)
    return {"bytes": sum(ctx) * kvh * d * 4 + 2 * len(ctx) * p * heads * d * 2, "flops": 4.0 * attended * heads * d}


def _attention64(q, k, v, base):
    """Causal attention in 64 bits: q [t][heads][d] at positions base.., k and v [n][kvh][d]."""
    t, heads, d = q.shape
    n, kvh = k.shape[0], k.shape[1]
    qs = q.double().view(t, kvh, heads // kvh, d).permute(1, 2, 0, 3).reshape(kvh, -1, d)
    s = torch.bmm(qs, k.double().permute(1, 2, 0).contiguous()).view(kvh, heads // kvh, t, n) / math.sqrt(d)
    seen = torch.arange(n, device="cuda")[None, :] <= base + torch.arange(t, device="cuda")[:, None]
    s = torch.softmax(s.masked_fill(~seen, -math.inf), dim=-1)
    o = torch.bmm(s.view(kvh, -1, n), v.double().permute(1, 0, 2).contiguous())
    return o.view(kvh, heads // kvh, t, d).permute(2, 0, 1, 3).reshape(t, heads, d)


def _attend_exact(c, seed):
    ctx, q, k, v = _attend_inputs(c, seed)
    p, at, out = c["piece"], 0, []
    for i, n in enumerate(ctx):
        out.append(_attention64(q[i * p:(i + 1) * p], k[at:at + n], v[at:at + n], n - p))
        at += n
    return torch.cat(out)


# ---- pick ---------------------------------------------------------------------------------

def _pick_prepare(c, seed):
    L = A.lib()
    g = _gen("pick", seed, c["rows"], c["vocab"])
    # a model's logits: a broad bulk and a few dozen tokens that stand out of it
    logits = torch.randn(c["rows"], c["vocab"], device="cuda", generator=g) * 2.0
    at = torch.randint(0, c["vocab"], (c["rows"], 60), device="cuda", generator=g)
    logits.scatter_add_(1, at, torch.rand(c["rows"], 60, device="cuda", generator=g) * 10.0)
    agent = torch.arange(c["rows"], dtype=torch.int32, device="cuda")
    token = torch.zeros(c["rows"], dtype=torch.int32, device="cuda")
    drawn = torch.zeros(c["rows"], dtype=torch.int32, device="cuda")
    L.aotx_model_restream()
    return {"case": c, "logits": logits, "agent": agent, "token": token, "draw": drawn,
            "args": (A.ptr(logits), c["rows"], c["vocab"], A.ptr(agent), None, c["top_k"], c["top_p"], c["temperature"],
                     seed & 0xFFFFFFFF, A.ptr(token), A.ptr(drawn))}


def _pick_run(s):
    A.check(A.lib().aotx_pick(*s["args"], _stream()), "aotx_pick")
    return {"token": s["token"], "draw": s["draw"]}


def _pick_work(c):
    return {"bytes": c["rows"] * (c["vocab"] * 4 + 12), "flops": 0.0}


# ---- experts ------------------------------------------------------------------------------

def _experts_inputs(c, seed):
    hidden, ffn, experts, _ = EXPERTS[c["shape"]]
    g = _gen("experts", seed, c["tokens"], hidden)
    gate, up, down = _q8(experts * ffn, hidden, g), _q8(experts * ffn, hidden, g), _q8(experts * hidden, ffn, g)
    router = torch.randn(experts, hidden, device="cuda", generator=g) * 0.02
    return gate, up, down, router, torch.randn(c["tokens"], hidden, device="cuda", generator=g).half()


def _experts_prepare(c, seed):
    hidden, ffn, experts, used = EXPERTS[c["shape"]]
    gate, up, down, router, x = _experts_inputs(c, seed)
    t = c["tokens"]
    prob = torch.zeros(t, experts, device="cuda")
    ids = torch.zeros(t, used, dtype=torch.int32, device="cuda")
    out = torch.zeros(t, hidden, device="cuda")
    return {"case": c, "keep": (gate, up, down, router, x), "prob": prob, "ids": ids, "out": out,
            "route": (A.ptr(router), A.ptr(x), t, hidden, experts, used, A.ptr(prob), A.ptr(ids)),
            "ffn": (A.ptr(gate), A.ptr(up), A.ptr(down), experts, used, hidden, ffn, A.ptr(x), t, A.ptr(prob), A.ptr(ids), A.ptr(out))}


def _experts_run(s):
    L, st = A.lib(), _stream()
    A.check(L.aotx_expert_route(*s["route"], st), "aotx_expert_route")
    A.check(L.aotx_expert_ffn(*s["ffn"], st), "aotx_expert_ffn")
    return {"ids": s["ids"], "out": s["out"], "prob": s["prob"]}


def _experts_work(c):
    hidden, ffn, experts, used = EXPERTS[c["shape"]]
    t = c["tokens"]
    read = experts * (1.0 - (1.0 - used / experts) ** t)      # experts that some token chose
    return {"bytes": read * 3 * ffn * hidden * 34 / 32 + t * hidden * 6 + experts * hidden * 4,
            "flops": 2.0 * t * (used * 3 * ffn * hidden + experts * hidden)}


def _experts_exact(c, seed):
    hidden, ffn, experts, used = EXPERTS[c["shape"]]
    gate, up, down, router, x = _experts_inputs(c, seed)
    x64 = x.double()
    prob = torch.softmax(x64 @ router.double().t(), dim=1)
    ids = torch.sort(prob, dim=1, descending=True, stable=True).indices[:, :used]
    out = torch.zeros(c["tokens"], hidden, dtype=torch.float64, device="cuda")
    for e in range(experts):
        rows = (ids == e).any(dim=1).nonzero()[:, 0]
        if rows.numel():
            f = slice(e * ffn, (e + 1) * ffn)
            a = torch.nn.functional.silu(_product64(x64[rows], gate[f])) * _product64(x64[rows], up[f])
            out[rows] += prob[rows, e:e + 1] * _product64(a, down[e * hidden:(e + 1) * hidden])
    return {"ids": None, "out": out, "prob": prob}


# ---- model --------------------------------------------------------------------------------

def _cache(shape, slots, context, layer):
    """The cached keys and values of one layer, [slots * context][kv_heads][d]."""
    g = _gen("cache", layer, slots, context)
    size = (slots * context, shape.kv_heads, shape.head_dim)
    return torch.randn(size, device="cuda", generator=g).half(), torch.randn(size, device="cuda", generator=g).half()


def _model_world(c):
    shape, B, C = SHAPES[c["shape"]], c["slots"], c["context"]

    def make():
        region, lay = build_device(shape, seed=7)
        need = layout_pages(C + c["prompt"] + c["steps"] + 1, shape.layers, shape.kv_heads, shape.head_dim)
        rt = Runtime(region, lay.desc, max_tokens=max(B, B * c["prompt"]), pool_pages=need * B + 8)
        for slot in range(B):
            if rt.L.aotx_kv_request(slot, need) != 1:
                raise RuntimeError("page request refused")
        rt.L.aotx_kv_serve(ctypes.byref(rt.map), None)
        if C:
            pos = torch.arange(C, dtype=torch.int32, device="cuda").repeat(B)
            slot = torch.arange(B, dtype=torch.int32, device="cuda").repeat_interleave(C)
            for l in range(shape.layers):
                k, v = _cache(shape, B, C, l)
                A.check(rt.L.aotx_kv_write(A.ptr(k), A.ptr(v), A.ptr(pos), A.ptr(slot), B * C, shape.kv_heads, shape.head_dim,
                                           l, shape.layers, None), "aotx_kv_write")
                torch.cuda.synchronize()
        return rt, rt.close

    return _world(("model", c["shape"], B, C, c["prompt"], c["steps"]), make)


def _model_ids(c, seed):
    return torch.randint(0, SHAPES[c["shape"]].vocab, (c["slots"], c["prompt"] + c["steps"]), device="cuda",
                         dtype=torch.int32, generator=_gen("ids", seed, c["slots"]))


def _model_prepare(c, seed):
    rt, shape, B, P = _model_world(c), SHAPES[c["shape"]], c["slots"], c["prompt"]
    ids = _model_ids(c, seed)
    agent = torch.arange(B, dtype=torch.int32, device="cuda")
    keep, calls = [ids, agent], []
    logits = torch.zeros(c["steps"] + (1 if P else 0), B, shape.vocab, device="cuda")
    token = torch.zeros(B, dtype=torch.int32, device="cuda")
    for i, (first, rows) in enumerate(([(0, P)] if P else []) + [(P + j, 1) for j in range(c["steps"])]):
        one = ids[:, first:first + rows].contiguous()
        offset = torch.arange(B + 1, dtype=torch.int32, device="cuda") * rows
        keep += [one, offset]
        r = A.ModelRun()
        r.ids, r.offset, r.agent, r.token = one.data_ptr(), offset.data_ptr(), agent.data_ptr(), token.data_ptr()
        r.logits = logits[i].data_ptr()
        r.seqs, r.tokens, r.rows, r.select, r.top_p = B, B * rows, B, A.AOTX_MODEL_ROWS_LAST, 1.0
        calls.append((r, offset))
    torch.cuda.synchronize()
    return {"case": c, "rt": rt, "keep": keep, "agent": agent, "calls": calls, "logits": logits, "token": token}


def _model_run(s):
    c, rt = s["case"], s["rt"]
    L = rt.L
    if c["context"] == 0:
        L.aotx_model_forget()
    else:
        for slot in range(c["slots"]):
            L.aotx_model_seat(slot, c["context"])
    agent, kvm = A.ptr(s["agent"]), ctypes.byref(rt.map)
    for r, offset in s["calls"]:
        A.check(L.aotx_model_pages(rt.role, A.ptr(offset), c["slots"], agent), "aotx_model_pages")
        L.aotx_kv_serve(kvm, None)
        A.check(L.aotx_model_launch(rt.role, ctypes.byref(r)), "aotx_model_launch")
    return s["logits"]


def _model_work(c):
    s, B, C, P = SHAPES[c["shape"]], c["slots"], c["context"], c["prompt"]
    wide, narrow = s.heads * s.head_dim, s.kv_heads * s.head_dim
    per_layer = s.hidden * (2 * wide + 2 * narrow) + 3 * s.ffn * s.hidden
    weights = (s.layers * per_layer + s.vocab * s.hidden) * 34 / 32
    byte = flop = 0.0
    for first, rows in ([(C, P)] if P else []) + [(C + P + j, 1) for j in range(c["steps"])]:
        attended = rows * first + rows * (rows + 1) // 2
        byte += weights + B * ((first + rows) * narrow * 4 * s.layers + s.vocab * 4 + rows * s.hidden * 34 / 32)
        flop += 2.0 * B * (rows * s.layers * per_layer + s.vocab * s.hidden) + 4.0 * B * attended * wide * s.layers
    return {"bytes": byte, "flops": flop}


def _model_exact(c, seed):
    s, B, C, P, T = SHAPES[c["shape"]], c["slots"], c["context"], c["prompt"], c["prompt"] + c["steps"]
    region, lay = build_device(s, seed=7)
    d, slot = lay.desc, A.SLOT

    def q8(at, rows, k):
        return region[at:at + rows * (k // 32) * 34].view(rows, k // 32, 34)

    def norm(x):                                           # the norm weights are ones
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + s.eps)

    half = torch.arange(s.head_dim // 2, device="cuda", dtype=torch.float64)
    angle = torch.arange(C, C + T, device="cuda", dtype=torch.float64)[:, None] * s.theta ** (-2.0 * half / s.head_dim)
    cos, sin = angle.cos()[:, None, :], angle.sin()[:, None, :]

    def turn(x):                                           # [B][T][heads][d]
        if s.pairs == A.AOTX_ROPE_PAIRS_ADJACENT:
            a, b = x[..., 0::2], x[..., 1::2]
            return torch.stack([a * cos - b * sin, a * sin + b * cos], dim=-1).flatten(-2)
        a, b = x.chunk(2, dim=-1)
        return torch.cat([a * cos - b * sin, a * sin + b * cos], dim=-1)

    ids = _model_ids(c, seed).long().flatten()
    x = _values(q8(d.token_embd, s.vocab, s.hidden)[ids])
    wide, narrow = s.heads * s.head_dim, s.kv_heads * s.head_dim
    for l in range(s.layers):
        o = d.layer[l].offset
        y = norm(x)
        q = _product64(y, q8(o[slot["attn_q"]], wide, s.hidden)).view(B, T, s.heads, s.head_dim)
        k = _product64(y, q8(o[slot["attn_k"]], narrow, s.hidden)).view(B, T, s.kv_heads, s.head_dim)
        v = _product64(y, q8(o[slot["attn_v"]], narrow, s.hidden)).view(B, T, s.kv_heads, s.head_dim)
        if s.qk_norm:
            q, k = norm(q), norm(k)
        q, k = turn(q), turn(k)
        ck, cv = _cache(s, B, C, l)
        ck, cv = (t.double().view(B, C, s.kv_heads, s.head_dim) for t in (ck, cv))
        att = torch.stack([_attention64(q[b], torch.cat([ck[b], k[b]]), torch.cat([cv[b], v[b]]), C) for b in range(B)])
        x = x + _product64(att.view(B * T, wide), q8(o[slot["attn_o"]], s.hidden, wide))
        y = norm(x)
        a = torch.nn.functional.silu(_product64(y, q8(o[slot["ffn_gate"]], s.ffn, s.hidden)))
        a = a * _product64(y, q8(o[slot["ffn_up"]], s.ffn, s.hidden))
        x = x + _product64(a, q8(o[slot["ffn_down"]], s.hidden, s.ffn))
    rows = ([P - 1] if P else []) + list(range(P, T))
    y = norm(x).view(B, T, s.hidden)[:, rows].transpose(0, 1).reshape(-1, s.hidden)
    return _product64(y, q8(d.output, s.vocab, s.hidden)).view(len(rows), B, s.vocab)


# ---- text ---------------------------------------------------------------------------------

_made = {}


def _vocabulary():
    """A byte-level BPE vocabulary: 256 bytes, then the merges of a small seeded lexicon, most
    frequent pair first, as such vocabularies are trained. Returns (words, weights, tokens, merges)."""
    if not _made:
        keep = [b for b in range(256) if 33 <= b <= 126 or 161 <= b <= 172 or 174 <= b <= 255]
        char = {b: chr(b) for b in keep}
        for i, b in enumerate(b for b in range(256) if b not in char):
            char[b] = chr(256 + i)
        r = random.Random(11)
        part = ["ta", "ren", "mo", "li", "ske", "dor", "an", "ing", "us", "per", "ca", "ver", "ti", "on", "é", "ño", "дан", "ные", "中", "文"]
        words = [" " + "".join(r.choice(part[:14] if r.random() < 0.9 else part) for _ in range(r.randint(1, 4))) for _ in range(420)]
        words += [" the", " of", " and", "'s", "'t", ",", ".", " (", ")", "::", "\n\n", " 2024", "12", " 😀", " =", " x"]
        weight = [1.0 / (i + 3) for i in range(len(words))]
        parts = [[char[b] for b in w.encode()] for w in words]
        tokens, merges = [char[b] for b in range(256)], []
        have = set(tokens)
        for _ in range(900):
            count = {}
            for p, w in zip(parts, weight):
                for a, b in zip(p, p[1:]):
                    count[(a, b)] = count.get((a, b), 0.0) + w
            if not count:
                break
            a, b = max(count, key=lambda t: (count[t], t))
            merges.append(a + " " + b)
            if a + b not in have:
                have.add(a + b)
                tokens.append(a + b)
            for p in parts:
                i = 0
                while i + 1 < len(p):
                    if p[i] == a and p[i + 1] == b:
                        p[i:i + 2] = [a + b]
                    i += 1
        _made["all"] = (words, weight, tokens, merges)
    return _made["all"]


def _text_world():
    def make():
        _, _, tokens, merges = _vocabulary()
        tk = Tokenizer(tokens=tokens, merges=merges, family="llama3")
        return tk, tk.close

    return _world("text", make)


def _texts(c, seed):
    words, weight, _, _ = _vocabulary()
    sizes = random.Random("%d %d" % (c["texts"], c["bytes"]))    # the lengths are the case's, the words the seed's
    r = random.Random("%d %d %d" % (seed, c["texts"], c["bytes"]))
    run = [w.encode() for w in r.choices(words, weight, k=max(64, min(60000, c["texts"] * c["bytes"] // 3)))]
    out = []
    for _ in range(c["texts"]):
        want, at, have, size = int(c["bytes"] * sizes.uniform(0.5, 1.5)), r.randrange(len(run)), [], 0
        while size + len(run[at]) <= want:
            have.append(run[at])
            size += len(run[at])
            at = (at + 1) % len(run)
        out.append(b"".join(have) + b"." * (want - size))
    return out


def _offsets(lengths):
    at = np.zeros(len(lengths) + 1, dtype=np.int64)
    at[1:] = np.cumsum(lengths)
    return at


def _text_prepare(c, seed):
    tk, texts = _text_world(), _texts(c, seed)
    at = _offsets([len(t) for t in texts])
    data = torch.from_numpy(np.frombuffer(b"".join(texts), dtype=np.uint8).copy()).cuda()
    s = {"case": c, "tk": tk, "data": data, "at": torch.from_numpy(at).cuda(),
         "ids": torch.zeros(3 * int(at[-1]), dtype=torch.int32, device="cuda"),
         "count": torch.zeros(len(texts), dtype=torch.int32, device="cuda")}
    if c["way"] == "decode":
        # a reply's ids, as the sampler gave them
        _encode(s)
        ids, count = s["ids"].cpu().numpy(), s["count"].cpu().numpy()
        flat = np.concatenate([ids[3 * a:3 * a + n] for a, n in zip(at, count)])
        s["limit"] = max(len(t) for t in texts)
        s["flat"], s["flat_at"] = torch.from_numpy(flat).cuda(), torch.from_numpy(_offsets(count)).cuda()
        s["out"] = torch.zeros(len(texts), s["limit"], dtype=torch.uint8, device="cuda")
        s["length"] = torch.zeros(len(texts), dtype=torch.int32, device="cuda")
    return s


def _encode(s):
    A.check(s["tk"].L.aotx_text_encode(A.ptr(s["data"]), A.ptr(s["at"]), s["case"]["texts"], A.ptr(s["ids"]), A.ptr(s["count"]),
                                       _stream()), "aotx_text_encode")


def _text_run(s):
    if s["case"]["way"] == "encode":
        _encode(s)
        return {"count": s["count"], "ids": s["ids"]}
    A.check(s["tk"].L.aotx_text_detok(A.ptr(s["flat"]), A.ptr(s["flat_at"]), s["case"]["texts"], A.ptr(s["out"]), s["limit"],
                                      A.ptr(s["length"]), _stream()), "aotx_text_detok")
    return {"length": s["length"], "bytes": s["out"]}


def _text_work(c):
    n = c["texts"] * c["bytes"]
    return {"bytes": n + 4.0 * n / 4 + 12.0 * c["texts"], "flops": 0.0}   # about four bytes a token


# ---- the interface --------------------------------------------------------------------------

_KINDS = {"product": (_product_prepare, _product_run, _product_work, _product_exact),
          "attend": (_attend_prepare, _attend_run, _attend_work, _attend_exact),
          "pick": (_pick_prepare, _pick_run, _pick_work, None),
          "experts": (_experts_prepare, _experts_run, _experts_work, _experts_exact),
          "model": (_model_prepare, _model_run, _model_work, _model_exact),
          "text": (_text_prepare, _text_run, _text_work, None)}


def prepare(case, seed):
    return _KINDS[case["kind"]][0](case, seed)


def run(state):
    return _KINDS[state["case"]["kind"]][1](state)


def work(case):
    return _KINDS[case["kind"]][2](case)


def exact(case, seed):
    f = _KINDS[case["kind"]][3]
    return None if f is None else f(case, seed)


def tolerance(case):
    kind = case["kind"]
    if kind == "product":
        # fp32 sums in another order; an fp16 result adds its rounding
        return {"rel": 1e-3, "max": 4e-3} if case["half"] else {"rel": 1e-5, "max": 1e-4}
    if kind == "attend":
        # fp16 probabilities into fp32 sums, an fp16 result
        return {"rel": 1.2e-3, "max": 1e-2}
    if kind == "experts":
        # the gated unit's result is rounded to fp16 between the products
        return {"rel": 1e-3, "max": 1e-2, "differ": 0.01}
    if kind == "model":
        # fp16 rows between the layers: roundings travel through all that follow
        return {"rel": 2e-2, "max": 1e-1}
    return "exact"
