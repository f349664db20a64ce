"""The framework's timed cases: what a program that runs a model's full-attention layers asks of it.

A case is one pass through the public entry points of qwen3-local-test_amd (the Python mirror of
include/qwattn.h) over `layers` layers, each with its own K/V cache, weights and inputs. Kinds:
  attn       the attention layer body: decode / verify (`decode`) or a prefill chunk (`prefill`)
  proj       the projections around it: query + gate, key and value in one `mat_multi`, then the output `mat`
  layer      both: mat_multi, the attention layer body, mat
  qsa_step   a block-sparse layer step: `qsa_index`, then `decode_qsa` over the keys it left visible
  qsa_index  the indexer alone over a chunk of new tokens
  qsa_attn   the attention of a chunk of new tokens over given key visibility bits (`prefill_qsa`)

listed() holds the shapes of the repository's benchmark and tests plus ragged ones; draw() gives more of the
same ranges. exact() restates a pass in float64 with plain torch.
"""
import importlib.util
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda"
THETA, EPS = 1e7, 1e-6
# attention shapes of the tests: (query heads, key/value heads, head dim, rotated dims)
FULL, TINY, PAIR, D128 = (16, 2, 256, 64), (4, 1, 64, 16), (2, 1, 256, 64), (8, 2, 128, 32)
IH, ID = 4, 128  # the indexer: heads, dims


def package():
    """qwen3-local-test_amd as the module qwattn_amd (its folder's name has a hyphen: loaded by path)."""
    if "qwattn_amd" not in sys.modules:
        pkg = os.path.join(ROOT, "qwen3-local-test_amd")
        spec = importlib.util.spec_from_file_location("qwattn_amd", os.path.join(pkg, "__init__.py"),
                                                      submodule_search_locations=[pkg])
        sys.modules["qwattn_amd"] = mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
    return sys.modules["qwattn_amd"]


def case(kind, pos, n, shape=FULL, **more):
    nh, nkv, d, r = shape
    return {"kind": kind, "pos": pos, "n": n, "heads": nh, "kv_heads": nkv, "dim": d, "rope": r, "layers": 1, **more}


def named(name, *args, **kw):
    return {"name": name, **case(*args, **kw)}


def listed():
    return [
        # the smallest call: one token of the tiny test model, where the launch is all there is
        named("tiny_decode", "attn", 128, 1, TINY, dtype="f32"),
        # the ordinary decode step of a chat at 4K: whole layers, four of a model's
        named("layer_decode_4k", "layer", 4096, 1, hidden=2048, weights="q8", layers=4),
        # long-context decode, the benchmark's headline
        named("decode_32k", "attn", 32768, 1, dtype="f32", layers=4),
        # decode at the context limit, 1% of the keys eight times the others
        named("decode_256k", "attn", 262143, 1, dtype="f32", heavy=0.01),
        # speculative verify: one token and three drafts through whole layers
        named("layer_verify_32k", "layer", 32768, 4, hidden=2048, weights="q8", layers=4),
        # a chunk of a long prompt, bf16 activations
        named("prefill_2k_on_2k", "attn", 2048, 2048, dtype="bf16"),
        # a short chat prompt: whole layer, 77 tokens from position 0
        named("layer_prompt_77", "layer", 0, 77, hidden=2048, weights="q8"),
        # the engine's own chunk size deep in a prompt: whole layer, fp32 activations
        named("layer_chunk_1k_on_8k", "layer", 8192, 1024, hidden=2048, weights="q8"),
        # the four projections of a 2,048-token chunk
        named("proj_2k", "proj", 0, 2048, hidden=2048, weights="q8"),
        # block-sparse decode past the budget: index, then attend
        named("qsa_step_32k", "qsa_step", 32768, 1, cr=4, budget=2048, layers=4),
        # the indexer over a prompt chunk
        named("qsa_index_512_on_16k", "qsa_index", 16384, 512, cr=4, budget=2048, dtype="f32"),
        # the attention of the same kind of chunk over what an indexer with longer blocks left visible
        named("qsa_attn_512_on_16k", "qsa_attn", 16384, 512, cr=64, budget=2048, dtype="f32"),
    ]


def spread(rng, lo, hi):
    """A whole number from lo to hi, even over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    top = {}
    for c in listed():
        w = work(c)
        for k in (c["kind"], "all"):
            b, f = top.get(k, (0, 0))
            top[k] = (max(b, w["bytes"]), max(f, w["flops"]))
    while True:
        kind = rng.choice(["attn", "attn", "attn", "layer", "layer", "proj", "proj", "qsa_step", "qsa_index", "qsa_attn"])
        shape = rng.choice([FULL, FULL, FULL, FULL, D128, TINY, PAIR])
        decode = kind == "qsa_step" or (kind not in ("qsa_index", "qsa_attn") and rng.random() < 0.5)
        n = rng.choice([1, 1, 1, 2, 3, 4]) if decode else spread(rng, 33, 2048)
        pos = spread(rng, 1, 262144 - n) if decode else rng.choice([0, spread(rng, 1, 65536)])
        more = {}
        if kind == "proj":
            pos, n = 0, spread(rng, 1, 2048)
        if kind in ("proj", "layer"):
            more["weights"] = "f32" if rng.random() < 0.15 else "q8"
            more["hidden"] = rng.choice([512, 1024, 2048, 2048, 2048])
        elif kind != "qsa_step":
            more["dtype"] = rng.choice(["f32", "bf16"])
        if kind.startswith("qsa"):
            shape = FULL
            more["cr"] = rng.choice([4, 4, 8, 64])
            more["budget"] = 2048
            pos = spread(rng, 4096, 262144 - n if kind == "qsa_step" else 65536)
        if decode:
            more["layers"] = rng.choice([1, 2, 4])
        c = case(kind, pos, n, shape, **more)
        w, most = work(c), top[kind]
        # no drawn case costs more than the largest listed one of its kind
        if w["bytes"] <= most[0] and w["flops"] <= most[1]:
            return c


# ---- work and tolerance ------------------------------------------------------------------------------------

def matrices(c):
    """(rows, cols) of the query + gate, key, value and output projections."""
    h, d = c["hidden"], c["dim"]
    return [(c["heads"] * 2 * d, h), (c["kv_heads"] * d, h), (c["kv_heads"] * d, h), (h, c["heads"] * d)]


def work(c):
    kind, n, pos, d, nh, nkv = c["kind"], c["n"], c["pos"], c["dim"], c["heads"], c["kv_heads"]
    size = 2 if c.get("dtype") == "bf16" else 4
    rows = pos + n
    byts = flops = 0
    if kind in ("layer", "proj"):
        per = 1 + 4 / 32 if c["weights"] == "q8" else 4
        byts += sum(r * k * per for r, k in matrices(c)) + 2 * 4 * n * c["hidden"]
        flops += sum(2 * n * r * k for r, k in matrices(c))
        if kind == "proj":
            byts += 4 * n * (3 * nh * d + 2 * nkv * d)
    if kind in ("attn", "layer"):
        byts += 2 * rows * nkv * d * 2
        flops += 4 * d * nh * (n * pos + n * (n + 1) // 2)
    if kind == "attn":
        byts += n * (size * (2 * nh * d + 2 * nkv * d) + 4 * nh * d)
    if kind in ("qsa_step", "qsa_index"):
        blocks = rows // c["cr"]
        byts += blocks * ID * 4 + n * (size * (IH + 1) * ID + rows // 8)
        flops += 2 * n * blocks * IH * ID
    if kind in ("qsa_step", "qsa_attn"):
        seen = min(rows, c["budget"] + c["cr"])
        keys = seen if n == 1 else min(rows, n * seen)  # each visible key's rows once
        byts += 2 * keys * nkv * d * 2 + n * (size * (2 * nh * d + 2 * nkv * d) + 4 * nh * d + rows // 8)
        flops += 4 * d * nh * n * seen
    return {"bytes": byts * c["layers"], "flops": flops * c["layers"]}


def prefills(c):
    return c["kind"] in ("attn", "layer", "qsa_attn") and not decodes(c)


def decodes(c):
    return c["n"] <= 8 and c["n"] * (c["heads"] // c["kv_heads"]) <= 32


def tolerance(c):
    # "max": a new key's fp16 cache element may round the other way (one step: 2^-10 of it)
    if c["kind"] == "qsa_index":
        # fp32 scores: a block whose score is within rounding of the budget's last may swap with it
        return {"rel": 1e-5, "max": 2e-3, "differ": 2e-4}
    if prefills(c):
        # fp16 queries and probabilities (11 bits each): 3e-4 against float64
        return {"rel": 1.5e-3, "max": 1e-2}
    if c["kind"] == "proj":
        # fp32-level products and sums: 2.5e-6 against float64
        return {"rel": 1e-5, "max": 2e-4}
    # decode, verify: fp32-level products against the fp16 cache (4e-7; 2e-5 where a new key's element is
    # cached the other way)
    return {"rel": 8e-5, "max": 2e-3}


# ---- inputs ------------------------------------------------------------------------------------------------

def inputs(c, seed):
    """The tensors a program has in hand, per layer (rows form, on the GPU)."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    n, nh, nkv, d = c["n"], c["heads"], c["kv_heads"], c["dim"]
    rows = c["pos"] + n
    cap = (rows + 31) // 32 * 32
    dt = torch.bfloat16 if c.get("dtype") == "bf16" else torch.float32

    def rand(*shape, dtype=torch.float32):
        return torch.randn(shape, device=DEV, generator=g, dtype=dtype)

    def uniform(*shape):
        return torch.rand(shape, device=DEV, generator=g)

    got = []
    for _ in range(c["layers"]):
        s = {"cap": cap}
        if c["kind"] in ("layer", "proj"):
            s["x"] = rand(n, c["hidden"])
            s["w"] = []
            for r, k in matrices(c):
                if c["weights"] == "q8":
                    w8 = torch.randint(-127, 128, (r, k), dtype=torch.int8, device=DEV, generator=g)
                    s["w"].append((w8, 0.5 / math.sqrt(k) / 73 * (0.5 + uniform(r, k // 32))))
                else:
                    s["w"].append((rand(r, k) / math.sqrt(k), None))
            if c["kind"] == "proj":
                s["xo"] = rand(n, nh * d)
        elif c["kind"] != "qsa_index":
            s["qg"], s["k"], s["v"] = (rand(n, h, w).to(dt) for h, w in ((nh, 2 * d), (nkv, d), (nkv, d)))
        if c["kind"] not in ("proj", "qsa_index"):
            s["qn"], s["kn"] = 0.1 * rand(d), 0.1 * rand(d)
            s["krows"], s["vrows"] = rand(cap, nkv, d, dtype=torch.float16), rand(cap, nkv, d, dtype=torch.float16)
            if c.get("heavy"):
                s["krows"][uniform(cap) < c["heavy"]] *= 8
        if c["kind"] in ("qsa_step", "qsa_index"):
            s["ik"], s["iq"] = rand(n, ID).to(dt), rand(n, IH, ID).to(dt)
            s["ik_gamma"], s["iq_gamma"] = 1 + 0.1 * rand(ID), 1 + 0.1 * rand(ID)
            s["raw"], s["pooled"] = rand(cap, ID), rand(cap // c["cr"] + 1, ID)
        if c["kind"] == "qsa_attn":
            # neighbouring tokens want much the same blocks: half of a block's score is the chunk's own
            blocks = rows // c["cr"]
            s["visible"] = visible(c, rand(blocks)[None] + rand(n, blocks))
        got.append(s)
    return got


def visible(c, scores):
    """[n, pos + n] truth values from block scores [n, blocks]: the budget's best complete blocks and the
    tail block; everything while there are no more blocks than the budget holds."""
    n, pos, cr = c["n"], c["pos"], c["cr"]
    top, dev = c["budget"] // cr, scores.device
    done = (pos + 1 + torch.arange(n, device=dev)) // cr  # each token's complete blocks
    b = torch.arange(scores.shape[1], device=dev)
    scores = scores.masked_fill(b[None] >= done[:, None], -math.inf)
    order = scores.sort(dim=1, descending=True, stable=True).indices[:, :top]
    taken = torch.zeros_like(scores, dtype=torch.bool).scatter_(1, order, True)
    taken |= (done <= top)[:, None]
    j = torch.arange(pos + n, device=dev)
    key = taken.new_zeros((n, pos + n))
    whole = scores.shape[1] * cr
    key[:, :whole] = taken.repeat_interleave(cr, dim=1)
    return key | (j[None] >= (done * cr)[:, None])


def packed(bits):
    """[n, keys] truth values as int32 words of 32, key j in bit j % 32."""
    n, keys = bits.shape
    words = (keys + 31) // 32
    full = torch.zeros((n, words * 32), dtype=torch.int64, device=bits.device)
    full[:, :keys] = bits
    w = (full.view(n, words, 32) << torch.arange(32, device=bits.device)).sum(dim=2)
    return torch.where(w >= 1 << 31, w - (1 << 32), w).to(torch.int32)


def prepare(c, seed):
    """A context of the model's shape, the caches, weights, inputs and output buffers of each layer."""
    qw = package()
    n, nh, nkv, d = c["n"], c["heads"], c["kv_heads"], c["dim"]
    layers = inputs(c, seed)
    att = qw.Attention(nh, nkv, d, c["rope"], THETA, EPS, max_ctx=layers[0]["cap"], max_tokens=n)
    for s in layers:
        if "krows" in s:
            s["kc"], s["vc"] = qw.k_block(s.pop("krows")), qw.v_block(s.pop("vrows"))
            s["out"] = torch.zeros((n, nh, d), device=DEV)
        if "w" in s:
            s["qg"], s["k"], s["v"] = (torch.zeros((n, r), device=DEV) for r, _ in matrices(c)[:3])
            s["h"] = torch.zeros((n, c["hidden"]), device=DEV)
        if "visible" in s:
            s["bits"] = packed(s.pop("visible"))
        elif c["kind"].startswith("qsa"):
            s["bits"] = torch.zeros((n, (c["pos"] + n + 31) // 32), dtype=torch.int32, device=DEV)
    torch.cuda.synchronize()
    return {"case": c, "att": att, "rope": att.rope_table(), "layers": layers}


# ---- the pass ------------------------------------------------------------------------------------------------

def attend(st, s):
    """The attention layer body of one layer."""
    c, a = st["case"], st["att"]
    args = (s["qg"], s["k"], s["v"], s["qn"], s["kn"], st["rope"], s["kc"], s["vc"], s["cap"], s["out"], c["pos"],
            c["n"])
    if c["kind"] == "qsa_step":
        a.decode_qsa(*args, 0, s["bits"])
    elif c["kind"] == "qsa_attn":
        a.prefill_qsa(*args, s["bits"])
    elif decodes(c):
        a.decode(*args)
    else:
        a.prefill(*args)


def run(st):
    c, a = st["case"], st["att"]
    kind = c["kind"]
    for s in st["layers"]:
        if "w" in s:
            a.mat_multi(s["x"], [(s["qg"], *s["w"][0]), (s["k"], *s["w"][1]), (s["v"], *s["w"][2])])
        if kind in ("qsa_step", "qsa_index"):
            a.qsa_index(s["ik"], s["iq"], s["ik_gamma"], s["iq_gamma"], c["cr"], c["budget"], s["raw"], s["pooled"],
                        s["cap"], c["pos"], c["n"], None, s["bits"])
        if kind not in ("proj", "qsa_index"):
            attend(st, s)
        if "w" in s:
            a.mat(s["xo"] if kind == "proj" else s["out"].view(c["n"], -1), s["h"], *s["w"][3])
    keep = {"attn": ("out", "kc", "vc"), "proj": ("qg", "k", "v", "h"), "layer": ("h", "kc", "vc"),
            "qsa_step": ("out", "bits", "kc", "vc", "raw"), "qsa_index": ("bits", "raw", "pooled"),
            "qsa_attn": ("out", "kc", "vc")}[kind]
    return [{k: s[k] for k in keep} for s in st["layers"]]


# ---- the same in float64 ---------------------------------------------------------------------------------------

def angles(pos, r):
    """(cos, sin) [len(pos), r / 2] of the fp32 angle p * inv_freq, as the rope table is defined."""
    i = torch.arange(r // 2, dtype=torch.float64, device=DEV)
    a = (pos.float()[:, None] * (1.0 / THETA ** (2 * i / r)).float()[None]).double()
    return a.cos(), a.sin()


def norm_rope(x, mult, pos, r):
    """RMS norm with multipliers `mult`, then rotate-half RoPE of the first r dims; x [n, heads, dims] float64."""
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * mult.double()
    cs, sn = (t[:, None] for t in angles(pos, r))
    a, b = x[..., : r // 2], x[..., r // 2: r]
    return torch.cat([a * cs - b * sn, b * cs + a * sn, x[..., r:]], -1)


def blocked_k(rows):
    """[cap][kv heads][dims] rows in the K cache's element order (include/qwattn.h)."""
    cap, nkv, d = rows.shape
    return rows.view(cap // 32, 4, 2, 4, nkv, d // 32, 4, 8).permute(4, 0, 5, 2, 6, 1, 3, 7).reshape(-1)


def blocked_v(rows):
    cap, nkv, d = rows.shape
    return rows.view(cap // 32, 4, 8, nkv, d // 16, 16).permute(3, 0, 4, 1, 5, 2).reshape(-1)


def weight(w, s):
    return w.double() if s is None else w.double() * s.double().repeat_interleave(32, dim=1)


def exact(c, seed):
    if c["kind"] == "layer" and decodes(c):
        # the new keys and values come from fp32 projections and are cached in fp16: which way one near the
        # middle of a step is cached moves the layer's output by far more than the precision of its products
        # (4e-7 or 1e-5 of it, by chance); attn and proj look at the two halves of the path
        return None
    kind, n, pos = c["kind"], c["n"], c["pos"]
    nh, nkv, d, r = c["heads"], c["kv_heads"], c["dim"], c["rope"]
    rows, p = pos + n, pos + torch.arange(n, device=DEV)
    got = []
    for s in inputs(c, seed):
        o, seen = {}, s.get("visible")
        if "w" in s:
            qg, k, v = (s["x"].double() @ weight(*w).T for w in s["w"][:3])
            if kind == "proj":
                got.append({"qg": qg, "k": k, "v": v, "h": s["xo"].double() @ weight(*s["w"][3]).T})
                continue
            s["qg"], s["k"], s["v"] = qg.view(n, nh, 2 * d), k.view(n, nkv, d), v.view(n, nkv, d)
        if "ik" in s:
            s["raw"][pos:rows] = s["ik"].float()
            cr, pooled = c["cr"], s["pooled"].double()
            b = torch.arange(pos // cr, rows // cr, device=DEV)
            if len(b):
                mean = s["raw"][pos // cr * cr: rows // cr * cr].double().view(-1, cr, ID).mean(1)
                pooled[b] = norm_rope(mean[:, None], s["ik_gamma"], b * cr, r)[:, 0]
            o["bits"], o["raw"], o["pooled"] = None, s["raw"].double(), pooled
            if kind == "qsa_index":
                got.append(o)
                continue
            q = norm_rope(s["iq"].double(), s["iq_gamma"], p, r)
            seen = visible(c, torch.einsum("thd,bd->thb", q, pooled[: rows // cr]).clamp(min=0).sum(1))
            del o["pooled"]
        q = norm_rope(s["qg"][..., :d].double(), 1 + s["qn"].double(), p, r)
        kr, vr = s["krows"], s["vrows"]
        kr[pos:rows] = norm_rope(s["k"].double(), 1 + s["kn"].double(), p, r).half()
        vr[pos:rows] = s["v"].half()
        out = torch.zeros((n, nh, d), dtype=torch.float64, device=DEV)
        past = torch.arange(rows, device=DEV)[None] > p[:, None]
        hidden = past if seen is None else past | ~seen
        for h in range(nkv):
            kd, vd = kr[:rows, h].double(), vr[:rows, h].double()
            for e in range(h * (nh // nkv), (h + 1) * (nh // nkv)):
                sc = (q[:, e] @ kd.T / math.sqrt(d)).masked_fill(hidden, -math.inf)
                out[:, e] = torch.softmax(sc, -1) @ vd
        out *= torch.sigmoid(s["qg"][..., d:].double())
        o["kc"], o["vc"] = blocked_k(kr).double(), blocked_v(vr).double()
        if "w" in s:
            o["h"] = out.view(n, -1) @ weight(*s["w"][3]).T
        else:
            o["out"] = out
        got.append(o)
    return got
