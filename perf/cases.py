"""Performance cases of the speculative-decoding framework.

Each case is one call, or one layer's calls, as an engine built on this package
makes them:
  attend   q/k-norm + RoPE + KV store + attention over the paged cache, for
           verify, decode and prefill steps (Attention.attend_qkv)
  prefill  attention over the step's own k / v rows, prompts without a cached
           prefix (Attention.forward with no block table and no bound cache)
  layer    a whole decoder layer (Qwen3Layer) of the 8B target
  decode   a forward of the 0.6B draft's geometry with its logits, replayed from a
           HIP graph as the runner replays it; its depth is a setting, kept at a few
           layers so that bf16 rounding does not outgrow the comparison of logits
  accept   the acceptance sampler (ops.spec_accept)
  sample   the draft-step row sampler: probabilities and tokens
           (ops.sample_rows)
Sizes follow the framework's benchmark configurations: batch 1 with gamma 3
(target 32/8 heads, draft 16/8), 64 sequences with contexts of 64..2048, 32
sequences growing to 8192 tokens over an FP8 cache, vocabulary 151936.
"""
from __future__ import annotations

import importlib
import random

import torch
import torch.nn.functional as F

hv = importlib.import_module("hilda-vllm_amd")
ops = hv.ops
attention = importlib.import_module("hilda-vllm_amd.layers.attention")
host = importlib.import_module("hilda-vllm_amd.engine.qwen3_host")
context = importlib.import_module("hilda-vllm_amd.utils.context")

VOCAB = 151936
BLOCK = 256  # tokens per KV block, the framework's default
D = 128
EPS = 1e-6
DEV = "cuda"
GEOMETRY = {"8b": host.QWEN3_8B, "0.6b": host.QWEN3_0_6B}


def listed():
    return [
        # the batch-1 verify step's attention, 4 query rows on a 320-token context: the
        # smallest call, 36 of them in every step of an interactive user
        dict(name="attend-verify-b1", kind="attend", model="8b", batch=1, q_min=4, q_max=4,
             k_min=320, k_max=320, bound=4096, kv="bf16"),
        # a serving batch of draft / small-model verify rows with ragged contexts
        dict(name="attend-verify-b64", kind="attend", model="0.6b", batch=64, q_min=4, q_max=4,
             k_min=64, k_max=2048, bound=2048, kv="bf16"),
        # long generations over the FP8 cache, 8B target heads
        dict(name="attend-verify-b32-fp8", kind="attend", model="8b", batch=32, q_min=4, q_max=4,
             k_min=1024, k_max=8192, bound=8192, kv="fp8"),
        # admission of a few prompts of ordinary, odd lengths (no cached prefix)
        dict(name="prefill-ragged", kind="prefill", model="8b", batch=4, q_min=61, q_max=1021),
        # a long conversation read back in after a preemption: one sequence's whole
        # history through one layer's attention, into its cache blocks
        dict(name="attend-prefill-long", kind="attend", model="8b", batch=1, q_min=6301,
             q_max=6301, k_min=6301, k_max=6301, bound=8192, kv="bf16"),
        # one target layer of the batch-1 verify step (4 rows)
        dict(name="layer-verify-b1", kind="layer", model="8b", batch=1, q_min=4, q_max=4,
             k_min=320, k_max=320, bound=4096, kv="bf16"),
        # one target layer of a batch-8 verify step (32 rows)
        dict(name="layer-verify-b8", kind="layer", model="8b", batch=8, q_min=4, q_max=4,
             k_min=256, k_max=1280, bound=4096, kv="bf16"),
        # one draft decode step of the batch-1 run: embedding, layers, logits
        dict(name="decode-draft-b1", kind="decode", model="0.6b", batch=1, q_min=1, q_max=1,
             k_min=320, k_max=320, bound=4096, kv="bf16", layers=6),
        # acceptance of the batch-1 step
        dict(name="accept-b1", kind="accept", batch=1, gamma=3, logits="bf16",
             mode="reference", settings="plain"),
        # acceptance of a large serving batch, every sequence its own temperature
        dict(name="accept-b256", kind="accept", batch=256, gamma=5, logits="bf16",
             mode="reference", settings="mixed"),
        # acceptance with per-sequence temperature / top-k / top-p
        dict(name="accept-b64-filtered", kind="accept", batch=64, gamma=3, logits="bf16",
             mode="filtered", settings="mixed"),
        # the draft side of the same batch: filtered probabilities and the drawn tokens
        dict(name="sample-b64-filtered", kind="sample", rows=64, logits="bf16",
             mode="filtered", settings="mixed"),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["attend", "attend", "prefill", "layer", "decode", "accept", "accept",
                       "sample"])
    if kind == "attend" and rng.random() < 0.6:  # verify or decode rows
        batch = _log_int(rng, 1, 64)
        q = rng.choice([1, 2, 3, 4, 5, 6, 9])
        top = max(64, min(8192, 150000 // batch))
        hi = _log_int(rng, 64, top)
        lo = max(q, int(hi * rng.choice([0.05, 0.3, 1.0])))
        return dict(kind=kind, model=rng.choice(["8b", "0.6b"]), batch=batch, q_min=q, q_max=q,
                    k_min=lo, k_max=hi, bound=4096 if hi <= 4096 else 8192,
                    kv=rng.choice(["bf16", "fp8"]))
    if kind == "attend":  # prompts, half of them behind a cached prefix
        batch = _log_int(rng, 1, 8)
        hi = _log_int(rng, 17, 5000 // batch)
        lo = max(1, int(hi * rng.choice([0.1, 0.5, 1.0])))
        prefix = rng.choice([0, 256 * rng.randint(1, 4)])
        return dict(kind=kind, model=rng.choice(["8b", "0.6b"]), batch=batch, q_min=lo, q_max=hi,
                    k_min=0, k_max=prefix, bound=4096 if hi + prefix <= 4096 else 8192,
                    kv=rng.choice(["bf16", "fp8"]))
    if kind == "prefill":
        batch = _log_int(rng, 1, 8)
        hi = _log_int(rng, 17, 5000 // batch)
        return dict(kind=kind, model=rng.choice(["8b", "0.6b"]), batch=batch,
                    q_min=max(1, int(hi * rng.choice([0.1, 0.5, 1.0]))), q_max=hi)
    if kind == "layer":
        batch = _log_int(rng, 1, 16)
        q = rng.choice([1, 2, 4, 6])
        hi = _log_int(rng, 64, 4096)
        return dict(kind=kind, model=rng.choice(["8b", "8b", "0.6b"]), batch=batch, q_min=q,
                    q_max=q, k_min=max(q, int(hi * rng.choice([0.1, 1.0]))), k_max=hi, bound=4096,
                    kv=rng.choice(["bf16", "fp8"]))
    if kind == "decode":
        batch = rng.choice([1, 1, 2, 3, 4, 8])
        q = rng.choice([1, 2]) if batch <= 4 else 1
        hi = _log_int(rng, 33, 4000)
        return dict(kind=kind, model="0.6b", batch=batch, q_min=q, q_max=q,
                    k_min=max(q, int(hi * rng.choice([0.3, 1.0]))), k_max=hi, bound=4096,
                    kv="bf16", layers=rng.randint(2, 6))
    if kind == "accept":
        return dict(kind=kind, batch=_log_int(rng, 1, 200), gamma=rng.choice([1, 2, 3, 3, 5]),
                    logits=rng.choice(["bf16", "bf16", "f32"]),
                    mode=rng.choice(["reference", "reference", "filtered", "filtered", "greedy"]),
                    settings=rng.choice(["plain", "mixed"]))
    return dict(kind=kind, rows=_log_int(rng, 1, 256), logits=rng.choice(["bf16", "bf16", "f32"]),
                mode=rng.choice(["reference", "filtered"]),
                settings=rng.choice(["plain", "mixed"]))


# ---------------------------------------------------------------- shapes of a case

def _lens(case):
    """(query rows, keys) of every sequence: from the case alone, so that inputs of
    another seed are of the same shapes. For prompts (q_max > 16) k_min .. k_max is
    the range of the cached prefix, or equal to the prompt where there is none."""
    rng = random.Random(f"{case['batch']}-{case['q_min']}-{case['q_max']}-{case.get('k_max', 0)}")
    out = []
    for i in range(case["batch"]):
        first = i == 0  # the longest of the range is always there
        q = case["q_max"] if first else rng.randint(case["q_min"], case["q_max"])
        if case["kind"] == "prefill" or case["q_max"] > 16:
            prefix = case.get("k_max", 0)
            out.append((q, q if prefix in (0, q) else q + prefix))
        else:
            k = case["k_max"] if first else rng.randint(case["k_min"], case["k_max"])
            out.append((q, max(q, k)))
    return out


def _cu(values):
    c = [0]
    for v in values:
        c.append(c[-1] + v)
    return c


def _ints(values, dtype=torch.int32):
    return torch.tensor(values, dtype=dtype, device=DEV)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(gen, *shape, dtype=torch.bfloat16, scale=1.0):
    return (torch.randn(*shape, generator=gen, device=DEV, dtype=torch.float32) * scale).to(dtype)


def _paged(case, gen, layers=1):
    """The block pool of a running batch (blocks in no order) and the staging of a step."""
    g = GEOMETRY[case["model"]]
    lens = _lens(case)
    nblk = [-(-k // BLOCK) for _, k in lens]
    pool = sum(nblk) + 2
    perm = torch.randperm(pool, generator=gen, device=DEV).to(torch.int32)
    width = -(-(case["bound"] + 10) // BLOCK)
    tables = torch.full((case["batch"], width), -1, dtype=torch.int32, device=DEV)
    at = 0
    for b, n in enumerate(nblk):
        tables[b, :n] = perm[at:at + n]
        at += n
    pos = torch.cat([torch.arange(k - q, k, device=DEV) for q, k in lens])
    seq = torch.cat([torch.full((q,), b, device=DEV) for b, (q, _) in enumerate(lens)])
    slots = (tables[seq, pos // BLOCK].long() * BLOCK + pos % BLOCK).to(torch.int32)
    fp8 = case["kv"] == "fp8"
    caches = []
    for _ in range(layers):
        kv = []
        for _ in range(2):
            c = torch.empty(pool, BLOCK, g.num_kv_heads, D, device=DEV,
                            dtype=torch.float8_e4m3fn if fp8 else torch.bfloat16)
            for i in range(0, pool, 64):
                x = _normal(gen, *c[i:i + 64].shape, dtype=torch.float32)
                c[i:i + 64] = ((x / KV_SCALE) if fp8 else x).to(c.dtype)
            kv.append(c)
        caches.append(kv)
    return dict(lens=lens, tables=tables, pos=pos, slots=slots, caches=caches,
                cu_q=_ints(_cu([q for q, _ in lens])), cu_k=_ints(_cu([k for _, k in lens])),
                max_q=max(q for q, _ in lens), tokens=sum(q for q, _ in lens))


# per-tensor scale of the FP8 caches: twice the largest normalised key over 448
KV_SCALE = 2.0 * 5.5 / 448.0


def _bind(attn, cache, case):
    attn.k_cache, attn.v_cache = cache
    attn.max_model_len = case["bound"] + case["q_max"] + 2 if case["q_max"] <= 16 else case["bound"]
    if case["kv"] == "fp8":
        attn.kv_cache_dtype = "fp8"
        attn.k_scale = attn.v_scale = KV_SCALE


def _enter(s):
    context.set_context(True, s["cu_q"], s["cu_k"], s["max_q"], 0, s["slots"], None, s["tables"])


def _seen(cache):
    """A cache as it is compared: FP8 codes as bytes."""
    return [c.view(torch.uint8) if c.dtype == torch.float8_e4m3fn else c for c in cache]


# ---------------------------------------------------------------- prepare

def prepare(case, seed):
    with torch.inference_mode():
        return _PREPARE[case["kind"]](case, seed)


def _prepare_attend(case, seed):
    g, gen = GEOMETRY[case["model"]], _gen(seed)
    s = _paged(case, gen)
    s["case"] = case
    s["qkv"] = _normal(gen, s["tokens"], (g.num_heads + 2 * g.num_kv_heads) * D)
    s["q_norm"] = _normal(gen, D, scale=0.1) + 1
    s["k_norm"] = _normal(gen, D, scale=0.1) + 1
    s["rope"] = host.Rope(D, g.max_position, g.rope_theta, DEV)
    s["attn"] = attention.Attention(g.num_heads, D, D ** -0.5, g.num_kv_heads)
    _bind(s["attn"], s["caches"][0], case)
    return s


def _prepare_prefill(case, seed):
    g, gen = GEOMETRY[case["model"]], _gen(seed)
    lens = _lens(case)
    n = sum(q for q, _ in lens)
    cu = _ints(_cu([q for q, _ in lens]))
    return dict(case=case, lens=lens, cu=cu, max_q=max(q for q, _ in lens),
                q=_normal(gen, n, g.num_heads, D), k=_normal(gen, n, g.num_kv_heads, D),
                v=_normal(gen, n, g.num_kv_heads, D),
                attn=attention.Attention(g.num_heads, D, D ** -0.5, g.num_kv_heads))


def _prepare_layer(case, seed):
    g, gen = GEOMETRY[case["model"]], _gen(seed)
    s = _paged(case, gen)
    s["case"] = case
    torch.cuda.manual_seed(seed)
    s["layer"] = host.Qwen3Layer(g, DEV, torch.bfloat16,
                                 host.Rope(D, g.max_position, g.rope_theta, DEV))
    # rows of the embedding the step's tokens come from: a fresh hidden state every pass
    s["embed"] = _normal(gen, 1024, g.hidden)
    s["ids"] = torch.randint(1024, (s["tokens"],), generator=gen, device=DEV)
    _bind(s["layer"].attn, s["caches"][0], case)
    return s


def _prepare_decode(case, seed):
    g, gen = GEOMETRY[case["model"]], _gen(seed)
    s = _paged(case, gen, layers=case["layers"])
    s["case"] = case
    s["model"] = host.Qwen3Host(g, DEV, torch.bfloat16, seed=seed, num_layers=case["layers"])
    s["ids"] = torch.randint(VOCAB, (s["tokens"],), generator=gen, device=DEV)
    for a, c in zip(s["model"].attention_layers(), s["caches"]):
        _bind(a, c, case)

    def step():
        _enter(s)
        h = s["model"](s["ids"], s["pos"])
        context.reset_context()
        return s["model"].compute_logits(h)

    # the runner's own sequence: eager steps, then a captured one that is replayed
    step()
    torch.cuda.synchronize()
    s["graph"] = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        with torch.cuda.graph(s["graph"], stream=side):
            s["logits"] = step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    return s


def _settings(case, n, gen):
    """Temperatures, top-k and top-p of n sequences."""
    if case["settings"] == "mixed":
        t = torch.rand(n, generator=gen, device=DEV) * 0.7 + 0.5
        ks = _ints([0, 20, 50])[torch.randint(3, (n,), generator=gen, device=DEV)]
        ps = torch.tensor([1.0, 0.9, 0.8], device=DEV)[
            torch.randint(3, (n,), generator=gen, device=DEV)]
        return t, ks, ps
    one = torch.ones(n, device=DEV)
    return one * 0.6, _ints([50]).expand(n).contiguous(), one * 0.9


def _filtered(x, k, p):
    """Softmax of one row's x = logits / T over its top-k, then top-p ranks."""
    v, at = torch.sort(x, descending=True, stable=True)
    if 0 < k < v.numel():
        v, at = v[:k], at[:k]
    e = torch.softmax(v, 0)
    if p < 1.0:
        n = max(1, int((torch.cumsum(e, 0) < p).sum()))
        e, at = torch.softmax(v[:n], 0), at[:n]
    out = torch.zeros_like(x)
    out[at] = e
    return out


def _prepare_accept(case, seed):
    gen, B, gamma = _gen(seed), case["batch"], case["gamma"]
    dtype = torch.bfloat16 if case["logits"] == "bf16" else torch.float32
    t, ks, ps = _settings(case, B, gen)
    logits = torch.empty(B, gamma + 1, VOCAB, device=DEV, dtype=dtype)
    probs = torch.empty(B, gamma, VOCAB, device=DEV)
    tokens = torch.empty(B, gamma, dtype=torch.int64, device=DEV)
    kp = list(zip(ks.tolist(), ps.tolist()))
    for b in range(B):
        # logits of spread 2, the draft's those and noise of spread 1
        x = torch.randn(gamma + 1, VOCAB, generator=gen, device=DEV) * 2
        logits[b] = x.to(dtype)
        y = x[:gamma] + torch.randn(gamma, VOCAB, generator=gen, device=DEV)
        y = y.to(dtype).float() / t[b]
        if case["mode"] == "filtered":
            for j in range(gamma):
                probs[b, j] = _filtered(y[j], *kp[b])
        else:
            probs[b] = torch.softmax(y, -1)
        tokens[b] = torch.multinomial(probs[b], 1, generator=gen).flatten()
    return dict(case=case, logits=logits, probs=probs, tokens=tokens, t=t, ks=ks, ps=ps,
                u_acc=torch.rand(B, gamma, generator=gen, device=DEV),
                u_res=torch.rand(B, generator=gen, device=DEV))


def _prepare_sample(case, seed):
    gen, n = _gen(seed), case["rows"]
    dtype = torch.bfloat16 if case["logits"] == "bf16" else torch.float32
    t, ks, ps = _settings(case, n, gen)
    return dict(case=case, logits=_normal(gen, n, VOCAB, dtype=dtype, scale=2.0), t=t, ks=ks,
                ps=ps, u=torch.rand(n, generator=gen, device=DEV))


_PREPARE = dict(attend=_prepare_attend, prefill=_prepare_prefill, layer=_prepare_layer,
                decode=_prepare_decode, accept=_prepare_accept, sample=_prepare_sample)


# ---------------------------------------------------------------- run

@torch.inference_mode()
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "attend":
        _enter(s)
        out = s["attn"].attend_qkv(s["qkv"], s["q_norm"], s["k_norm"], s["rope"].cos_sin,
                                   s["pos"], EPS)
        context.reset_context()
        return [out] + _seen(s["caches"][0])
    if kind == "prefill":
        context.set_context(True, s["cu"], s["cu"], s["max_q"], s["max_q"])
        out = s["attn"](s["q"], s["k"], s["v"])
        context.reset_context()
        return out
    if kind == "layer":
        h = F.embedding(s["ids"], s["embed"])
        _enter(s)
        h, residual = s["layer"](s["pos"], h, None)
        context.reset_context()
        return [h, residual] + _seen(s["caches"][0])
    if kind == "decode":
        s["graph"].replay()
        return s["logits"]
    if kind == "accept":
        topk = case["mode"] == "filtered" and case["settings"] == "plain"
        return list(ops.spec_accept(
            s["logits"], s["probs"], s["tokens"], s["t"], s["u_acc"], s["u_res"],
            mode=case["mode"], top_ks=s["ks"], top_ps=s["ps"], topk_le64=topk))
    r = ops.sample_rows(s["logits"], s["t"], s["ks"], s["ps"], mode=case["mode"],
                        uniforms=s["u"], want_probs=True)
    return [r["probs"], r["tokens"]]


# ---------------------------------------------------------------- work

def _attention_work(case):
    g = GEOMETRY[case["model"]]
    size = 1 if case.get("kv") == "fp8" else 2
    q = sum(a for a, _ in _lens(case))
    keys = sum(k for _, k in _lens(case))
    pairs = sum(a * (k - a) + a * (a + 1) // 2 for a, k in _lens(case))
    row = g.num_kv_heads * D
    # the cached keys and values read (the step's own come with its rows), the q / k / v
    # rows read, the attention's rows written
    nbytes = 2 * (keys - q) * row * size + q * (g.num_heads + 2 * row // D) * D * 2
    nbytes += q * g.num_heads * D * 2
    if case["kind"] != "prefill":
        nbytes += 2 * q * row * size  # the new keys and values stored
    return nbytes, 4 * pairs * g.num_heads * D


def work(case):
    kind = case["kind"]
    if kind in ("attend", "prefill"):
        nbytes, flops = _attention_work(case)
        return {"bytes": nbytes, "flops": flops}
    if kind in ("layer", "decode"):
        g = GEOMETRY[case["model"]]
        rows = sum(q for q, _ in _lens(case))
        weights = g.hidden * (g.num_heads + 2 * g.num_kv_heads) * D
        weights += g.hidden * g.num_heads * D + 3 * g.hidden * g.ffn
        keys, flops = _attention_work(case)
        # the layer's activations between its calls can stay on the chip
        nbytes = 2 * weights + keys - rows * (2 * g.num_heads + 2 * g.num_kv_heads) * D * 2
        flops += 2 * rows * weights
        if kind == "layer":
            return {"bytes": nbytes + 3 * rows * g.hidden * 2, "flops": flops}
        head = g.vocab * g.hidden
        return {"bytes": case["layers"] * nbytes + 2 * head + rows * (g.hidden + g.vocab) * 2,
                "flops": case["layers"] * flops + 2 * rows * head}
    size = 2 if case["logits"] == "bf16" else 4
    if kind == "accept":
        n = case["batch"]
        target = n * (case["gamma"] + 1) * VOCAB * size
        if case["mode"] == "greedy":
            return {"bytes": target, "flops": 0}
        # the row of draft probabilities that a resample subtracts
        return {"bytes": target + n * VOCAB * 4, "flops": 0}
    return {"bytes": case["rows"] * VOCAB * (size + 4), "flops": 0}


# ---------------------------------------------------------------- tolerance

def tolerance(case):
    # about four times what the path measures against exact() (rel): bf16 inputs,
    # probabilities and outputs; an FP8 code may move by its rounding
    kind = case["kind"]
    if kind == "attend":
        return {"rel": 1.4e-2, "differ": 1e-3}
    if kind == "prefill":
        return {"rel": 8e-3}
    if kind == "layer":
        return {"rel": 1.8e-2, "differ": 1e-3}
    if kind == "decode":
        return {"rel": 3e-2}
    if kind == "accept":
        return "exact"  # counts and tokens on given uniforms
    return {"rel": 1.2e-6, "differ": 0.0}  # f32 probabilities; the tokens as they are


# ---------------------------------------------------------------- exact

def exact(case, seed):
    if case["kind"] == "accept":
        return None  # whole numbers
    s = prepare(case, seed)
    with torch.inference_mode():
        return _EXACT[case["kind"]](case, s)


def _softmax_attention(q, k, v, lens, out):
    """q [N, Hq, D], k / v lists per sequence [Lk, Hkv, D], float64, bottom-right causal."""
    at = 0
    for b, (nq, nk) in enumerate(lens):
        mask = (torch.arange(nk, device=DEV)[None, :]
                > torch.arange(nk - nq, nk, device=DEV)[:, None])
        rep = q.shape[1] // k[b].shape[1]
        for h in range(q.shape[1]):
            x = q[at:at + nq, h] @ k[b][:, h // rep].T * D ** -0.5
            x = torch.softmax(x.masked_fill(mask, float("-inf")), -1)
            out[at:at + nq, h] = x @ v[b][:, h // rep]
        at += nq
    return out


def _norm64(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x, pos, g):
    inv = g.rope_theta ** (-torch.arange(0, D, 2, device=DEV, dtype=torch.float64) / D)
    a = pos.double()[:, None, None] * inv
    x1, x2 = x.chunk(2, -1)
    return torch.cat([x1 * a.cos() - x2 * a.sin(), x2 * a.cos() + x1 * a.sin()], -1)


def _attend64(s, case, qkv, q_norm, k_norm, cache):
    g = GEOMETRY[case["model"]]
    nq, nk = g.num_heads * D, g.num_kv_heads * D
    q, k, v = qkv.double().split([nq, nk, nk], -1)
    q = _rope64(_norm64(q.reshape(-1, g.num_heads, D), q_norm), s["pos"], g)
    k = _rope64(_norm64(k.reshape(-1, g.num_kv_heads, D), k_norm), s["pos"], g)
    v = v.reshape(-1, g.num_kv_heads, D)
    scale = KV_SCALE if case["kv"] == "fp8" else 1.0
    if case["kv"] == "fp8":  # what the cache holds is what is attended to
        k, v = ((x / scale).float().to(torch.float8_e4m3fn).double() * scale for x in (k, v))
    ks, vs, at = [], [], 0
    for b, (a, n) in enumerate(s["lens"]):
        blocks = s["tables"][b, :-(-n // BLOCK)].long()
        for c, new, to in ((cache[0], k, ks), (cache[1], v, vs)):
            old = c[blocks].reshape(-1, g.num_kv_heads, D)[:n - a].float().double() * scale
            to.append(torch.cat([old, new[at:at + a]]))
        at += a
    return _softmax_attention(q, ks, vs, s["lens"], torch.empty_like(q))


def _exact_attend(case, s):
    return [_attend64(s, case, s["qkv"], s["q_norm"], s["k_norm"], s["caches"][0]), None, None]


def _exact_prefill(case, s):
    at = _cu([q for q, _ in s["lens"]])
    ks, vs = ([x[a:b].double() for a, b in zip(at, at[1:])] for x in (s["k"], s["v"]))
    q = s["q"].double()
    return _softmax_attention(q, ks, vs, s["lens"], torch.empty_like(q))


def _layer64(case, s, layer, h, residual, cache):
    residual = h if residual is None else residual + h
    o = _attend64(s, case, _norm64(residual, layer.ln1) @ layer.qkv.double().T, layer.q_norm,
                  layer.k_norm, cache)
    residual = residual + o.reshape(o.shape[0], -1) @ layer.o.double().T
    gate, up = (_norm64(residual, layer.ln2) @ layer.gate_up.double().T).chunk(2, -1)
    return (F.silu(gate) * up) @ layer.down.double().T, residual


def _exact_layer(case, s):
    h = F.embedding(s["ids"], s["embed"]).double()
    h, residual = _layer64(case, s, s["layer"], h, None, s["caches"][0])
    return [h, residual, None, None]


def _exact_decode(case, s):
    m = s["model"]
    h, residual = F.embedding(s["ids"], m.embed).double(), None
    for layer, cache in zip(m.layers, s["caches"]):
        h, residual = _layer64(case, s, layer, h, residual, cache)
    h = _norm64(residual + h, m.norm)
    return torch.cat([h @ w.double().T for w in m.lm_head.split(16384)], -1)


def _exact_sample(case, s):
    x = s["logits"].double() / s["t"].double()[:, None]
    if case["mode"] != "filtered":
        return [torch.softmax(x, -1), None]
    rows = [_filtered(r, k, p) for r, k, p in zip(x, s["ks"].tolist(), s["ps"].tolist())]
    return [torch.stack(rows), None]


_EXACT = dict(attend=_exact_attend, prefill=_exact_prefill, layer=_exact_layer,
              decode=_exact_decode, sample=_exact_sample)
