"""What the framework is timed on, from one small compression call to a mixture of experts over 16 384 prompt
tokens.  Every case goes through an entry point that an engine or a model calls once per step:

  compress    compress_layers: one chunk of layers of the KV compression (score, select, compact in place)
  prefill     Qwen3.forward and compute_logits over whole prompts of several requests
  decode      the same over one token per request, keys and values in pages
  attention   GroupedAttention.attend: the attention of a hybrid layer, prompts in runs or decoded tokens
  latent      LatentAttention.forward and the residual step behind it
  recurrent   the scan of a recurrent mixer (delta rule, matrix memory, linear attention, retention)
  experts     Experts.forward and the residual step behind it

Sizes are those of the repository's benchmark: Qwen3-8B and Qwen3-0.6B attention (32 or 16 query heads over 8 key
heads of 128), windows of 16 and 32 queries, a budget of 8 pages of 256 tokens, and the "1k" and "4k" widths of the
model comparison.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch
import torch.nn.functional as F

DEV = "cuda:0"
PAGE = 256
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one sequence reached its budget, one layer, fp32: latency and launches count
        _compress("compress-one", dtype="fp32", batch=1, heads=16, window=32, pool=7),
        # 64 sequences with the switches of the reference's scripts: window 16, carried scores, lightning redundancy
        _compress("compress-64-scripts", batch=64, window=16, pool=5, carry=True, redundancy="lightning"),
        # the headline: 256 ragged sequences, groups of 16 share two prefix pages that are copied on write
        _compress("compress-256-shared", batch=256, window=32, pool=7, most_pages=10, share=16),
        # 128 sequences in fp32, carried scores added up, lightning redundancy, average pooling at every compression
        _compress("compress-128-fp32", dtype="fp32", batch=128, heads=16, window=32, pool=7, mode="avg", carry=True,
                  redundancy="lightning"),
        # prompts of different lengths in one step, as requests arrive
        dict(name="qwen3-prefill-ragged", kind="prefill", width=4096, heads=32, ff=12288, layers=2, requests=16, shortest=256,
             longest=768),
        # one decode step in the steady state of a compressed cache
        dict(name="qwen3-decode-256", kind="decode", width=4096, heads=32, ff=12288, layers=2, requests=256, shortest=2049,
             longest=2304),
        # a prompt step of a hybrid model's window layer whose values turn
        dict(name="attention-window-prefill", kind="attention", phase="prefill", heads=32, kv_heads=8, dim=128, sight="window",
             reach=1024, sinks=False, turning=True, requests=8, shortest=2048, longest=2048),
        # decoded tokens over shared latents with a rotated key part
        dict(name="latent-decode-256", kind="latent", phase="decode", width=4096, heads=32, dim=128, q_rank=1536, kv_rank=512,
             rot=64, window=0, requests=256, shortest=1800, longest=2304),
        # prompts through the gated delta rule
        dict(name="delta-prefill", kind="recurrent", mixer="delta", phase="prefill", width=4096, heads=32, dim=128, requests=8,
             shortest=2048, longest=2048),
        # decoded tokens through linear attention with a decay per key channel
        dict(name="linear-decode-256", kind="recurrent", mixer="linear", phase="decode", width=4096, heads=32, dim=128,
             requests=256, shortest=1, longest=1),
        # a full prompt step of the mixture of experts
        dict(name="experts-prefill", kind="experts", tokens=16384, width=4096, ff=3072, experts=32, top=3, groups=4, keep=2,
             shared=True, score="softmax", act="clamped"),
        # and a decode step, which reads nearly every expert for a few rows
        dict(name="experts-decode-64", kind="experts", tokens=64, width=4096, ff=3072, experts=32, top=3, groups=4, keep=2,
             shared=True, score="softmax", act="clamped"),
    ]


def _compress(name, dtype="bf16", layers=1, batch=64, heads=32, window=32, pool=7, mode="max", carry=False, redundancy="none",
              most_pages=9, share=0):
    c = dict(kind="compress", dtype=dtype, layers=layers, batch=batch, heads=heads, window=window, pool=pool, mode=mode,
             carry=carry, redundancy=redundancy, most_pages=most_pages, share=share)
    return dict(name=name, **c) if name else c


def draw(rng):
    spread = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    kind = rng.choice(["compress"] * 4 + ["prefill", "decode", "attention", "latent", "recurrent", "recurrent", "experts", "experts"])
    if kind == "compress":
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
        redundancy = rng.choice(["none", "none", "lightning", "raw"])
        batch = spread(1, 48 if redundancy == "raw" else 256)
        layers = rng.choice([n for n in (1, 2, 4, 8) if n * batch <= (48 if redundancy == "raw" else 256)])
        return _compress(None, dtype=dtype, layers=layers, batch=batch, heads=rng.choice([16, 32]), window=rng.choice([16, 32]),
                         pool=rng.choice([3, 5, 7]), mode=rng.choice(["max", "max", "avg"]), carry=rng.random() < 0.4,
                         redundancy=redundancy, most_pages=rng.choice([9, 10]),
                         share=16 if batch >= 16 and rng.random() < 0.3 else 0)
    wide = rng.random() < 0.5
    width, heads = (4096, 32) if wide else (1024, 16)
    if kind in ("prefill", "decode"):
        # up to the listed case's tokens; a decode step of a few requests too
        requests = spread(1, 16) if kind == "prefill" else spread(8, 256)
        lo, hi = sorted(rng.sample(range(64, 1024), 2)) if kind == "prefill" else sorted(rng.sample(range(300, 2304), 2))
        return dict(kind=kind, width=width, heads=heads, ff=3 * width, layers=2, requests=requests, shortest=lo, longest=hi)
    if kind == "attention":
        phase = rng.choice(["prefill", "decode"])
        sight = rng.choice(["window", "chunk", "all"])
        turning = sight == "window" and rng.random() < 0.5
        requests = spread(1, 8) if phase == "prefill" else spread(8, 256)
        lo, hi = sorted(rng.sample(range(100, 2049), 2))
        return dict(kind=kind, phase=phase, heads=heads, kv_heads=8, dim=rng.choice([64, 128, 128]), sight=sight,
                    reach=0 if sight == "all" else rng.choice([512, 1024]), sinks=not turning and rng.random() < 0.5,
                    turning=turning, requests=requests, shortest=lo, longest=hi)
    if kind == "latent":
        phase = rng.choice(["prefill", "decode"])
        window = rng.choice([0, 1024])
        requests = spread(1, 8) if phase == "prefill" else spread(8, 256)
        lo, hi = sorted(rng.sample(range(100, 2049), 2))
        return dict(kind=kind, phase=phase, width=width, heads=heads, dim=128, q_rank=1536 if wide else 512,
                    kv_rank=512 if wide else 256, rot=0 if window else 64, window=window, requests=requests, shortest=lo,
                    longest=hi)
    if kind == "recurrent":
        phase = rng.choice(["prefill", "decode"])
        mixer = rng.choice(["delta", "memory", "linear", "retention"])
        requests = spread(1, 8) if phase == "prefill" else spread(16, 256)
        lo, hi = sorted(rng.sample(range(100, 2049), 2)) if phase == "prefill" else (1, 1)
        return dict(kind=kind, mixer=mixer, phase=phase, width=width, heads=heads // 2 if mixer in ("memory", "retention") else heads,
                    dim=128, requests=requests, shortest=lo, longest=hi)
    top = rng.choice([3, 4])
    return dict(kind=kind, tokens=spread(1, 16384), width=width, ff=width * 3 // 4, experts=32, top=top,
                groups=4 if top == 3 else 1, keep=2 if top == 3 else 1, shared=top == 3,
                score="softmax" if top == 3 else "sigmoid", act="clamped" if top == 3 else "silu")


# ---------------------------------------------------------------- inputs
class _Draw:
    """Tensors and numbers from one seed."""

    def __init__(self, seed):
        self.dev = torch.Generator(device=DEV).manual_seed(seed)
        self.cpu = torch.Generator().manual_seed(seed)

    def normal(self, *shape, dtype=torch.bfloat16, std=1.0, mean=0.0):
        return torch.empty(*shape, dtype=dtype, device=DEV).normal_(mean, std, generator=self.dev)

    def uniform(self, *shape, lo=0.0, hi=1.0, dtype=torch.float32):
        return torch.empty(*shape, dtype=torch.float32, device=DEV).uniform_(lo, hi, generator=self.dev).to(dtype)

    def integers(self, lo, hi, n):
        """n of lo .. hi, both included."""
        return torch.randint(lo, hi + 1, (n,), generator=self.cpu).tolist()

    def order(self, n):
        return torch.randperm(n, generator=self.cpu).tolist()


def _i32(a):
    return torch.as_tensor(a, dtype=torch.int32, device=DEV)


def prepare(case, seed):
    with torch.inference_mode():
        return globals()["_prepare_" + case["kind"]](case, _Draw(seed), seed)


def run(state):
    with torch.inference_mode():
        return globals()["_run_" + state.kind](state)


def work(case):
    return globals()["_work_" + case["kind"]](case)


def exact(case, seed):
    if case["kind"] == "compress":
        return None                       # flags, and copies of cached rows: no value is computed but compared
    with torch.inference_mode():
        return globals()["_exact_" + case["kind"]](case, prepare(case, seed))


def tolerance(case):
    if case["kind"] == "compress":
        return "exact"                    # kept indices and compacted keys and values are bit-exact
    return TOLERANCE[case["kind"]]


# four times what the path is off its 64-bit value (16-bit weights, caches and activations; sums in 32 bits)
TOLERANCE = {
    "prefill": {"rel": 0.03, "max": 0.5},
    "decode": {"rel": 0.03, "max": 0.9},      # the query ring is mostly empty, so its root mean square is small
    "attention": {"rel": 0.012, "max": 0.3},
    "latent": {"rel": 0.009, "max": 0.05},
    "recurrent": {"rel": 0.007, "max": 0.08},
    "experts": {"rel": 0.01, "max": 0.07},
}


def _lengths(lo, hi, n, d):
    """n lengths of lo .. hi that belong to the case, in an order that belongs to the seed."""
    lens = torch.randint(lo, hi + 1, (n,), generator=torch.Generator().manual_seed(n * 4099 + hi)).tolist()
    return [lens[i] for i in d.order(n)]


def _case_lengths(case, d):
    return _lengths(case["shortest"], case["longest"], case["requests"], d)


def _mean_lengths(case, f=lambda n: n):
    lo, hi = case["shortest"], case["longest"]
    return case["requests"] * sum(f(n) for n in (lo, (lo + hi) // 2, hi)) / 3


# ---------------------------------------------------------------- compress
BUDGET = 8         # pages that survive
REFILLS = 8        # last pages per sequence, taken in turn: a decode fills the page between two compressions


def _prepare_compress(c, d, seed):
    from zipage_amd.compress import CompressConfig
    B, L, G, D, dt = c["batch"], c["layers"], 8, 128, DTYPES[c["dtype"]]
    pages = [-(-n // PAGE) for n in _lengths(BUDGET * PAGE + 1, c["most_pages"] * PAGE, B, d)]
    pool = sum(pages) + (REFILLS - 1 + (2 if c["share"] else 0)) * B
    free = iter(d.order(pool))
    take = lambda n: [next(free) for _ in range(n)]
    tables, targets = [], []
    for b in range(B):
        if c["share"]:
            if b % c["share"] == 0:
                prefix = take(2)
            t = prefix + take(pages[b] - 2)
            targets.append(take(2) + t[2:BUDGET + 1])
        else:
            t = take(pages[b])
            targets.append(t[:BUDGET + 1])
        tables.append(t)
    width = max(pages)
    encode = lambda t: t[:-1] + [-t[-1] - 2] + [-1] * (width - len(t))
    steps = []
    for r in range(REFILLS):
        if r:
            fresh = take(B)
            swap = lambda row, t, f: [f if p == t[-1] else p for p in row]
            now = [t[:-1] + [f] for t, f in zip(tables, fresh)]
            goal = [swap(row, t, f) for row, t, f in zip(targets, tables, fresh)]
        else:
            now, goal = tables, targets
        steps.append((_i32([encode(t) for t in now]), _i32(goal)))
    kv = d.normal(2, L, pool, PAGE, G, D, dtype=dt)
    cfg = CompressConfig(budget_blocks=BUDGET, query_cache_len=c["window"], enable_pooling=True, pooling_size=c["pool"],
                         pooling_mode=c["mode"], continues_pooling=c["mode"] == "avg", use_global_score=c["carry"],
                         decay_factor=0.9 if c["mode"] == "avg" else 0.8, activate_method="sum" if c["mode"] == "avg" else "max",
                         use_redudancy=c["redundancy"] != "none", lightning_redudancy=c["redundancy"] == "lightning")
    return SimpleNamespace(kind="compress", cfg=cfg, k=kv[0], v=kv[1], q=d.normal(L, B, c["window"], c["heads"], D, dtype=dt),
                           scores=d.uniform(L, pool, PAGE, G, dtype=dt) if c["carry"] else None, rows=_i32(list(range(B))),
                           again=torch.full((B,), c["carry"], device=DEV), steps=steps, at=0)


def _run_compress(s):
    from zipage_amd.compress import compress_layers
    tables, targets = s.steps[s.at]
    s.at = (s.at + 1) % len(s.steps)
    keep = compress_layers(s.k, s.v, s.q, s.scores, s.rows, tables, s.again, targets, s.cfg)
    return [keep, s.k, s.v] + ([] if s.scores is None else [s.scores])


def _work_compress(c):
    es, G, D = 4 if c["dtype"] == "fp32" else 2, 8, 128
    units, tokens = c["layers"] * c["batch"], (BUDGET + c["most_pages"] + 1) / 2 * PAGE
    b = tokens * G * D * es + c["window"] * c["heads"] * D * es + 4 * BUDGET * PAGE * G * D * es + tokens * G
    f = 2 * c["heads"] * c["window"] * tokens * D
    if c["carry"]:
        b += (tokens + BUDGET * PAGE) * G * es
    if c["redundancy"] == "lightning":
        f += tokens * PAGE * D * G
    if c["redundancy"] == "raw":
        f += tokens * tokens * D * G
    return {"bytes": units * b, "flops": units * f}


# ---------------------------------------------------------------- Qwen3 steps
VOCAB, WINDOW = 32768, 16


def _qwen3(c, seed):
    from zipage_amd.engine import Qwen3Shape
    from zipage_amd.engine.qwen3 import Qwen3
    return Qwen3(Qwen3Shape(c["layers"], c["width"], c["heads"], 8, 128, c["ff"], VOCAB, max_position=8192), DEV, seed=seed)


def _tables(lens, d):
    """Pages of sequences of `lens` tokens, drawn from a pool that just holds them: tables, pool size."""
    order = iter(d.order(sum(-(-n // PAGE) for n in lens)))
    tables = [[next(order) for _ in range(-(-n // PAGE))] for n in lens]
    return tables, sum(map(len, tables))


def _slots(table, lo, hi):
    return [table[t // PAGE] * PAGE + t % PAGE for t in range(lo, hi)]


def _padded(tables):
    w = max(map(len, tables))
    return _i32([t + [-1] * (w - len(t)) for t in tables])


def _prepare_prefill(c, d, seed):
    from zipage_amd.engine.qwen3 import StepContext
    m, lens = _qwen3(c, seed), _case_lengths(c, d)
    tables, pool = _tables(lens, d)
    m.attach_caches(torch.zeros(2, c["layers"], pool, PAGE, 8, 128, dtype=torch.bfloat16, device=DEV),
                    torch.zeros(c["layers"], len(lens), WINDOW, c["heads"], 128, dtype=torch.bfloat16, device=DEV))
    triples, at = [], 0
    for i, n in enumerate(lens):                      # tokens in the last WINDOW places of their prompt's last page
        full = -(-n // PAGE) * PAGE - WINDOW
        triples += [(at + p, i, p - full) for p in range(full, n)]
        at += n
    ctx = StepContext(True, _i32([s for t, n in zip(tables, lens) for s in _slots(t, 0, n)]),
                      _i32(triples) if triples else None, None, None, list(lens), list(lens))
    ids = torch.tensor(d.integers(0, VOCAB - 1, sum(lens)), device=DEV)
    return SimpleNamespace(kind="prefill", m=m, lens=lens, ids=ids, ctx=ctx, triples=triples,
                           pos=torch.tensor([p for n in lens for p in range(n)], device=DEV),
                           ends=torch.tensor(lens, device=DEV).cumsum(0) - 1)


def _run_prefill(s):
    hidden = s.m.forward(s.ids, s.pos, s.ctx)
    return [s.m.compute_logits(hidden[s.ends]), s.m.k_cache, s.m.v_cache, s.m.q_cache]


def _prepare_decode(c, d, seed):
    from zipage_amd.engine.qwen3 import StepContext
    m, lens = _qwen3(c, seed), _case_lengths(c, d)
    tables, pool = _tables(lens, d)
    m.attach_caches(d.normal(2, c["layers"], pool, PAGE, 8, 128),
                    torch.zeros(c["layers"], len(lens), WINDOW, c["heads"], 128, dtype=torch.bfloat16, device=DEV))
    last = [(n - 1) % PAGE - (PAGE - WINDOW) for n in lens]
    ctx = StepContext(False, _i32([_slots(t, n - 1, n)[0] for t, n in zip(tables, lens)]),
                      _i32([(i, i, w) if w >= 0 else (-1, i, -1) for i, w in enumerate(last)]), _i32(lens), _padded(tables))
    return SimpleNamespace(kind="decode", m=m, lens=lens, tables=tables, last=last, ctx=ctx,
                           ids=torch.tensor(d.integers(0, VOCAB - 1, len(lens)), device=DEV),
                           pos=torch.tensor([n - 1 for n in lens], device=DEV))


def _run_decode(s):
    return [s.m.compute_logits(s.m.forward(s.ids, s.pos, s.ctx)), s.m.k_cache, s.m.v_cache, s.m.q_cache]


def _qwen3_weights(c):
    W, H, ff = c["width"], c["heads"], c["ff"]
    return c["layers"] * (W * (H + 16) * 128 + H * 128 * W + 3 * W * ff), VOCAB * W


def _work_prefill(c):
    layers, head = _qwen3_weights(c)
    n, pairs = _mean_lengths(c), _mean_lengths(c, lambda n: n * (n + 1) / 2)
    return {"bytes": 2 * (layers + head + n * c["layers"] * 16 * 128 + c["requests"] * VOCAB),
            "flops": 2 * n * layers + 2 * c["requests"] * head + 4 * pairs * c["heads"] * 128 * c["layers"]}


def _work_decode(c):
    layers, head = _qwen3_weights(c)
    n, B = _mean_lengths(c), c["requests"]
    return {"bytes": 2 * (layers + head + n * c["layers"] * 16 * 128 + B * VOCAB),
            "flops": 2 * B * (layers + head) + 4 * n * c["heads"] * 128 * c["layers"]}


def _rms(x, eps, n=None):
    return x / torch.sqrt((x * x).sum(-1, keepdim=True) / (n or x.shape[-1]) + eps)


def _angles(pos, freqs):
    return pos.double()[:, None] * freqs.double()[None]


def _turn(x, a, pairs="halves", back=False):
    """x (n, heads, dim): pairs of its first 2 a.shape[1] elements turn by the angles a (n, pairs)."""
    h = a.shape[1]
    c, s = a.cos()[:, None], (-a.sin() if back else a.sin())[:, None]
    out = x.clone()
    one, two = (slice(0, h), slice(h, 2 * h)) if pairs == "halves" else (slice(0, 2 * h, 2), slice(1, 2 * h, 2))
    out[..., one] = x[..., one] * c - x[..., two] * s
    out[..., two] = x[..., two] * c + x[..., one] * s
    return out


def _attend(q, k, v, scale, q_from=0, window=0, chunk=0, sinks=None):
    """q (n, H, D) at positions q_from .., k (T, G, D), v (T, G, V) -> (n, H, V)."""
    n, H, _ = q.shape
    T, G, V = v.shape
    i = torch.arange(q_from, q_from + n, device=q.device)[:, None]
    j = torch.arange(T, device=q.device)[None]
    hidden = (j > i) | ((j <= i - window) if window else False) | ((j // chunk != i // chunk) if chunk else False)
    s = torch.matmul(q.view(n, G, H // G, -1).permute(1, 2, 0, 3), k.permute(1, 2, 0).contiguous().unsqueeze(1)) * scale
    s = s.masked_fill(hidden, -math.inf)
    if sinks is not None:
        s = torch.cat([s, sinks.double().view(G, H // G, 1, 1).expand(-1, -1, n, 1)], -1)
    p = torch.softmax(s, -1)[..., :T]
    return torch.matmul(p, v.permute(1, 0, 2).contiguous().unsqueeze(1)).permute(2, 0, 1, 3).reshape(n, H, V)


def _exact_qwen3(c, s, attend):
    m, sh = s.m, s.m.shape
    w = lambda t: t.double()
    inv = sh.rope_theta ** (-torch.arange(0, 128, 2, dtype=torch.float64, device=DEV) / 128)
    a = _angles(s.pos, inv)
    x = w(m.embed)[s.ids]
    n, H = x.shape[0], sh.heads
    k_cache, v_cache, q_cache = w(m.k_cache), w(m.v_cache), w(m.q_cache)
    for li, p in enumerate(m.layers):
        qkv = (_rms(x, sh.eps) * w(p["ln1"])) @ w(p["wqkv"]).T
        q, k, v = qkv.view(n, H + 16, 128).split([H, 8, 8], 1)
        q, k = _turn(_rms(q, sh.eps) * w(p["qn"]), a), _turn(_rms(k, sh.eps) * w(p["kn"]), a)
        slots = s.ctx.slot_mapping.long()
        k_cache[li].view(-1, 8, 128)[slots] = k
        v_cache[li].view(-1, 8, 128)[slots] = v
        x = x + attend(li, q, k, v, k_cache[li], v_cache[li], q_cache[li]).reshape(n, -1) @ w(p["wo"]).T
        g, u = ((_rms(x, sh.eps) * w(p["ln2"])) @ w(p["wgu"]).T).chunk(2, -1)
        x = x + (F.silu(g) * u) @ w(p["wd"]).T
    return _rms(x, sh.eps) * w(m.final_norm), [k_cache, v_cache, q_cache]


def _exact_prefill(c, s):
    def attend(li, q, k, v, kc, vc, qc):
        for row, i, at in s.triples:
            qc[i, at] = q[row]
        parts = [t.split(s.lens) for t in (q, k, v)]
        return torch.cat([_attend(*p, 128 ** -0.5) for p in zip(*parts)])
    hidden, caches = _exact_qwen3(c, s, attend)
    return [hidden[s.ends] @ s.m.lm_head.double().T, *caches]


def _exact_decode(c, s):
    def attend(li, q, k, v, kc, vc, qc):
        out = torch.empty_like(q)
        for i, (t, n) in enumerate(zip(s.tables, s.lens)):
            if s.last[i] >= 0:
                qc[i, s.last[i]] = q[i]
            rows = lambda cache: cache[t].reshape(-1, 8, 128)[:n]
            out[i] = _attend(q[i:i + 1], rows(kc), rows(vc), 128 ** -0.5, n - 1)[0]
        return out
    hidden, caches = _exact_qwen3(c, s, attend)
    return [hidden @ s.m.lm_head.double().T, *caches]


# ---------------------------------------------------------------- steps of portions
def _context(c, lens, tables, sight):
    """What the engine hands a mixer: whole prompts as runs, or one token per sequence."""
    from zipage_amd.engine.inputs import plan_runs
    from zipage_amd.engine.qwen3 import Segments, StepContext
    from zipage_amd.engine.sequence import Portion, Sequence
    n, B = len(lens), _i32(list(range(len(lens))))
    if c["phase"] == "decode":
        return StepContext(False, _i32([_slots(t, m - 1, m)[0] for t, m in zip(tables, lens)]), None, _i32(lens), _padded(tables),
                           table_rows=B, runs={}, segments=Segments(B, _i32([1] * n), B, _i32([m - 1 for m in lens]), max_count=1))
    portions = []
    for t, m in zip(tables, lens):
        seq = Sequence([0] * m)
        seq.block_table = t
        portions.append(Portion(seq, 0, m))
    plan = plan_runs(portions, PAGE, sight)
    plan.tiles = _i32(plan.tiles)
    first = [sum(lens[:i]) for i in range(n)]
    return StepContext(False, _i32([x for t, m in zip(tables, lens) for x in _slots(t, 0, m)]), None, _i32([]), _padded(tables),
                       table_rows=_i32([]), runs={sight: plan},
                       run_segments=Segments(_i32(first), _i32(lens), B, _i32([0] * n), longest=max(lens)))


def _positions(c, lens):
    return _i32([n - 1 for n in lens] if c["phase"] == "decode" else [p for n in lens for p in range(n)])


def _seen(n, window, chunk):
    """Keys the token at place n - 1 sees."""
    return min(n, window) if window else (n - 1) % chunk + 1 if chunk else n


# ---------------------------------------------------------------- grouped attention
def _prepare_attention(c, d, seed):
    from zipage_amd.layers import GroupedAttention, Rotary
    from zipage_amd.sight import Chunk
    H, G, D = c["heads"], c["kv_heads"], c["dim"]
    sight = {"window": c["reach"], "chunk": Chunk(c["reach"]), "all": None}[c["sight"]]
    # rotary pairs as neighbours where values turn, which the layer puts in its own order at load
    m = GroupedAttention(32, H, G, D, D, D ** -0.5, sight, Rotary(5e5, D, interleaved=c["turning"]), sinks=c["sinks"],
                         turn_values=c["turning"])
    w = {k: d.normal(*s, std=0.02) for k, s in m.shapes().items()}
    if c["sinks"]:
        w["sink"] = d.normal(H, dtype=torch.float32)
    m.load(w, torch.bfloat16, DEV, 32)
    lens = _case_lengths(c, d)
    tables, pool = _tables(lens, d)
    rows = len(lens) if c["phase"] == "decode" else sum(lens)
    cache = m.allocate(pool, PAGE, torch.bfloat16, DEV)
    if c["phase"] == "decode":
        cache.normal_(generator=d.dev)
    return SimpleNamespace(kind="attention", m=m, lens=lens, tables=tables, cache=cache, ctx=_context(c, lens, tables, sight),
                           pos=_positions(c, lens), proj=d.normal(rows, m.columns),
                           out=torch.empty(rows, m.out_columns, dtype=torch.bfloat16, device=DEV))


def _run_attention(s):
    s.m.attend(s.proj, s.pos, s.cache, s.ctx, s.out)
    return [s.out, s.cache]


def _limits(c):
    return c["reach"] if c["sight"] == "window" else 0, c["reach"] if c["sight"] == "chunk" else 0


def _work_attention(c):
    H, G, D, lim = c["heads"], c["kv_heads"], c["dim"], _limits(c)
    if c["phase"] == "decode":
        seen = _mean_lengths(c, lambda n: _seen(n, *lim))
        return {"bytes": 2 * (seen * 2 * G * D + c["requests"] * (2 * H + 4 * G) * D), "flops": 4 * seen * H * D}
    n, pairs = _mean_lengths(c), _mean_lengths(c, lambda n: sum(_seen(i + 1, *lim) for i in range(n)))
    return {"bytes": 2 * n * (2 * H + 4 * G) * D, "flops": 4 * pairs * H * D}


def _exact_attention(c, s):
    H, G, D, m = c["heads"], c["kv_heads"], c["dim"], s.m
    window, chunk = _limits(c)
    proj, n = s.proj.double(), s.proj.shape[0]
    a = _angles(s.pos, 5e5 ** (-torch.arange(0, D, 2, dtype=torch.float64, device=DEV) / D))
    q, k, v = proj.view(n, H + 2 * G, D).split([H, G, G], 1)
    q, k = _turn(q, a), _turn(k, a)
    if c["turning"]:
        v = _turn(v, a, "neighbours")
    cache = s.cache.double()
    cache.view(-1, 2 * G * D)[s.ctx.slot_mapping.long()] = torch.cat([k.reshape(n, -1), v.reshape(n, -1)], 1)
    if c["phase"] == "decode":
        out = torch.empty(n, H, D, dtype=torch.float64, device=DEV)
        for i, (t, L) in enumerate(zip(s.tables, s.lens)):
            both = cache[t].reshape(-1, 2 * G, D)[:L]
            out[i] = _attend(q[i:i + 1], both[:, :G], both[:, G:], D ** -0.5, L - 1, window, chunk, m.sinks)[0]
    else:
        out = torch.cat([_attend(*p, D ** -0.5, 0, window, chunk, m.sinks) for p in zip(*(t.split(s.lens) for t in (q, k, v)))])
    if c["turning"]:
        out = _turn(out, a, "neighbours", back=True)
    return [out.reshape(n, H * D), cache]


# ---------------------------------------------------------------- latent attention
EPS = 1e-6


def _prepare_latent(c, d, seed):
    from zipage_amd.layers import LatentAttention, Rotary
    W, P, window = c["width"], c["rot"], c["window"] or None
    m = LatentAttention(W, c["heads"], c["dim"], c["dim"], c["q_rank"], c["kv_rank"], (c["dim"] + P) ** -0.5, window, EPS,
                        rotary=Rotary(5e5, P) if P else None)
    w = {k: d.uniform(*s, lo=0.5, hi=1.5, dtype=torch.bfloat16) if k.endswith("norm") else d.normal(*s, std=s[1] ** -0.5)
         for k, s in m.shapes().items()}
    m.load(w, torch.bfloat16, DEV)
    lens = _case_lengths(c, d)
    tables, pool = _tables(lens, d)
    rows = len(lens) if c["phase"] == "decode" else sum(lens)
    cache = m.allocate(pool, PAGE, torch.bfloat16, DEV)
    if c["phase"] == "decode":
        cache.normal_(generator=d.dev)
    x, f32 = d.normal(rows, W, dtype=torch.float32), dict(dtype=torch.float32, device=DEV)
    return SimpleNamespace(kind="latent", m=m, w=w, lens=lens, tables=tables, cache=cache, ctx=_context(c, lens, tables, window),
                           pos=_positions(c, lens), h=x.to(torch.bfloat16), x=x, norm=torch.ones(W, **f32),
                           stream=torch.empty(rows, W, **f32))


def _run_latent(s):
    from zipage_amd.layers import residual_norm
    y = s.m.forward(s.h, s.cache, s.ctx, positions=s.pos)
    h = residual_norm(s.x, y, s.norm, EPS, s.x.shape[1], x_out=s.stream)
    return [h, s.stream, s.cache]


def _work_latent(c):
    W, H, D, Q, R, P = c["width"], c["heads"], c["dim"], c["q_rank"], c["kv_rank"], c["rot"]
    weights = W * (Q + R + P) + Q * H * (D + P) + 2 * R * H * D + H * D * W
    seen = lambda n: _seen(n, c["window"], 0)
    rows = c["requests"] if c["phase"] == "decode" else _mean_lengths(c)
    byts = 2 * weights + rows * W * (2 + 4 + 4 + 2) + 2 * rows * (R + P)
    if c["phase"] == "decode":
        keys = _mean_lengths(c, seen)
        return {"bytes": byts + 2 * keys * (R + P), "flops": 2 * rows * weights + 2 * keys * H * (2 * R + P)}
    pairs = _mean_lengths(c, lambda n: sum(seen(i + 1) for i in range(n)))
    return {"bytes": byts, "flops": 2 * rows * weights + 2 * pairs * H * (2 * D + P)}


def _exact_latent(c, s):
    H, D, R, P, W = c["heads"], c["dim"], c["kv_rank"], c["rot"], c["width"]
    w = {k: t.double() for k, t in s.w.items()}
    h, n = s.h.double(), s.h.shape[0]
    a = _angles(s.pos, 5e5 ** (-torch.arange(0, P, 2, dtype=torch.float64, device=DEV) / max(P, 1)))
    q = ((_rms(h @ w["dq"].T, EPS) * w["dq.norm"]) @ w["uq"].T).view(n, H, D + P)
    q = torch.cat([q[..., :D], _turn(q[..., D:], a)], -1)
    down = h @ w["dkv"].T
    row = torch.cat([_rms(down[:, :R], EPS) * w["dkv.norm"], _turn(down[:, None, R:], a)[:, 0]], -1)
    cache = s.cache.double()
    cache.view(-1, R + P)[s.ctx.slot_mapping.long()] = row

    def attend(q, rows, at):
        k = torch.cat([(rows[:, :R] @ w["uk"].T).view(-1, H, D), rows[:, None, R:].expand(-1, H, -1)], -1)
        return _attend(q, k, (rows[:, :R] @ w["uv"].T).view(-1, H, D), (D + P) ** -0.5, at, c["window"])
    if c["phase"] == "decode":
        o = torch.cat([attend(q[i:i + 1], cache[t].reshape(-1, R + P)[:L], L - 1)
                       for i, (t, L) in enumerate(zip(s.tables, s.lens))])
    else:
        o = torch.cat([attend(a, b, 0) for a, b in zip(q.split(s.lens), row.split(s.lens))])
    x = s.x.double() + o.reshape(n, -1) @ w["o"].T
    return [_rms(x, EPS), x, cache]


# ---------------------------------------------------------------- recurrent mixers
RANK, TAPS, TAU = 128, 4, 16.0


def _prepare_recurrent(c, d, seed):
    from zipage_amd.layers import ChannelDelta, LinearAttention, MatrixMemory, Rotary
    W, H, D, kind = c["width"], c["heads"], c["dim"], c["mixer"]
    if kind == "delta":
        m = ChannelDelta(W, H, H // 2, D, D, TAPS, EPS)
        shapes = m.shapes(RANK, RANK)
    elif kind == "memory":
        m = MatrixMemory(W, H, D, D, 15.0, EPS)
        shapes = m.shapes()
    elif kind == "linear":
        m = LinearAttention(W, H, D, D, EPS, q_scale=D ** -0.5, tau=TAU, weighted=True)
        shapes = m.shapes(RANK)
    else:
        m = LinearAttention(W, H, D, D, EPS, k_scale=D ** -0.5, decay=tuple(1 - 2.0 ** (-5 - 3 * i / H) for i in range(H)),
                            rotary=Rotary(1e4, D))
        shapes = m.shapes()
    w = {k: d.normal(*s, std=s[-1] ** -0.5) for k, s in shapes.items()}
    spread = lambda k, lo, hi: w.update({k: d.uniform(*shapes[k], lo=lo, hi=hi, dtype=torch.bfloat16)})
    for k, lo, hi in (("norm", 0.5, 1.5), ("A_log", -1.0, 1.0), ("dt_bias", -5.0, -1.0), ("i.b", -1.0, 1.0), ("f.b", 3.0, 6.0),
                      ("a2.b", 0.0, 2.0)):
        if k in w:
            spread(k, lo, hi)
    m.load(w, torch.bfloat16, DEV, W)
    lens = _case_lengths(c, d)
    decode = c["phase"] == "decode"
    rows = len(lens) if decode else sum(lens)
    state = m.allocate(len(lens), torch.bfloat16, DEV)
    if decode:                                        # as earlier tokens left it
        (state[0] if kind == "delta" else state).normal_(0.0, 0.1 if kind == "delta" else 1.0, generator=d.dev)
        if kind == "delta":
            state[1].copy_(d.normal(len(lens), H // 2, TAPS - 1, 3 * D).repeat_interleave(2, 1))
            state[1][..., 2 * D:] = d.normal(len(lens), H, TAPS - 1, D)
        if kind == "memory":
            state[..., D * D + D] = d.uniform(len(lens), H, lo=-1.0, hi=1.0)
            state[..., D * D + D + 1:] = 0.0
        lens = [1000 + n for n in d.integers(0, 1000, len(lens))]      # places of the decoded tokens
    tables = [[0] * (-(-n // PAGE)) for n in lens]
    return SimpleNamespace(kind="recurrent", mixer=kind, m=m, w=w, lens=lens, state=state, ctx=_context(c, lens, tables, None),
                           h=d.normal(rows, W), proj=d.normal(rows, m.columns),
                           out=torch.empty(rows, m.out_columns, dtype=torch.bfloat16, device=DEV))


def _run_recurrent(s):
    if s.mixer == "memory":
        s.m.scan(s.h, s.proj, s.state, s.ctx, s.out)
    else:
        s.m.scan(s.proj, s.state, s.ctx, s.out)
    return [s.out, s.state]


def _work_recurrent(c):
    W, H, D, kind = c["width"], c["heads"], c["dim"], c["mixer"]
    rows = c["requests"] if c["phase"] == "decode" else _mean_lengths(c)
    columns = {"delta": 2 * H * D + H + 2 * RANK, "memory": 4 * H * D, "linear": 4 * H * D + RANK, "retention": 4 * H * D}[kind]
    low = {"delta": 2 * H * D * RANK, "memory": 2 * H * W, "linear": H * D * RANK, "retention": 0}[kind]
    state = c["requests"] * H * D * D * 4 * (2 if c["phase"] == "decode" else 1)
    return {"bytes": state + 2 * rows * (columns + H * D) + 2 * low + (2 * rows * W if kind == "memory" else 0),
            "flops": rows * (2 * low + (7 if kind == "delta" else 5) * H * D * D)}


def _exact_recurrent(c, s):
    """One token after the other, all sequences side by side; shorter ones stop earlier."""
    W, H, D, kind, B = c["width"], c["heads"], c["dim"], c["mixer"], c["requests"]
    f64 = dict(dtype=torch.float64, device=DEV)
    decode = c["phase"] == "decode"
    counts = torch.tensor([1] * B if decode else s.lens, device=DEV)
    first = counts.cumsum(0) - counts
    N, proj, w = s.proj.shape[0], s.proj.double(), {k: t.double() for k, t in s.w.items()}
    pos = torch.cat([torch.tensor([n - 1], device=DEV) if decode else torch.arange(n, device=DEV) for n in s.lens])
    cut = lambda *sizes: proj[:, :sum(sizes)].split(sizes, 1)
    old = s.state[0] if kind == "delta" else s.state
    if kind == "memory":
        S = old[..., :D * D].double().view(B, H, D, D).clone()
        z, m0 = old[..., D * D:D * D + D].double().clone(), old[..., D * D + D].double().clone()
    else:
        S = old.double().clone()
    beta = None
    if kind == "delta":
        G = H // 2
        x = proj[:, :2 * G * D + H * D]
        taps = torch.cat([w["q.conv"], w["k.conv"], w["v.conv"]])                       # (channels, taps)
        y = torch.zeros_like(x)
        for j in range(TAPS):                          # the input of j tokens ago; before a prompt there is none
            back = torch.zeros_like(x)
            if decode and j:
                t = s.state[1][:, :, TAPS - 1 - j].double()
                back = torch.cat([t[:, ::2, :D].flatten(1), t[:, ::2, D:2 * D].flatten(1), t[:, :, 2 * D:].flatten(1)], 1)
            elif j == 0:
                back = x
            else:
                back[j:] = x[:-j]
                back[pos < j] = 0
            y += taps[:, TAPS - 1 - j] * back
        y = F.silu(y)
        unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)
        q, k, v = y.split([G * D, G * D, H * D], 1)
        q = unit(q.reshape(N, G, D)).repeat_interleave(2, 1) * D ** -0.5
        k, v = unit(k.reshape(N, G, D)).repeat_interleave(2, 1), v.reshape(N, H, D)
        at = 2 * G * D + H * D
        beta = torch.sigmoid(proj[:, at:at + H])
        a1, g1 = proj[:, at + H:at + H + RANK], proj[:, at + H + RANK:at + H + 2 * RANK]
        g = torch.exp(-torch.exp(w["A_log"])[:, None] * F.softplus(a1 @ w["a2"].T + w["dt_bias"]).view(N, H, D))
        gate = torch.sigmoid(g1 @ w["g2"].T).view(N, H, D)
    else:
        q, k, v, gate = (t.reshape(N, H, D) for t in cut(*[H * D] * 4))
        if kind == "memory":
            q, gate, h = q * D ** -0.5, torch.sigmoid(gate), s.h.double()
            cap = lambda t: 15.0 * torch.tanh(t / 15.0)
            i, f = cap(h @ w["i"].T + w["i.b"]), F.logsigmoid(cap(h @ w["f"].T + w["f.b"]))
        elif kind == "linear":
            q, gate = q * D ** -0.5, F.silu(gate)
            g = (torch.sigmoid(proj[:, 4 * H * D:] @ w["a2"].T + w["a2.b"]) ** (1 / TAU)).view(N, H, D)
        else:
            a = _angles(pos, 1e4 ** (-torch.arange(0, D, 2, **f64) / D))
            q, k, gate = _turn(q, a), _turn(k, a) * D ** -0.5, F.silu(gate)
            g = torch.tensor(s.m.decay, **f64)[None, :, None].expand(N, H, D)
    o = torch.empty(N, H, D, **f64)
    for t in range(int(counts.max())):
        live = (t < counts).nonzero()[:, 0]
        r = first[live] + t
        if kind == "memory":
            new = torch.maximum(f[r] + m0[live], i[r])
            keep, write = torch.exp(f[r] + m0[live] - new), torch.exp(i[r] - new)
            m0[live] = new
            z[live] = keep[..., None] * z[live] + write[..., None] * k[r]
            S[live] = keep[..., None, None] * S[live] + (write[..., None] * k[r])[..., None] * v[r][:, :, None]
            den = torch.maximum((z[live] * q[r]).sum(-1).abs(), torch.exp(-new)) + 1e-6
            o[r] = (S[live] * q[r][..., None]).sum(2) / den[..., None]
            continue
        A = g[r][..., None] * S[live]
        u = v[r] if beta is None else beta[r][..., None] * (v[r] - (A * k[r][..., None]).sum(2))
        A = A + k[r][..., None] * u[:, :, None]
        S[live] = A
        o[r] = (A * q[r][..., None]).sum(2)
    norm = {"delta": lambda: w["norm"], "memory": lambda: w["norm"].view(H, D), "linear": lambda: w["norm"]}.get(kind, lambda: 1.0)()
    out = (_rms(o, EPS) * norm * gate).reshape(N, H * D)
    if kind == "memory":
        state = old.double().clone()
        state[..., :D * D], state[..., D * D:D * D + D], state[..., D * D + D] = S.flatten(2), z, m0
        return [out, state]
    return [out, [S, None] if kind == "delta" else S]


# ---------------------------------------------------------------- experts
LIMIT = 7.0


def _prepare_experts(c, d, seed):
    from zipage_amd.layers import Experts
    W, ff, E = c["width"], c["ff"], c["experts"]
    m = Experts(W, E, c["top"], ff, LIMIT, c["groups"], c["keep"], ff if c["shared"] else None, LIMIT, score=c["score"], act=c["act"])
    w = {k: d.normal(*s, std=s[1] ** -0.5) for k, s in m.shapes().items()}
    m.load(w, torch.bfloat16, DEV)
    f32 = dict(dtype=torch.float32, device=DEV)
    return SimpleNamespace(kind="experts", m=m, w=w, h=d.normal(c["tokens"], W), x=d.normal(c["tokens"], W, dtype=torch.float32),
                           norm=torch.ones(W, **f32), branch=d.uniform(W, lo=0.5, hi=1.5) if c["act"] == "clamped" else None,
                           stream=torch.empty(c["tokens"], W, **f32))


def _run_experts(s):
    from zipage_amd.layers import residual_norm
    y = s.m.forward(s.h)
    return [residual_norm(s.x, y, s.norm, EPS, s.x.shape[1], x_out=s.stream, y_weight=s.branch), s.stream]


def _work_experts(c):
    n, W, ff, E, top = c["tokens"], c["width"], c["ff"], c["experts"], c["top"]
    used = E * (1 - (1 - top / E) ** n) + c["shared"]
    return {"bytes": 2 * (used * 3 * W * ff + E * W) + n * W * (2 + 4 + 4 + 2),
            "flops": 2 * n * W * E + 6 * n * (top + c["shared"]) * W * ff}


def _exact_experts(c, s):
    h, E, top = s.h.double(), c["experts"], c["top"]
    z = h @ s.w["router"].double().T
    score = torch.softmax(z, -1) if c["score"] == "softmax" else torch.sigmoid(z)
    groups = score.view(-1, c["groups"], E // c["groups"])
    best = groups.amax(-1).topk(c["keep"], -1).indices
    allowed = torch.zeros(groups.shape[:2], dtype=torch.bool, device=DEV).scatter_(1, best, True)
    chosen = groups.masked_fill(~allowed[..., None], -1.0).flatten(1).topk(top, -1).indices

    def expert(x, p):
        g, u = x @ s.w[p + ".gate"].double().T, x @ s.w[p + ".up"].double().T
        if c["act"] == "silu":
            return (F.silu(g) * u) @ s.w[p + ".down"].double().T
        g, u = g.clamp(max=LIMIT), u.clamp(-LIMIT, LIMIT)
        return (g * torch.sigmoid(1.702 * g) * (u + 1)) @ s.w[p + ".down"].double().T
    y = expert(h, "shared") if c["shared"] else torch.zeros_like(h)
    for e in range(E):
        rows = (chosen == e).any(-1).nonzero()[:, 0]
        if len(rows):
            a = score[rows, e][:, None]
            y[rows] += a * expert(h[rows], f"e{e}") if c["act"] == "clamped" else expert(a * h[rows], f"e{e}")
    x = s.x.double() + (y if s.branch is None else _rms(y, EPS) * s.branch.double())
    return [_rms(x, EPS), x]
