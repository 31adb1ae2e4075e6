"""Kernels that come in several forms, at the sizes where the choice falls and at the forms' edges."""
import pytest
import torch

from oracle import kapolorn_oracle as K
from oracle import rutevik_oracle as R
from oracle import zipage_oracle as O
from zipage_amd.sight import Chunk

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _rand(*shape, seed, std=1.0, dtype=BF16):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * std).to(dtype)


# ------------------------------------------------------------------ compaction
# pairs of (row, tensor): up to 512 take workgroups of sixteen waves, up to 256 workgroups are cut by columns; 513 and
# more take the general form
@pytest.mark.parametrize("dtype,L,B,Hkv,D", [(torch.float32, 1, 1, 1, 256), (torch.float32, 1, 1, 8, 128), (BF16, 1, 1, 2, 128),
                                             (BF16, 2, 8, 8, 128), (torch.float16, 1, 32, 8, 64), (BF16, 1, 33, 8, 64),
                                             (BF16, 1, 2, 3, 48), (torch.float32, 1, 16, 8, 64)])
@pytest.mark.parametrize("style", ["aliased", "cow"])
def test_compaction_of_few_rows(dev, dtype, L, B, Hkv, D, style):
    from zipage_amd.kernel import compress_kv
    BS, budget, NB = 32, 3, 5
    g = torch.Generator().manual_seed(B * 7 + D)
    pages = torch.randperm(B * (NB + 2), generator=g).tolist()
    tables = [[pages.pop() for _ in range(NB - b % 2)] for b in range(B)]
    enc = O.encode_block_table(tables)
    head = [t[:budget + 1] for t in tables]
    if style == "cow":
        head = [[pages.pop(), pages.pop()] + t[2:] for t in head]
    target = torch.tensor(head, dtype=torch.int32)
    k, v = (_rand(L, B * (NB + 2), BS, Hkv, D, seed=s, dtype=dtype) for s in (1, 2))
    scores = O.pad_mask(torch.rand((L, B, Hkv, NB, BS), generator=g), enc).view(L, B, Hkv, NB * BS)
    flag = O.topk_mask(scores, budget * BS).view(L, B, Hkv, NB, BS)
    wk, wv = k.clone(), v.clone()
    O.compress_kv_loop(wk, wv, flag, enc, target)
    gk, gv = k.to(dev), v.to(dev)
    compress_kv(gk, gv, flag.to(dev), enc.to(dev), target.to(dev))
    assert torch.equal(gk.cpu().view(torch.uint8), wk.view(torch.uint8))
    assert torch.equal(gv.cpu().view(torch.uint8), wv.view(torch.uint8))


# columns of 32 bytes where a row's workgroups share an XCD, which multiples of eight pairs do, and of whole lines elsewhere;
# rounds of half as many pieces up to 8192 of them: exactly as many, and a page more
@pytest.mark.parametrize("dtype,Hkv,D,width", [(BF16, 4, 128, 128), (BF16, 4, 128, 129), (torch.float32, 4, 128, 64), (BF16, 3, 128, 32),
                                               (BF16, 3, 128, 33), (torch.float32, 12, 64, 61), (torch.float16, 8, 32, 40)])
def test_compaction_in_parts_of_lines(dev, dtype, Hkv, D, width):
    from zipage_amd.kernel import compress_kv
    BS, NB = 32, width + 2
    g = torch.Generator().manual_seed(width)
    table = torch.randperm(NB + 3, generator=g).tolist()
    enc = O.encode_block_table([table[:NB]])
    target = torch.tensor([[table[NB]] + table[1:width]], dtype=torch.int32)
    k, v = (_rand(1, NB + 3, BS, Hkv, D, seed=s, dtype=dtype) for s in (1, 2))
    flag = torch.zeros(1, 1, Hkv, NB * BS, dtype=torch.bool)
    for h in range(Hkv):                                                 # the first of as many as there is room for
        flag[0, 0, h, torch.randperm(NB * BS, generator=g)[:width * BS - 7 * h]] = True
    flag = flag.view(1, 1, Hkv, NB, BS)
    wk, wv = k.clone(), v.clone()
    O.compress_kv(wk, wv, flag, enc, target)
    gk, gv = k.to(dev), v.to(dev)
    compress_kv(gk, gv, flag.to(dev), enc.to(dev), target.to(dev))
    assert torch.equal(gk.cpu().view(torch.uint8), wk.view(torch.uint8)) and torch.equal(gv.cpu().view(torch.uint8), wv.view(torch.uint8))


# the list of 65 536 tokens and its pages, which fill the LDS but for 16 or 64 bytes: the former leaves no room for the
# sums of sixteen waves
@pytest.mark.parametrize("width", [4092, 4080])
def test_compaction_of_the_longest_list(dev, width):
    from zipage_amd.kernel import compress_kv
    BS, NB, D = 16, 4096, 64
    g = torch.Generator().manual_seed(width)
    table = torch.randperm(NB, generator=g).tolist()
    enc, target = O.encode_block_table([table]), torch.tensor([table[:width]], dtype=torch.int32)
    k, v = (_rand(1, NB, BS, 1, D, seed=s) for s in (1, 2))
    flag = (torch.rand((1, 1, 1, NB, BS), generator=g) < 0.9)
    wk, wv = k.clone(), v.clone()
    O.compress_kv(wk, wv, flag, enc, target)
    gk, gv = k.to(dev), v.to(dev)
    compress_kv(gk, gv, flag.to(dev), enc.to(dev), target.to(dev))
    assert torch.equal(gk.cpu(), wk) and torch.equal(gv.cpu(), wv)


# ------------------------------------------------------------------ attention scores
# pages of 256 tokens with groups of two or four heads and a mean over the window have forms of their own; the same
# tokens in pages of 128 take the general one: same bits.  Of few blocks of rows, too, whose tiles lie side by side where there is
# room, and which walk them where there is not.
@pytest.mark.parametrize("dtype", [BF16, torch.float16, torch.float32])
@pytest.mark.parametrize("group,W", [(2, 32), (2, 16), (2, 5), (4, 32), (3, 20)])
def test_scores_by_page_size_and_group(dev, dtype, group, W):
    from zipage_amd.kernel import attention_score
    from tests.test_hip_kernels import _score_one_sweep
    B, Hkv, D, P = 3, 2, 128, 9
    g = torch.Generator().manual_seed(group * 64 + W)
    pages = torch.randperm(P, generator=g).tolist()
    tables = [[pages.pop() for _ in range(n)] for n in (4, 3, 1)]
    k, q = _rand(1, P, 256, Hkv, D, seed=W, dtype=dtype).to(dev), _rand(1, B, W, group * Hkv, D, seed=W + 1, dtype=dtype).to(dev)
    seq = torch.arange(B, dtype=torch.int32, device=dev)
    whole, halves = (O.encode_block_table(t).to(dev) for t in (tables, [[2 * p + i for p in t for i in (0, 1)] for t in tables]))
    want = _score_one_sweep(k.view(1, 2 * P, 128, Hkv, D), q, seq, halves)
    for got in (_score_one_sweep(k, q, seq, whole), attention_score(k, q, seq, whole),
                attention_score(k.view(1, 2 * P, 128, Hkv, D), q, seq, halves)):
        assert torch.equal(got.reshape(want.shape), want)


# up to 64 blocks of query rows (32, fp32: 16) have their tiles side by side, more walk them: same bits for a sequence alone and
# in a batch, and where the scratch holds only what the walk needs.
@pytest.mark.parametrize("dtype", [BF16, torch.float16, torch.float32])
@pytest.mark.parametrize("group,W,BS,D,reduced,B", [(1, 32, 256, 128, "mean", 65), (2, 16, 256, 128, "mean", 65), (3, 9, 128, 64, "mean", 65),
                                                    (4, 32, 256, 96, "max", 17), (8, 5, 256, 128, "mean", 33), (8, 3, 128, 40, "max", 65),
                                                    (16, 4, 128, 128, "mean", 33), (1, 20, 128, 128, "max", 65)])
def test_scores_of_few_sequences(dev, dtype, group, W, BS, D, reduced, B):
    from zipage_amd.kernel import attention_score
    from tests.test_hip_kernels import _score_one_sweep
    NB = 6
    g = torch.Generator().manual_seed(group * 64 + W)
    pages = torch.randperm(B * NB, generator=g).tolist()
    enc = O.encode_block_table([[pages.pop() for _ in range(NB - b % 5)] for b in range(B)])
    k, q = _rand(1, B * NB, BS, 1, D, seed=W, dtype=dtype, std=2.0).to(dev), _rand(1, B, W, group, D, seed=W + 1, dtype=dtype).to(dev)
    seq = torch.randperm(B, generator=g).int().to(dev)
    many = attention_score(k, q, seq, enc.to(dev), reduced=reduced)
    for n in (1, 3):
        args = (k, q, seq[:n].contiguous(), enc[:n].contiguous().to(dev), reduced)
        for few in (attention_score(*args[:4], reduced=reduced), _score_one_sweep(*args)):
            assert torch.equal(few, many[:, :n])
    want = O.attention_score(k[:, :, :, :, :].cpu(), q.cpu(), seq[:3].cpu(), enc[:3], reduced=reduced)
    torch.testing.assert_close(many[:, :3].cpu().float(), want.float(), rtol=2.0 ** -6 if dtype != torch.float32 else 1e-4, atol=1e-6)


# Units of groups of two and four, up to 128 of them, go in halves of their rows where the selection adds up what they leave and there is
# room for it: the flags of whole units.
@pytest.mark.parametrize("dtype,L,B,Hkv,G,W", [(BF16, 1, 1, 8, 4, 32), (BF16, 1, 5, 8, 2, 32), (torch.float16, 1, 3, 8, 4, 32), (BF16, 1, 16, 8, 2, 16),
                                               (torch.float16, 1, 4, 8, 4, 28), (BF16, 2, 4, 4, 3, 20), (BF16, 1, 9, 5, 4, 5), (BF16, 1, 17, 8, 2, 16)])
@pytest.mark.parametrize("carry", [False, True])
def test_scores_in_halves_of_units(dev, monkeypatch, dtype, L, B, Hkv, G, W, carry):
    from zipage_amd import _lib
    from zipage_amd.compress import CompressConfig, compress_layers
    BS, D, budget = 256, 128, 2
    g = torch.Generator().manual_seed(B * 8 + W)
    counts = [3 + (b * 3 + 4) % 7 for b in range(B)]
    pages = torch.randperm(sum(counts), generator=g).tolist()
    tables = [[pages.pop() for _ in range(n)] for n in counts]
    enc, target = O.encode_block_table(tables).to(dev), torch.tensor([t[:budget + 1] for t in tables], dtype=torch.int32, device=dev)
    k, v = (_rand(L, sum(counts), BS, Hkv, D, seed=i, dtype=dtype).to(dev) for i in (1, 2))
    q = _rand(L, B, W, Hkv * G, D, seed=3, std=2.0, dtype=dtype).to(dev)
    old = torch.rand((L, sum(counts), BS, Hkv), generator=g).to(dtype).to(dev) if carry else None
    cfg = CompressConfig(budget_blocks=budget, query_cache_len=W, enable_pooling=True, pooling_size=5, use_global_score=carry)
    seq, again = torch.arange(B, dtype=torch.int32, device=dev), torch.full((B,), carry, device=dev)
    run = lambda: [t for x in [(k.clone(), v.clone(), None if old is None else old.clone())]
                   for t in (compress_layers(x[0], x[1], q, x[2], seq, enc, again, target, cfg), *x) if t is not None]
    halves, size = run(), _lib.size
    monkeypatch.setattr(_lib, "size", lambda name, *a: size(name.replace("_layers_workspace_few", "_layers_workspace"), *a))
    for got, want in zip(halves, run()):
        assert torch.equal(got, want)


# ------------------------------------------------------------------ redundancy inside pages
# workgroups walk whole rows where 512 of them (fp32: 256), or a multiple, are at least 90 % full (461 rows on), and
# take a page each otherwise.  Same bits for a sequence alone, in a batch that is walked and in one
# that is not; pages the caller did not list score as none.
@pytest.mark.parametrize("dtype", [BF16, torch.float16, torch.float32])
@pytest.mark.parametrize("B", [57, 58, 64, 65, 116])
def test_redundancy_of_pages_walked_or_alone(dev, dtype, B):
    from zipage_amd.kernel import lightning_redudancy_score
    BS, Hkv, D, NB = 64, 8, 32, 3
    g = torch.Generator().manual_seed(B)
    pages = torch.randperm(B * NB, generator=g).tolist()
    enc = O.encode_block_table([[pages.pop() for _ in range(1 + b % NB)] for b in range(B)]).contiguous()
    k = _rand(1, B * NB, BS, Hkv, D, seed=B, dtype=dtype).to(dev)
    got = lightning_redudancy_score(k, enc.to(dev))
    for b in (0, 1, 2, B - 1):
        alone = lightning_redudancy_score(k, enc[b:b + 1].contiguous().to(dev))
        assert torch.equal(got[:, b:b + 1], alone)
    want = O.lightning_redudancy_score(k.cpu()[:, :, :, :1].contiguous(), enc[:3])
    torch.testing.assert_close(got[:, :3, :1].cpu().float(), want.float(), atol=1e-7, rtol=2.0 ** -6 if dtype != torch.float32 else 1e-4)


# ------------------------------------------------------------------ experts
# rows per tile go by the average expert (16, 32, 64, 128, 256); 16-row tiles take 128 rows of W per workgroup from six
# tokens per expert, 40 tiles and 1280 workgroups on; 256-row tiles are worked off whole from a contraction of 2560 on, in
# two halves below it.  Odd numbers of steps, results that end inside a workgroup's columns, and experts without a token are
# among them.
@pytest.mark.parametrize("n,width,E,top,ff", [(60, 96, 64, 2, 800), (61, 2080, 64, 2, 544), (1, 4096, 4, 2, 32),
                                              (260, 160, 4, 1, 288), (1100, 2144, 3, 2, 96), (1100, 96, 2, 1, 2112),
                                              (1300, 256, 2, 1, 96), (515, 2112, 1, 1, 48),
                                              (1100, 2592, 3, 2, 96), (1100, 96, 2, 1, 2592), (515, 2624, 1, 1, 48),
                                              (200, 96, 64, 2, 800), (225, 2080, 64, 2, 544),
                                              (200, 96, 64, 2, 1120)])
@pytest.mark.parametrize("act", ["clamped", "silu"])
def test_experts_by_rows_and_contraction(dev, n, width, E, top, ff, act, shared_ff=None):
    from zipage_amd.layers import Experts
    clamped = act == "clamped"
    m = Experts(width, E, top, ff, 7.0, shared_ff=(shared_ff or ff + 32) if clamped else None, shared_limit=5.0, act=act,
                score="softmax" if clamped else "sigmoid")
    w = {k: _rand(*s, seed=i, std=2.0 * s[-1] ** -0.5) for i, (k, s) in enumerate(m.shapes().items())}
    if E > 2:
        w["router"][E - 1] = w["router"][0] - 4.0 * w["router"][0].sign()     # hardly anyone's choice
    m.load(w, BF16, dev)
    h = torch.zeros(n, m.width_p, dtype=BF16, device=dev)
    x = _rand(n, width, seed=99)
    h[:, :width] = x.to(dev)
    x64, w64 = x.double(), {k: v.double() for k, v in w.items()}
    z = (x64 @ w64["router"].T).sort(-1, descending=True).values
    sure = torch.ones(n, dtype=torch.bool) if top == E else z[:, top - 1] - z[:, top] > 1e-3
    got = m.forward(h).double().sum(0)[:, :width].cpu()
    groups = {"count": 1, "keep": 1}
    if clamped:
        want = K.experts(x64, w64, {"router": {"experts": E, "top": top, "groups": groups}, "expert": {"limit": 7.0},
                                    "shared": {"limit": 5.0}})
    else:
        want = R.experts(x64, w64, {"router": {"experts": E, "top": top}})
    assert int(sure.sum()) >= 0.8 * n
    # bf16 activations and planes: each of top + 2 roundings is at most 2^-9 of its own value
    err = (got - want)[sure].norm() / want[sure].norm()
    assert float(err) < 2.0 ** -8 and bool(torch.isfinite(got).all())


# averages of 8, 9, 16, 17 and 48 rows; tiles that eight XCDs cannot have as many of each, over several blocks of columns;
# launches of few rows that are no multiple of eight workgroups; a shared expert of one to three tiles of 16
@pytest.mark.parametrize("n,width,E,top,ff", [(40, 96, 5, 1, 544), (45, 96, 5, 1, 544), (80, 544, 5, 1, 800), (85, 544, 5, 1, 800),
                                              (240, 800, 5, 1, 288), (130, 800, 11, 2, 1056), (7, 160, 5, 1, 32), (17, 160, 5, 1, 96),
                                              (33, 288, 6, 1, 160), (48, 96, 9, 1, 352)])
@pytest.mark.parametrize("act", ["clamped", "silu"])
def test_experts_among_xcds(dev, n, width, E, top, ff, act):
    test_experts_by_rows_and_contraction(dev, n, width, E, top, ff, act)


# Tiles of 64 rows, staged where tiles and 256 rows of W make 128 workgroups: both products, the first alone (exactly as many), neither;
# averages of 17 to 48, experts of more than one tile; contractions that leave each remainder of what the loop takes
@pytest.mark.parametrize("n,width,E,top,ff", [(600, 1056, 32, 1, 544), (1000, 992, 32, 1, 512), (816, 768, 48, 1, 352), (700, 1088, 64, 2, 544),
                                              (272, 2048, 16, 1, 1056), (272, 1024, 16, 1, 512)])
@pytest.mark.parametrize("act", ["clamped", "silu"])
def test_experts_staged_in_tiles_of_64(dev, n, width, E, top, ff, act):
    from zipage_amd import _lib
    assert _lib.size("zp_moe_tile_rows", n, E, top, 0) == 64
    test_experts_by_rows_and_contraction(dev, n, width, E, top, ff, act)


# tokens that lie so far apart that the staged form cannot address them are read where they lie
@pytest.mark.parametrize("n,E,top,shared_ff", [(160, 8, 1, 0), (384, 8, 1, 96), (200, 9, 1, 0), (60, 8, 4, 32)])
def test_experts_of_tokens_far_apart(dev, n, E, top, shared_ff):
    from zipage_amd.layers import Experts
    W, ff = 544, 2048
    m = Experts(W, E, top, ff, 7.0, shared_ff=shared_ff or None)
    m.random(BF16, dev, torch.Generator(device=dev).manual_seed(1))
    ids = (torch.arange(n * top, device=dev) % (E - 1)).to(torch.int32).view(n, top)
    weights = torch.rand(n, top, device=dev, generator=torch.Generator(device=dev).manual_seed(2))
    m.route = lambda h: (ids, weights, torch.zeros(E + 1, dtype=torch.int32, device=dev))
    h = torch.empty(n, -(-2 ** 30 // n) + 8 & -8, dtype=BF16, device=dev)[:, :W]
    h.copy_(_rand(n, W, seed=3))
    want, got = m.forward(h.contiguous()).float(), m.forward(h).float()
    # the same products, whose sums are split over other waves: roundings of activations and of rows, a bf16 step of 2^-8 where they differ
    assert float((got - want).norm() / want.norm()) < 2.0 ** -9 and bool(torch.isfinite(got).all())


def test_experts_of_many_weights_spread_over_xcds(dev):
    """Few rows against 380 MB of weights: every expert as by itself, whose weights are one XCD's share."""
    from zipage_amd.layers import Experts
    from zipage_amd.layers.moe import Plan
    E, n, W, ff = 7, 24, 4096, 3328
    m = Experts(W, E, 1, ff, 7.0)
    m.random(BF16, dev, torch.Generator(device=dev).manual_seed(1))
    plan = lambda ids_, experts: Plan(ids_, torch.zeros(experts + 1, dtype=torch.int32, device=dev), experts, False, BF16)
    h, ids_ = _rand(n, W, seed=2).to(dev), (torch.arange(n, device=dev) * 5 % E).to(torch.int32)[:, None]
    p, one = plan(ids_, E), torch.ones(n, 1, device=dev)
    act = m.gate_up_rows(h, p, one)
    down, order = m.down_planes(act, p)[0], p.sorted.long()
    assert p.rows == 16
    for e in range(E):
        mine = (ids_[:, 0] == e).nonzero()[:, 0]
        alone = Experts(W, 1, 1, ff, 7.0)
        alone.gate_up, alone.down, alone.shared_gate_up, alone.shared_down = m.gate_up[e:e + 1], m.down[e:e + 1], None, None
        q = plan(torch.zeros(len(mine), 1, dtype=torch.int32, device=dev), 1)
        a = alone.gate_up_rows(h[mine].contiguous(), q, one)
        at = (order[:, None] == mine[q.sorted.long()]).nonzero()
        assert torch.equal(act[at[at[:, 1].argsort(), 0]], a)
        assert torch.equal(down[mine], alone.down_planes(a, q)[0])


# 256-row tiles whose contraction leaves 0 to 3 steps behind the loop, which takes four at a time, in either product; a
# shared expert that has fewer steps than the loop takes
@pytest.mark.parametrize("n,width,ff,shared_ff", [(530, 2560, 48, 0), (530, 2592, 48, 0), (530, 2624, 48, 0), (530, 2656, 48, 0),
                                                  (530, 2688, 48, 0), (530, 96, 2656, 0), (700, 160, 2688, 32),
                                                  (700, 160, 2656, 64), (700, 2656, 2592, 96), (530, 96, 2624, 128),
                                                  (530, 96, 2560, 160), (530, 96, 2560, 224)])
def test_experts_of_long_contractions(dev, n, width, ff, shared_ff):
    test_experts_by_rows_and_contraction(dev, n, width, 1, 1, ff, "clamped" if shared_ff else "silu", shared_ff)


# ------------------------------------------------------------------ attention of runs
def _attended(q, k, v, lens, scale):
    """64-bit attention of runs: lens of (queries, keys), queries being the last positions."""
    H, rep, want, a, b = q.shape[1], q.shape[1] // k.shape[1], [], 0, 0
    for n, m in lens:
        kk, vv = (t[b:b + m].double().repeat_interleave(rep, 1) for t in (k, v))
        sc = torch.einsum("qhd,khd->hqk", q[a:a + n].double(), kk) * scale
        seen = torch.arange(m)[None] <= torch.arange(m - n, m)[:, None]
        want.append(torch.einsum("hqk,khd->qhd", torch.softmax(sc.masked_fill(~seen, float("-inf")), -1), vv))
        a, b = a + n, b + m
    return torch.cat(want)


def _tiles(lens):
    made, a, b = [], 0, 0
    for n, m in lens:
        made += [(a + i, min(128, n - i), b, m - n + i) for i in range(0, n, 128)]
        a, b = a + n, b + m
    return torch.tensor(made, dtype=torch.int32)


# queries as projected, which the attention turns itself, against queries that the store has turned: heads as long as what turns
# and longer, 8 and 16 steps of a key, runs that take either form and both
@pytest.mark.parametrize("H,G,D,V,rot", [(4, 2, 64, 64, 64), (2, 1, 128, 128, 128), (3, 3, 128, 64, 64), (4, 1, 72, 128, 64), (2, 2, 104, 56, 64),
                                         (16, 8, 128, 128, 128)])
@pytest.mark.parametrize("lens", ["few", "short", "long"])
def test_runs_turn_their_queries(dev, H, G, D, V, rot, lens, first=5):
    from zipage_amd.layers import run_attention
    from zipage_amd.layers.grouped import rotary_store, store_form
    from zipage_amd.layers.runs import attention_form
    lens = {"few": FEW_KEYS, "short": MANY_SHORT, "long": [(385, 385), (1, 900), (129, 193), (33, 600)]}[lens]
    N, M = (sum(t) for t in zip(*lens))
    rows, edge = first + N, H * D
    proj = _rand(rows, edge + G * (D + V) + 8, seed=1).to(dev)[:, :edge + G * (D + V)]
    pos = torch.randint(0, 3000, (rows,), generator=torch.Generator().manual_seed(2), dtype=torch.int32).to(dev)
    freqs = (1e4 ** (-torch.arange(0, rot, 2) / rot)).float().to(dev)
    slots = torch.arange(rows, dtype=torch.int32, device=dev)
    cache, other = (torch.zeros(rows, 1, G * (D + V), dtype=BF16, device=dev) for _ in range(2))
    q = rotary_store(proj, pos, freqs, H, G, D, V, cache, slots)
    turns = torch.full((rot // 4, rows, 2, 2), float("nan"), device=dev)
    some, kv = rotary_store(proj, pos, freqs, H, G, D, V, other, slots, return_kv=True, form=store_form(q_turns=turns, q_rows=first))
    assert torch.equal(some, q[:first]) and torch.equal(cache, other) and torch.equal(kv, cache[:, 0])
    keys, sinks = _rand(M, G * (D + V), seed=3).to(dev), _rand(H, seed=4, dtype=torch.float32).to(dev)
    for scale in (D ** -0.5, -0.1):
        got, want = (torch.empty(N, H * V, dtype=BF16, device=dev) for _ in range(2))
        run_attention(q[first:], keys, H, G, D, V, _tiles(lens).to(dev), scale, want, window=200, sinks=sinks)
        run_attention(proj[first:, :edge], keys, H, G, D, V, _tiles(lens).to(dev), scale, got, window=200, sinks=sinks,
                      form=attention_form(q_turns=turns[:, first:]))
        # both turn in 32 bits and round once, but a compiler may round a product on the way: seldom another last bit of a query
        assert (got != want).float().mean() < 1e-3 and (got.float() - want.float()).abs().max() <= 2.0 ** -6 * want.float().abs().max()


# the scale joins the subtraction of the maximum: a negative one turns the queries round, zero takes them away
@pytest.mark.parametrize("scale", [-0.25, 0.0, 1e-30, 0.25])
@pytest.mark.parametrize("H,G,D,V", [(2, 1, 40, 24), (2, 2, 64, 64), (3, 1, 128, 56), (4, 2, 128, 128), (3, 3, 136, 136)])
def test_runs_of_any_scale(dev, H, G, D, V, scale, lens=((1, 1), (63, 63), (65, 65), (32, 64), (33, 129), (130, 200))):
    from zipage_amd.layers import run_attention
    N, M = (sum(t) for t in zip(*lens))
    q, k = (_rand(N, H, D, seed=1), _rand(M, G, D, seed=2))
    v = _rand(M, G, V, seed=3)
    out = torch.empty(N, H * V, dtype=BF16, device=dev)
    run_attention(q.flatten(1).to(dev), torch.cat([k.flatten(1), v.flatten(1)], 1).to(dev), H, G, D, V,
                  _tiles(lens).to(dev), scale, out)
    want = _attended(q, k, v, lens, scale)
    # bf16 keeps 8 bits: 2^-8 of the result, and 2^-8 of each weight times its value's distance from the result
    assert bool(((out.view(N, H, V).cpu().double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -7 * v.abs().max()).all())


# The launch hands key heads and tiles to eight parts: heads that divide into them, tiles that do not; key heads that share a
# part; key and value rows of 8 and 16 pieces in each combination, not all of them there
@pytest.mark.parametrize("H,G,D,V", [(16, 8, 128, 128), (32, 16, 64, 128), (12, 12, 72, 40), (10, 10, 40, 24), (6, 2, 64, 64),
                                     (9, 3, 128, 104), (5, 1, 56, 72)])
def test_runs_over_the_parts_of_a_launch(dev, H, G, D, V):
    test_runs_of_any_scale(dev, H, G, D, V, 0.25, ((385, 385), (1, 900), (127, 191), (128, 192), (129, 193), (33, 600)))


# up to 256 keys, and up to 32 per tile on average: steps of 32 keys, whatever a run has
FEW_KEYS = [(1, 1)] * 5 + [(16, 16), (17, 33), (64, 65), (96, 137)]


@pytest.mark.parametrize("H,G,D,V", [(2, 1, 128, 128), (3, 3, 136, 128), (4, 2, 40, 72), (2, 2, 64, 64), (2, 1, 200, 256)])
def test_runs_of_few_keys(dev, H, G, D, V):
    test_runs_of_any_scale(dev, H, G, D, V, 0.25, FEW_KEYS)


# launches of many workgroups take runs of up to 128 keys apart from 1024 workgroups on, of up to 64 from 512 on; beside them
# longer runs, and runs with cached context
MANY_SHORT = [(n, n) for n in (1, 16, 31, 33, 63, 64, 65, 100, 127, 128, 129)] * 6 + [(40, 90), (3, 300), (200, 264), (300, 300)]


@pytest.mark.parametrize("H,G,D,V", [(16, 8, 128, 128), (15, 5, 72, 104), (8, 8, 56, 128), (4, 2, 128, 72)])
def test_many_short_runs(dev, H, G, D, V):
    test_runs_of_any_scale(dev, H, G, D, V, -0.25 if G == 8 else 0.25, MANY_SHORT)


@pytest.mark.parametrize("H,G,D", [(16, 4, 128), (8, 2, 104)])
def test_causal_attention_of_many_short_prompts(dev, H, G, D):
    test_causal_attention(dev, H, G, D, MANY_SHORT)


def test_causal_attention_of_few_keys(dev):
    test_causal_attention(dev, 8, 2, 128, FEW_KEYS)


@pytest.mark.parametrize("H,G,D", [(2, 1, 8), (4, 4, 64), (6, 2, 72), (8, 2, 128)])
def test_causal_attention(dev, H, G, D, lens=((1, 1), (31, 31), (128, 128), (129, 129), (5, 300), (64, 65), (257, 257))):
    """Prompts with and without cached context, of lengths about a tile's and a step's; queries that point at one key."""
    from zipage_amd.engine.inputs import plan_prompts
    from zipage_amd.layers import causal_attention
    N, M = (sum(t) for t in zip(*lens))
    qkv = _rand(N, (H + 2 * G) * D, seed=1)
    k, v = _rand(M, G, D, seed=2), _rand(M, (H + 2 * G) * D, seed=3)
    q = qkv[:, :H * D].view(N, H, D)
    q[::3] = (k[torch.arange(0, N, 3) % M].repeat_interleave(H // G, 1).float() * (8.0 / D ** 0.5)).to(BF16)
    at = (H + G) * D
    tiles = plan_prompts(*zip(*lens))
    assert sorted(map(tuple, tiles.tolist())) == sorted(map(tuple, _tiles(lens).tolist()))
    got = causal_attention(qkv.to(dev)[:, :H * D].view(N, H, D), k.to(dev), v.to(dev)[:, at:].view(M, G, D),
                           torch.from_numpy(tiles).to(dev), D ** -0.5)
    vv = v[:, at:].view(M, G, D)
    want = _attended(q, k, vv, lens, D ** -0.5)
    # bf16 keeps 8 bits: 2^-8 of the result; two planes of it 16: 2^-16 of each weight times its value's distance from the
    # result, and as much for the fp32 sums of scores up to 32
    assert bool(((got.view(N, H, D).cpu().double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -14 * vv.abs().max()).all())


# ------------------------------------------------------------------ products of few rows
# token tiles of 1, 2 and 4, row tiles of 1, 2 and 4; contractions of one step, of stages that end early and of more than
# the ring; outputs that end inside a tile; rows of x further apart than they are long
@pytest.mark.parametrize("dtype", [BF16, torch.float16])
@pytest.mark.parametrize("n", [1, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("K,M", [(32, 4), (96, 20), (128, 4096), (1056, 4100), (1312, 68), (2048, 4128), (160, 16388), (2176, 16400), (1984, 8196)])
def test_products_of_few_rows(dev, dtype, n, K, M):
    from zipage_amd import _lib
    wide = _rand(n, K + 24, seed=1, dtype=dtype).to(dev)
    x, w = wide[:, 8:8 + K], (_rand(M, K, seed=2).float() * K ** -0.5).to(dtype).to(dev)
    out = torch.full((n, M + 4), 7.0, dtype=dtype, device=dev)
    _lib.call_models("zp_few_rows_linear", x.data_ptr(), w.data_ptr(), out.data_ptr(), n, K, M, x.stride(0), out.stride(0),
                     _lib.dtype_tag(x), _lib.stream_ptr(x))
    assert bool((out[:, M:] == 7).all())
    want = x.double() @ w.double().T
    # rounding to 8 or 11 bits, and K terms in fp32, each sum within 2^-24 sqrt(K) of its terms' root of squares
    bits = 2.0 ** (-8 if dtype == BF16 else -11)
    assert bool(((out[:, :M].double() - want).abs() <= bits * want.abs() + 2.0 ** -20).all())


# a mixer whose runs turn their queries, against the same with stored ones: whole prompts, portions that look back on pages, both beside
# decoded tokens; values that turn too; heads as long as what turns and longer
@pytest.mark.parametrize("H,G,D,V,rot,turning,sight", [(4, 2, 64, 64, 64, False, None), (4, 1, 128, 128, 128, True, 100),
                                                       (2, 2, 96, 64, 64, True, Chunk(64)), (2, 1, 128, 48, 64, False, 100)])
@pytest.mark.parametrize("portions", [[(0, 150), (0, 33)], [(70, 140), (5, 20)], [(40, 1), (0, 129), (99, 1), (64, 64)]])
def test_mixers_turn_queries_late(dev, monkeypatch, H, G, D, V, rot, turning, sight, portions):
    from zipage_amd.engine.inputs import Runs, plan_portions
    from zipage_amd.engine.qwen3 import StepContext
    from zipage_amd.engine.sequence import Portion, Sequence
    from zipage_amd.layers import GroupedAttention, Rotary, grouped
    mix = GroupedAttention(32, H, G, D, V, D ** -0.5, sight, Rotary(5e5, rot, interleaved=turning), turn_values=turning)
    mix.load({k: _rand(*t, seed=i) for i, (k, t) in enumerate(mix.shapes().items())}, BF16, dev, 32)
    assert mix._turns_late(1 << 20) and not mix._turns_late(200)
    BS, work, free = 16, [], iter(torch.randperm(80, generator=torch.Generator().manual_seed(D)).tolist())
    for start, count in portions:
        seq = Sequence([0] * (start + count), block_size=BS)
        seq.block_table = [next(free) for _ in range(-(-(start + count) // BS))]
        work.append(Portion(seq, start, count))
    plan = plan_portions(work, BS, [sight], 16)
    t = lambda a: None if a is None else torch.as_tensor(a).to(dev)
    ctx = StepContext(False, t(plan.slots), None, t(plan.context_lens), t(plan.tables), table_rows=t(plan.table_rows),
                      runs={k: Runs(t(r.tiles), t(r.key_slots)) for k, r in plan.runs.items()})
    N, singles, asked = len(plan.positions), len(plan.context_lens), []
    held = _rand(80, BS, mix.row, seed=1).to(dev)
    wide = _rand(N, mix.columns + mix.out_columns, seed=2).to(dev)
    attention = grouped.run_attention
    monkeypatch.setattr(grouped, "run_attention", lambda *a, form=None, **k: (asked.append(form is not None and bool(form.q_turns)),
                                                                              attention(*a, form=form, **k)))

    def go(late, proj, out):
        monkeypatch.setattr(GroupedAttention, "_turns_late", lambda self, n: late)
        cache = held.clone()
        mix.attend(proj, t(plan.positions), cache, ctx, out)
        return out.clone(), cache
    proj = wide[:, :mix.columns]
    want, cache = go(False, proj, torch.full((N, mix.out_columns), float("nan"), dtype=BF16, device=dev))
    got, other = go(True, proj, torch.full((N, mix.out_columns), float("nan"), dtype=BF16, device=dev))
    assert asked == [False, True] and torch.equal(cache, other) and torch.equal(got[:singles], want[:singles])
    # as above
    assert (got != want).float().mean() < 1e-3 and (got.float() - want.float()).abs().max() <= 2.0 ** -6 * want.float().abs().max()
    # results beside the projections, between them, and where the queries are
    for both, at in ((wide.clone(), mix.columns), (wide.clone(), 0)):
        again, other = go(True, both[:, :mix.columns], both[:, at:at + mix.out_columns])
        assert torch.equal(again, want) and torch.equal(cache, other)
    assert asked == [False, True, False, False]


# up to 256 rows: each of the four tile sizes at the most outputs that make 256 workgroups with it and at more; rows that leave one,
# 33 and 63 of a tile of 64; a contraction of less than a stage, and of one step more than whole stages
@pytest.mark.parametrize("dtype", [BF16, torch.float16])
@pytest.mark.parametrize("n", [65, 97, 127, 128, 193, 256])
@pytest.mark.parametrize("K,M", [(96, 4), (128, 340), (160, 2048), (1056, 4100), (1312, 1364), (2048, 516), (384, 8196)])
def test_products_of_row_tiles(dev, dtype, n, K, M):
    from zipage_amd import _lib
    wide = _rand(n, K + 24, seed=1, dtype=dtype).to(dev)
    x, w = wide[:, 8:8 + K], (_rand(M, K, seed=2).float() * K ** -0.5).to(dtype).to(dev)
    out = torch.full((n + 1, M + 4), 7.0, dtype=dtype, device=dev)
    args = (K, M, x.stride(0), out.stride(0), _lib.dtype_tag(x), _lib.stream_ptr(x))
    _lib.call_models("zp_row_tiles_linear", x.data_ptr(), w.data_ptr(), out.data_ptr(), n, *args)
    assert bool((out[:n, M:] == 7).all()) and bool((out[n:] == 7).all())
    want = x.double() @ w.double().T                           # bounds as for few rows
    bits = 2.0 ** (-8 if dtype == BF16 else -11)
    assert bool(((out[:n, :M].double() - want).abs() <= bits * want.abs() + 2.0 ** -20).all())
    with pytest.raises(RuntimeError, match="at most 256"):
        _lib.call_models("zp_row_tiles_linear", x.data_ptr(), w.data_ptr(), out.data_ptr(), 257, *args)
    with pytest.raises(RuntimeError, match="at most 64"):
        _lib.call_models("zp_few_rows_linear", x.data_ptr(), w.data_ptr(), out.data_ptr(), n, *args)


# every tile size, in one part and in several; a contraction that ends inside a stage, and parts of unequal length; rows and outputs
# that end inside a tile; the largest number of parts
@pytest.mark.parametrize("dtype", [BF16, torch.float16])
@pytest.mark.parametrize("n", [1, 32, 33, 64, 65, 127, 129, 192, 193, 256])
@pytest.mark.parametrize("K,M", [(32, 4), (96, 516), (1056, 1540), (4128, 512), (2080, 4100), (1024, 6148), (160, 24580), (3072, 132)])
def test_products_in_parts(dev, dtype, n, K, M):
    from zipage_amd import _lib
    wide = _rand(n, K + 24, seed=1, dtype=dtype).to(dev)
    x, w = wide[:, 8:8 + K], (_rand(M, K, seed=2).float() * K ** -0.5).to(dtype).to(dev)
    out = torch.full((n + 1, M + 4), 7.0, dtype=dtype, device=dev)
    size = _lib.size("zp_split_rows_workspace", n, K, M)
    room = torch.full((size // 4 + 4,), 7.0, device=dev)
    args = lambda n, size: (x.data_ptr(), w.data_ptr(), out.data_ptr(), n, K, M, x.stride(0), out.stride(0), _lib.dtype_tag(x),
                            room.data_ptr(), size, _lib.stream_ptr(x))
    _lib.call_models("zp_split_rows_linear", *args(n, size))
    assert bool((out[:n, M:] == 7).all()) and bool((out[n:] == 7).all()) and bool((room[size // 4:] == 7).all())
    want = x.double() @ w.double().T                           # bounds as for few rows
    bits = 2.0 ** (-8 if dtype == BF16 else -11)
    assert bool(((out[:n, :M].double() - want).abs() <= bits * want.abs() + 2.0 ** -20).all())
    if size:
        with pytest.raises(RuntimeError, match="workspace"):
            _lib.call_models("zp_split_rows_linear", *args(n, size - 16))
    with pytest.raises(RuntimeError, match="at most 256"):
        _lib.call_models("zp_split_rows_linear", *args(257, size))


@pytest.mark.parametrize("dtype", [BF16, torch.float16])
@pytest.mark.parametrize("n,K,M", [(17, 12288, 4096), (40, 4096, 1024), (100, 6144, 2048), (256, 8192, 1288), (40, 128, 4096), (5, 4096, 4096)])
def test_norms_of_products_in_parts(dev, dtype, n, K, M):
    """The norm that adds the parts up: what the product and the norm after it give; products that are made whole stay what they are."""
    from zipage_amd.layers import linear, linear_parts, rms_norm, rms_norm_parts
    x, w = _rand(n, K, seed=1, dtype=dtype).to(dev), (_rand(M, K, seed=2).float() * K ** -0.5).to(dtype).to(dev)
    weight, resid = _rand(M, seed=3, dtype=dtype).to(dev), _rand(n, M, seed=4, dtype=dtype).to(dev)
    parts, whole = linear_parts(x, w), linear(x, w)
    assert parts.dim() == (3 if 16 < n and K > 128 else 2)
    if parts.dim() == 2:
        assert torch.equal(parts, whole)
        return
    want, got = rms_norm(whole, weight, 1e-6, resid.clone()), rms_norm_parts(parts, weight, 1e-6, resid.clone())
    assert torch.equal(want[1].view(torch.int16), got[1].view(torch.int16))
    # fp16: one instruction may multiply and round to 16 bits, or two, which round a value beside a tie twice: a unit in the last place
    # (2^-10) before the weight, and the rounding after it; bf16 has no such instruction
    assert bool(((want[0].double() - got[0].double()).abs() <= (2.0 ** -9 if dtype == torch.float16 else 0.0) * want[0].double().abs()).all())
    assert float((want[0] == got[0]).float().mean()) > 0.999


@torch.inference_mode()
@pytest.mark.parametrize("n", [0, 8, 40, 65, 256])
def test_products_without_outputs(dev, n):
    from zipage_amd.layers import linear, linear_parts
    x, w = _rand(n, 1024, seed=1).to(dev), torch.empty(0, 1024, dtype=BF16, device=dev)
    assert linear(x, w).shape == linear_parts(x, w).shape == (n, 0)


@torch.inference_mode()
def test_products_in_parts_under_capture(dev):
    """Through the entry point, in a graph that is replayed on new rows."""
    from zipage_amd.layers import linear
    x, w = _rand(40, 5120, seed=3).to(dev), (_rand(2048, 5120, seed=4).float() / 72).to(BF16).to(dev)
    linear(x, w)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = linear(x, w)
    for seed in range(3):
        x.copy_(_rand(40, 5120, seed=seed).to(dev))
        g.replay()
        assert torch.equal(y, linear(x, w))
        want = x.double() @ w.double().T
        assert bool(((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -20).all())


@pytest.fixture
def few_rows_calls(monkeypatch):
    """Says whether the kernel for few rows was called since it last did."""
    from zipage_amd import _lib
    made, call = [], _lib.call_models
    monkeypatch.setattr(_lib, "call_models", lambda name, *args: (made.append(name), call(name, *args))[1])

    def called():
        n = made.count("zp_few_rows_linear")
        made.clear()
        return n > 0
    return called


def test_which_products_are_of_few_rows(dev, few_rows_calls):
    from zipage_amd.layers import linear
    w = (_rand(96, 64, seed=1).float() / 8).to(BF16).to(dev)
    wide = _rand(5, 96, seed=10).to(dev)
    for few, x in ((True, _rand(5, 64, seed=2).to(dev)), (True, _rand(1, 64, seed=2).to(dev)), (True, wide[:, 8:72]),
                   (False, _rand(65, 64, seed=4).to(dev)), (False, _rand(5, 128, seed=5).to(dev)[:, ::2]),
                   (False, _rand(5, 65, seed=6).to(dev)[:, 1:]), (False, wide[:, 1:65]), (False, _rand(2, 3, 64, seed=7).to(dev)),
                   (False, _rand(0, 64, seed=8).to(dev)), (False, _rand(64, 5, seed=9).to(dev).T)):
        want = torch.nn.functional.linear(x, w)
        got = linear(x, w)
        assert few_rows_calls() == few, x.shape
        assert got.shape == want.shape and got.dtype == want.dtype
        assert bool(((got.double() - want.double()).abs() <= 2.0 ** -7 * want.double().abs() + 2.0 ** -18).all())
    x = _rand(5, 64, seed=2).to(dev)
    with torch.inference_mode():
        linear(x, w)
    assert few_rows_calls()
    grad = w.clone().requires_grad_()
    linear(x, grad).sum().backward()
    assert grad.grad is not None and not few_rows_calls()
    with torch.no_grad():
        linear(x, grad)
    assert few_rows_calls()
    assert linear(x.float(), w.float()).dtype == torch.float32 and not few_rows_calls()
    with torch.autocast("cuda", dtype=torch.float16):
        assert linear(x, w).dtype == torch.float16 and not few_rows_calls()


def test_products_of_few_rows_keep_tangents(dev, few_rows_calls):
    import torch.autograd.forward_ad as fwd
    from zipage_amd.layers import linear
    x, t, w = (_rand(*s, seed=i, dtype=torch.float16).to(dev) / 8 for i, s in enumerate([(5, 64), (5, 64), (96, 64)]))
    with fwd.dual_level():
        got = fwd.unpack_dual(linear(fwd.make_dual(x, t), w)).tangent
    assert torch.equal(got, torch.nn.functional.linear(t, w)) and not few_rows_calls()


# ------------------------------------------------------------------ raw redundancy of few sequences
# pages of few sequences are worked on in parts (five, three, two; the claims' in eight, four and two), of twelve whole: the same bits.  Odd and
# even numbers of pages, padding, near copies of keys in their own page, in others and across the parts' edges
@pytest.mark.parametrize("dtype", [BF16, torch.float16])
@pytest.mark.parametrize("BS,pages", [(128, (9, 9, 8, 9)), (256, (3, 4, 4, 1)), (384, (2, 1, 2, 2))])
def test_raw_redundancy_in_parts(dev, dtype, BS, pages):
    from zipage_amd.kernel import raw_redudancy_score
    B, G, D = 12, 8, 64
    g = torch.Generator().manual_seed(BS)
    lens = [pages[b % 4] for b in range(B)]
    order = iter(torch.randperm(sum(lens), generator=g).tolist())
    enc = O.encode_block_table([[next(order) for _ in range(n)] for n in lens])
    keys = torch.randn(sum(lens) * BS, G, D, generator=g)
    copies = torch.randint(0, len(keys), (2, len(keys) // 4), generator=g)
    keys[copies[0]] = keys[copies[1]] + 0.3 * torch.randn(len(keys) // 4, G, D, generator=g)
    keys[BS:BS + 30] = keys[:30]
    k = keys.view(1, sum(lens), BS, G, D).to(dtype).to(dev)
    logits, red = raw_redudancy_score(k, enc.to(dev), threshold=0.5, temperature=0.4, return_logits=True)
    assert bool(torch.isfinite(logits).any())
    for first, n in ((0, 1), (1, 1), (3, 1), (0, 2), (2, 2), (1, 3), (4, 4), (0, 8)):
        few = enc[first:first + n].contiguous().to(dev)
        a, b = raw_redudancy_score(k, few, threshold=0.5, temperature=0.4, return_logits=True)
        assert torch.equal(a.view(1, n, G, -1), logits.view(1, B, G, -1)[:, first:first + n]) and torch.equal(b, red[:, first:first + n]), (first, n)


# ------------------------------------------------------------------ recurrences over runs, in pieces
# Few heads walk long runs in pieces of at least four blocks of 16 tokens: one run, runs of which some have fewer pieces than
# others or none, pieces whose last has one token or a whole block, states of earlier tokens and none; key and value sizes
# apart (the delta rule stays whole there).  The same kernels take runs whole where the workspace has room for blocks alone; token by
# token in fp32 the same sums stand in another order.
@pytest.mark.parametrize("kind", ["delta", "memory", "linear", "retention"])
@pytest.mark.parametrize("H,D,V,lens", [(1, 128, 128, (700,)), (16, 128, 128, (705, 161, 64, 1377)), (2, 32, 32, (16, 1025, 31)),
                                        (24, 64, 96, (1024, 496)), (40, 64, 64, (400, 15, 401)), (128, 32, 32, (640,))])
def test_recurrences_in_pieces(dev, monkeypatch, kind, H, D, V, lens):
    import types
    from zipage_amd import _lib
    from zipage_amd.engine.qwen3 import Segments
    from zipage_amd.layers import ChannelDelta, LinearAttention, MatrixMemory, Rotary
    W, n, rows = 64, len(lens), sum(lens)
    m = {"delta": lambda: ChannelDelta(W, H, H // 2 if H % 2 == 0 else H, D, V, 4, 1e-3),
         "memory": lambda: MatrixMemory(W, H, D, V, 15.0, 1e-3),
         "linear": lambda: LinearAttention(W, H, D, V, 1e-3, q_scale=D ** -0.5, tau=16.0, weighted=True),
         "retention": lambda: LinearAttention(W, H, D, V, 1e-3, k_scale=D ** -0.5, rotary=Rotary(1e4, D),
                                              decay=tuple(1 - 2.0 ** (-3 - 4 * i / H) for i in range(H)))}[kind]()
    shapes = m.shapes(8, 8) if kind == "delta" else m.shapes(8) if kind == "linear" else m.shapes()
    w = {k: _rand(*s, seed=i) * s[-1] ** -0.5 for i, (k, s) in enumerate(shapes.items())}
    if kind == "memory":
        w["f.b"] = (3 + _rand(H, seed=50).float()).to(BF16)
    if kind == "linear":
        w["a2.b"] = (1 + _rand(H * D, seed=51).float()).to(BF16)
    if kind == "delta":
        w["dt_bias"] = (_rand(H * D, seed=52).float() - 3).to(BF16)
    into, _ = m.load(w, BF16, dev, W)
    h = _rand(rows, W, seed=60).to(dev)
    proj = (h.float() @ into.to(dev).float().T).to(BF16)
    t = lambda a: torch.tensor(a, dtype=torch.int32, device=dev)
    first, starts = [sum(lens[:i]) for i in range(n)], [0 if i % 2 == 0 else 333 for i in range(n)]

    lib = _lib.load_models("recurrent" if kind in ("delta", "memory") else "linear")
    name = {"delta": "zp_delta_runs_workspace", "memory": "zp_mlstm_runs_workspace"}.get(kind, "zp_linear_runs_workspace")
    size = getattr(lib, name)

    def scan(runs, left=None):
        # so many heads' runs stay whole: the room that their blocks take, and `left` bytes
        room = size if left is None else lambda rows, segments, heads, *dims: size(rows, segments, 1000, *dims) // 1000 * heads + left
        monkeypatch.setattr(lib, name, room)
        state = m.allocate(n + 1, BF16, dev)
        S = state[0] if kind == "delta" else state
        S.copy_((0.1 * _rand(*S.shape, seed=61).float()).to(dev))
        if kind == "delta":
            state[1].copy_(_rand(*state[1].shape, seed=62))
        seg = Segments(t(first), t(lens), t(list(range(n, 0, -1))), t(starts), longest=max(lens))
        out = torch.empty(rows, m.out_columns, dtype=BF16, device=dev)
        ctx = types.SimpleNamespace(segments=None if runs else seg, run_segments=seg if runs else None)
        m.scan(*([h] if kind == "memory" else []), proj, state, ctx, out)
        return out.float(), S.double(), state[1] if kind == "delta" else None
    (got, gs, gt), (want, ws, wt) = scan(True), scan(False)
    for left in (0, 64):                         # and too little for the first state
        one, os, ot = scan(True, left)
        # whole runs and pieces: the planes' products leave out 2^-24 of each, sums of up to 1400 terms in fp32 stand in another order
        assert float((gs - os).norm() / os.norm()) < 2.0 ** -20, float((gs - os).norm() / os.norm())
        # rows: one in 2^12 lies so near the middle of two bf16 values that 2^-20 moves it to the other, 2^-8 away
        assert float((got - one).norm() / one.norm()) < 2.0 ** -13, float((got - one).norm() / one.norm())
        if gt is not None:
            assert torch.equal(gt[1:], ot[1:])
    with pytest.raises(RuntimeError, match="workspace too small"):
        scan(True, -4)
    # the state: sums of up to 1400 terms in fp32, each way within 2^-24 sqrt(1400) of their size, decays of 2^-23 each token
    # that forgets little; the token-by-token form takes its exponentials from another function
    assert float((gs - ws).norm() / ws.norm()) < 2.0 ** -13
    # rows: bf16 rounds both to 2^-9, one step apart where they lie on either side; small denominators amplify the rest
    assert float((got - want).norm() / want.norm()) < 2.0 ** -8
    assert bool(((got - want).abs() <= 2.0 ** -6 * want.abs() + 2.0 ** -6 * want.square().mean().sqrt()).float().mean() > 0.999)
    if gt is not None:
        assert torch.equal(gt[1:], wt[1:])       # the convolutions' last inputs

# The gates of matrix memories: as many waves as the longest run keeps busy.  A wave's remainder, all that it has, one token more; runs
# shorter than the longest; the same bits as with the sixteen that a longest run of 1100 tokens gets (whole runs: no room for pieces).
@pytest.mark.parametrize("lens", [(1,), (63, 64, 5), (65, 16), (128, 129, 17), (449, 448), (960, 961, 2), (1023,), (1025, 1024)])
def test_matrix_memory_gates_by_the_longest_run(dev, monkeypatch, lens):
    import types
    from zipage_amd import _lib
    from zipage_amd.engine.qwen3 import Segments
    from zipage_amd.layers import MatrixMemory
    W, H, D, n, rows = 64, 3, 32, len(lens), sum(lens)
    m = MatrixMemory(W, H, D, D, 15.0, 1e-3)
    w = {k: _rand(*s, seed=i) * s[-1] ** -0.5 for i, (k, s) in enumerate(m.shapes().items())}
    into, _ = m.load(w, BF16, dev, W)
    h = _rand(rows, W, seed=60).to(dev)
    proj = (h.float() @ into.to(dev).float().T).to(BF16)
    t = lambda a: torch.tensor(a, dtype=torch.int32, device=dev)
    lib = _lib.load_models("recurrent")
    size = lib.zp_mlstm_runs_workspace
    monkeypatch.setattr(lib, "zp_mlstm_runs_workspace", lambda rows, segments, heads: size(rows, segments, 1000) // 1000 * heads)

    def scan(longest):
        S = m.allocate(n + 1, BF16, dev)
        S.copy_((0.1 * _rand(*S.shape, seed=61).float()).to(dev))
        seg = Segments(t([sum(lens[:i]) for i in range(n)]), t(lens), t(list(range(n, 0, -1))), t([7 * i for i in range(n)]), longest=longest)
        out = torch.empty(rows, m.out_columns, dtype=BF16, device=dev)
        m.scan(h, proj, S, types.SimpleNamespace(segments=None, run_segments=seg), out)
        return out, S
    for got, want in zip(scan(max(lens)), scan(1100)):
        assert bool(torch.isfinite(got).all()) and torch.equal(got, want)



# ------------------------------------------------------------------ rotary store of heads of 128
# aligned rows take sixteen lanes a vector, fewer than 2^18 of them with a workgroup per sixteen; others take a wave a vector
@pytest.mark.parametrize("N,Hq,Hkv", [(1, 1, 1), (37, 32, 8), (700, 5, 2), (2047, 64, 32), (2048, 64, 32)])
@pytest.mark.parametrize("dtype", [BF16, torch.float16])
def test_rotary_store_of_wide_rows(dev, dtype, N, Hq, Hkv):
    from zipage_amd.layers import qk_norm_rope_store
    D, total, max_pos = 128, Hq + 2 * Hkv, 300
    rows = _rand(N, total * D + 16, seed=1, dtype=dtype).to(dev)
    odd = torch.empty(N * (total * D + 17) + 1, dtype=dtype, device=dev)[1:].view(N, -1)     # not on 16 bytes
    odd[:, :total * D] = rows[:, :total * D]
    qn, kn = (1 + 0.1 * _rand(D, seed=2).float()).to(dtype).to(dev), (1 + 0.1 * _rand(D, seed=3).float()).to(dtype).to(dev)
    ang = torch.arange(max_pos)[:, None] * 1e4 ** (-torch.arange(0, D, 2) / D)[None]
    cos, sin = ang.cos().to(dev), ang.sin().to(dev)
    pos = (torch.arange(N, dtype=torch.int32) * 7 % max_pos).to(dev)
    slots = torch.randperm(N + 8, generator=torch.Generator().manual_seed(2))[:N].int()
    slots[::5] = -1
    ring = torch.tensor([[i, i % 3, i // 3] if i % 2 == 0 and i < 12 else [-1] * 3 for i in range(N)], dtype=torch.int32).to(dev)
    got = []
    for x in (rows[:, :total * D], odd[:, :total * D]):
        kc, vc = (torch.zeros(N + 8, 1, Hkv, D, dtype=dtype, device=dev) for _ in range(2))
        qc = torch.zeros(3, 4, Hq, D, dtype=dtype, device=dev)
        q, k = qk_norm_rope_store(x, pos, cos, sin, qn, kn, Hq, Hkv, D, 1e-6, kc, vc, slots.to(dev), qc, ring, return_k=True)
        got.append([t.cpu() for t in (q, k, kc, vc, qc)])
    for a, b in zip(*got):                               # the same sums in the same order
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


# ------------------------------------------------------------------ recurrences over runs
def _run_segments(dev, counts):
    import types
    from zipage_amd.engine.qwen3 import Segments
    at = lambda x: torch.as_tensor(x, dtype=torch.int32).to(dev)
    rows = [sum(counts[:i]) for i in range(len(counts))]
    seg = Segments(at(rows), at(counts), at(range(len(counts))), at([0] * len(counts)), first_row=0, longest=max(counts))
    return rows, types.SimpleNamespace(segments=None, run_segments=seg)


# Blocks of 16 tokens go in pairs: one block, a second one of one token to all, a third; channels that forget little, some that
# forget everything within a block, and all of them.  Low-rank products of ranks that share a step of 32 columns, that
# fill the most that the kernels make, and that are left to the library.
@pytest.mark.parametrize("bias,spread", [(-3.0, 1.0), (-2.0, 6.0), (12.0, 1.0)])
@pytest.mark.parametrize("H,G,D,V,taps,ranks", [(2, 1, 128, 128, 4, (128, 128)), (3, 3, 64, 64, 2, (40, 72)), (2, 1, 32, 96, 8, (8, 8)),
                                                (1, 1, 128, 32, 1, (136, 8)), (2, 2, 64, 128, 3, (100, 16))])
def test_delta_runs_in_pairs_of_blocks(dev, H, G, D, V, taps, ranks, bias, spread):
    import types
    from zipage_amd.engine.qwen3 import Segments
    from zipage_amd.layers import ChannelDelta
    counts, W = [1, 15, 16, 17, 31, 32, 33, 48, 49, 64, 65, 97], 64
    m, n, rows = ChannelDelta(W, H, G, D, V, taps, 1e-3), len(counts), sum(counts)
    shapes = m.shapes(*ranks)
    w = {k: _rand(*s, seed=i) * s[-1] ** -0.5 for i, (k, s) in enumerate(shapes.items())}
    w["dt_bias"] = (bias + spread * _rand(H * D, seed=52).float()).to(BF16)
    into, _ = m.load(w, BF16, dev, W)
    assert (m.low_tiles is None) == (max(ranks) > 128)
    proj = (_rand(rows, W, seed=60).to(dev).float() @ into.to(dev).float().T).to(BF16)
    t = lambda a: torch.tensor(a, dtype=torch.int32, device=dev)
    seg = Segments(t([sum(counts[:i]) for i in range(n)]), t(counts), t(list(range(n, 0, -1))),
                   t([0 if i % 2 or c < taps else 333 for i, c in enumerate(counts)]), longest=max(counts))

    def scan(runs):
        state = m.allocate(n + 1, BF16, dev)
        state[0].copy_((0.1 * _rand(*state[0].shape, seed=61).float()).to(dev))
        state[1].copy_(_rand(*state[1].shape, seed=62))
        out = torch.empty(rows, m.out_columns, dtype=BF16, device=dev)
        m.scan(proj, state, types.SimpleNamespace(segments=None if runs else seg, run_segments=seg if runs else None), out)
        return out.float(), state[0].double()
    (got, gs), (want, ws) = scan(True), scan(False)
    # as in pieces of runs: sums of up to 100 terms in fp32, exponentials of another function; rows rounded to 2^-9
    assert float((gs - ws).norm() / ws.norm()) < 2.0 ** -15
    assert float((got - want).norm() / want.norm()) < 2.0 ** -8 and bool(torch.isfinite(got).all())


# Decoded tokens and short portions beside runs: a row's low-rank products are made once, by the library for portions and by the kernels for
# runs, which get what they would of a step of their own; by the library for all rows where the portions' may be any.
@pytest.mark.parametrize("short,known", [((1, 1, 1), True), ((3, 15), True), ((3, 15), False), ((), True)])
def test_delta_steps_of_runs_and_portions(dev, monkeypatch, short, known):
    import types
    from zipage_amd import _lib
    from zipage_amd.engine.qwen3 import Segments
    from zipage_amd.layers import ChannelDelta, recurrent
    H, G, D, taps, W, counts = 4, 2, 128, 4, 64, [*short, 64, 100]
    m, n, rows, first = ChannelDelta(W, H, G, D, D, taps, 1e-3), len(counts), sum(counts), sum(short)
    into, _ = m.load({k: _rand(*s, seed=i) * s[-1] ** -0.5 for i, (k, s) in enumerate(m.shapes(128, 128).items())}, BF16, dev, W)
    proj = (_rand(rows, W, seed=60).to(dev).float() @ into.to(dev).float().T).to(BF16)
    t = lambda a: torch.tensor(a, dtype=torch.int32, device=dev)

    def segments(i, j, **kw):
        return Segments(t([sum(counts[:k]) for k in range(i, j)]), t(counts[i:j]), t(list(range(i, j))), t([7] * (j - i)), **kw) if j > i else None
    portions = segments(0, len(short), end=first if known else 0)
    runs = segments(len(short), n, first_row=first, longest=max(counts))

    def scan(portions, runs, tiles=True):
        calls, call, product = [], _lib.call_models, recurrent.step_product
        with monkeypatch.context() as patch:
            patch.setattr(_lib, "call_models", lambda name, *a: (calls.append(name), call(name, *a)))
            patch.setattr(recurrent, "step_product", lambda ctx: lambda x, w: (calls.append(x.shape[0]), product(ctx)(x, w))[1])
            patch.setattr(m, "low_tiles", m.low_tiles if tiles else None)
            state = m.allocate(n, BF16, dev)
            state[0].copy_((0.1 * _rand(*state[0].shape, seed=61).float()).to(dev))
            out = torch.empty(rows, m.out_columns, dtype=BF16, device=dev)
            m.scan(proj, state, types.SimpleNamespace(segments=portions, run_segments=runs), out)
        return calls, out, state[0]
    calls, got, gs = scan(portions, runs)
    made = known or not short
    assert calls == ([first if known else rows, "zp_delta_scan"] if short else []) + ["zp_delta_runs_projected" if made else "zp_delta_runs"]
    _, alone, state = scan(None, runs, made)
    assert torch.equal(got[first:], alone[first:]) and torch.equal(gs[len(short):], state[len(short):])
    if short:
        _, other, state = scan(portions, None)
        # pre-activations that another order of sums rounds to the next bf16 value, one in some hundred
        assert float((got[:first] - other[:first]).float().norm() / other[:first].float().norm()) < 2.0 ** -7
        assert float((gs[:len(short)] - state[:len(short)]).norm() / state[:len(short)].norm()) < 2.0 ** -9


# operands enter the bf16 matrix cores in three planes: the state has to stay as good as fp32's
@pytest.mark.parametrize("H,G,D,V", [(2, 1, 128, 128), (2, 2, 32, 96), (3, 1, 64, 32), (1, 1, 128, 64)])
def test_delta_state_of_runs(dev, H, G, D, V):
    from zipage_amd.layers import ChannelDelta
    W, taps, counts = 64, 2, [16, 47, 100]
    m, n = ChannelDelta(W, H, G, D, V, taps, 1e-3), sum(counts)
    r = lambda *s, seed, std=1.0: _rand(*s, seed=seed, std=std)
    w = {"q": r(G * D, W, seed=1, std=.2), "k": r(G * D, W, seed=2, std=.2), "v": r(H * V, W, seed=3, std=.2),
         "q.conv": r(G * D, taps, seed=4), "k.conv": r(G * D, taps, seed=5), "v.conv": r(H * V, taps, seed=6),
         "b": r(H, W, seed=7, std=.2), "A_log": r(H, seed=8, std=.5), "norm": 1 + r(V, seed=9, std=.3),
         "a1": r(5, W, seed=10, std=.1), "a2": r(H * D, 5, seed=11, std=.4), "dt_bias": -3 + 6 * r(H * D, seed=12),
         "g1": r(7, W, seed=13, std=.1), "g2": r(H * V, 7, seed=14, std=.4), "o": r(W, H * V, seed=15)}
    into, _ = m.load(w, BF16, dev, W)
    proj = (r(n, W, seed=16).float() @ into.float().cpu().T).to(BF16).to(dev)
    state = m.allocate(len(counts), BF16, dev)
    rows, ctx = _run_segments(dev, counts)
    m.scan(proj, state, ctx, torch.empty(n, H * V, dtype=BF16, device=dev))
    P, head = proj.double().cpu(), torch.arange(H) // (H // G)
    low = torch.nn.functional.linear(proj[:, m.low_at:m.low_at + m.low_rank], m.low).double().cpu()
    a = low[:, :H * D].view(n, H, D) + w["dt_bias"].double().view(H, D)
    g = torch.exp(-torch.exp(w["A_log"].double())[None, :, None] * torch.nn.functional.softplus(a))
    for i, c in enumerate(counts):
        p, gg = P[rows[i]:rows[i] + c], g[rows[i]:rows[i] + c]
        conv = lambda f, t, k: K.short_conv(p[:, f:t], w[k + ".conv"].double())
        k = K.unit(conv(G * D, 2 * G * D, "k").view(c, G, D))[:, head]
        v = conv(2 * G * D, 2 * G * D + H * V, "v").view(c, H, V)
        beta, S = torch.sigmoid(p[:, m.b_at:m.b_at + H]), torch.zeros(H, D, V, dtype=torch.float64)
        for t in range(c):
            S = gg[t][:, :, None] * S
            u = beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
            S = S + k[t][:, :, None] * u[:, None, :]
        # roundings of 2^-24 by the products, decays and unit vectors of the tokens that a state remembers; a product of
        # planes that is left out costs 2^-17 and more
        err = (state[0][i].double().cpu().view(H, D, V) - S).norm() / S.norm()
        assert float(err) < 2.0 ** -19, float(err)


# Channels that forget `bits` a token, or hardly anything but 5 to 14 at every sixteenth: A, P and what the state gets of a key are
# sums of running products, which carry no rounding of what was forgotten before.  Low-rank products of one term each, which are exact.
@pytest.mark.parametrize("bits", [0.05, 0.5, 3.0, 8.0, "spikes"])
def test_delta_state_of_channels_that_forget(dev, bits):
    from zipage_amd.layers import ChannelDelta
    H, G, D, V, W, taps, rank, counts = 4, 2, 128, 128, 64, 4, 64, [160, 96, 47]
    m, n, g = ChannelDelta(W, H, G, D, V, taps, 1e-6), sum(counts), torch.Generator().manual_seed(3)
    r = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(BF16)
    w = {k: r(*s) for k, s in m.shapes(rank, rank).items()} | {k: r(*m.shapes(rank, rank)[k], std=.5) for k in ("q.conv", "k.conv", "v.conv")}
    w |= {"A_log": torch.zeros(H, dtype=BF16), "dt_bias": torch.zeros(H * D, dtype=BF16), "a2": torch.zeros(H * D, rank, dtype=BF16)}
    column = torch.randint(rank, (H * D,), generator=g)
    w["a2"][torch.arange(H * D), column] = 1
    m.load(w, BF16, dev, W)
    P = r(n, m.columns, std=.5)
    if bits == "spikes":
        forgets = torch.where(torch.rand(n, rank, generator=g) < 1 / 16, 5 + 9 * torch.rand(n, rank, generator=g), 0.01)
    else:
        forgets = bits * torch.exp(.3 * torch.randn(n, rank, generator=g))
    P[:, m.low_at:m.low_at + rank] = torch.log(torch.expm1(forgets.double() * 0.6931471805599453)).to(BF16)      # softplus gives it back
    state = m.allocate(len(counts), BF16, dev)
    rows, ctx = _run_segments(dev, counts)
    m.scan(P.to(dev), state, ctx, torch.empty(n, H * V, dtype=BF16, device=dev))
    P, head = P.double(), torch.arange(H) // (H // G)
    decay = torch.exp(-torch.nn.functional.softplus(P[:, m.low_at:m.low_at + rank]))[:, column].view(n, H, D)
    for i, c in enumerate(counts):
        p, gg = P[rows[i]:rows[i] + c], decay[rows[i]:rows[i] + c]
        conv = lambda f, t, k: K.short_conv(p[:, f:t], w[k + ".conv"].double())
        k = K.unit(conv(G * D, 2 * G * D, "k").view(c, G, D))[:, head]
        v = conv(2 * G * D, 2 * G * D + H * V, "v").view(c, H, V)
        beta, S = torch.sigmoid(p[:, m.b_at:m.b_at + H]), torch.zeros(H, D, V, dtype=torch.float64)
        for t in range(c):
            S = gg[t][:, :, None] * S
            u = beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
            S = S + k[t][:, :, None] * u[:, None, :]
        # Roundings of 2^-24 by the products, decays and unit vectors of the tokens that a state remembers: one or two of them where
        # channels forget 3 bits and more, each with a unit vector, a step size, a value and a few decays (1.1e-7 measured for 3 bits; 5.9e-7
        # with quotients of decays).
        err = float((state[0][i].double().cpu().view(H, D, V) - S).norm() / S.norm())
        assert err < (2.0 ** -22 if bits in (3.0, 8.0) else 2.0 ** -20), err


# linear attention and matrix memory likewise; rows of values, and of the memory's keys, are bf16 as they come
@pytest.mark.parametrize("H,D,V", [(2, 128, 128), (2, 32, 96), (3, 64, 32), (1, 128, 64)])
@pytest.mark.parametrize("mixer", ["linear", "memory"])
def test_states_of_runs(dev, mixer, H, D, V):
    from zipage_amd.layers import LinearAttention, MatrixMemory
    W, counts, tau, cap = 64, [16, 47, 100], 8.0, 3.0
    r = lambda *s, seed, std=1.0: _rand(*s, seed=seed, std=std)
    w = {k: r(H * (V if k in "vg" else D), W, seed=i, std=.2) for i, k in enumerate("qkvg")} | {"o": r(W, H * V, seed=5)}
    if mixer == "linear":
        m = LinearAttention(W, H, D, V, 1e-3, k_scale=0.5, tau=tau, weighted=True)
        w |= {"norm": r(V, seed=6), "a1": r(5, W, seed=7, std=.1), "a2": r(H * D, 5, seed=8, std=.4), "a2.b": 6 * r(H * D, seed=9)}
    else:
        m = MatrixMemory(W, H, D, V, cap, 1e-3)
        w |= {"norm": r(H * V, seed=6), "i": r(H, W, seed=7, std=.3), "i.b": r(H, seed=8), "f": r(H, W, seed=9, std=.2),
              "f.b": 3 + r(H, seed=10)}
    into, _ = m.load(w, BF16, dev, W)
    n = sum(counts)
    h = r(n, W, seed=16)
    proj = (h.float() @ into.float().cpu().T).to(BF16).to(dev)
    state, out = m.allocate(len(counts), BF16, dev), torch.empty(n, H * V, dtype=BF16, device=dev)
    rows, ctx = _run_segments(dev, counts)
    m.scan(*([h.to(dev)] if mixer == "memory" else []), proj, state, ctx, out)
    P, hh = proj.double().cpu(), h.double()
    k, v = P[:, H * D:2 * H * D].view(n, H, D), P[:, 2 * H * D:2 * H * D + H * V].view(n, H, V)
    if mixer == "linear":
        low = torch.nn.functional.linear(proj[:, m.low_at:m.low_at + m.low_rank], m.low).double().cpu()
        g = (torch.sigmoid(low.view(n, H, D) + w["a2.b"].double().view(H, D)) ** (1 / tau))[..., None]
        k = k * 0.5
    else:
        i = cap * torch.tanh((hh @ w["i"].double().T + w["i.b"].double()) / cap)
        f = torch.nn.functional.logsigmoid(cap * torch.tanh((hh @ w["f"].double().T + w["f.b"].double()) / cap))
    for s, (a, c) in enumerate(zip(rows, counts)):
        S, top = torch.zeros(H, D, V, dtype=torch.float64), torch.zeros(H, dtype=torch.float64)
        for t in range(a, a + c):
            if mixer == "linear":
                S = g[t] * S + k[t][:, :, None] * v[t][:, None, :]
            else:
                new = torch.maximum(f[t] + top, i[t])
                S = torch.exp(f[t] + top - new)[:, None, None] * S + (torch.exp(i[t] - new)[:, None] * k[t])[:, :, None] * v[t][:, None, :]
                top = new
        # as above; the memory's gates are sums of 64 products in fp32, whose error their exponentials take over
        err = (state[s][..., :D * V].flatten(1).double().cpu().view(H, D, V) - S).norm() / S.norm() if mixer == "memory" else \
            (state[s].double().cpu().view(H, D, V) - S).norm() / S.norm()
        assert float(err) < 2.0 ** -19, float(err)


# ------------------------------------------------------------------ latent rows
# up to 32 heads of up to 256 columns a wave goes its own way; more of either: a ring of stages of 32 keys, page ids
# fetched 64 at a time, a token's keys cut into ranges of at least four stages
@pytest.mark.parametrize("H,R,P,BS,window", [(1, 288, 8, 16, None), (17, 512, 64, 16, 1100), (33, 128, 24, 16, None),
                                             (48, 256, 0, 32, 65), (65, 384, 40, 16, 1), (32, 256, 8, 16, None),
                                             (16, 512, 0, 64, None), (128, 32, 64, 16, 700), (24, 352, 24, 16, 300),
                                             (9, 416, 16, 32, None)])
def test_latent_rows_by_width_and_heads(dev, H, R, P, BS, window):
    from zipage_amd.layers import latent_rows_attention
    ctx = [0, 1, 31, 32, 33, 63, 64, 65, 96, 97, 128, 129, 130, 160, 193, 1023, 1024, 1025, 2080, 2500]
    n, NB = len(ctx), -(-2500 // BS)
    g = torch.Generator().manual_seed(H + R)
    tables = torch.randperm(n * NB, generator=g).view(n, NB).int()
    cache, q = _rand(n * NB, BS, R + P, seed=3), _rand(n, H, R + P, seed=4, std=4.0 * (R + P) ** -0.5)
    want = torch.zeros(n, H, R, dtype=torch.double)
    absolute = torch.zeros_like(want)
    for i, c in enumerate(ctx):
        low = max(0, c - window) if window else 0
        if c:
            rows = cache[tables[i].long()].reshape(-1, R + P)[low:c].double()
            p = (q[i].double() @ rows.T).softmax(-1)
            want[i], absolute[i] = p @ rows[:, :R], p @ rows[:, :R].abs()
        tables[i, :low // BS] = -1                       # in front of the window: never read
        tables[i, -(-c // BS):] = 1 << 30                # nor past the last key
    t = lambda a: torch.as_tensor(a, dtype=torch.int32).to(dev)
    qd, cd, td = q.to(dev), cache.to(dev), t(tables)
    # probabilities in bf16 (2^-8 of a term and as much of the sum they are over), the result once more (2^-8); in two
    # planes 2^-17 of a term, and fp32 scores of up to 20 and their exponentials 2^-14 of it
    weights = 2 * 2.0 ** -8 if R <= 256 and H <= 32 else 2.0 ** -13
    allowed = (weights * absolute + 2.0 ** -8 * want.abs()) * 1.01 + 1e-6
    got = latent_rows_attention(qd, cd, td, t(ctx), 1.0, window, rank=R).cpu().double()
    assert not got[0].any()
    assert ((got - want).abs() <= allowed).all()
    for i in (8, 16, 19):                                # alone: its keys cut into more ranges
        one = latent_rows_attention(qd[i:i + 1], cd, td[i:i + 1], t(ctx[i:i + 1]), 1.0, window, rank=R).cpu().double()
        assert ((one - want[i:i + 1]).abs() <= allowed[i:i + 1]).all()


def _contexts_past_the_cache(row_bytes):
    """As many contexts as make tokens of 2500 keys take the call to read 320 MB, and those of 700 not."""
    once = [0, 1, 33, 700, 1024, 2500]
    ctx = once * (-(-(320 << 20) // (2500 * row_bytes)) // len(once) + 1)
    assert len(ctx) * 700 * row_bytes < 320 << 20 <= len(ctx) * 2500 * row_bytes
    return ctx


# a pool and tables of 320 MB and more: rows are asked for past the last-level cache, in some kernels by the tokens whose contexts
# say so, by the same sums
@pytest.mark.parametrize("H,R,P", [(16, 512, 64), (20, 320, 64), (33, 512, 64), (40, 128, 64), (65, 512, 0),
                                   (20, 256, 64), (16, 128, 0), (32, 256, 0)])
def test_latent_rows_past_the_cache(dev, H, R, P):
    from zipage_amd.layers import latent_rows_attention
    BS, used, ctx = 1024, 8, _contexts_past_the_cache((R + P) * 2)
    pages = (320 << 20) // (BS * (R + P) * 2) + 1
    cache = torch.zeros(pages, BS, R + P, dtype=torch.bfloat16, device=dev)
    cache[:used] = _rand(used, BS, R + P, seed=H).to(dev)
    tables = torch.full((len(ctx), pages), -1, dtype=torch.int32)
    for i, c in enumerate(ctx):
        tables[i, :-(-c // BS)] = (torch.arange(-(-c // BS)) * 3 + i).int() % used
    q = _rand(len(ctx), H, R + P, seed=R, std=4.0 * (R + P) ** -0.5).to(dev)
    t, n = tables.to(dev), torch.tensor(ctx, dtype=torch.int32, device=dev)
    past = latent_rows_attention(q, cache, t, n, 1.0, None, rank=R)
    assert torch.equal(past, latent_rows_attention(q, cache[:used].clone(), t, n, 1.0, None, rank=R))
    assert past[n > 0].any(-1).all()


@pytest.mark.parametrize("H,G,D,V", [(8, 2, 128, 128), (16, 1, 64, 64), (6, 2, 96, 256), (34, 2, 128, 128)])
def test_grouped_rows_past_the_cache(dev, H, G, D, V):
    from zipage_amd.layers.grouped import grouped_rows_attention
    BS, used, row = 1024, 8, G * (D + V)
    ctx = _contexts_past_the_cache(row * 2)
    pages = (320 << 20) // (BS * row * 2) + 1
    cache = torch.zeros(pages, BS, row, dtype=torch.bfloat16, device=dev)
    cache[:used] = _rand(used, BS, row, seed=H).to(dev)
    tables = torch.full((len(ctx), pages), -1, dtype=torch.int32)
    for i, c in enumerate(ctx):
        tables[i, :-(-c // BS)] = (torch.arange(-(-c // BS)) * 3 + i).int() % used
    q = _rand(len(ctx), H * D, seed=D).to(dev)
    t, n = tables.to(dev), torch.tensor(ctx, dtype=torch.int32, device=dev)
    got = [torch.empty(len(ctx), H * V, dtype=torch.bfloat16, device=dev) for _ in range(2)]
    for out, c in zip(got, (cache, cache[:used].clone())):
        grouped_rows_attention(q, c, H, G, D, V, t, n, D ** -0.5, out)
    assert torch.equal(*got) and got[0][n > 0].any(-1).all()


# ------------------------------------------------------------------ per-head products
# through LDS: tiles of 64 outputs by 16, 32 or 64 tokens, stages of 128 elements in a ring of four; straight from
# memory: contractions below 256 (512 with fewer than 64 outputs) and below 8192 matrix products
@pytest.mark.parametrize("n,H,K,M,tail", [(1, 2, 160, 16, 0), (16, 3, 128, 80, 8), (16, 65, 128, 272, 0), (17, 3, 544, 48, 0),
                                          (33, 64, 128, 144, 64), (65, 8, 1056, 64, 0), (129, 130, 96, 112, 8),
                                          (64, 256, 32, 16, 24), (200, 72, 640, 128, 0), (9, 3, 256, 64, 8), (9, 3, 224, 64, 8),
                                          (40, 171, 64, 128, 0), (39, 171, 64, 128, 0), (33, 4, 480, 48, 0), (24, 512, 128, 48, 8),
                                          (1300, 33, 32, 64, 8), (70, 3, 192, 80, 40), (200, 70, 64, 64, 64)])
def test_headwise_by_tokens_and_contraction(dev, n, H, K, M, tail):
    from zipage_amd.layers.latent import headwise_linear
    x, w = _rand(n, H, K + tail, seed=6), _rand(H, M, K, seed=7)
    x[n - 1, H - 1, :K] = float("inf")                   # a row of its own: nothing else may see it
    got = headwise_linear(x.to(dev), w.to(dev)).cpu().double()
    assert torch.equal(got[..., M:], x[..., K:].double())
    live = torch.ones(n, H, dtype=torch.bool)
    live[n - 1, H - 1] = False
    a, b = x[..., :K].double().transpose(0, 1), w.double().transpose(1, 2)
    a[H - 1, n - 1] = 0
    want, absolute = (a @ b).transpose(0, 1), (a.abs() @ b.abs()).transpose(0, 1)
    # fp32 sums of K products, then bf16
    allowed = K * 2.0 ** -24 * absolute + 2.0 ** -8 * want.abs() + 1e-30
    assert ((got[..., :M] - want).abs() <= allowed)[live].all()
    assert not got[n - 1, H - 1, :M].isfinite().any()


# ------------------------------------------------------------------ few outputs
# from 4 081 rows, 17 outputs, a contraction of 256 and 2.2 million elements of x on through LDS: 32 tokens by 32 or 64
# outputs, stages of 128 elements
@pytest.mark.parametrize("n,K,M", [(4080, 160, 20), (4081, 32, 20), (4099, 160, 32), (4095, 1056, 36), (4100, 96, 100),
                                   (5000, 640, 64), (4113, 4128, 132), (8594, 256, 20), (8593, 256, 20), (8100, 224, 36),
                                   (6900, 320, 100), (4099, 544, 32)])
def test_small_linear_of_many_rows(dev, n, K, M):
    from zipage_amd.layers import small_linear
    x, w = _rand(n, K + 8, seed=8)[:, :K], _rand(M, K, seed=9)
    got = small_linear(x.to(dev)[:, :K], w.to(dev)).cpu().double()
    want, absolute = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    assert ((got - want).abs() <= K * 2.0 ** -24 * absolute + 1e-30).all()


# decoded tokens: a layer's states of 320 MB and more go past the cache; those of inert segments count, but aren't there
@pytest.mark.parametrize("mixer", ["linear", "delta"])
def test_decoded_states_past_the_cache(dev, mixer):
    from zipage_amd.engine.qwen3 import Segments
    from zipage_amd.layers import ChannelDelta, LinearAttention
    import types
    W, H, D, live, n = 64, 8, 128, 4, 640                # 640 states of 8 x 128 x 128 in fp32: 320 MB
    r = lambda *s, seed, std=1.0: _rand(*s, seed=seed, std=std)
    if mixer == "linear":
        m = LinearAttention(W, H, D, D, 1e-3, k_scale=0.5, decay=tuple(1 - 2.0 ** -(2 + h) for h in range(H)), weighted=True)
        w = {k: r(H * D, W, seed=i, std=.2) for i, k in enumerate("qkvg")} | {"o": r(W, H * D, seed=5), "norm": r(D, seed=6)}
    else:
        m = ChannelDelta(W, H, H, D, D, 2, 1e-3)
        w = {k: r(H * D, W, seed=i, std=.2) for i, k in enumerate("qkv")}
        w |= {k + ".conv": r(H * D, 2, seed=i) for i, k in enumerate("qkv", 4)}
        w |= {"b": r(H, W, seed=7, std=.2), "A_log": r(H, seed=8, std=.5), "norm": 1 + r(D, seed=9, std=.3),
              "a1": r(5, W, seed=10, std=.1), "a2": r(H * D, 5, seed=11, std=.4), "dt_bias": -3 + 6 * r(H * D, seed=12),
              "g1": r(7, W, seed=13, std=.1), "g2": r(H * D, 7, seed=14, std=.4), "o": r(W, H * D, seed=15)}
    into, _ = m.load(w, BF16, dev, W)
    proj = (r(n, W, seed=16).float() @ into.float().cpu().T).to(BF16).to(dev)
    t = lambda *a: torch.tensor(a, dtype=torch.int32, device=dev)
    results = []
    for size in (live, n):
        state, out = m.allocate(live, BF16, dev), torch.empty(size, H * D, dtype=BF16, device=dev)
        for step in range(3):                            # the second reads what the first wrote
            rest = [0] * (size - live)
            ctx = types.SimpleNamespace(segments=Segments(None, t(1, 1, 1, 1, *rest), t(2, 0, 3, 1, *rest),
                                                          t(step, 5 + step, step, 0, *rest), max_count=1), run_segments=None)
            m.scan(proj[:size], state, ctx, out)
        assert not out[live:].any()
        results.append((out[:live].double(), [x.double() for x in state]))
    (a, sa), (b, sb) = results
    close = lambda x, y: float((x - y).norm()) <= (0.0 if mixer == "linear" else 2.0 ** -7) * float(x.norm())
    # linear: the same sums.  The delta rule's low-rank products are the library's, which may round other row counts otherwise
    assert close(a, b) and all(close(x, y) for x, y in zip(sa, sb)) and a.any()


# ------------------------------------------------------------------ products of a step
@pytest.mark.parametrize("model", ["kapolorn", "mefupel", "pedivik", "rutevik"])
def test_prompts_keep_the_librarys_products(dev, few_rows_calls, tmp_path, model):
    """Portions of prompts, attended as runs or token by token, and a portion beside a decoded token: none of their products is one of few
    rows, as none of a whole prompt is; those of decoded tokens alone are."""
    import importlib
    import json
    from zipage_amd.engine import EngineConfig, ZipageEngine, read_shape
    from zipage_amd.engine.weights import write_safetensors
    C = importlib.import_module(f"tests.{model}_cases")
    cfg, w = C.case("wide" if "wide" in C.CONFIGS else sorted(C.CONFIGS)[0])
    (tmp_path / "config.json").write_text(json.dumps(cfg))
    write_safetensors(str(tmp_path / "model.safetensors"), w)
    eng = ZipageEngine(EngineConfig(shape=read_shape(str(tmp_path)), model_folder=str(tmp_path), dtype=BF16, num_kvcache_blocks=64,
                                    kvcache_block_size=16, max_concurrency=6, use_graph=False))
    toks = C.tokens(cfg, 60, 1)
    a, b = eng.open_request(), eng.open_request()
    for step in ([(a, toks[:24], [])], [(a, toks[24:29], [])], [(a, toks[29:30], []), (b, toks[:20], [])]):
        eng.feed(step)
        assert not few_rows_calls(), [len(t) for _, t, _ in step]
    eng.feed([(a, toks[30:31], []), (b, toks[20:21], [])])
    assert few_rows_calls()


# ------------------------------------------------------------------ redundancy over all pairs, 16 bit
# Pages of one or two tiles of 128 keys are their own first tiles, larger ones read their rows apart and take several rounds; pages
# that are no whole tiles take the general form.  Rows of a multiple of eight share an XCD; few pages go in parts.  Chains of 16, 8,
# 24, 32 and 12 chunks a page, whose ends fall anywhere among the 32 that are taken at a time.  The longest row of pages of 256.
@pytest.mark.parametrize("dtype,BS,D,Hkv,pages,thr", [
    (BF16, 256, 128, 3, (5, 2), 0.5), (BF16, 256, 64, 8, (4, 1), 0.5), (torch.float16, 128, 128, 4, (7, 3), 0.3), (BF16, 384, 96, 1, (3,), 0.5),
    (torch.float16, 512, 32, 2, (2, 3), 0.9), (BF16, 192, 128, 2, (3, 5), 0.5), (BF16, 256, 128, 8, (4, 3) * 8, 0.5), (BF16, 128, 128, 8, (9,) * 6, 0.5),
    (BF16, 256, 128, 8, (4, 3) * 8, 0.0), (BF16, 256, 64, 1, (51,), 0.5)])
def test_all_pairs_forms(dev, dtype, BS, D, Hkv, pages, thr):
    from tests.test_redundancy_planted import _clear_of_norm_boundaries, _close_in_ulps
    from zipage_amd.kernel import raw_redudancy_score
    g = torch.Generator().manual_seed(BS + D)
    order = torch.randperm(sum(pages), generator=g).tolist()
    tables = [[order.pop() for _ in range(n)] for n in pages]
    enc = O.encode_block_table(tables)
    k = torch.randn((1, sum(pages), BS, Hkv, D), generator=g)
    for t in tables:                                 # a quarter of a sequence's keys are another one's direction, some of them longer
        rows = k[0, t].reshape(-1, Hkv, D)
        n = rows.shape[0] // 4
        to, src = torch.randperm(rows.shape[0], generator=g)[:n], torch.randint(rows.shape[0], (n,), generator=g)
        rows[to] = rows[src] * torch.where(torch.rand(n, 1, 1, generator=g) < 0.2, 4.0, 1.0)
        k[0, t] = rows.view(len(t), BS, Hkv, D)
    k = _clear_of_norm_boundaries(k.to(dtype))
    want, scale = O.raw_redudancy_logits(k, enc, thr, return_partial_max=True)
    got, _ = raw_redudancy_score(k.to(dev), enc.to(dev), threshold=thr, temperature=0.4, return_logits=True)
    _close_in_ulps(got, want, dtype, ulps=1, frac_exact=0.95, chain_scale=scale)
