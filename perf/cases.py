"""What a serving host has this framework do, as cases that can be timed and compared.

Every case is one unit of a decode loop's work through the public entry points (``cpm.cu_amd.ops``, ``cpm.cu_amd.driver``):

  step      one speculative verify step (``VerifyStep``): per layer KV append + tree attention, target head with arg-max, greedy
            acceptance, compaction, and the read-back of (accept length, ids) the host needs before it can go on.  Enqueued call by
            call, or replayed from a HIP graph as a decode loop with static buffers does.
  decode    one token without a drafter: rotary table, per layer append + attention of one query (rotation fused), target head.
  draft     one whole draft: per round FR-Spec head + log-softmax + top-k, drafter-layer attention behind its block window, tree
            bookkeeping, and the final tree.
  prefill   the cache side of one prompt chunk: K/V rows of every layer appended to the paged cache.
  logprobs  target head with logits, log-softmax and top-k: what a sampler or a logprobs request takes from the head.

The listed shapes are those of ``synth.CONFIGS`` / ``synth.MINICPM4_8B`` with the odd lengths, element types, head counts and weight
layouts that the tests and the sweeps cover.  Head weights and hidden rows sit on a 16-level and an 8-bit grid (the values a 4-bit
checkpoint dequantises to): every dot product is then exact in fp32 whatever the order of summation, so that token ids and
positions are the same whole numbers for every correct implementation.
"""
import math

import numpy as np
import torch

from cpm.cu_amd import lib, ops, synth
from cpm.cu_amd.driver import VerifyStep
from cpm.cu_amd.kvcache import HEAD_DIM, PAGE, PagedKVCache

WINDOW = 1024             # the drafter layer's block window, in tokens
HEAD_SCALE = 0.0625       # the target head's pre-scale
LARGEST_ROWS = 32 * 131072 * 60  # layers * context * query rows, and
LARGEST_CACHE = 32 * 131072 * 2  # layers * context * KV heads: what no drawn case exceeds


def _step(name, layers, prefix, nodes, iters, topk, vocab=73448, hidden=4096, q_heads=32, kv_heads=2, bf16=False, graph=True):
    return dict(name=name, kind="step", layers=layers, prefix=prefix, nodes=nodes, iters=iters, topk=topk, vocab=vocab, hidden=hidden,
                q_heads=q_heads, kv_heads=kv_heads, bf16=bf16, graph=graph)


def listed():
    return [
        # a one-layer model with a small vocabulary, called operator by operator: launches and host calls are the time
        _step("step_1layer_1k_16", 1, 1024, 16, 4, 4, vocab=8192, graph=False),
        # the headline: 60-node tree behind 4K tokens, 32 layers
        _step("step_4k_60", 32, 4096, 60, 6, 10),
        # the same trees behind long prompts
        _step("step_32k_60", 32, 32768, 60, 6, 10),
        _step("step_128k_60", 32, 131072, 60, 6, 10),
        # a tree wider than one mask word
        _step("step_32k_128", 32, 32768, 128, 8, 16),
        # bfloat16, four query heads per KV head, odd sizes, enqueued call by call
        _step("step_bf16_10007_33", 32, 10007, 33, 5, 8, kv_heads=8, bf16=True, graph=False),
        # generation without a drafter: short and long context
        dict(name="decode_4k", kind="decode", layers=32, prefix=4096, vocab=73448, hidden=4096, q_heads=32, kv_heads=2, bf16=False),
        dict(name="decode_60001", kind="decode", layers=32, prefix=60001, vocab=73448, hidden=4096, q_heads=32, kv_heads=2, bf16=True),
        # one draft at the reference's settings (6 rounds of 10 on a 32768-row sub-vocabulary), replayed from a graph
        dict(name="draft_6x10_32768", kind="draft", prefix=4096, nodes=60, iters=6, topk=10, vocab=73448, sub=32768, hidden=4096, bf16=False, graph=True),
        # a shallow drafter with a small sub-vocabulary, called operator by operator
        dict(name="draft_4x4_8192", kind="draft", prefix=1000, nodes=16, iters=4, topk=4, vocab=73448, sub=8192, hidden=4096, bf16=False, graph=False),
        # one 2048-token chunk of a prompt into the caches of 32 layers, in the middle of a page
        dict(name="prefill_2048", kind="prefill", layers=32, prefix=4000, rows=2048, kv_heads=2),
        # log-probabilities of a few rows over a full vocabulary of odd length, from the row-major matrix as a checkpoint holds it
        dict(name="logprobs_5_73449", kind="logprobs", rows=5, topk=20, vocab=73449, hidden=4096, tiled=False, bf16=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "decode", "draft", "draft", "prefill", "logprobs"])
    bf16 = rng.random() < 0.3
    heads = dict(q_heads=32, kv_heads=rng.choice([2, 2, 2, 4, 8]))
    if kind == "step":
        topk = rng.choice([4, 8, 10, 16])
        iters = rng.randint(3, 64 // topk if topk > 8 else 8)
        nodes = _log(rng, 4, min(128, topk + topk * topk * (iters - 1)))
        layers = rng.choice([1, 8, 32])
        prefix = min(_log(rng, 100, 131072), LARGEST_ROWS // (layers * nodes), LARGEST_CACHE // (layers * heads["kv_heads"]))
        return dict(kind=kind, layers=layers, prefix=prefix, nodes=nodes, iters=iters, topk=topk, vocab=_log(rng, 8192, 151936), hidden=4096,
                    bf16=bf16, graph=rng.random() < 0.6, **heads)
    if kind == "decode":
        layers = rng.choice([1, 8, 32])
        prefix = min(_log(rng, 100, 131072), LARGEST_CACHE // (layers * heads["kv_heads"]))
        return dict(kind=kind, layers=layers, prefix=prefix, vocab=_log(rng, 8192, 151936), hidden=4096, bf16=bf16, **heads)
    if kind == "draft":
        topk = rng.randint(4, 12)
        iters = rng.randint(3, min(6, 64 // topk))
        return dict(kind=kind, prefix=_log(rng, 100, 32768), nodes=rng.randint(topk + 1, min(64, topk + topk * topk * (iters - 1))), iters=iters, topk=topk, vocab=73448,
                    sub=_log(rng, 4096, 73448), hidden=4096, bf16=bf16, graph=rng.random() < 0.6)
    if kind == "prefill":
        return dict(kind=kind, layers=rng.choice([1, 8, 32]), prefix=_log(rng, 1, 65536), rows=_log(rng, 32, 4096), kv_heads=heads["kv_heads"])
    return dict(kind=kind, rows=_log(rng, 1, 64), topk=rng.choice([1, 5, 20, 50]), vocab=_log(rng, 8192, 151936), hidden=4096,
                tiled=rng.random() < 0.5, bf16=bf16)


class _Maker:
    """Seeded device tensors in the 16-bit container the entry points take (bfloat16 travels as its bit pattern)."""

    def __init__(self, seed, bf16):
        self.gen = torch.Generator(device="cuda").manual_seed(int(seed))
        self.bf16 = bool(bf16)

    def pack(self, t):
        return t.to(torch.bfloat16).view(torch.float16) if self.bf16 else t.to(torch.float16)

    def normal(self, *shape):
        t = torch.empty(shape, dtype=torch.bfloat16 if self.bf16 else torch.float16, device="cuda").normal_(generator=self.gen)
        return t.view(torch.float16)

    def weight_grid(self, V, H):
        """[V, H] on the levels -8 .. 7, before the scale of 1/128."""
        t = torch.empty((V, H), dtype=torch.float16, device="cuda").normal_(0.0, 2.2, generator=self.gen)
        return t.round_().clamp_(-8, 7)

    def weight(self, grid):
        return self.pack(grid * 0.0078125)

    def hidden(self, grid, picks, strength):
        """[n, H] on an 8-bit grid of 1/32: noise plus `strength[j]` times row picks[i, j] of the weights, so that those tokens lead."""
        n, m = picks.shape
        h = torch.empty((n, grid.shape[1]), dtype=torch.float32, device="cuda").normal_(0.0, 20.0, generator=self.gen)
        for j in range(m):
            h += strength[j] * grid[picks[:, j]].float()
        return self.pack(h.round_().clamp_(-127, 127) / 32.0)

    def ints(self, n, high):
        return torch.randint(0, high, (n,), device="cuda", generator=self.gen)


def _paged_cache(make, layers, kv_heads, tokens, seed, empty=False):
    """A paged cache of `layers` layers in two allocations, behind a shuffled page table."""
    pages = (tokens + PAGE - 1) // PAGE + 1
    shape_k, shape_v = (layers, pages, kv_heads, PAGE, HEAD_DIM), (layers, pages, kv_heads, HEAD_DIM, PAGE)
    if empty:
        k, v = (torch.zeros(s, dtype=torch.float16, device="cuda") for s in (shape_k, shape_v))
    else:
        k, v = make.normal(*shape_k), make.normal(*shape_v)
    table = torch.from_numpy(synth.rng(seed, 4).permutation(pages).astype(np.int32)).cuda()
    return PagedKVCache.from_pools(list(k.unbind(0)), list(v.unbind(0)), table), k, v


def _device(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


class _Replay:
    """fn recorded into a HIP graph.  The graph holds bare addresses, so fn -- and with it every buffer it uses -- stays with it."""

    def __init__(self, fn):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            fn()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        self.fn, self.graph = fn, torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            self.out = fn()

    def __call__(self):
        self.graph.replay()
        return self.out


def _prepare_step(c, seed):
    make = _Maker(seed, c["bf16"])
    T, L, P, Hq, Hkv = c["nodes"], c["layers"], c["prefix"], c["q_heads"], c["kv_heads"]
    tree = synth.eagle_tree(c["iters"], c["topk"], T, seed)
    cache, k_pool, v_pool = _paged_cache(make, L, Hkv, P + T, seed)
    grid = make.weight_grid(c["vocab"], c["hidden"])
    gt = make.ints(T, c["vocab"])
    hidden = make.hidden(grid, gt[:, None], [6.0])
    w = ops.tile_head_weight(make.weight(grid))
    # two of the tree's levels are accepted, as deep as its nodes allow
    draft, _ = synth.draft_ids_for_accept(tree, gt.cpu().numpy(), min(2, int(tree.depth.max())), c["vocab"], seed)
    st = VerifyStep(cache, w, _device(tree.mask.view(np.int64)), _device(tree.parent), _device(tree.positions(P)), P, head_scale=HEAD_SCALE)
    q, attn = make.normal(L, T, Hq, HEAD_DIM), torch.empty((L, T, Hq, HEAD_DIM), dtype=torch.float16, device="cuda")
    k_new, v_new = make.normal(L, T, Hkv, HEAD_DIM), make.normal(L, T, Hkv, HEAD_DIM)
    args = ([list(t.unbind(0)) for t in (q, k_new, v_new)], hidden, _device(draft), list(attn.unbind(0)))

    def enqueue():
        (ql, kl, vl), h, d, outs = args
        st.enqueue(ql, kl, vl, h, d, attn_out=outs)

    one_pass = _Replay(enqueue) if c["graph"] else enqueue

    def run():
        one_pass()
        a, ids = st.result()
        return dict(accept=a, ids=ids, gt=st.gt, best=st.best, attn=_typed(attn, c), k=_typed(k_pool, c), v=_typed(v_pool, c))
    return run


def _typed(t, c):
    return t.view(torch.bfloat16) if c["bf16"] else t


def _prepare_decode(c, seed):
    make = _Maker(seed, c["bf16"])
    L, P, Hq, Hkv = c["layers"], c["prefix"], c["q_heads"], c["kv_heads"]
    cache, k_pool, v_pool = _paged_cache(make, L, Hkv, P + 1, seed)
    grid = make.weight_grid(c["vocab"], c["hidden"])
    hidden = make.hidden(grid, make.ints(1, c["vocab"])[:, None], [6.0])
    w = ops.tile_head_weight(make.weight(grid))
    q, k_new, v_new = make.normal(L, 1, Hq, HEAD_DIM), make.normal(L, 1, Hkv, HEAD_DIM), make.normal(L, 1, Hkv, HEAD_DIM)
    attn, gt = torch.empty_like(q), torch.empty(1, dtype=torch.int32, device="cuda")
    inv_freq = (10000.0 ** (-torch.arange(0, HEAD_DIM, 2, dtype=torch.float64) / HEAD_DIM)).float().cuda()
    position = torch.tensor([P], dtype=torch.int32, device="cuda")
    kv_len = torch.tensor([P + 1], dtype=torch.int32, device="cuda")
    padded = (P + 1 + 127) // 128 * 128

    def token():
        table = ops.rope_table(position, inv_freq)
        for l in range(L):
            ops.tree_attention(q[l], cache, l, kv_len, padded, out=attn[l], k_new=k_new[l], v_new=v_new[l], rope=table)
        ops.lm_head_argmax(hidden, w, head_scale=HEAD_SCALE, gt=gt)

    one_pass = _Replay(token)

    def run():
        one_pass()
        return dict(gt=gt, attn=_typed(attn, c), k=_typed(k_pool, c), v=_typed(v_pool, c))
    return run


def _prepare_draft(c, seed):
    make = _Maker(seed, c["bf16"])
    k, iters, P, Hq, Hkv = c["topk"], c["iters"], c["prefix"], 32, 2
    cache, k_pool, v_pool = _paged_cache(make, 1, Hkv, P + k * iters, seed)
    grid = make.weight_grid(c["vocab"], c["hidden"])
    remap = _device(synth.frspec_remap(c["vocab"], c["sub"], seed))
    w = ops.tile_head_weight(make.weight(grid), remap)
    strength = np.linspace(5.0, 1.5, 2 * k)
    hidden = [make.hidden(grid, remap.long()[make.ints(n * 2 * k, c["sub"])].reshape(n, 2 * k), strength) for n in [1] + [k] * (iters - 1)]
    rounds = range(1, iters)
    q = {d: make.normal(k, Hq, HEAD_DIM) for d in rounds}
    k_new = {d: make.normal(k, Hkv, HEAD_DIM) for d in rounds}
    v_new = {d: make.normal(k, Hkv, HEAD_DIM) for d in rounds}
    kv_len = {d: torch.tensor([P + k * d], dtype=torch.int32, device="cuda") for d in rounds}
    cache_length = torch.tensor([P], dtype=torch.int32, device="cuda")
    padded = (P + k * iters + 127) // 128 * 128
    tree = ops.DraftTree(k, iters, remap)

    def draft():
        heads, attn = [], []
        r = ops.frspec_head_topk(hidden[0], w, remap, k)
        heads.append(r)
        tree.begin(r["val"][0], r["pos"][0])
        for d in rounds:
            attn.append(ops.tree_attention(q[d], cache, 0, kv_len[d], padded, mask=tree.draft_mask, k_new=k_new[d], v_new=v_new[d],
                                           mask_k_range=k * d, block_window_size=WINDOW))
            r = ops.frspec_head_topk(hidden[d], w, remap, k)
            heads.append(r)
            tree.extend(d, r["val"], r["pos"])
        return heads, attn, tree.finish(c["nodes"], cache_length)

    one_pass = _Replay(draft) if c["graph"] else draft

    def run():
        heads, attn, (ids, pos, mask, parent) = one_pass()
        # (entry 0 of the ids and the parent of the root are the caller's)
        return dict(ids=ids[1:], pos=pos, mask=mask, parent=parent[1:], logp=[_typed(r["val"], c) for r in heads],
                    logits=[_typed(r["logits"], c) for r in heads], stats=[r["row_stats"] for r in heads], attn=[_typed(t, c) for t in attn],
                    k=_typed(k_pool, c), v=_typed(v_pool, c))
    return run


def _prepare_prefill(c, seed):
    make = _Maker(seed, False)
    L, P, n, Hkv = c["layers"], c["prefix"], c["rows"], c["kv_heads"]
    cache, k_pool, v_pool = _paged_cache(make, L, Hkv, P + n, seed, empty=True)
    k_rows, v_rows = make.normal(L, n, Hkv, HEAD_DIM), make.normal(L, n, Hkv, HEAD_DIM)
    kv_len = torch.tensor([P + n], dtype=torch.int32, device="cuda")

    def run():
        for l in range(L):
            ops.kv_append(cache, l, k_rows[l], v_rows[l], kv_len)
        return dict(k=k_pool, v=v_pool)
    return run


def _prepare_logprobs(c, seed):
    make = _Maker(seed, c["bf16"])
    grid = make.weight_grid(c["vocab"], c["hidden"])
    n, m = c["rows"], 2 * c["topk"]
    hidden = make.hidden(grid, make.ints(n * m, c["vocab"]).reshape(n, m), np.linspace(5.0, 1.5, m) * min(1.0, math.sqrt(40.0 / m)))
    w = make.weight(grid)
    if c["tiled"]:
        w = ops.tile_head_weight(w)

    def run():
        gt, logits = ops.lm_head_argmax(hidden, w, head_scale=1.0, want_logits=True)
        stats = ops.log_softmax_(logits)
        val, pos = ops.topk(logits, c["topk"])
        return dict(gt=gt, logp=_typed(logits, c), stats=stats, val=_typed(val, c), pos=pos)
    return run


_PREPARE = dict(step=_prepare_step, decode=_prepare_decode, draft=_prepare_draft, prefill=_prepare_prefill, logprobs=_prepare_logprobs)


def prepare(case, seed):
    # the element type of the 16-bit tensors is a process-wide option of the library
    lib.get().set_option(b"dtype", 1 if case.get("bf16") else 0)
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return state()


def _attention_work(rows, keys, q_heads, kv_heads):
    """Keys and values read once, the new rows read and written, queries in, outputs out."""
    return dict(bytes=2 * keys * kv_heads * HEAD_DIM * 2 + 4 * rows * kv_heads * HEAD_DIM * 2 + 2 * rows * q_heads * HEAD_DIM * 2,
                flops=4 * q_heads * rows * keys * HEAD_DIM)


def _head_work(rows, vocab, hidden, out_bytes):
    return dict(bytes=vocab * hidden * 2 + rows * hidden * 2 + out_bytes, flops=2 * rows * vocab * hidden)


def _sum(*parts):
    return {m: sum(n * w[m] for n, w in parts) for m in ("bytes", "flops")}


def work(case):
    c, kind = case, case["kind"]
    if kind == "step":
        return _sum((c["layers"], _attention_work(c["nodes"], c["prefix"] + c["nodes"], c["q_heads"], c["kv_heads"])),
                    (1, _head_work(c["nodes"], c["vocab"], c["hidden"], 4 * c["nodes"])))
    if kind == "decode":
        return _sum((c["layers"], _attention_work(1, c["prefix"] + 1, c["q_heads"], c["kv_heads"])),
                    (1, _head_work(1, c["vocab"], c["hidden"], 4)))
    if kind == "draft":
        k = c["topk"]
        parts = [(1, _head_work(1, c["sub"], c["hidden"], 2 * c["sub"] + 10 * k))]
        for d in range(1, c["iters"]):
            parts += [(1, _head_work(k, c["sub"], c["hidden"], 2 * k * c["sub"] + 10 * k * k)),
                      (1, _attention_work(k, min(c["prefix"], WINDOW) + k * d, 32, 2))]
        return _sum(*parts)
    if kind == "prefill":
        return dict(bytes=c["layers"] * 2 * 2 * c["rows"] * c["kv_heads"] * HEAD_DIM * 2, flops=0)
    n = c["rows"]
    return _head_work(n, c["vocab"], c["hidden"], 2 * n * c["vocab"] + n * (12 + 6 * c["topk"]))


def tolerance(case):
    kind = case["kind"]
    if kind == "prefill":
        return "exact"
    # attention outputs: probabilities and split results rounded to the element type; heads: one rounding of an exact sum
    rel = 1e-2 if case["bf16"] else 2e-3
    # a log-probability on the edge of a rounding step can move one rank
    return dict(rel=rel, differ=0.01 if kind in ("draft", "logprobs") else 0.0)
