"""The direct shape of tree attention at its edges: block and row-tile remainders, splits with one block and with none, appended
rows in more than one step, windows that start inside a page, both element types -- against the oracle, and the cache against
what the other shapes leave behind, slots past the end included."""
import numpy as np
import pytest

from cpm.cu_amd import synth
from util import assert_close_f16, to_dev, to_np

pytestmark = pytest.mark.gpu
D = 128


@pytest.fixture
def option():
    from cpm.cu_amd import lib
    L = lib.get()
    yield lambda name, value: L.set_option(name.encode(), int(value))
    L.set_option(b"attn_direct", -1)
    L.set_option(b"dtype", 0)


@pytest.mark.parametrize("P,T,hq,hkv,splits,window,rope,fused", [
    (0, 1, 32, 2, 1, 0, False, True), (0, 33, 32, 2, 0, 0, True, True), (1, 1, 32, 2, 2, 0, True, True), (127, 1, 32, 2, 1, 0, False, True),
    (128, 9, 32, 2, 0, 0, True, True), (129, 16, 32, 2, 3, 0, False, True), (255, 60, 32, 2, 0, 0, False, True), (256, 31, 32, 8, 0, 0, True, True),
    (777, 128, 32, 8, 0, 0, False, True), (300, 7, 24, 8, 2, 0, True, True), (500, 13, 28, 4, 0, 0, False, True), (90, 3, 12, 12, 0, 0, False, True),
    (4090, 4, 32, 2, 0, 0, True, True), (4096, 1, 32, 2, 36, 0, False, True), (4700, 1, 32, 2, 37, 0, False, True), (9000, 2, 32, 4, 128, 0, True, True),
    (20000, 1, 32, 2, 1, 0, False, True), (1500, 10, 32, 2, 0, 1024, False, True), (1537, 12, 32, 2, 3, 1024, True, True),
    (700, 10, 32, 2, 0, 128, False, True), (640, 17, 32, 2, 0, 0, False, False), (2000, 64, 32, 2, 4, 512, False, False)])
def test_direct_shape_against_the_oracle(gpu, orc, option, P, T, hq, hkv, splits, window, rope, fused):
    from cpm.cu_amd import ops
    from cpm.cu_amd.kvcache import PagedKVCache
    torch = gpu
    S, seed = P + T, 7 * P + T
    tree = synth.random_tree(T, seed, max_children=4, max_depth=9)
    q, k, v = (synth.normal_f16(s, seed, i) for i, s in enumerate([(T, hq, D), (S, hkv, D), (S, hkv, D)]))
    max_len = (S + 127) // 128 * 128 + [0, 640][seed % 2]
    npages = (max_len + 255) // 256 + 1
    pages = synth.rng(seed, 4).permutation(npages).astype(np.int32)
    kv_len = torch.tensor([S], dtype=torch.int32, device="cuda")
    table, q_ref, k_ref = None, q, k
    if rope:
        inv_freq = (10000.0 ** (-np.arange(D // 2, dtype=np.float64) / (D // 2))).astype(np.float32)
        table = ops.rope_table(to_dev(torch, tree.positions(P)), to_dev(torch, inv_freq))
        q_ref, k_rot = orc.rope(q, k[P:], table=to_np(table))
        k_ref = np.concatenate([k[:P], k_rot], 0)
    n = P if fused else S
    new = dict(k_new=to_dev(torch, k[P:]), v_new=to_dev(torch, v[P:])) if fused else {}
    outs, pools = [], []
    for direct in (0, 1):
        option("attn_direct", direct)
        c = PagedKVCache(1, hkv, npages, block_table=pages, fill=float("nan"))
        if n:
            c.write_logical(0, 0, to_dev(torch, k[:n]), to_dev(torch, v[:n]))
        assert (ops.attention_plan(T, hq, hkv, max_len, rope, window)[0].startswith("tree_attn_direct")) == bool(direct)
        outs.append(ops.tree_attention(to_dev(torch, q), c, 0, kv_len, max_len, to_dev(torch, tree.mask), num_splits=splits if direct else 0,
                                       rope=table, block_window_size=window, **new))
        torch.cuda.synchronize()
        pools.append([t.view(torch.int16) for t in (c.k[0], c.v[0])])
    ref = orc.tree_attention(q_ref, k_ref, v, tree.mask, P, block_window_size=window)
    assert_close_f16(to_np(outs[1]), ref, "direct shape")
    assert all(torch.equal(a, b) for a, b in zip(*pools)), "the cache differs from what the split shapes leave"


@pytest.mark.parametrize("P,T,kd", [(900, 10, 30), (130, 8, 64), (61, 4, 128)])
def test_direct_shape_bf16_with_a_wider_mask(gpu, option, P, T, kd):
    """bf16, a mask whose range reaches into the cached rows, replayed from a graph: the merge's arrival words are at rest behind
    every launch."""
    from cpm.cu_amd import ops
    from cpm.cu_amd.kvcache import PagedKVCache
    torch = gpu
    option("dtype", 1)
    P += kd - T
    g = torch.Generator(device="cuda").manual_seed(P)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g).to(torch.bfloat16).view(torch.float16)
    S = P + T
    q, k, v = rnd(T, 32, D), rnd(S, 2, D), rnd(S, 2, D)
    mask = torch.randint(-2 ** 62, 2 ** 62, (T, (kd + 63) // 64), device="cuda", generator=g)
    cache = PagedKVCache(1, 2, (S + 255) // 256)
    cache.write_logical(0, 0, k[:P], v[:P])
    kv_len = torch.tensor([S], dtype=torch.int32, device="cuda")
    call = lambda out: ops.tree_attention(q, cache, 0, kv_len, S, mask, k_new=k[P:], v_new=v[P:], mask_k_range=kd, out=out)
    option("attn_direct", 0)
    ref = call(torch.empty_like(q)).view(torch.bfloat16).float()
    option("attn_direct", 1)
    out = call(torch.empty_like(q))
    torch.cuda.synchronize()
    first = out.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(3):
            call(out)
    for _ in range(4):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), first.view(torch.int16))
    err = (first.view(torch.bfloat16).float() - ref).norm() / ref.norm()
    assert err < 8e-3, float(err)


@pytest.mark.parametrize("P,T,hq,hkv,splits,rope", [
    (1900, 1, 32, 2, 15, False), (2040, 1, 32, 2, 16, True), (2100, 1, 32, 8, 17, False), (4090, 2, 32, 8, 32, True), (4200, 2, 28, 4, 33, False),
    (4500, 1, 32, 1, 40, False), (8190, 1, 32, 2, 64, False), (8300, 5, 4, 1, 65, True), (8400, 3, 16, 2, 64, False), (16500, 1, 32, 2, 128, False),
    (700, 1, 32, 2, 128, False), (8000, 2, 32, 2, 128, False)])
def test_merge_in_shares_against_the_oracle(gpu, orc, option, P, T, hq, hkv, splits, rope):
    """Around the split counts where the merge changes its form (one to eight waves an item, two row tiles, splits without a share,
    rows that fill a tile in part, more workgroups than CUs) and with splits that have no keys."""
    test_direct_shape_against_the_oracle(gpu, orc, option, P, T, hq, hkv, splits, 0, rope, True)


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("hkv,splits", [(2, 20), (2, 100), (8, 32)])
def test_shares_left_behind_are_merged_by_the_last_arrival(gpu, option, hkv, splits, dtype):
    """A wait limit of 1 us, which the arrivals of 20 workgroups and more on one word do not keep: those that it runs out for give their
    share up; the output is the same to the bit, and the launch behind it is whole again.  That the launches are direct ones with a CU for every workgroup, and that
    shares were given up, is asserted: without either the outputs would be the same."""
    from cpm.cu_amd import lib, ops
    from cpm.cu_amd.kvcache import PagedKVCache
    torch, L = gpu, lib.get()
    option("dtype", dtype)
    option("attn_direct", 1)
    option("attn_merge_in_launch", 1)
    S = 12901
    g = torch.Generator(device="cuda").manual_seed(S + splits)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g).to(torch.bfloat16 if dtype else torch.float16).view(torch.float16)
    cache = PagedKVCache(1, hkv, (S + 255) // 256)
    cache.write_logical(0, 0, rnd(S, hkv, D), rnd(S, hkv, D))
    q, kv_len = rnd(1, 32, D), torch.tensor([S], dtype=torch.int32, device="cuda")
    kernel, used, _, workgroups = ops.attention_plan(1, 32, hkv, S, num_splits=splits)
    assert (kernel, used) == ("tree_attn_direct_shares%s_kernel" % ("_bf16" if dtype else ""), splits)
    assert workgroups <= torch.cuda.get_device_properties(0).multi_processor_count
    L.synchronize()
    option("attn_merge_in_launch", 1)
    ref = ops.tree_attention(q, cache, 0, kv_len, S, num_splits=splits)
    L.synchronize()
    before = L.raw.cpmcu_attention_abandoned_waits()
    try:
        for wait_us in (1, 1, 2000, 1, 1, 1, 1):
            option("attn_merge_wait_us", wait_us)
            out = torch.full_like(q, float("nan"))
            ops.tree_attention(q, cache, 0, kv_len, S, num_splits=splits, out=out)
            torch.cuda.synchronize()
            assert torch.equal(out.view(torch.int16), ref.view(torch.int16)), wait_us
    finally:
        option("attn_merge_wait_us", 2000)
        L.synchronize()
        option("attn_merge_in_launch", 1)  # (nobody had waited in these workspaces' launches from the synchronisation on)
    assert L.raw.cpmcu_attention_abandoned_waits() > before, "no share was left behind"


@pytest.mark.parametrize("zero_limit", [False, True])
@pytest.mark.parametrize("hkv,T,splits", [(2, 1, 2), (2, 4, 15), (2, 1, 16), (8, 2, 32), (2, 1, 37), (1, 1, 128), (2, 3, 0)])
def test_direct_launches_after_an_abandoned_wait(gpu, option, hkv, T, splits, zero_limit):
    """After a merge wait that ran out on the device a launch of the direct shape stays one: nobody waits in it, and the last arrival
    merges.  Its partials, in the workspace, are those of the launch that waits: bit for bit up to 15 splits, whose partials are there as well; merged in shares, from 16 on,
    that launch leaves nothing in the workspace, and its output is what a merge of these partials in float64 rounds to.  A wait limit of zero does the same from the
    first launch on: nothing is left behind for the last arrival to merge share by share."""
    import ctypes
    from cpm.cu_amd import lib, ops
    from cpm.cu_amd.kvcache import PagedKVCache
    torch, L = gpu, lib.get()
    option("attn_direct", 1)
    S = 16500
    g = torch.Generator(device="cuda").manual_seed(S + splits)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g).half()
    cache = PagedKVCache(1, hkv, (S + 255) // 256)
    k, v = rnd(S, hkv, D), rnd(S, hkv, D)
    cache.write_logical(0, 0, k, v)
    q, kv_len = rnd(T, 32, D), torch.tensor([S], dtype=torch.int32, device="cuda")
    hidden = torch.arange(S, device="cuda")[None] > S - T + torch.arange(T, device="cuda")[:, None]
    exact = torch.empty((T, 32, D), dtype=torch.float64, device="cuda")
    for h in range(32):
        x = (q[:, h].double() @ k[:, h * hkv // 32].double().t().contiguous()) * D ** -0.5
        exact[:, h] = torch.softmax(x.masked_fill(hidden, -float("inf")), 1) @ v[:, h * hkv // 32].double()
    key = ("attn", q.device)
    ws = torch.empty(L.raw.cpmcu_tree_attention_workspace_bytes(T, 32, hkv, S), dtype=torch.uint8, device="cuda")
    saved, ops._workspaces[key] = ops._workspaces.get(key), ws

    def call():
        ws.zero_()
        out = torch.full_like(q, float("nan"))
        ops.tree_attention(q, cache, 0, kv_len, S, num_splits=splits, out=out)
        torch.cuda.synchronize()
        return out, ws.clone()

    def merged(parts, splits):
        """The output that the workspace's partials make: [unit][split][16 rows][128] of 16 bits, behind them [unit][split][16 rows] of (exponent, sum)."""
        group, tiles = 32 // hkv, -(-32 // hkv * T // 16)
        n = hkv * tiles * splits * 16
        x = parts[:n * D * 2].view(torch.float16).double().view(hkv, tiles, splits, 16, D)
        m, l = parts[n * D * 2:][:n * 8].view(torch.float32).double().view(hkv, tiles, splits, 16, 2).unbind(-1)
        w = l * torch.exp2(m - m.amax(2, keepdim=True))
        o = (w[..., None] * x).sum(2) / w.sum(2)[..., None]
        return o.view(hkv, tiles * 16, D)[:, :group * T].view(hkv, T, group, D).transpose(0, 1).reshape(T, 32, D)

    def nearly_all_bits(a, b):
        """The same fp32 sums in other orders (1e-5 of the value at most, where 128 partials cancel each other), rounded to fp16 once: a unit in the last place apart in one
        of 50 values.  Partials rounded otherwise move a third of them."""
        assert float(((a.double() - b).abs() - 2.0 ** -10 * b.abs()).max()) <= 2.0 ** -24
        assert float((a != b.half()).double().mean()) <= 0.02
    try:
        if not L.raw.cpmcu_tree_attention_merge_mode(ctypes.c_void_p(ws.data_ptr())):
            option("attn_merge_in_launch", 1)
        if not L.raw.cpmcu_tree_attention_merge_mode(ctypes.c_void_p(ws.data_ptr())):
            pytest.skip("this process has used up the library's counter blocks")
        ref, ref_parts = call()
        assert bool(ref_parts.any()) == (0 < splits <= 15)  # (three queries take more than 15 by themselves)
        L.synchronize()
        seen = L.raw.cpmcu_attention_abandoned_waits()
        option("attn_merge_wait_us", 0)
        if not zero_limit:
            # a wait that runs out: with a limit of zero the split shapes leave shares behind
            option("attn_direct", 0)
            for _ in range(4):
                ops.tree_attention(q[:1], cache, 0, kv_len, S, num_splits=32)
            before = seen
            L.synchronize()
            seen = L.raw.cpmcu_attention_abandoned_waits()
            assert seen > before and L.raw.cpmcu_tree_attention_merge_mode(ctypes.c_void_p(ws.data_ptr())) == 0
            option("attn_direct", 1)
            option("attn_merge_wait_us", 2000)
        for _ in range(2):
            out, parts = call()
            used = splits or ops.attention_plan(T, 32, hkv, S)[1]
            if zero_limit or splits:  # (else the plan is that of a launch that waits)
                nearly_all_bits(out, merged(parts, used))
            if splits:  # (else the number of splits is chosen anew)
                if splits <= 15:
                    assert torch.equal(parts, ref_parts)
                else:
                    nearly_all_bits(ref, merged(parts, splits))
                # two orders of the same fp32 sums, rounded to fp16 once: a unit in the last place apart, at most
                assert float((out.float() - ref.float()).abs().max()) <= 2.0 ** -10 * float(ref.float().abs().max())
            # three roundings to fp16 (probabilities, partials, output) of 2.1e-4 of the norm each, added up in full
            assert float((out.double() - exact).norm() / exact.norm()) < 6.3e-4
        L.synchronize()
        assert L.raw.cpmcu_attention_abandoned_waits() == seen, "somebody waited"
    finally:
        option("attn_merge_wait_us", 2000)
        L.synchronize()
        option("attn_merge_in_launch", 1)
        ops.release_attention_workspace(ws)
        ops._workspaces.pop(key)
        if saved is not None:
            ops._workspaces[key] = saved


def test_words_of_launches_of_changing_shapes(gpu, option):
    """Launches that merge in shares pass their partials on in the same slots, other splits and units in them each time (the edges of
    one to eight waves an item, shares of several turns, 256 workgroups): no launch takes an older one's words for its own.  Reference: the same
    launch merged by its last arrival, two orders of the same fp32 sums, rounded to fp16 once."""
    from cpm.cu_amd import ops
    from cpm.cu_amd.kvcache import PagedKVCache
    torch = gpu
    option("attn_direct", 1)
    option("attn_merge_in_launch", 1)
    shapes = [(1, 2, 34), (4, 2, 17), (1, 8, 32), (2, 4, 16), (1, 1, 128), (3, 4, 30), (4, 2, 32), (1, 2, 64), (1, 2, 65), (3, 2, 33), (1, 2, 16)]
    S, g = 9000, torch.Generator(device="cuda").manual_seed(5)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g).half()
    kv_len, caches, calls = torch.tensor([S], dtype=torch.int32, device="cuda"), {}, []
    for hkv in (1, 2, 4, 8):
        caches[hkv] = PagedKVCache(1, hkv, (S + 255) // 256)
        caches[hkv].write_logical(0, 0, rnd(S, hkv, D), rnd(S, hkv, D))
    for turn in range(3):
        for T, hkv, splits in shapes[turn:] + shapes[:turn]:
            q = rnd(T, 32, D)
            calls.append((lambda q=q, hkv=hkv, splits=splits: ops.tree_attention(q, caches[hkv], 0, kv_len, S, num_splits=splits), (T, hkv, splits)))
            assert ops.attention_plan(T, 32, hkv, S, num_splits=splits)[0] == "tree_attn_direct_shares_kernel"
    outs = [call() for call, _ in calls]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        replayed = [call() for call, _ in calls]
    for _ in range(3):
        for r in replayed:
            r.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        for r, o, (_, shape) in zip(replayed, outs, calls):
            assert torch.equal(r.view(torch.int16), o.view(torch.int16)), shape
    option("attn_merge_wait_us", 0)
    try:
        for o, (call, shape) in zip(outs, calls):
            ref = call()
            assert float((o.float() - ref.float()).abs().max()) <= 2.0 ** -10 * float(ref.float().abs().max()), shape
    finally:
        option("attn_merge_wait_us", 2000)


@pytest.mark.parametrize("splits", [8, 16, 20, 40, 128])
def test_merges_of_large_values_stay_finite(gpu, option, splits):
    """bfloat16 V of 1e34, keys of equal weight: no split's sum (at most 60001 / 8 x 1e34) and no output leaves the range of an fp32, and no merge of them does, by
    the last arrival or in shares on one to eight waves.  The mean of equal values is the value, but for fp32 roundings far below bfloat16's."""
    from cpm.cu_amd import ops
    from cpm.cu_amd.kvcache import PagedKVCache
    torch, S = gpu, 60001
    option("dtype", 1)
    option("attn_direct", 1)
    bits = lambda t: t.to(torch.bfloat16).view(torch.float16)
    cache = PagedKVCache(1, 2, (S + 255) // 256)
    v = torch.full((S, 2, D), 1e34, device="cuda")
    v[:, 1] *= -1
    cache.write_logical(0, 0, bits(torch.randn(S, 2, D, device="cuda")), bits(v))
    kv_len = torch.tensor([S], dtype=torch.int32, device="cuda")
    out = ops.tree_attention(bits(torch.zeros(1, 32, D, device="cuda")), cache, 0, kv_len, S, num_splits=splits).view(torch.bfloat16)
    assert torch.equal(out, v[:1].to(torch.bfloat16).repeat_interleave(16, 1))
