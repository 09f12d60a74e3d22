"""Tree attention whose workgroups merge their partials through the L2 of one XCD."""
import pytest

from cpm.cu_amd import synth
from util import to_dev

pytestmark = pytest.mark.gpu
D = 128


@pytest.mark.parametrize("P,T,hq,hkv,splits,groups", [
    (4548, 60, 32, 2, 16, 2), (4549, 60, 32, 2, 16, 2), (4000, 60, 32, 2, 15, 2), (2000, 60, 32, 2, 2, 2), (3000, 32, 32, 2, 32, 2), (3001, 128, 32, 2, 8, 2),
    (3000, 128, 32, 2, 16, 1), (1500, 60, 32, 2, 32, 1), (4500, 96, 32, 4, 10, 1), (2500, 33, 32, 8, 16, 2), (9001, 33, 32, 8, 31, 1), (6000, 128, 32, 8, 8, 1), (4480, 128, 32, 8, 8, 1), (5000, 65, 32, 8, 10, 2), (5000, 64, 32, 8, 16, 2),
    (700, 20, 48, 16, 16, 2), (5000, 17, 24, 8, 9, 2),
    (4076, 20, 32, 2, 16, 2), (1000, 24, 32, 2, 32, 2), (4560, 48, 32, 2, 16, 2), (2527, 33, 32, 2, 16, 2), (2504, 56, 32, 2, 13, 2), (1300, 40, 16, 1, 32, 2)])
def test_merge_on_one_xcd_equals_separate_merge(gpu, P, T, hq, hkv, splits, groups):
    """Launches whose units merge through the L2 of an XCD (one to three units on each, full, half empty and idle XCDs, XCDs with units of two heads, the longest context
    that is numbered for it, any length on a multiple of 8 KV heads and up to 256 rows of each), in both types: the bits of the separate merge launch, also where waits run out at
    once, and in replays.  The next longer context, more rows of 8 heads, and three M-tiles of 4 heads at 4596 keys, are merged through memory.  That the plan is the one meant, that the workspace has counters, and
    that waits ran out, is asserted: without any of them the bits would be the same."""
    torch = gpu
    import ctypes
    from cpm.cu_amd import lib, ops
    from cpm.cu_amd.kvcache import PagedKVCache
    L = lib.get()
    option = lambda name, value: L.set_option(name.encode(), int(value))
    L.synchronize()
    seen = L.raw.cpmcu_attention_abandoned_waits()
    option("attn_kv_groups", groups)
    option("attn_direct", 0)
    S = P + T
    on_one_xcd = (P, T, hkv) not in ((4549, 60, 2), (4500, 96, 4), (6000, 128, 8), (5000, 65, 8))
    g = torch.Generator(device="cuda").manual_seed(S)
    mask = to_dev(torch, synth.random_tree(T, S, max_children=4, max_depth=9).mask)
    kv_len = torch.tensor([S], dtype=torch.int32, device="cuda")
    try:
        for dtype in (0, 1):
            option("dtype", dtype)
            rnd = lambda *s: torch.randn(s, device="cuda", generator=g).to(torch.bfloat16 if dtype else torch.float16).view(torch.float16)
            cache = PagedKVCache(1, hkv, (S + 255) // 256 + 1)
            cache.write_logical(0, 0, rnd(S, hkv, D), rnd(S, hkv, D))
            q = rnd(T, hq, D)
            call = lambda out: ops.tree_attention(q, cache, 0, kv_len, S, mask, num_splits=splits, out=out)
            names, used, _, _ = ops.attention_plan(T, hq, hkv, S, num_splits=splits)
            assert (names, used) == ("tree_attn_split%s_kernel<%d,false,%s>" % ("_bf16" if dtype else "", groups, str(on_one_xcd).lower()), splits)
            option("attn_merge_in_launch", 0)
            ref = call(torch.empty_like(q))
            option("attn_merge_in_launch", 1)
            out = torch.empty_like(q)
            call(out)
            assert L.raw.cpmcu_tree_attention_merge_mode(ctypes.c_void_p(ops._workspaces["attn", q.device].data_ptr())) == 1
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                for _ in range(2):
                    call(out)
            for wait_us in (2000, 2000, 0, 2000):
                option("attn_merge_wait_us", wait_us)
                out.fill_(float("nan"))
                if wait_us:
                    graph.replay()
                else:
                    call(out)
                torch.cuda.synchronize()
                assert torch.equal(out.view(torch.int16), ref.view(torch.int16)), (dtype, wait_us)
    finally:
        option("attn_kv_groups", 0)
        option("attn_direct", -1)
        option("dtype", 0)
        option("attn_merge_wait_us", 2000)
        L.synchronize()
        option("attn_merge_in_launch", 1)
    assert L.raw.cpmcu_attention_abandoned_waits() > seen


@pytest.mark.parametrize("P,T,hq,hkv,splits,groups", [
    (4000, 60, 32, 2, 16, 2), (2000, 60, 32, 2, 2, 2), (3000, 32, 32, 2, 32, 2), (1500, 128, 32, 2, 8, 2), (9001, 33, 32, 8, 31, 1), (2527, 33, 32, 2, 16, 2), (4076, 20, 32, 2, 16, 2)])
def test_units_on_several_xcds_are_merged_all_the_same(gpu, set_option, P, T, hq, hkv, splits, groups):
    """Launches numbered for one XCD a unit whose workgroups are then on several (each split of a unit on the next one; with 2 splits two, else all
    eight): the bits are those of the separate merge, in replays, with launches on one XCD between them, and where waits run out (60 launches each; a mark or a count
    that outlived its launch would complete a unit that is not there yet).  All units of those launches are counted as spread, and none of the others."""
    torch = gpu
    from cpm.cu_amd import lib, ops
    from cpm.cu_amd.kvcache import PagedKVCache
    L = lib.get()
    set_option("attn_kv_groups", groups)
    set_option("attn_direct", 0)
    S = P + T
    g = torch.Generator(device="cuda").manual_seed(S)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g).half()
    cache = PagedKVCache(1, hkv, (S + 255) // 256 + 1)
    cache.write_logical(0, 0, rnd(S, hkv, D), rnd(S, hkv, D))
    q, kv_len = rnd(T, hq, D), torch.tensor([S], dtype=torch.int32, device="cuda")
    mask = to_dev(torch, synth.random_tree(T, S, max_children=4, max_depth=9).mask)

    def launch(out):
        out.fill_(float("nan"))
        if ("attn", q.device) in ops._workspaces:
            ops._workspaces["attn", q.device].fill_(255)  # (no partials of the launch before: NaN)
        ops.tree_attention(q, cache, 0, kv_len, S, mask, num_splits=splits, out=out)

    def same(out, *what):
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), ref.view(torch.int16)), what

    L.synchronize()
    set_option("attn_merge_in_launch", 0)
    ref = torch.empty_like(q)
    launch(ref)
    set_option("attn_merge_in_launch", 1)
    out, graphs, seen = torch.empty_like(q), {}, L.raw.cpmcu_attention_abandoned_waits()
    launch(out)  # (the workspace gets its counters outside the captures)
    for spread in (0, 1):
        set_option("attn_spread_units", spread)
        graphs[spread] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graphs[spread]):
            launch(out)
    set_option("attn_spread_units", 0)
    for spread in (0, 0):
        graphs[spread].replay()
        same(out, spread)
    L.synchronize()
    spread_units = L.raw.cpmcu_attention_spread_units()
    for spread in (1, 0, 1, 1, 0, 0, 1):
        graphs[spread].replay()
        same(out, spread)
    L.synchronize()
    units = hkv * -(-hq // hkv * T // (128 if groups == 2 else 256))
    assert L.raw.cpmcu_attention_spread_units() - spread_units == 4 * units
    assert L.raw.cpmcu_attention_abandoned_waits() == seen
    try:
        set_option("attn_merge_in_launch", 1)
        for wait_us in (0, 1):
            set_option("attn_merge_wait_us", wait_us)
            for turn in range(60):
                set_option("attn_spread_units", turn & 1)
                launch(out)
                same(out, wait_us, turn)
    finally:
        set_option("attn_merge_wait_us", 2000)
        set_option("attn_spread_units", 0)
        L.synchronize()
        set_option("attn_merge_in_launch", 1)
    assert L.raw.cpmcu_attention_abandoned_waits() > seen
