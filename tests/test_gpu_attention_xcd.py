"""Tree attention whose workgroups merge their partials through the L2 of one XCD."""
import pytest

from cpm.cu_amd import synth
from util import to_dev

pytestmark = pytest.mark.gpu
D = 128


@pytest.mark.parametrize("P,T,hq,hkv,splits,groups", [
    (4548, 60, 32, 2, 16, 2), (4549, 60, 32, 2, 16, 2), (4000, 60, 32, 2, 15, 2), (2000, 60, 32, 2, 2, 2), (3000, 32, 32, 2, 32, 2), (3001, 128, 32, 2, 8, 2),
    (3000, 128, 32, 2, 16, 1), (1500, 60, 32, 2, 32, 1), (4500, 96, 32, 4, 10, 1), (2500, 33, 32, 8, 16, 2), (9001, 33, 32, 8, 31, 1), (6000, 128, 32, 8, 8, 1),
    (700, 20, 48, 16, 16, 2), (5000, 17, 24, 8, 9, 2),
    (4076, 20, 32, 2, 16, 2), (1000, 24, 32, 2, 32, 2), (4560, 48, 32, 2, 16, 2), (2527, 33, 32, 2, 16, 2), (2504, 56, 32, 2, 13, 2), (1300, 40, 16, 1, 32, 2)])
def test_merge_on_one_xcd_equals_separate_merge(gpu, P, T, hq, hkv, splits, groups):
    """Launches whose units merge through the L2 of an XCD (one to three units on each, full, half empty and idle XCDs, XCDs with units of two heads, the longest context
    that is numbered for it and the next one, any length on a multiple of 8 KV heads), in both types: the bits of the separate merge launch, also where every wait runs out at
    once, and in replays."""
    torch = gpu
    from cpm.cu_amd import lib, ops
    from cpm.cu_amd.kvcache import PagedKVCache
    L = lib.get()
    option = lambda name, value: L.set_option(name.encode(), int(value))
    option("attn_kv_groups", groups)
    option("attn_direct", 0)
    S = P + T
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
            assert "combine" not in names and used == splits
            option("attn_merge_in_launch", 0)
            ref = call(torch.empty_like(q))
            option("attn_merge_in_launch", 1)
            out = torch.empty_like(q)
            call(out)
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
