"""Split counts and shapes that the library chooses, on both sides of the lines where it changes them."""
import pytest

from cpm.cu_amd import synth
from util import to_dev

pytestmark = pytest.mark.gpu
D = 128


@pytest.mark.parametrize("S,T,hkv,splits,shape", [
    (59 * 64, 24, 2, 16, 2), (61 * 64, 24, 2, 32, 2),           # 32 splits or 16
    (90 * 64, 33, 2, 16, 2), (91 * 64, 33, 2, 24, 2),           # 24 or 16
    (150 * 64, 48, 2, 16, 2), (151 * 64, 48, 2, 20, 2),         # 20 or 16
    (17 * 64, 40, 4, 16, 2), (16 * 64, 40, 4, 16, 2), (15 * 64, 40, 4, 15, 2),
    (1019 * 64, 17, 2, 32, 2), (1020 * 64, 17, 2, 64, 1),       # two KV groups on 32 splits or the 256-row shape on 64: 6 units of 128 rows
    (1359 * 64, 32, 2, 32, 2), (1360 * 64, 32, 2, 64, 1),       # 8 units
    (1360 * 64, 16, 4, 64, 2)])                                  # (two groups have 64 splits as well)
def test_plans_beside_their_lines(gpu, S, T, hkv, splits, shape):
    """The plan is the one that the line says, and its output is that of 5 splits (another shape, the separate merge): the normalised partials, the probabilities
    and the outputs are rounded to fp16, each by at most 2^-11 of values that a softmax over N(0, 1) keeps below 1.5, in either form: 6 x 1.5 x 2^-11 = 4.4e-3."""
    torch = gpu
    from cpm.cu_amd import lib, ops
    from cpm.cu_amd.kvcache import PagedKVCache
    L = lib.get()
    option = lambda name, value: L.set_option(name.encode(), int(value))
    g = torch.Generator(device="cuda").manual_seed(S)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g).to(torch.float16)
    cache = PagedKVCache(1, hkv, (S + 255) // 256)
    cache.write_logical(0, 0, rnd(S, hkv, D), rnd(S, hkv, D))
    q = rnd(T, 32, D)
    mask = to_dev(torch, synth.random_tree(T, S, max_children=4, max_depth=9).mask)
    kv_len = torch.tensor([S], dtype=torch.int32, device="cuda")
    option("attn_direct", 0)
    try:
        kernel, used, groups, _ = ops.attention_plan(T, 32, hkv, S)
        assert (used, groups) == (splits, shape), kernel
        out = ops.tree_attention(q, cache, 0, kv_len, S, mask)
        option("attn_kv_groups", 3 - shape)
        option("attn_merge_in_launch", 0)
        ref = ops.tree_attention(q, cache, 0, kv_len, S, mask, num_splits=5)
        torch.cuda.synchronize()
    finally:
        option("attn_kv_groups", 0)
        option("attn_direct", -1)
        option("attn_merge_in_launch", 1)
    assert (out.float() - ref.float()).abs().max().item() <= 4.4e-3


@pytest.mark.parametrize("S,T,hkv,splits,shares", [
    (2200, 6, 4, 19, True), (8200, 6, 4, 17, False), (8200, 3, 4, 22, True), (16500, 5, 4, 19, False), (8200, 8, 2, 14, False), (6000, 8, 2, 16, False), (6050, 4, 2, 25, True),
    (4300, 4, 2, 18, True), (4300, 4, 8, 18, False), (4300, 3, 8, 18, True), (6000, 8, 1, 16, True), (5400, 5, 2, 22, True), (8200, 6, 2, 17, False)])
def test_merges_of_the_direct_shape_beside_their_lines(gpu, set_option, S, T, hkv, splits, shares):
    """The splits and the merge are those that the lines say, and both merges have the same partials: two orders of their fp32 sums, rounded to fp16 once."""
    torch = gpu
    from cpm.cu_amd import ops
    from cpm.cu_amd.kvcache import PagedKVCache
    g = torch.Generator(device="cuda").manual_seed(S)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g).to(torch.float16)
    cache = PagedKVCache(1, hkv, (S + 255) // 256)
    cache.write_logical(0, 0, rnd(S, hkv, D), rnd(S, hkv, D))
    q, kv_len = rnd(T, 32, D), torch.tensor([S], dtype=torch.int32, device="cuda")
    assert ops.attention_plan(T, 32, hkv, S)[:2] == ("tree_attn_direct%s_kernel" % ("_shares" if shares else ""), splits)
    out = ops.tree_attention(q, cache, 0, kv_len, S)
    set_option("attn_direct", 1)
    set_option("attn_merge_wait_us", 0)
    ref = ops.tree_attention(q, cache, 0, kv_len, S, num_splits=splits)
    assert float((out.float() - ref.float()).abs().max()) <= 2.0 ** -10 * float(ref.float().abs().max())
