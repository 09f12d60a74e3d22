"""CPU-only checks of the boundary: the shared library loads without a GPU and exports every symbol
that include/cpmcu_amd.h declares; the ctypes table covers them all; argument validation that needs
no device works; the pybind11 module `C` exposes the reference's entry-point names."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "cpmcu_amd.h")


def declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(cpmcu_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from cpm.cu_amd import lib
    raw = ctypes.CDLL(lib.LIB_PATH)
    names = declared_symbols()
    assert len(names) >= 30
    for name in names:
        assert hasattr(raw, name), "libcpmcu_amd.so does not export %s" % name


def test_timeline_library_is_the_product_plus_its_readers():
    """The build with the in-kernel stamps (csrc/timeline.h) exports everything the product library does, and the two
    functions that hand the records over; the product library has neither."""
    from cpm.cu_amd import build, lib
    tl = ctypes.CDLL(build.TIMELINE_LIB_PATH)
    for name in declared_symbols():
        assert hasattr(tl, name), "libcpmcu_amd_timeline.so does not export %s" % name
    product = ctypes.CDLL(lib.LIB_PATH)
    for name in ("cpmcu_timeline_read_attention", "cpmcu_timeline_read_head", "cpmcu_timeline_read_topk"):
        assert hasattr(tl, name)
        assert not hasattr(product, name)


def test_ctypes_table_matches_header():
    from cpm.cu_amd import lib
    assert sorted(lib.SIGNATURES) == declared_symbols()
    lib.load_raw()


def test_argument_validation_without_device():
    """Checks that run before any HIP call: status codes, messages, exception mapping."""
    from cpm.cu_amd import lib
    L = lib.get()
    assert b"gfx950" in L.raw.cpmcu_version()
    with pytest.raises(ValueError, match="null pointer"):
        L.tree_accept(60, None, None, None, None, None, 1, None, None, None)
    with pytest.raises(ValueError, match="tree size 129"):
        p = ctypes.c_void_p(16)
        L.tree_accept(129, p, p, p, p, p, 3, p, p, None)
    with pytest.raises(ValueError, match="mask_words"):
        p = ctypes.c_void_p(16)
        L.tree_accept(100, p, p, p, p, p, 1, p, p, None)
    with pytest.raises(ValueError, match="top=200"):
        p = ctypes.c_void_p(16)
        L.topk(p, 1, 1000, 200, p, p, None, 0, None)
    with pytest.raises(RuntimeError, match="outside the verify/draft path"):
        L.decode(1, 128, 0, 0, 0, 0, 0, 0)
    with pytest.raises(RuntimeError, match="no model"):
        L.load_model(b"lm_head.weight", 1)
    assert L.raw.cpmcu_tree_attention_workspace_bytes(60, 32, 2, 4156) > 0
    assert L.raw.cpmcu_head_workspace_bytes(60, 73448) > 0


def test_pybind_module_has_reference_names():
    """Names of src/entry.cu:510-534."""
    from cpm.cu_amd import C
    for name in ("init_base_model", "init_minicpm4_model", "init_w4a16_gptq_marlin_base_model",
                 "init_w4a16_gptq_marlin_minicpm4_model", "init_eagle_model", "init_minicpm4_eagle_model",
                 "init_w4a16_gm_spec_w4a16_gm_model", "init_hier_eagle_w4a16_gm_spec_w4a16_gm_model",
                 "init_hier_eagle_w4a16_gm_rot_spec_w4a16_gm_model", "init_storage", "load_model", "prefill",
                 "decode", "draft", "verify_and_fix", "print_perf_summary"):
        assert callable(getattr(C, name)), name
    with pytest.raises(RuntimeError, match="outside the verify/draft path"):
        C.decode(1, 128, 0, 0, 0, 0, 0, False)
    with pytest.raises(RuntimeError):
        C.init_minicpm4_model(0.9, 1, 1, 1, 1, 1, 1, 128, 1e-5, 0, 1, 1.0, 1.0, 1.0, 0, 0, 0, 0, False)
    with pytest.raises(RuntimeError, match="dtype"):
        C.init_base_model(0.5, 100, 1, 512, 1024, 32, 2, 128, 1e-5, 2, 2048, 1.0, 1.0, 1.0)
    with pytest.raises(ValueError, match="head_dim"):
        C.init_base_model(0.5, 100, 1, 512, 1024, 32, 2, 64, 1e-5, 0, 2048, 1.0, 1.0, 1.0)


@pytest.mark.parametrize("args, error", [
    ((None,) * 6 + (1, 1), (ValueError, RuntimeError)),           # null pointers; without a device there is no stream either
    ((None,) * 6 + (1,), TypeError),                              # one argument short
    (("k",) + (None,) * 5 + (1, 1), TypeError),                   # neither a tensor nor an address
    ((None,) * 6 + (1 << 40, 1), OverflowError),
])
def test_torch_binding_checks_its_arguments(args, error):
    from cpm.cu_amd import ops
    with pytest.raises(error):
        ops._calls().kv_append(*args)


def test_torch_binding_refuses_host_tensors():
    import torch
    from cpm.cu_amd import ops
    with pytest.raises(AssertionError, match="device-resident"):
        ops._calls().kv_append(torch.zeros(4), None, None, None, None, None, 1, 1)


@pytest.mark.parametrize("address", [4096, True, 0, 2.5, object()])
def test_torch_binding_takes_no_bare_addresses(address):
    """Where a pointer goes, only tensors, None and what pinned() has looked at: a number that strayed there is refused, not written to."""
    import torch
    from cpm.cu_amd import ops
    native = ops._calls()
    for pos in range(6):
        args = [None] * 6 + [1, 1]
        args[pos] = address
        with pytest.raises(TypeError, match="a tensor or None required"):
            native.kv_append(*args)
    with pytest.raises(TypeError, match="a tensor or None required"):
        native.tree_attention_rows(None, None, None, None, None, 256, None, None, None, 0, address, 0, 2, 1.0, None, None, 0)
    with pytest.raises(AssertionError, match="pinned"):
        ops._ptr_result(torch.zeros(4, dtype=torch.int32))
    with pytest.raises(AssertionError, match="device-resident"):
        native.empty(torch.zeros(4), "h", 4, 0)


def test_tree_attention_takes_masks_that_reshape_makes_contiguous(monkeypatch):
    """Mask rows that lie in another order in memory reach the binding as a contiguous copy in row order; contiguous ones as they are."""
    import types
    import torch
    from cpm.cu_amd import ops
    seen = []
    monkeypatch.setattr(ops, "_native", types.SimpleNamespace(tree_attention_rows=lambda *args: seen.append(args[10])))
    cache = types.SimpleNamespace(k=[None], v=[None], block_table=None, Hkv=2)
    q = torch.zeros((6, 32, 128), dtype=torch.float16)
    halves = torch.arange(12, dtype=torch.int64).reshape(2, 3, 2)
    for mask in (halves.transpose(0, 1), halves.transpose(0, 1).contiguous(), None):
        ops.tree_attention(q, cache, 0, None, 256, mask)
    assert seen[0].is_contiguous() and seen[0].shape == (6, 2) and torch.equal(seen[0].flatten(), halves.transpose(0, 1).flatten())
    assert seen[1].shape == (3, 2, 2) and seen[2] is None


@pytest.mark.parametrize("prefixes, error", [([], None), ([None], TypeError)])
def test_attention_timeline_gives_the_choice_of_shape_back(prefixes, error):
    import contextlib
    import types
    import torch
    from cpm.cu_amd import timeline
    told = []
    with pytest.raises(error) if error else contextlib.nullcontext():
        timeline.attention(types.SimpleNamespace(set_option=lambda *a: told.append(a)), torch, prefixes, 1)
    assert told == [(b"attn_direct", 0), (b"attn_direct", -1)]


def test_outgrown_workspaces_stay(monkeypatch):
    """Captured launches hold the addresses of the workspace they were recorded with: a larger one does not give it away, and what
    is kept stays below what is in use."""
    import torch
    from cpm.cu_amd import ops
    monkeypatch.setattr(ops, "_workspaces", {})
    monkeypatch.setattr(ops, "_outgrown", [])
    monkeypatch.setattr(ops, "release_attention_workspace", lambda ws: None)
    cpu = torch.device("cpu")
    for kind in ("topk", "attn"):
        seen = []
        for nbytes in (10, 300, 301, 40000, 39999, 70000, 10 ** 6):
            ws = ops._workspace(kind, nbytes, cpu)
            assert ws.numel() >= nbytes
            seen += [ws.data_ptr()] if ws.data_ptr() not in seen else []
        kept = [t for t in ops._outgrown if t.data_ptr() in seen]
        assert [t.data_ptr() for t in kept] == seen[:-1] and sum(t.numel() for t in kept) < ws.numel()


_NOT_MEMORY = """
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from cpm.cu_amd import ops
native = ops._calls()
with FakeTensorMode(allow_non_fake_inputs=True):
    fake = torch.empty((4, 2, 128), dtype=torch.float16, device="cuda")
sparse = torch.sparse_coo_tensor(torch.zeros((1, 0), dtype=torch.int64), torch.zeros(0), (4,))
calls = [lambda t: native.kv_append(t, None, None, None, None, None, 1, 1), lambda t: native.kv_append_rows(None, None, None, t, t, t, 2),
         lambda t: native.tree_attention_rows(t, None, None, None, t, 256, None, None, None, 0, None, 0, 2, 1.0, None, None, 0),
         lambda t: native.lm_head_partials(t, t, 0, 1, 16, 512, 0, 1.0, None, None, 0), lambda t: native.empty(t, "h", 4, 0), lambda t: native.topk(t, 1, 4, 1, t, t, t, 0)]
seen = []
def vmapped(t):
    seen.append(t)
    for call in calls:
        refused(call, t)
    return t
def refused(call, t):
    try:
        call(t)
    except (RuntimeError, AssertionError):
        return
    raise SystemExit("accepted: %r" % t)
for t in (fake, sparse):
    for call in calls:
        refused(call, t)
with FakeTensorMode(allow_non_fake_inputs=True):
    torch.func.vmap(vmapped)(fake)
assert len(seen) == 1
print("all refused")
"""


def test_torch_binding_raises_for_tensors_without_memory():
    """Vmapped, fake and sparse tensors throw when they are asked for their layout or memory: a Python error, not the end of the
    process (hence one of its own)."""
    import subprocess
    import sys
    res = subprocess.run([sys.executable, "-c", _NOT_MEMORY], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert res.returncode == 0 and "all refused" in res.stdout, res.stdout


def test_requests_into_lds_set_their_own_lds_address():
    """A load into LDS takes its LDS address from m0, which the compiler may use between two statements: every inline assembly
    statement with such a load sets m0 itself, in front of the load, and says that it does."""
    csrc = os.path.join(ROOT, "cpm", "cu_amd", "csrc")
    found = 0
    for name in sorted(os.listdir(csrc)):
        if not name.endswith((".hip", ".h")):
            continue
        for statement in re.findall(r"\basm\b[^;]*?;", open(os.path.join(csrc, name)).read(), flags=re.S):
            if re.search(r"load_lds|\blds\b", statement):
                found += 1
                assert 0 <= statement.find("s_mov_b32 m0") < re.search(r"load_lds|\blds\b", statement).start(), (name, statement)
                assert '"m0"' in statement, (name, statement)
    assert found >= 5


@pytest.mark.parametrize("n,V,H,sliced", [
    (96, 65536, 4096, True), (97, 30304, 4096, True), (97, 30320, 4096, False), (128, 32768, 2048, True), (128, 32784, 4096, True), (97, 52416, 4096, True), (97, 52432, 4096, False), (128, 60000, 4096, False),
    (128, 65536, 2048, False), (128, 65552, 4096, True), (100, 57344, 2048, True), (100, 57360, 2048, False), (128, 120000, 4096, False),
    (128, 104848, 4096, True), (128, 104864, 4096, False), (100, 151936, 4096, False)])
def test_row_major_heads_of_many_rows_take_the_faster_kernel(n, V, H, sliced):
    """More than 96 rows: the K slices unless the chunked kernel's passes over the wave slots are nearly full, 37 fortieths of one, 32 of several
    (2048 columns: always with one, 35 of several).
    (The plan counts 256 CUs where there is no device.)"""
    from cpm.cu_amd import lib
    name, wg = ctypes.create_string_buffer(96), ctypes.c_int(0)
    lib.get().head_plan(n, V, H, 0, name, 96, ctypes.byref(wg))
    assert ("slice_kernel" in name.value.decode()) == sliced, name.value


@pytest.mark.parametrize("hkv,T", [(1, 1), (1, 4), (1, 8), (2, 1), (2, 2), (2, 4), (2, 5), (2, 8), (4, 1), (4, 4), (4, 6), (8, 1), (8, 2), (8, 4)])
def test_direct_splits_have_the_same_number_of_blocks(hkv, T):
    """No more splits than give each the same number of 128-key blocks, but for the last ones: more of them are slower but for lengths that are whole
    multiples of 128 keys per split.  (The plan counts 256 CUs where there is no device.)"""
    from cpm.cu_amd import ops
    direct = 0
    for S in [*range(1024, 20000, 128), 32896, 37376, 60032, 65664, 99072]:
        kernel, splits, _, _ = ops.attention_plan(T, 32, hkv, S)
        if "direct" in kernel:
            blocks = -(-S // 128) + 1
            direct += 1
            assert splits == -(-blocks // -(-blocks // splits)), S
    assert direct > 50


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("T,S,rope,splits,name", [
    (1, 512, False, 0, "tree_attn_direct{}_kernel"), (1, 4224, True, 0, "tree_attn_direct_shares{}_kernel"), (60, 32896, False, 0, "tree_attn_split{}_kernel<1,false,false>"), (60, 4224, True, 0, "tree_attn_split{}_kernel<2,true,true>"),
    (16, 32896, True, 0, "tree_attn_split{}_kernel<2,true,false>+tree_attn_combine_wide{}_kernel"),
    (60, 4224, False, 5, "tree_attn_split{}_kernel<2,false,false>+tree_attn_combine{}_kernel"), (60, 4224, False, 1, "tree_attn_split{}_kernel<2,false,false>")])
def test_plans_name_the_kernels_that_are_launched(set_option, dtype, T, S, rope, splits, name):
    """Direct or split, merged in shares or by the last arrival, rotary embedding, element type and merge launch, through an XCD's L2 or memory.
    (The plan counts 256 CUs where there is no device.)"""
    from cpm.cu_amd import ops
    set_option("dtype", dtype)
    if "combine{}_k" in name:
        set_option("attn_merge_in_launch", 0)
    kernel, used, _, _ = ops.attention_plan(T, 32, 2, S, rope, num_splits=splits)
    assert kernel == name.format(*["_bf16" * dtype] * 2) and (not splits or used == splits)
