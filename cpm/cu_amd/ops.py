"""The operators of the verify/draft path on torch device tensors.

torch only supplies device memory and the current stream; every function here is a thin call into
``libcpmcu_amd.so`` through the C-ABI (``include/cpmcu_amd.h``), made by the native binding
``_torch_call``.  Nothing falls back to torch math.
"""
import ctypes
import math

import torch

from . import lib as _libmod
from .kvcache import HEAD_DIM

_native = None


def _lib():
    return _libmod.get()


def _calls():
    """The library's operators as native calls on tensors (csrc/torch_call.cpp), bound to the library lib.py has loaded.
    Pointer arguments are tensors (device-resident and contiguous, or AssertionError) or None; the stream is torch's current one."""
    global _native
    if _native is None:
        lib = _libmod.get()
        try:
            from . import _torch_call
        except ImportError as e:
            raise ImportError("the torch binding is not built or does not fit this torch (%s); run `python -m cpm.cu_amd.build`" % e) from e
        _torch_call.bind(lib.raw._handle)
        _native = _torch_call
    return _native


def _ptr_result(t):
    """A device tensor, or a pinned host tensor in its place: the GPU writes it through the mapped address."""
    return t if t is None or t.is_cuda else (_native or _calls()).pinned(t)


# One scratch buffer per operator family and device, handed to every call: calls that use it have to follow one another (one stream, or
# streams that wait for each other).  A call that needs more gets a buffer of at least twice the size, and the old one is
# kept, because captured launches go on writing to the addresses they were recorded with; all those kept are less than the one in use.
_workspaces = {}
_outgrown = []


def _workspace(kind, nbytes, device):
    key = (kind, device)
    ws = _workspaces.get(key)
    if ws is None or ws.numel() < nbytes:
        if ws is not None:
            if kind == "attn":
                release_attention_workspace(ws)
            if kind == "head":
                release_head_workspace(ws)
            _outgrown.append(ws)
            nbytes = max(nbytes, 2 * ws.numel())
        ws = torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device=device)
        _workspaces[key] = ws
    return ws


def release_attention_workspace(ws):
    """Before an attention workspace tensor is dropped: the library gives its merge counters to another workspace.
    The device is synchronised first (no launch on the workspace may be in flight)."""
    torch.cuda.synchronize()
    _lib().tree_attention_release_workspace(ctypes.c_void_p(ws.data_ptr()))


def release_head_workspace(ws):
    """Before a head workspace tensor is dropped: the library takes back the states its one-launch FR-Spec head
    publishes through.  The device is synchronised first (no launch on the workspace may be in flight)."""
    torch.cuda.synchronize()
    _lib().head_release_workspace(ctypes.c_void_p(ws.data_ptr()))


_SCALE = 1.0 / math.sqrt(HEAD_DIM)


def synchronize():
    """Wait for torch's current stream."""
    (_native or _calls()).synchronize()


def mask_words(T):
    return (T + 63) // 64


def kv_append(cache, layer, k_new, v_new, kv_len):
    """copy_to_kvcache (src/model/attn.cuh:14-21): rows go to positions [*kv_len - T, *kv_len)."""
    (_native or _calls()).kv_append_rows(cache.k[layer], cache.v[layer], cache.block_table, k_new, v_new, kv_len, cache.Hkv)


def rope_table(position_ids, inv_freq):
    """(cos, sin) of float(position) * inv_freq for every tree row: [T, 64, 2] fp32 (src/model/rotary.cuh:11-17)."""
    T = position_ids.numel()
    assert position_ids.dtype == torch.int32 and inv_freq.dtype == torch.float32 and inv_freq.numel() == HEAD_DIM // 2
    out = torch.empty((T, HEAD_DIM // 2, 2), dtype=torch.float32, device=position_ids.device)
    _calls().rope_table(position_ids, inv_freq, T, out)
    return out


def rope_apply_(table, q, k):
    """In-place rotary embedding of q [T,Hq,128] and k [T,Hkv,128] (rotary_embedding_kernel, src/model/rotary.cuh:7-34)."""
    T, Hq, D = q.shape
    assert D == HEAD_DIM and k.shape[0] == T and k.shape[2] == D and table.shape[0] == T
    _calls().rope_apply(table, T, Hq, k.shape[1], q, k)


def tree_attention(q, cache, layer, kv_len, max_kv_len, mask=None, scale=None, num_splits=0, out=None,
                   k_new=None, v_new=None, mask_k_range=0, rope=None, block_window_size=0):
    """mha_fwd_kvcache with a tree mask (src/flash_attn/flash_api.hpp:292-392) on the paged cache.

    q [T, Hq, 128] fp16; kv_len int32[1] on the device = P + T; mask uint64 [T, W] or None (chain).
    k_new / v_new [T, Hkv, 128]: the tree rows' K/V; when given the kernel appends them to the cache
    itself (src/model/attn.cuh:200) instead of expecting them there.
    mask_k_range (0 = T): number of trailing keys the mask bits refer to; k*d for the drafter's layers.
    rope [T, 64, 2] fp32 from rope_table: q and k_new are taken unrotated and rotated inside the kernel.
    block_window_size (0 = none, else >= 128 tokens): the drafter layer's block sliding window
    (src/flash_attn/src/flash_blockmask.h:32): key blocks of 128 below ceil(P/128) - window/128 are skipped.
    """
    native = _native or _calls()
    if out is None:
        out = torch.empty_like(q)
    if mask is not None and not mask.is_contiguous():
        mask = mask.reshape(q.shape[0], -1)  # (a copy where the rows' order in memory is another one)
    ws = _workspaces.get(("attn", q.device))
    # (shapes and types are checked there)
    args = (q, cache.k[layer], cache.v[layer], cache.block_table, kv_len, int(max_kv_len), k_new, v_new, rope, int(block_window_size),
            mask, int(mask_k_range), cache.Hkv, _SCALE if scale is None else scale, out)
    need = native.tree_attention_rows(*args, ws, int(num_splits))
    if need is not None:
        native.tree_attention_rows(*args, _workspace("attn", need, q.device), int(num_splits))
    return out


def gather_rows(src, remap):
    """remap_copy (src/model/tree_drafter.cuh:79-86): dst[r] = src[remap[r]]."""
    assert src.dtype == torch.float16 and remap.dtype == torch.int32
    dst = torch.empty((remap.numel(), src.shape[1]), dtype=torch.float16, device=src.device)
    _calls().gather_rows(src, remap, remap.numel(), src.shape[1], dst)
    return dst


W_ROW_MAJOR, W_TILED = 0, 1
COMMIT_ADVANCE_LENGTH = 1
COMMIT_NEXT_ROOT = 2


class TiledWeight:
    """A head weight matrix in MFMA operand order (CPMCU_W_TILED): built once, streamed ~20 % faster."""

    def __init__(self, data, V, H):
        self.data, self.V, self.H = data, int(V), int(H)
        self.shape = (self.V, self.H)


def tile_head_weight(w, row_remap=None):
    """[*, H] row-major fp16 -> TiledWeight of V rows; with row_remap (int32 [V]) row r is w[row_remap[r]]
    (remap_copy, src/model/tree_drafter.cuh:79-86, fused with the re-tiling)."""
    assert w.dtype == torch.float16 and w.is_contiguous()
    H = w.shape[1]
    V = w.shape[0] if row_remap is None else row_remap.numel()
    out = torch.empty(_lib().raw.cpmcu_head_weight_tiled_bytes(V, H) // 2, dtype=torch.float16, device=w.device)
    _calls().head_weight_tile(w, row_remap, V, H, out)
    return TiledWeight(out, V, H)


def _weight(w):
    if isinstance(w, TiledWeight):
        return w.data, W_TILED, w.V
    return w, W_ROW_MAJOR, w.shape[0]


def frspec_head_topk(hidden, w, token_id_remap, k):
    """FR-Spec draft head: logits -> log-softmax -> top-k -> full-vocabulary ids.

    Returns dict(logits [n,V] f16 raw, row_stats [n,2] f32 (max, ln sum), val [n,k] f16, pos [n,k] i32, ids [n,k] i32).
    """
    n, H = hidden.shape
    w, layout, V = _weight(w)
    native = _native or _calls()
    logits, stats, val, pos, ids = native.empty(hidden, "h", n, V, "f", n, 2, "h", n, k, "i", n, k, "i", n, k)
    ws = _workspace("head", native.head_workspace_bytes(n, V), hidden.device)
    native.frspec_head_topk(hidden, w, layout, token_id_remap, n, V, H, k, logits, stats, val, pos, ids, ws, ws.numel())
    return dict(logits=logits, row_stats=stats, val=val, pos=pos, ids=ids)


def frspec_head_plan(n, w, k):
    """Kernel name(s) of a frspec_head_topk call with n hidden rows on matrix w: the one-launch kernel when the shape
    allows it and the library has a publication state for the head workspace, else GEMM + top-k."""
    w_, layout, V = _weight(w)
    H = w.H if isinstance(w, TiledWeight) else w.shape[1]
    gemm = head_plan(n, w)[0]
    ws = _workspace("head", _lib().raw.cpmcu_head_workspace_bytes(n, V), w_.device)
    if _lib().raw.cpmcu_frspec_head_mode(ctypes.c_void_p(ws.data_ptr()), layout, n, V, H, k) == 1:
        nb, fp, kc = gemm[gemm.index("<") + 1:-1].split(",")
        return "frspec_head_topk_kernel<%s,%s>" % (fp, kc)
    # the row kernel: on the whole row up to 32768 elements (in its short form up to 8192), on slices of it beyond
    slices = (V + 8191) // 8192
    short = V <= 8192 or (V > 32768 and n * slices <= 512 and slices * k <= 256)
    return gemm + ("+topk_short_row_kernel<true>" if short else "+topk_row_kernel<true>") + ("" if V <= 32768 else "+topk_slice_merge_kernel<true>")


def lm_head_argmax(hidden, w, head_scale=None, want_logits=False, gt=None):
    """Target head + arg-max (src/model/linear.cuh:82-101 + torch argmax of tree_drafter.py:233)."""
    n, H = hidden.shape
    w, layout, V = _weight(w)
    native = _native or _calls()
    logits = native.empty(hidden, "h", n, V)[0] if want_logits else None
    if gt is None:
        gt = torch.empty(n, dtype=torch.int32, device=hidden.device)
    ws = _workspace("head", native.head_workspace_bytes(n, V), hidden.device)
    native.lm_head_argmax(hidden, w, layout, n, V, H, 0 if head_scale is None else 1, 1.0 if head_scale is None else head_scale, logits, gt,
                          ws, ws.numel())
    return (gt, logits) if want_logits else gt


class HeadPartials:
    """The target head's arg-max left as per-workgroup partials (cpmcu_lm_head_partials): finished by verify_tail."""

    def __init__(self, workspace, num_partials, stride, n):
        self.workspace, self.num_partials, self.stride, self.n = workspace, int(num_partials), int(stride), int(n)


def lm_head_partials(hidden, w, head_scale=None, logits=None):
    """The target head's GEMM without the launch that finishes its arg-max; see verify_tail."""
    n, H = hidden.shape
    w, layout, V = _weight(w)
    native = _native or _calls()
    ws = _workspace("head", native.head_workspace_bytes(n, V), hidden.device)
    num, stride = native.lm_head_partials(hidden, w, layout, n, V, H, 0 if head_scale is None else 1,
                                          1.0 if head_scale is None else head_scale, logits, ws, ws.numel())
    return HeadPartials(ws, num, stride, n)


def verify_tail(cache, draft_ids, gt, position_ids, cache_length, attn_mask, tree_parent, hidden=None, prev_hidden=None,
                gt_out=None, best=None, path=None, accepted_ids=None, next_position_ids=None, result=None):
    """The whole tail of verify() in one launch (src/model/minicpm4/minicpm4_eagle.cuh:398-418): arg-max finish
    when `gt` is a HeadPartials, acceptance, compaction of every layer, accepted ids, hidden-row gather.
    draft_ids is read only; results go to best (a, node), path [T], accepted_ids [T], gt_out [T], ..."""
    T = draft_ids.numel()
    W = attn_mask.numel() // T
    parts = gt if isinstance(gt, HeadPartials) else None
    hidden_dim = 0 if hidden is None else hidden.shape[-1]
    (_native or _calls()).verify_tail(
        cache.k_ptrs, cache.v_ptrs, cache.num_layers, cache.block_table, cache.Hkv, T, draft_ids, None if parts else gt,
        parts.workspace if parts else None, parts.num_partials if parts else 0, parts.stride if parts else 0, position_ids, cache_length,
        attn_mask, W, tree_parent, hidden, hidden_dim, prev_hidden, gt_out, best, path, accepted_ids, next_position_ids, _ptr_result(result))


def verify_tail_inplace(best, accepted_ids, pred=None, cache_length=None, kv_len=None, position_ids=None, advance_length=False,
                        next_root=False):
    """The in-place updates behind verify_tail: pred[:a] <- ids (or pred[0] <- last id), lengths and positions += a."""
    flags = (COMMIT_ADVANCE_LENGTH if advance_length else 0) | (COMMIT_NEXT_ROOT if next_root else 0)
    _calls().verify_tail_inplace(best, accepted_ids, accepted_ids.numel(), pred, cache_length, kv_len, position_ids, flags)


def log_softmax_(x):
    """In place (src/model/eagle.cuh:29-89); returns row_stats [n,2] (max, ln sum)."""
    n, dim = x.shape
    native = _native or _calls()
    # (the slices' few bytes are the call's own, as the outputs are: calls on several streams or threads, and captured ones, share nothing)
    stats, ws = native.empty(x, "f", n, 2, "f", native.log_softmax_workspace_bytes(n, dim) // 4, 0)
    native.log_softmax_sliced(x, n, dim, stats, ws, ws.nbytes)
    return stats


def topk(x, top):
    """TopK::prefill (src/model/topk.cuh:255-288): value descending, ties -> lower index."""
    n, dim = x.shape
    native = _native or _calls()
    val, pos = native.empty(x, "h", n, top, "i", n, top)
    ws = _workspace("topk", native.topk_workspace_bytes(n, dim, top), x.device)
    native.topk(x, n, dim, top, val, pos, ws, ws.numel())
    return val, pos


def remap(pos, token_id_remap):
    out = torch.empty_like(pos)
    _calls().remap(pos, pos.numel(), token_id_remap, out)
    return out


def tree_accept(pred, gt, position_ids, cache_length, attn_mask, tree_parent, best=None):
    """verify_kernel (src/model/tree_drafter.cuh:5-46). pred is overwritten with the path; returns best[2]."""
    T = pred.numel()
    if best is None:
        best = torch.empty(2, dtype=torch.int32, device=pred.device)
    W = attn_mask.numel() // T
    _calls().tree_accept(T, pred, gt, position_ids, cache_length, attn_mask, W, tree_parent, best)
    return best


def kv_compact(cache, pred, gt, cache_length, best, max_accept):
    """fix_kv_cache (src/model/tree_drafter.cuh:48-77) on every layer of the paged cache."""
    _calls().kv_compact(cache.k_ptrs, cache.v_ptrs, cache.num_layers, cache.block_table, cache.Hkv, pred, gt, cache_length, best, int(max_accept))


def accept_commit(cache, pred, gt, cache_length, best, max_accept, hidden=None, prev_hidden=None,
                  next_position_ids=None, result=None, advance_length=False, next_root=False, kv_len=None):
    """The rest of verify() after the acceptance (src/model/minicpm4/minicpm4_eagle.cuh:398-418): compaction,
    accepted ids, gather of the accepted hidden rows, next position ids, packed (a, ids) result and the
    device-side advance of cache_length, in two launches with the accept length staying on the device."""
    flags = (COMMIT_ADVANCE_LENGTH if advance_length else 0) | (COMMIT_NEXT_ROOT if next_root else 0)
    hidden_dim = 0 if hidden is None else hidden.shape[-1]
    _calls().accept_commit(cache.k_ptrs, cache.v_ptrs, cache.num_layers, cache.block_table, cache.Hkv, pred, gt, cache_length, kv_len, best,
                           int(max_accept), hidden, hidden_dim, prev_hidden, next_position_ids, _ptr_result(result), flags)


class DraftTree:
    """Tree bookkeeping of the drafter (src/model/minicpm4/minicpm4_eagle.cuh:319-393) on the device.

    One object per draft model; ``begin`` / ``extend`` / ``finish`` are one kernel each and never
    synchronise, so a whole draft can be enqueued (or graph-captured) without a host round trip.
    """

    def __init__(self, k, num_iter, token_id_remap=None, device="cuda"):
        self.k, self.num_iter = int(k), int(num_iter)
        self.remap = token_id_remap
        nbytes = _lib().raw.cpmcu_draft_tree_state_bytes(self.k, self.num_iter)
        self.state = torch.zeros(max(nbytes, 256), dtype=torch.uint8, device=device)
        self.next_ids = torch.empty(self.k, dtype=torch.int32, device=device)
        self.parent_rows = torch.empty(self.k, dtype=torch.int32, device=device)
        self.draft_mask = torch.empty(self.k, dtype=torch.int64, device=device)

    def begin(self, topk_val, topk_pos):
        """topk_val fp16[k], topk_pos int32[k] (first row). Returns next_ids [k]."""
        assert topk_val.dtype == torch.float16 and topk_pos.dtype == torch.int32 and topk_val.numel() == self.k
        (_native or _calls()).draft_tree_begin(self.state, self.k, self.num_iter, topk_val, topk_pos, self.remap, self.next_ids, self.draft_mask)
        return self.next_ids

    def extend(self, d, topk_val, topk_pos):
        """topk_val fp16[k,k] (cumulated in place), topk_pos int32[k,k] of iteration d >= 1.
        Returns (next_ids [k], parent_rows [k], draft_mask [k])."""
        assert topk_val.dtype == torch.float16 and topk_pos.dtype == torch.int32 and topk_val.numel() == self.k * self.k
        (_native or _calls()).draft_tree_extend(self.state, self.k, self.num_iter, int(d), topk_val, topk_pos, self.remap, self.next_ids,
                                                self.parent_rows, self.draft_mask)
        return self.next_ids, self.parent_rows, self.draft_mask

    def finish(self, tree_size, cache_length, tree_draft_ids=None):
        """cache_length int32[1] on the device = P.  Returns (ids [T] -- entry 0 untouched --, positions [T],
        mask [T, W] as int64 bit patterns, parent [T])."""
        native, T = _native or _calls(), int(tree_size)
        W = mask_words(T)
        if tree_draft_ids is not None:
            pos, mask, parent = native.empty(self.state, "i", T, 0, "l", T, W, "i", T, 0)
            native.draft_tree_finish(self.state, self.k, self.num_iter, T, cache_length, self.remap, tree_draft_ids, pos, mask, parent)
        else:
            tree_draft_ids, pos, mask, parent = native.empty(self.state, "i", T, 0, "i", T, 0, "l", T, W, "i", T, 0)
            native.draft_tree_finish_root(self.state, self.k, self.num_iter, T, cache_length, self.remap, -1, tree_draft_ids, pos, mask, parent)
        return tree_draft_ids, pos, mask, parent


def attention_plan(T, Hq, Hkv, max_kv_len, rope=False, block_window_size=0, num_splits=0):
    """(kernel names, KV splits, KV groups per workgroup, workgroups) of a tree-attention call of this shape."""
    buf = ctypes.create_string_buffer(160)
    ns, g, wg = ctypes.c_int(0), ctypes.c_int(0), ctypes.c_int(0)
    _lib().tree_attention_plan(T, Hq, Hkv, int(max_kv_len), 1 if rope else 0, int(block_window_size), int(num_splits), buf, 160,
                               ctypes.byref(ns), ctypes.byref(g), ctypes.byref(wg))
    return buf.value.decode(), ns.value, g.value, wg.value


def head_plan(n, w):
    """(GEMM kernel name, workgroups) of a head call with n hidden rows on weight matrix w."""
    _, layout, V = _weight(w)
    H = w.H if isinstance(w, TiledWeight) else w.shape[1]
    buf = ctypes.create_string_buffer(96)
    wg = ctypes.c_int(0)
    _lib().head_plan(n, V, H, layout, buf, 96, ctypes.byref(wg))
    return buf.value.decode(), wg.value
