"""GPU parity of the draft-tree construction kernels (through the C-ABI) against the CPU oracle:
every output is integer or a bit pattern, so the bar is equality."""
import numpy as np
import pytest

from cpm.cu_amd import synth
from test_draft_tree_cpu import make_rows, run_oracle
from util import to_dev, to_np

pytestmark = pytest.mark.gpu


def run_gpu(torch, k, num_iter, T, P, vals, poss, remap):
    from cpm.cu_amd import ops
    t = ops.DraftTree(k, num_iter, None if remap is None else to_dev(torch, remap))
    trace = [to_np(t.begin(to_dev(torch, vals[0][0]), to_dev(torch, poss[0][0]))).copy()]
    cums = []
    for d in range(1, num_iter):
        v = to_dev(torch, vals[d])
        ids, rows, mask = t.extend(d, v, to_dev(torch, poss[d]))
        torch.cuda.synchronize()
        trace.append((to_np(ids).copy(), to_np(rows).copy(), to_np(mask).view(np.uint64).copy()))
        cums.append(to_np(v))
    cl = torch.tensor([P], dtype=torch.int32, device="cuda")
    ids, pos, mask, parent = t.finish(T, cl)
    torch.cuda.synchronize()
    return (to_np(ids), to_np(pos), to_np(mask).view(np.uint64), to_np(parent)), trace, cums


@pytest.mark.parametrize("k,num_iter,T,seed,with_remap,dyadic", [(2, 2, 4, 1, False, True), (3, 3, 10, 2, True, False),
                                                                  (10, 6, 60, 4, True, False), (10, 6, 64, 5, False, True),
                                                                  (8, 8, 32, 6, True, False), (10, 3, 128, 7, True, False),
                                                                  (32, 2, 100, 8, True, False), (1, 5, 5, 9, False, False)])
def test_draft_tree_equals_oracle(gpu, orc, k, num_iter, T, seed, with_remap, dyadic):
    torch = gpu
    vocab, full = 500, 2000
    remap = synth.frspec_remap(full, vocab, seed) if with_remap else None
    vals, poss = make_rows(k, num_iter, vocab, seed, dyadic=dyadic)
    P = 4096 + seed
    (o_ids, o_pos, o_mask, o_parent), o_trace = run_oracle(orc, k, num_iter, T, P, vals, poss, remap)
    (g_ids, g_pos, g_mask, g_parent), g_trace, _ = run_gpu(torch, k, num_iter, T, P, vals, poss, remap)
    assert np.array_equal(g_trace[0], o_trace[0])
    for d in range(1, num_iter):
        for a, b in zip(g_trace[d], o_trace[d]):
            assert np.array_equal(a, b), "iteration %d" % d
    assert np.array_equal(g_ids[1:], o_ids[1:]) and g_ids[0] == -1
    assert np.array_equal(g_pos, o_pos) and np.array_equal(g_parent, o_parent)
    assert np.array_equal(g_mask, o_mask)


@pytest.mark.parametrize("k,num_iter,T,with_remap", [(15, 4, 64, True), (16, 4, 64, True), (16, 2, 30, False), (17, 3, 60, True), (24, 2, 128, False)])
def test_rounds_of_one_and_of_several_candidates_a_thread(gpu, orc, k, num_iter, T, with_remap):
    """Up to 256 candidates a thread of the extend kernel holds one, beyond up to four: both sides of that line, with ties and with
    zeros of either sign (whose bits the running log-probs keep)."""
    torch = gpu
    remap = synth.frspec_remap(2000, 500, k) if with_remap else None
    vals, poss = make_rows(k, num_iter, 500, k, dyadic=True)
    for d in range(num_iter):
        vals[d][:, 0] = np.float16(-0.0 if d % 2 == 0 else 0.0)
    (o_ids, o_pos, o_mask, o_parent), o_trace = run_oracle(orc, k, num_iter, T, 99, vals, poss, remap)
    (g_ids, g_pos, g_mask, g_parent), g_trace, _ = run_gpu(torch, k, num_iter, T, 99, vals, poss, remap)
    assert np.array_equal(g_trace[0], o_trace[0])
    for d in range(1, num_iter):
        for a, b in zip(g_trace[d], o_trace[d]):
            assert np.array_equal(a, b), "iteration %d" % d
    assert np.array_equal(g_ids[1:], o_ids[1:]) and np.array_equal(g_pos, o_pos)
    assert np.array_equal(g_parent, o_parent) and np.array_equal(g_mask, o_mask)


@pytest.mark.parametrize("bits", [0xFC00, 0xFFFF])  # -inf of a padded list, and what an unfinished row of a one-launch head holds
@pytest.mark.parametrize("k,num_iter,T,rows_lost,cols_lost", [(4, 4, 30, 1, 2), (10, 3, 60, 9, 3), (17, 3, 128, 5, 0), (6, 2, 40, 6, 6)])
def test_positions_of_minus_one_stay_inside_the_table(gpu, orc, k, num_iter, T, rows_lost, cols_lost, bits):
    """Candidates that are none (position -1, the lowest value): they read the table's first entry and not the one in front of it,
    ranked among the chosen or not.  The last rows of every round lost, and the last columns of the first."""
    from cpm.cu_amd import ops
    torch = gpu
    vals, poss = make_rows(k, num_iter, 500, k, dyadic=True)
    table = synth.frspec_remap(2000, 500, k)
    lost = [np.zeros(p.shape, bool) for p in poss]
    lost[0][:, k - cols_lost:] = True
    for d in range(1, num_iter):
        lost[d][k - rows_lost:] = True
    o_vals = [np.where(m, np.float16(-np.inf), v) for m, v in zip(lost, vals)]
    (o_ids, o_pos, o_mask, o_parent), o_trace = run_oracle(orc, k, num_iter, T, 99, o_vals, [np.where(m, 0, p) for m, p in zip(lost, poss)], table)
    g_vals = [np.where(m, np.uint16(bits), v.view(np.uint16)).view(np.float16) for m, v in zip(lost, vals)]
    g_poss = [np.where(m, -1, p).astype(np.int32) for m, p in zip(lost, poss)]
    around = to_dev(torch, np.concatenate([[-777], table]).astype(np.int32))
    t = ops.DraftTree(k, num_iter, around[1:])
    assert np.array_equal(to_np(t.begin(to_dev(torch, g_vals[0][0]), to_dev(torch, g_poss[0][0]))), o_trace[0])
    for d in range(1, num_iter):
        ids, rows, mask = t.extend(d, to_dev(torch, g_vals[d]), to_dev(torch, g_poss[d]))
        for a, b in zip((to_np(ids), to_np(rows), to_np(mask).view(np.uint64)), o_trace[d]):
            assert np.array_equal(a, b), "iteration %d" % d
    ids, pos, mask, parent = (to_np(x) for x in t.finish(T, torch.tensor([99], dtype=torch.int32, device="cuda")))
    assert np.array_equal(ids[1:], o_ids[1:]) and np.array_equal(pos, o_pos)
    assert np.array_equal(parent, o_parent) and np.array_equal(mask.view(np.uint64), o_mask)


@pytest.mark.parametrize("k,num_iter,T,equal", [(8, 3, 64, 0.), (9, 3, 60, 0.), (8, 4, 2, 0.), (8, 4, 64, 0.), (8, 4, 65, 0.), (8, 4, 66, 0.), (12, 2, 60, 0.), (14, 2, 60, .3), (10, 6, 60, 1.), (10, 6, 60, .9), (8, 8, 65, .99),
                                                (32, 2, 64, .5), (32, 2, 2, 0.), (10, 6, 30, -1.)])
def test_entries_below_the_bound_are_left_out(gpu, orc, k, num_iter, T, equal):
    """Histories around the length from which the last step bounds its entries, one and several entries a thread, the smallest and the largest tree that it is done
    for and the next one, with ties at the bound (`equal` of the log-probs the same; -1: all of them -inf but for one a row)."""
    torch = gpu
    vals, poss = make_rows(k, num_iter, 500, k + T)
    rng = np.random.default_rng(T)
    for v in vals:
        v[rng.random(v.shape) < equal] = np.float16(-0.5)
        if equal < 0:
            v[:, 1:] = np.float16(-np.inf)
    (o_ids, o_pos, o_mask, o_parent), _ = run_oracle(orc, k, num_iter, T, 99, vals, poss, None)
    (g_ids, g_pos, g_mask, g_parent), _, _ = run_gpu(torch, k, num_iter, T, 99, vals, poss, None)
    assert np.array_equal(g_ids[1:], o_ids[1:]) and np.array_equal(g_pos, o_pos)
    assert np.array_equal(g_parent, o_parent) and np.array_equal(g_mask, o_mask)


def test_heavy_ties(gpu, orc):
    """All log-probs equal: every choice is made by the index rule alone."""
    torch = gpu
    k, num_iter, T = 4, 4, 20
    vals = [np.full((1 if d == 0 else k, k), -0.5, np.float16) for d in range(num_iter)]
    poss = [np.arange((1 if d == 0 else k) * k, dtype=np.int32).reshape(-1, k) + 10 * d for d in range(num_iter)]
    (o_ids, o_pos, o_mask, o_parent), _ = run_oracle(orc, k, num_iter, T, 7, vals, poss, None)
    (g_ids, g_pos, g_mask, g_parent), _, _ = run_gpu(torch, k, num_iter, T, 7, vals, poss, None)
    assert np.array_equal(g_ids[1:], o_ids[1:]) and np.array_equal(g_pos, o_pos)
    assert np.array_equal(g_parent, o_parent) and np.array_equal(g_mask, o_mask)


def test_tree_feeds_the_verify_path(gpu, orc):
    """The tree the draft kernels build is consumed as is by acceptance: plant the target's choices
    along one root path of the built tree and check the accept length."""
    from cpm.cu_amd import ops
    torch = gpu
    k, num_iter, T, P = 10, 6, 60, 4096
    vocab, full = 500, 2000
    remap = synth.frspec_remap(full, vocab, 11)
    vals, poss = make_rows(k, num_iter, vocab, 11, dyadic=False)
    t = ops.DraftTree(k, num_iter, to_dev(torch, remap))
    t.begin(to_dev(torch, vals[0][0]), to_dev(torch, poss[0][0]))
    for d in range(1, num_iter):
        t.extend(d, to_dev(torch, vals[d]), to_dev(torch, poss[d]))
    cl = torch.tensor([P], dtype=torch.int32, device="cuda")
    ids = torch.full((T,), -1, dtype=torch.int32, device="cuda")
    ids[0] = 1234  # the root token is the caller's
    ids, pos, mask, parent = t.finish(T, cl, tree_draft_ids=ids)
    torch.cuda.synchronize()
    ids_np, par_np = to_np(ids), to_np(parent)
    depth = to_np(pos) - P
    leaf = int(np.argmax(depth))  # a deepest node
    path = [leaf]
    while path[-1] != 0:
        path.append(int(par_np[path[-1]]))
    path = path[::-1]
    gt = np.full(T, full + 5, np.int32)  # matches nothing ...
    for a, b in zip(path[:-1], path[1:]):
        gt[a] = ids_np[b]                # ... except along the chosen path
    pred = ids.clone()
    best = ops.tree_accept(pred, to_dev(torch, gt), pos, cl, mask, parent)
    torch.cuda.synchronize()
    assert int(best[0]) == len(path) and int(best[1]) == leaf
    assert to_np(pred)[:len(path)].tolist() == path


def test_argument_errors(gpu):
    from cpm.cu_amd import ops
    with pytest.raises(ValueError):
        ops.DraftTree(10, 7).begin(gpu.zeros(10, dtype=gpu.float16, device="cuda"), gpu.zeros(10, dtype=gpu.int32, device="cuda"))
