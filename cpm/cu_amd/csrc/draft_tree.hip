// Draft-tree construction around the FR-Spec head for gfx950: the tree bookkeeping of the
// reference's draft() (src/model/minicpm4/minicpm4_eagle.cuh:319-393) as three single-workgroup
// kernels that keep all state on the device:
//   begin  -- d = 0: record the first k candidates, init_tree (src/model/eagle.cuh:91-93);
//   extend -- d >= 1: cumsum (eagle.cuh:103-106), history append, top-k over k*k -> k,
//             set_parent / update_tree (eagle.cuh:95-101), id remap (eagle.cuh:121-127) and the row
//             indices the hidden-state gather needs (remap_hidden, eagle.cuh:108-115);
//   finish -- top-(T-1) over the whole history, build_dynamic_tree (eagle.cuh:188-214) and the id
//             remap of the chosen nodes.
// The reference spends about ten launches and a device-to-host copy per iteration on these; here
// the prefix length is read from device memory, so building the tree needs no host round trip.
// Selection follows the ordering of the top-k kernels (value descending, lower index first).  The
// histories are short (k*k = 100 and k + 5*k*k = 510 entries at the reference's settings), so it is
// done by counting: every entry becomes a unique 32-bit key in LDS, every thread counts the keys above
// its own, and that count is the entry's place in the sorted order -- no rounds, two barriers.
#include "common.h"
#include "internal.h"
#include "topk_keys.h"

namespace cpmcu {
namespace {

constexpr int kMaxK = 32;        // topk_per_iter
constexpr int kMaxTried = kTopkThreads * kPerThread;  // history entries one workgroup can rank

// (order-preserving 16-bit image of the fp16 value) << 16 | (0xFFFF - index): unique, never 0 for index < kMaxTried.
__device__ inline uint32_t key32(uint16_t bits, int idx) { return (ord16(bits) << 16) | (uint32_t)(0xFFFF - idx); }
static_assert(kMaxTried <= 0x10000, "the index must fit the low half of a 32-bit key");

// How many of s_keys[0, n) are larger: the place of a key among them.  s_keys must be padded with zeros to a multiple of 4 and be
// visible (barrier) on entry.
__device__ inline int keys_above(const uint32_t* s_keys, int n, uint32_t mine) {
    const int n4 = (n + 3) & ~3;
    int above = 0;
#pragma unroll 8
    for (int j = 0; j < n4; j += 4) {  // every lane reads the same 16 bytes: an LDS broadcast
        const uint4 o = *reinterpret_cast<const uint4*>(s_keys + j);
        above += (o.x > mine) + (o.y > mine) + (o.z > mine) + (o.w > mine);
    }
    return above;
}

// Vocabulary id of a candidate.  A position of -1 stands for no candidate (a row that a one-launch FR-Spec head left unfinished, a list that
// was padded): it reads the table's first entry rather than what lies in front of the table.  Without a table the position itself.
__device__ inline const int32_t* id_address(const int32_t* remap, const int32_t* pos) { return remap ? remap + max(*pos, 0) : pos; }

struct DraftState {
    uint16_t* tried_val;    // [total] fp16 bits
    int32_t* tried_pos;     // [total]
    int32_t* tried_parent;  // [k * (num_iter - 1)]
    uint64_t* mask;         // [k] eagle_mask_2d
    uint16_t* cum;          // [k] running log-prob of the k live nodes
};

__host__ __device__ inline size_t draft_state_layout(int k, int num_iter, size_t* off_pos, size_t* off_parent, size_t* off_mask,
                                                     size_t* off_cum) {
    const size_t total = (size_t)k + (size_t)(num_iter - 1) * k * k;
    size_t o = (total * 2 + 15) / 16 * 16;
    *off_pos = o;
    o += total * 4;
    *off_parent = o;
    o += (size_t)k * (num_iter > 1 ? num_iter - 1 : 1) * 4;
    o = (o + 15) / 16 * 16;
    *off_mask = o;
    o += (size_t)k * 8;
    *off_cum = o;
    o += (size_t)k * 2;
    return (o + 255) / 256 * 256;
}

inline DraftState draft_state(void* state, int k, int num_iter) {
    size_t op, opar, om, oc;
    draft_state_layout(k, num_iter, &op, &opar, &om, &oc);
    char* b = (char*)state;
    return DraftState{(uint16_t*)b, (int32_t*)(b + op), (int32_t*)(b + opar), (uint64_t*)(b + om), (uint16_t*)(b + oc)};
}

__global__ void draft_begin_kernel(DraftState s, int k, const uint16_t* val, const int32_t* pos, const int32_t* remap,
                                   int32_t* next_ids, uint64_t* mask_out) {
    const int i = threadIdx.x;
    if (i >= k) return;
    s.tried_val[i] = val[i];
    s.tried_pos[i] = pos[i];
    s.cum[i] = val[i];
    s.mask[i] = 1ull << i;
    if (mask_out) mask_out[i] = 1ull << i;
    next_ids[i] = *id_address(remap, pos + i);
}

// A chain of round trips (arguments, candidates, vocabulary ids) around a short count, so an entry stays with its thread: what a chosen one
// needs -- its id is looked up for every candidate, under the count -- is in registers when its place is known.  (Against looking the chosen ones' ids up behind the
// count, replayed graphs, three runs of either build in turn within 0.2 us: the launch 3.06 -> 2.69 us with 10 x 10 candidates, 2.41 -> 2.00 with 4 x 4,
// 38.4 -> 37.9 with 32 x 32; a draft of 6 rounds of 10 361.3 -> 358.4, one of 4 rounds of 4 104.5 -> 102.6.  A first pass on new inputs shows no gain.)
// kEntries: entries of a thread, at most.  The loads have no branches around them (an entry past the end repeats the last one): behind a
// branch the compiler would wait for the ids in front of the count.
template <int kEntries>
__global__ __launch_bounds__(kTopkThreads) void draft_extend_kernel(DraftState s, int k, int d, uint16_t* val, const int32_t* pos,
                                                                    const int32_t* remap, int32_t* next_ids, int32_t* parent_rows,
                                                                    uint64_t* mask_out, int is_bf16) {
    __shared__ __attribute__((aligned(16))) uint32_t s_keys[kEntries * kTopkThreads];
    const int tid = threadIdx.x;
    const int kk = k * k;
    const int base = k + (d - 1) * kk;
    uint32_t key[kEntries];
    int32_t id[kEntries];
    int parent[kEntries];
    uint64_t mask[kEntries];
    uint16_t cum[kEntries];
#pragma unroll
    for (int e = 0; e < kEntries; ++e) {
        const int x = tid + e * kTopkThreads, at = min(x, kk - 1);
        parent[e] = (unsigned)at / (unsigned)k;
        const uint16_t v = val[at], c = s.cum[parent[e]];
        const int32_t p = pos[at];
        mask[e] = s.mask[parent[e]];
        id[e] = *id_address(remap, pos + at);
        // the running log-prob of the parent is added in the element type: 16 bits += 16 bits, rounded to 16 bits
        const uint16_t sum_f16 = Elem<f16>::to_bits(Elem<f16>::from_bits(v) + Elem<f16>::from_bits(c));
        const uint16_t sum_bf16 = Elem<bf16>::to_bits(Elem<bf16>::from_bits(v) + Elem<bf16>::from_bits(c));
        cum[e] = is_bf16 ? sum_bf16 : sum_f16;
        key[e] = x < kk ? key32(cum[e], x) : 0;
        s_keys[x] = key[e];
        if (x < kk) {
            val[x] = cum[e];
            s.tried_val[base + x] = cum[e];
            s.tried_pos[base + x] = p;
        }
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kEntries; ++e) {
        const int x = tid + e * kTopkThreads;
        if (x >= kk) break;
        const int place = keys_above(s_keys, kk, key[e]);
        if (place >= k) continue;
        const uint64_t m = mask[e] | (1ull << (k * d + place));
        s.tried_parent[(d - 1) * k + place] = x + base;
        s.mask[place] = m;
        if (mask_out) mask_out[place] = m;
        if (parent_rows) parent_rows[place] = parent[e];
        next_ids[place] = id[e];
        s.cum[place] = cum[e];
    }
}

// One thread per history entry up to 1024 entries (two beyond).  A count over all entries is two vector instructions per entry and wave on
// one CU, 4 us of 7.2 with 510 entries, so entries that cannot be among the T - 1 largest are left out first: the (T - 1)-th largest of the 64
// maxima over every 64th entry has T - 1 entries at or above it.  us a launch in replayed graphs, all entries counted /
// those kept, with their vocabulary ids looked up under the count: 7.4 / 5.0 with 510 entries and a tree of 60, 7.0 / 4.5 with 456 and 32, 15.3 / 6.6 with
// 784 and 60, 21.4 / 8.7 with 1056 and 64, 3.9 / 4.0 with 136 and 30.  A draft of 6 rounds of 10 360.6 -> 357.8.
constexpr int kFinishThreads = 1024;
constexpr int kFinishCountsAll = 192;  // entries

template <bool BOUND>
__global__ __launch_bounds__(kFinishThreads) void draft_finish_kernel(DraftState s, int k, int num_iter, int T, const int32_t* cache_length,
                                                                      const int32_t* remap, bool set_root, int32_t root_id, int32_t* ids_out, int32_t* tree_pos,
                                                                      uint64_t* tree_mask, int32_t* tree_parent) {
    __shared__ __attribute__((aligned(16))) uint32_t s_keys[kMaxTried];
    __shared__ int32_t s_pos[kMaxTried];     // FR-Spec index of every history entry
    __shared__ int32_t s_reverse[kMaxTried]; // history index -> tree node (0: not selected, stands for the root)
    __shared__ int32_t s_hpar[64];           // history parent of the entries chosen in rounds >= 1 (k * num_iter <= 64 of them)
    __shared__ int32_t s_sel[kMaxTree];      // history index of tree node i + 1
    __shared__ int32_t s_par[kMaxTree];
    __shared__ __attribute__((aligned(16))) uint32_t s_kept[BOUND ? kMaxTried : 4];
    __shared__ int s_kept_count;
    const int tid = threadIdx.x;
    const int kk = k * k;
    const int total = k + (num_iter - 1) * kk;
    const int W = (T + 63) / 64;
    // everything the later phases need comes into LDS in one round trip to memory
    for (int x = tid; x < ((total + 3) & ~3); x += kFinishThreads) {
        const bool in = x < total;
        s_keys[x] = in ? key32(s.tried_val[x], x) : 0;
        if constexpr (BOUND) s_kept[x] = 0;
        if (in) {
            s_pos[x] = s.tried_pos[x];
            s_reverse[x] = 0;  // a parent that was not selected maps to the root
        }
    }
    if (tid < k * (num_iter - 1)) s_hpar[tid] = s.tried_parent[tid];
    const int P = cache_length[0];
    if (BOUND && tid == 0) s_kept_count = 0;
    __syncthreads();
    const uint32_t* keys = s_keys;
    int count = total;
    if constexpr (BOUND) {
        const int lane = tid & 63;
        if (tid - lane < total) {
            uint32_t top = 0;
            for (int x = lane; x < total; x += 64) top = max(top, s_keys[x]);
            uint32_t bound = 0;  // of the values (a key's upper half)
            for (int b = 15; b >= 0; --b) {
                const uint32_t higher = bound | (1u << b);
                if (__popcll(__ballot((top >> 16) >= higher)) >= T - 1) bound = higher;
            }
            for (int x = tid; x - lane < total; x += kFinishThreads) {
                const uint32_t key = x < total ? s_keys[x] : 0;
                const bool kept = x < total && (key >> 16) >= bound;
                const uint64_t who = __ballot(kept);
                int first = 0;
                if (lane == 0) first = atomicAdd(&s_kept_count, __popcll(who));
                first = __builtin_amdgcn_readfirstlane(first);
                if (kept) s_kept[first + __popcll(who & ((1ull << lane) - 1))] = key;
            }
        }
        __syncthreads();
        keys = s_kept;
        count = s_kept_count;
    }
    for (int j = tid; j < count; j += kFinishThreads) {
        const uint32_t key = keys[j];
        const int x = BOUND ? 0xFFFF - (int)(key & 0xFFFF) : j;
        auto id_of = [&]() {
            const int32_t fr = s_pos[x];
            return remap ? remap[max(fr, 0)] : fr;
        };
        int32_t id = 0;
        if constexpr (BOUND) id = id_of();
        const int place = keys_above(keys, count, key);
        if (place < T - 1) {
            s_sel[place] = x;
            s_reverse[x] = place + 1;
            ids_out[place + 1] = BOUND ? id : id_of();
        }
    }
    __syncthreads();
    // build_dynamic_tree (src/model/eagle.cuh:188-214), every node on its own thread: its parent is the
    // tree node of its history parent; its mask row is its own bit plus those of its ancestors.
    // Parents come before children (cumulative log-probs fall along a path, ties go to the older
    // entry), which the sequential form of the reference relies on as well.
    if (tid < T) {
        int parent = 0;
        if (tid == 0) {
            tree_pos[0] = P;
            if (set_root) ids_out[0] = root_id;
        } else {
            int p = s_sel[tid - 1];
            tree_pos[tid] = P + (p < k ? 1 : (p - k) / kk + 2);
            if (p >= k) {
                p -= k;
                p = p < kk ? p / k : s_hpar[(p - kk) / k];
                parent = s_reverse[p];
            }
        }
        s_par[tid] = parent;
        tree_parent[tid] = parent;
    }
    __syncthreads();
    if (tid < T) {
        uint64_t m0 = 1, m1 = 0;  // the root is everybody's ancestor
        int node = tid;
        for (int hop = 0; hop < T && node != 0; ++hop) {
            if (node < 64) m0 |= 1ull << node;
            else m1 |= 1ull << (node - 64);
            const int up = s_par[node];
            node = up < node ? up : 0;  // never walks downwards, so it ends
        }
        tree_mask[(size_t)tid * W] = m0;
        if (W > 1) tree_mask[(size_t)tid * W + 1] = m1;
    }
}

int check_shape(const char* what, int k, int num_iter) {
    CPMCU_CHECK_ARG(k >= 1 && k <= kMaxK, "%s: k=%d outside [1, %d]", what, k, kMaxK);
    CPMCU_CHECK_ARG(num_iter >= 1 && k * num_iter <= 64, "%s: k * num_iter = %d does not fit the 64-bit draft mask", what, k * num_iter);
    CPMCU_CHECK_ARG((size_t)k + (size_t)(num_iter - 1) * k * k <= (size_t)kMaxTried, "%s: history of %d entries exceeds %d", what,
                    k + (num_iter - 1) * k * k, kMaxTried);
    return CPMCU_OK;
}

}  // namespace
}  // namespace cpmcu

using namespace cpmcu;

extern "C" size_t cpmcu_draft_tree_state_bytes(int k, int num_iter) {
    if (k < 1 || num_iter < 1) return 0;
    size_t a, b, c, d;
    return draft_state_layout(k, num_iter, &a, &b, &c, &d);
}

extern "C" int cpmcu_draft_tree_begin(void* state, int k, int num_iter, const void* topk_val, const int32_t* topk_pos,
                                      const int32_t* token_id_remap, int32_t* next_ids, uint64_t* draft_mask, void* stream) {
    CPMCU_CHECK_ARG(state && topk_val && topk_pos && next_ids, "draft_tree_begin: null pointer argument");
    if (int rc = check_shape("draft_tree_begin", k, num_iter)) return rc;
    hipLaunchKernelGGL(draft_begin_kernel, dim3(1), dim3(64), 0, resolve_stream(stream), draft_state(state, k, num_iter), k,
                       (const uint16_t*)topk_val, topk_pos, token_id_remap, next_ids, draft_mask);
    CPMCU_LAUNCH_CHECK();
    return CPMCU_OK;
}

extern "C" int cpmcu_draft_tree_extend(void* state, int k, int num_iter, int d, void* topk_val, const int32_t* topk_pos,
                                       const int32_t* token_id_remap, int32_t* next_ids, int32_t* parent_rows,
                                       uint64_t* draft_mask, void* stream) {
    CPMCU_CHECK_ARG(state && topk_val && topk_pos && next_ids, "draft_tree_extend: null pointer argument");
    if (int rc = check_shape("draft_tree_extend", k, num_iter)) return rc;
    CPMCU_CHECK_ARG(d >= 1 && d < num_iter, "draft_tree_extend: iteration d=%d outside [1, %d)", d, num_iter);
    const auto kernel = k * k <= kTopkThreads ? draft_extend_kernel<1> : draft_extend_kernel<kMaxK * kMaxK / kTopkThreads>;
    hipLaunchKernelGGL(kernel, dim3(1), dim3(kTopkThreads), 0, resolve_stream(stream), draft_state(state, k, num_iter), k, d,
                       (uint16_t*)topk_val, topk_pos, token_id_remap, next_ids, parent_rows, draft_mask, options().dtype == 1 ? 1 : 0);
    CPMCU_LAUNCH_CHECK();
    return CPMCU_OK;
}

static int draft_tree_finish(void* state, int k, int num_iter, int tree_size, const int32_t* cache_length, const int32_t* token_id_remap,
                             const int32_t* root_id, int32_t* tree_draft_ids, int32_t* tree_position_ids, uint64_t* tree_attn_mask,
                             int32_t* tree_parent, void* stream) {
    CPMCU_CHECK_ARG(state && cache_length && tree_draft_ids && tree_position_ids && tree_attn_mask && tree_parent,
                    "draft_tree_finish: null pointer argument");
    if (int rc = check_shape("draft_tree_finish", k, num_iter)) return rc;
    const int total = k + (num_iter - 1) * k * k;
    CPMCU_CHECK_ARG(tree_size >= 2 && tree_size <= kMaxTree && tree_size - 1 <= total,
                    "draft_tree_finish: tree_size=%d outside [2, min(%d, history %d + 1)]", tree_size, kMaxTree, total);
    const auto kernel = total > kFinishCountsAll && tree_size - 1 <= 64 ? draft_finish_kernel<true> : draft_finish_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3(1), dim3(kFinishThreads), 0, resolve_stream(stream), draft_state(state, k, num_iter), k,
                       num_iter, tree_size, cache_length, token_id_remap, root_id != nullptr, root_id ? *root_id : 0, tree_draft_ids,
                       tree_position_ids, tree_attn_mask, tree_parent);
    CPMCU_LAUNCH_CHECK();
    return CPMCU_OK;
}
extern "C" int cpmcu_draft_tree_finish(void* state, int k, int num_iter, int tree_size, const int32_t* cache_length,
                                       const int32_t* token_id_remap, int32_t* tree_draft_ids, int32_t* tree_position_ids,
                                       uint64_t* tree_attn_mask, int32_t* tree_parent, void* stream) {
    return draft_tree_finish(state, k, num_iter, tree_size, cache_length, token_id_remap, nullptr, tree_draft_ids, tree_position_ids,
                             tree_attn_mask, tree_parent, stream);
}
extern "C" int cpmcu_draft_tree_finish_root(void* state, int k, int num_iter, int tree_size, const int32_t* cache_length,
                                            const int32_t* token_id_remap, int32_t root_id, int32_t* tree_draft_ids, int32_t* tree_position_ids,
                                            uint64_t* tree_attn_mask, int32_t* tree_parent, void* stream) {
    return draft_tree_finish(state, k, num_iter, tree_size, cache_length, token_id_remap, &root_id, tree_draft_ids, tree_position_ids,
                             tree_attn_mask, tree_parent, stream);
}
