// The direct shape of tree attention: for launches whose time is their chain of round trips, not their bytes or matrix work
// (plain decode, the drafter's rounds, small trees, short contexts).  Included by tree_attention.hip inside its namespace.
//
// A workgroup owns 16 packed query rows of one KV head and walks half pages (blocks of 128 keys), dealt out round-robin over the
// splits.  Its eight waves share the scores out by keys (16 each) and the second product by output dims (16 each), so a block is
// 4 KB of K and 4 KB of V^T per wave, in LDS of the wave's own:
//   * between a wave's keys and its dims only the row maxima and the probabilities (4 KB) change hands; the outputs never have to be
//     summed over the waves (64 KB of LDS writes and reads: 1 us);
//   * which pages a workgroup reads follows from its number alone: the page ids are requested beside the length instead of behind
//     it, and a bound above the length costs no imbalance;
//   * the appended rows are a block of their own, read from k_new / v_new (split 0 takes it first, while its pages are on their
//     way), so no tile has to be patched; workgroups of their own write them to the pool meanwhile;
//   * the partials of few splits are merged by the last workgroup of a unit to arrive: nobody polls or waits, so the launch may be larger
//     than the chip.  Those of many splits are merged in shares, by words that say themselves whether they are there: a kernel of its own
//     (tree_attn_direct_shares_kernel), since code that a launch jumps over is fetched all the same, 0.1-0.2 us.
// The products are the transposed ones of the other shapes (S^T = K.Q^T, O^T = V^T.P^T), on v_mfma_f32_16x16x32: lane (c, h) =
// (lane & 15, lane >> 4) of a score block holds query row c and four keys.  Which key sits in which row of the K operand is free;
// it is chosen so that the eight probabilities of a lane of the B operand belong to eight neighbouring slots of a V^T row.
// K and V go through LDS although no two waves share them: an operand fetched straight into registers has every lane on a row of
// its own, 64 address cycles for 1 KB (3.3 us per 256 keys, measured; 1 us this way).
// Every instruction of the eight waves is 8 cycles of the CU, so the paths that most workgroups take are kept short: row sums come
// out of an MFMA with ones, mask words are looked at where a block reaches the tree, merge weights are computed once per row.

constexpr int kDirectRows = 16;        // packed query rows per workgroup
constexpr int kBlockKeys = kPage / 2;  // keys per iteration
constexpr int kDirectItems = kDirectRows * 4;  // pieces of a unit's output that are merged by themselves: 32 dims of a row
constexpr int kDirectLastMerges = 15;          // up to here the last arrival merges all splits
constexpr float kSumScale = 1.f / kMaxSplits;
static_assert((kMaxSplits & (kMaxSplits - 1)) == 0, "kSumScale");
// A partial that is merged in shares changes hands through memory of the library: every 8-byte word carries two outputs (or half of a
// row's statistics) and the generation of its slot, so that a reader that sees the generation has the payload, and nothing is acknowledged
// or counted in front of the reads (acknowledgement, arrival, poll and read were four round trips, store and poll are two).  A slot's
// generation is read when a launch begins and advanced by the last arrival of its unit, so no older word passes for a fresh one (but for one
// of exactly 2^32 launches ago).  us per layer in replayed graphs, partials counted in / words: one query with the rotary embedding on 2 KV
// heads 7.4 / 7.1 at 4096 keys, 11.4 / 10.4 at 16384, 19.5 / 17.9 at 60001, 30.0 / 28.6 at 131072; on 8 heads 10.0 / 9.6 at 4096, 21.0 / 19.6 at
// 20000; two queries 9.0 / 8.6 at 9000; four 8.5 / 8.5 at 4096, on 4 heads 11.2 / 11.45 at 8192.  A plain copy of the partials beside the words: 0.1-0.4 more.
constexpr int kDirectSlots = 256;                           // workgroups of such a launch
constexpr int kSlotQuads = kDirectRows * 32 + kDirectRows;  // of 16 bytes: four dims of a row, then a row's maximum and sum
constexpr int kSlotBytes = kSlotQuads * 16;
struct DirectSlots {
    uint32_t generation[kDirectSlots];
    u32x4 words[kDirectSlots][kSlotQuads];
};
static_assert(kThreads == kDirectRows * 32, "the merge: 32 threads per row");
// The keys of a group of 32 make two operand blocks.  Row m of the K operand of block b of a group is its key direct_key_of_row(m) + 8 b;
// probability j of lane (., h) of the group's B operand belongs to key 16 (h / 2) + 4 (h % 2) + j % 4 + 8 (j / 4), whose slots in
// a V^T row are 8 h + j.
__device__ inline int direct_key_of_row(int m) { return 16 * (m >> 3) + 4 * ((m >> 2) & 1) + (m & 3); }
// Swizzled 16-byte pieces of a 256-byte row: the 16 lanes of an operand read touch 16 different columns.
__device__ inline int direct_off(int row, int piece) { return row * 256 + ((piece ^ (row & 15)) << 4); }
// Exchanges between lanes that take no LDS: max (or sum) with the lane 16 or 32 away, the value of the lane 8 or so away.
template <bool MAX>
__device__ inline float max_or_sum(float a, float b) {
    return MAX ? fmaxf(a, b) : a + b;
}
template <int CTRL>
__device__ inline float dpp(float v) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_mov_dpp((int)__float_as_uint(v), CTRL, 0xf, 0xf, true));
}
__device__ inline float lanes_8(float x) { return dpp<0x128>(x); }  // rotated by 8 in 16
template <bool MAX>
__device__ inline float with_lanes_16(float x) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return max_or_sum<MAX>(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
template <bool MAX>
__device__ inline float with_lanes_32(float x) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return max_or_sum<MAX>(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
// x over the four lanes of a column (lanes c, c + 16, c + 32, c + 48)
__device__ inline float column_max(float x) { return with_lanes_32<true>(with_lanes_16<true>(x)); }
// over the 32 lanes of a half wave
template <bool MAX>
__device__ inline float half_wave(float x) {
    x = max_or_sum<MAX>(x, dpp<0xB1>(x));   // lane ^ 1
    x = max_or_sum<MAX>(x, dpp<0x4E>(x));   // lane ^ 2
    x = max_or_sum<MAX>(x, dpp<0x141>(x));  // mirrored in 8
    x = max_or_sum<MAX>(x, dpp<0x140>(x));  // mirrored in 16
    return with_lanes_16<MAX>(x);
}
// over the 16 lanes of the same number modulo 4
template <bool MAX>
__device__ inline float over_splits(float x) {
    x = max_or_sum<MAX>(x, dpp<0x124>(x));  // rotated by 4 in 16
    x = max_or_sum<MAX>(x, lanes_8(x));
    return with_lanes_32<MAX>(with_lanes_16<MAX>(x));
}

template <bool SHARES, typename E>
__device__ __forceinline__ void tree_attn_direct_body(const AttnParams& p) {
    typedef typename Elem<E>::x8 X8;
    typedef typename Elem<E>::x4 X4;
    constexpr int kGroups = kBlockKeys / 32;
    constexpr int kWaveBytes = kDirectRows * kHeadDim * 2;  // a wave's 16 keys, and its 16 dims of 128 keys
    constexpr int kPartBytes = kDirectRows * kHeadDim * 2;  // a split's partial
    __shared__ __attribute__((aligned(1024))) union {
        struct {
            char k[kWaves][kWaveBytes];
            char v[kWaves][kWaveBytes];
        } block;
        AppendStage append[kThreads / kAppendThreads];
        float weight[kMaxSplits][kDirectRows];  // of the merge by the last arrival
    } s;
    __shared__ __attribute__((aligned(1024))) char s_q[kDirectRows * kHeadDim * 2];
    __shared__ X8 s_p[kGroups][64];                   // the probabilities of an iteration
    __shared__ f32x4 s_max[kDirectRows][kWaves / 4];  // each wave's row maxima
    __shared__ Arrival s_arrival;
    __shared__ int s_late[2];  // the merge in shares: a wave's wait for partials ran out
    asm volatile("" ::"s"(p.q), "s"(p.k_pool), "s"(p.v_pool), "s"(p.block_table), "s"(p.kv_len), "s"(p.k_new), "s"(p.v_new), "s"(p.rope),
                 "s"(p.mask), "s"(p.mask_words), "s"(p.mask_k_range), "s"(p.T), "s"(p.Hq), "s"(p.Hkv), "s"(p.group), "s"(p.group_inv),
                 "s"(p.hkv_inv), "s"(p.tile_groups), "s"(p.tile_groups_inv), "s"(p.num_splits), "s"(p.num_mtiles), "s"(p.table_pages), "s"(p.window_blocks), "s"(p.max_kv_len));
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int append = p.k_new != nullptr ? 1 : 0;
    const int wg = SHARES ? (int)blockIdx.x - p.append_groups : (int)blockIdx.x;
    const int append_wg = SHARES ? blockIdx.x : wg - p.tile_groups * p.num_mtiles;

    int S;
    auto clamp_length = [&]() {
        const int lo = max(p.T, p.mask_k_range);
        if (S > p.max_kv_len || S < lo) {
            if (blockIdx.x == 0 && tid == 0) g_attn_report.bad_length = S == 0 ? -1 : S;
            S = min(max(S, lo), p.max_kv_len);
        }
    };
    if (SHARES ? wg < 0 : append_wg >= 0) {  // the rows on their way into the pool
        const int runs = (p.T + kAppendRows - 1) / kAppendRows;
        constexpr int kHalves = kThreads / kAppendThreads;
        const int y = append_wg * kHalves + tid / kAppendThreads;
        if (y / kHalves * kHalves < runs * p.Hkv) {
            const Quotient y_of = divide(y, p.Hkv, p.hkv_inv);
            const int gg = y_of.r, run = y_of.q;
            kv_append_run<E, true>(p.k_pool_w, p.v_pool_w, p.block_table, p.k_new, p.v_new, p.rope, p.T, p.Hkv, gg, run * kAppendRows,
                             tid % kAppendThreads, s.append[tid / kAppendThreads], [&]() {
                                 S = scalar_load(p.kv_len);
                                 clamp_length();
                                 return S;
                             });
        }
        return;
    }
    const Quotient wg_of = divide(wg, p.tile_groups, p.tile_groups_inv);
    const int mt = wg_of.q, sh = wg_of.r;
    if (sh >= p.num_splits * p.Hkv) return;
    const Quotient sh_of = divide(sh, p.Hkv, p.hkv_inv);
    const int g = sh_of.r, split = sh_of.q;
    const int unit = g * p.num_mtiles + mt;
    const int c = lane & 15, h = lane >> 4;
    // lane i: the generation that the words of splits i and i + 64 carry in this launch
    uint32_t fresh[2] = {0, 0};
    if constexpr (SHARES) {
        const uint32_t* gen = p.slots->generation + unit * p.num_splits;
        fresh[0] = __hip_atomic_load(gen + min(lane, p.num_splits - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
        if (tid < 2) s_late[tid] = 0;
        if (p.num_splits > 64) fresh[1] = __hip_atomic_load(gen + min(lane + 64, p.num_splits - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
    }

    // This workgroup's blocks: base + block_of(i), i = 0, 1, ...  The appended rows come in front of the stream, as its block 0.
    const bool has_new = append && split == 0;
    const int block0 = (has_new ? p.num_splits : split) - append;
    auto block_of = [&](int i) { return block0 + i * p.num_splits; };
    int base = 0, first_key = 0;
    if (p.window_blocks > 0) {  // the window's first key depends on the length
        S = scalar_load(p.kv_len);
        clamp_length();
        first_key = max((S - p.T + 127) / 128 - p.window_blocks, 0) * 128;
        base = first_key / kBlockKeys;
    }
    auto table_entry = [&](int block) { return p.block_table + min((base + block) / (kPage / kBlockKeys), p.table_pages - 1); };
    // lane i holds the page of the workgroup's i-th block (of the current 64); the first one comes with the length
    const bool may_iterate = block_of(1) * kBlockKeys < p.max_kv_len;
    auto pages_from = [&](int i0) { return *table_entry(block_of(i0 + lane)); };
    int pages = 0;
    if (may_iterate) pages = pages_from(0);

    auto node_of = [&](int R) { return divide(R, p.group, p.group_inv).q; };
    // where row R of q and out begins
    auto row_at = [&](int R) {
        const Quotient row = divide(R, p.group, p.group_inv);
        return ((size_t)row.q * p.Hq + g * p.group + row.r) * kHeadDim;
    };
    const int last_row = p.group * p.T - 1;
    const int my_node = node_of(min(mt * kDirectRows + c, last_row));
    // What this lane's row sees of the tree: needed where keys of the mask's range are met.
    uint64_t mw0 = ~0ull, mw1 = ~0ull;
    if (p.mask != nullptr && (has_new || !append || p.mask_k_range > p.T)) {
        mw0 = p.mask[my_node * p.mask_words];
        mw1 = p.mask_words > 1 ? p.mask[my_node * p.mask_words + 1] : 0ull;
    }
    // The query rows and the appended K rows reach LDS through registers, rotated on the way: a thread has the pieces at d and
    // d + 64 of a row.
    const int t_row = tid >> 3, t_piece = tid & 7;
    auto fetch_row = [&](X8 (&x)[2], f32x4 (&cs)[4], const f16* src, int node) {
        x[0] = *reinterpret_cast<const X8*>(src + t_piece * 8);
        x[1] = *reinterpret_cast<const X8*>(src + t_piece * 8 + 64);
        if (p.rope != nullptr) {
            const f32x4* t = reinterpret_cast<const f32x4*>(p.rope + (size_t)node * (kHeadDim / 2) + t_piece * 8);
#pragma unroll
            for (int j = 0; j < 4; ++j) cs[j] = t[j];
        }
    };
    auto place_row = [&](X8 (&x)[2], const f32x4 (&cs)[4], char* rows, int row) {
        if (p.rope != nullptr) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                E a = x[0][j], b = x[1][j];
                rotate_pair(a, b, j & 1 ? make_float2(cs[j >> 1][2], cs[j >> 1][3]) : make_float2(cs[j >> 1][0], cs[j >> 1][1]));
                x[0][j] = a;
                x[1][j] = b;
            }
        }
        *reinterpret_cast<X8*>(rows + direct_off(row, t_piece)) = x[0];
        *reinterpret_cast<X8*>(rows + direct_off(row, t_piece + 8)) = x[1];
    };
    // (waits for the rows where it stands: behind the K/V requests the compiler would wait for those as well)
    auto arrived = [&](X8 (&x)[2], f32x4 (&cs)[4]) {
        asm volatile("" : "+v"(x[0]), "+v"(x[1]));
        if (p.rope != nullptr) asm volatile("" : "+v"(cs[0]), "+v"(cs[1]), "+v"(cs[2]), "+v"(cs[3]));
    };
    constexpr int kQThreads = kDirectRows * 8;
    X8 rq[2];
    f32x4 rq_cs[4];
    if (tid < kQThreads) {
        const int R = min(mt * kDirectRows + t_row, last_row);
        const int node = node_of(R);
        fetch_row(rq, rq_cs, p.q + row_at(R), node);
    }
    // 32 appended rows at a time, by the upper half of the threads: K row t is row m of block b, in the K area of wave b ...
    constexpr int kNewRows = 32;
    const int n_row = t_row - kThreads / 16;
    X8 rk[2];
    f32x4 rk_cs[4];
    auto fetch_new = [&](int t0) {
        const int t = min(t0 + n_row, p.T - 1);
        if (wave >= kWaves / 2) fetch_row(rk, rk_cs, p.k_new + ((size_t)t * p.Hkv + g) * kHeadDim, t);
    };
    auto place_new = [&]() {
        if (wave >= kWaves / 2) {
            const int b = (n_row >> 3) & 1, m = ((n_row >> 1) & 8) | (n_row & 7);
            place_row(rk, rk_cs, s.block.k[b], m);
        }
    };
    // ... and V rows stay as they are, in the K areas of the two waves behind.
    constexpr int kNewWaves = 2;
    char* const v_new_rows = s.block.k[kNewWaves];
    auto load_new_v = [&](int t0) {
        const int t = min(t0 + wave * 4 + h, p.T - 1);
        load_to_lds16_v(p.v_new + ((size_t)t * p.Hkv + g) * kHeadDim + c * 8, v_new_rows + wave * 1024);
    };
    if (has_new) fetch_new(0);
    int first_page;
    if (p.window_blocks == 0) {
        scalar_load2(p.kv_len, table_entry(block0), S, first_page);
        clamp_length();
    } else {
        first_page = scalar_load(table_entry(block0));
    }
    const int P = S - p.T;
    const int Pm = S - p.mask_k_range;       // first key column governed by the mask bits
    const int kend = append ? P : S;         // keys of the stream that come from the pool
    const int nblocks = (kend + kBlockKeys - 1) / kBlockKeys - base;
    auto has = [&](int i) { return block_of(i) < nblocks; };

    // One wave-level request fills 1 KB of LDS in lane order; the swizzle is applied on the global side.  From here on the wave
    // counts its outstanding requests by hand, four for its keys and four for its dims of a block: everything the compiler
    // has requested so far (page ids, mask words, rows) is waited for first.
    asm volatile("" : "+v"(mw0), "+v"(mw1), "+v"(pages));
    if constexpr (SHARES) asm volatile("" : "+v"(fresh[0]), "+v"(fresh[1]));
    if (tid < kQThreads) arrived(rq, rq_cs);
    if (has_new && wave >= kWaves / 2) arrived(rk, rk_cs);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const int grp = wave >> 1, blk = wave & 1;  // this wave's keys: operand block blk of group grp
    auto page_at = [&](int i) { return i == 0 ? first_page : __builtin_amdgcn_readlane(pages, i & 63); };
    // request x: rows 4 x + h of the wave's 16; of K, keys direct_key_of_row(4 x) + h of its operand block
    const uint32_t k_off = (uint32_t)(h * kHeadDim * 2 + ((c ^ h) << 4)), v_off = (uint32_t)(h * kPage * 2 + ((c ^ h) << 4));
    auto load_k = [&](int i) {
        const int first = (base + block_of(i)) * kBlockKeys % kPage + grp * 32 + blk * 8;
        const f16* kb = p.k_pool + (((size_t)page_at(i) * p.Hkv + g) * kPage + first) * kHeadDim;
#pragma unroll
        for (int x = 0; x < 4; ++x) load_to_lds16(kb + direct_key_of_row(4 * x) * kHeadDim, k_off ^ (x << 6), s.block.k[wave] + x * 1024);
    };
    auto load_v = [&](int i) {
        const int first = (base + block_of(i)) * kBlockKeys % kPage;
        const f16* vb = p.v_pool + (((size_t)page_at(i) * p.Hkv + g) * kHeadDim + wave * 16) * kPage + first;
#pragma unroll
        for (int x = 0; x < 4; ++x) load_to_lds16(vb + x * 4 * kPage, v_off ^ (x << 6), s.block.v[wave] + x * 1024);
    };
    auto wait_but_half = [&]() { asm volatile("s_waitcnt vmcnt(4)" ::: "memory"); };  // all but the newest half of a block
    auto wait_all = [&]() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
    const bool late_keys = has_new && wave < 2 * kNewWaves;  // the area holds appended rows first
    if (has_new) load_new_v(0);
    if (has(0)) {
        if (!late_keys) load_k(0);
        load_v(0);
    }
    if (tid < kQThreads) place_row(rq, rq_cs, s_q, t_row);
    if (has_new) {
        place_new();
        // the V rows are the oldest of the requests
        if (!has(0)) wait_all();
        else if (late_keys) wait_but_half();
        else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    }
    __syncthreads();
    // Q as the B operand of S^T = K.Q^T: lane (c, h) of ks holds row c, dims 32 ks + 8 h + [0, 8)
    X8 q[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) q[ks] = *reinterpret_cast<const X8*>(s_q + direct_off(c, ks * 4 + h));

    f32x4 o = {0.f, 0.f, 0.f, 0.f};  // O[row c][d = 16 wave + 4 h + 0..3]
    f32x4 l = {0.f, 0.f, 0.f, 0.f};  // the row's sum, four times
    float M = -INFINITY;             // exponent reference: follows the row maximum lazily, as in the other shapes; one for all waves
    X8 ones;
#pragma unroll
    for (int j = 0; j < 8; ++j) ones[j] = (E)1.f;
    // bits 0..3: keys first .. + 3 (first: the distance from Pm) are seen by this lane's row, as far as the mask goes
    auto tree_bits = [&](int first) {
        // the causal bound: nothing above the query's own key
        const int own = p.mask_k_range - p.T + my_node;
        const uint64_t w0 = mw0 & (own >= 63 ? ~0ull : ((2ull << own) - 1ull));
        const uint64_t w1 = mw1 & (own >= 127 ? ~0ull : (own < 64 ? 0ull : ((2ull << (own - 64)) - 1ull)));
        // the mask words extend by ones below their first bit
        const uint64_t below = first <= -64 ? ~0ull : ((w0 << (-first & 63)) | ((1ull << (-first & 63)) - 1ull));
        const uint64_t inside = (w0 >> (first & 63)) | ((w1 << 1) << (63 - (first & 63)));
        return (uint32_t)(first < 0 ? below : first < 64 ? inside : first < 128 ? w1 >> (first & 63) : 0ull);
    };
    auto first_bits = [&](int n) { return n <= 0 ? 0u : n >= 4 ? 15u : (1u << n) - 1u; };

    // One iteration: this wave's keys (in LDS) against all rows, then all keys of the iteration for its 16 dims.
    //   seen(key): which of the four keys from `key` of the group on exist and are visible (only if masked); keys_free(): the K area has been read;
    //   dims_ready(): waits for V; v_of(group): the A operand of the second product.
    auto iterate = [&](auto groups_c, bool have_keys, bool masked, auto&& seen, auto&& keys_free, auto&& dims_ready,
                       auto&& v_of) __attribute__((always_inline)) {
        constexpr int groups = decltype(groups_c)::value;
        f32x4 x = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        if (have_keys) {
            x = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
                x = Elem<E>::mfma_16x16x32(*reinterpret_cast<const X8*>(s.block.k[wave] + direct_off(c, ks * 4 + h)), q[ks], x);
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] *= p.scale_log2;
            if (masked) {
                const uint32_t see = seen(direct_key_of_row(4 * h) + 8 * blk);
#pragma unroll
                for (int i = 0; i < 4; ++i) x[i] = (see >> i) & 1u ? x[i] : -INFINITY;
            }
        }
        keys_free();
        const float mx = column_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
        if (h == 0) reinterpret_cast<float*>(&s_max[c])[wave] = mx;
        __syncthreads();
        const f32x4 ma = s_max[c][0], mb = s_max[c][1];
        const float m_all = fmaxf(fmaxf(fmaxf(ma[0], ma[1]), fmaxf(ma[2], ma[3])), fmaxf(fmaxf(mb[0], mb[1]), fmaxf(mb[2], mb[3])));
        if (__any(m_all > M + kLazyLog2)) {  // (the same decision in every wave)
            const float m = fmaxf(m_all, M);
            const float a = m == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(M - m);
            M = m;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                o[e] *= a;
                l[e] *= a;
            }
        }
        if (groups == kGroups || wave < kNewWaves) {
            const float m = M == -INFINITY ? 0.f : M;
            X4 pr;
#pragma unroll
            for (int i = 0; i < 4; ++i) pr[i] = (E)__builtin_amdgcn_exp2f(x[i] - m);
            reinterpret_cast<X4*>(&s_p[grp][lane])[blk] = pr;
        }
        dims_ready();
        __syncthreads();
#pragma unroll
        for (int u = 0; u < groups; ++u) {
            const X8 pr = s_p[u][lane];
            o = Elem<E>::mfma_16x16x32(v_of(u), pr, o);
            l = Elem<E>::mfma_16x16x32(ones, pr, l);  // the denominator weighs exactly what the numerator sees
        }
    };

    if (has_new) {
        for (int t0 = 0; t0 < p.T; t0 += kNewRows) {
            if (t0 > 0) {  // (trees of more than 32 nodes)
                __syncthreads();
                fetch_new(t0);
                load_new_v(t0);
                place_new();
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __syncthreads();
            }
            iterate(std::integral_constant<int, 1>{}, wave < kNewWaves, true,
                    [&](int key) { return tree_bits(P - Pm + t0 + key) & first_bits(p.T - t0 - key); },
                    [&]() {}, [&]() {},
                    [&](int) {
                        X8 v;
#pragma unroll
                        for (int j = 0; j < 8; ++j)
                            v[j] = reinterpret_cast<const E*>(v_new_rows)[(direct_key_of_row(4 * h) + (j & 3) + 8 * (j >> 2)) * kHeadDim + wave * 16 + c];
                        return v;
                    });
        }
        __syncthreads();
        if (late_keys && has(0)) load_k(0);
    }
    // A block's keys are requested ahead of its dims (but for late ones), each as soon as its area has been read.
    constexpr auto kAll = std::integral_constant<int, kGroups>{};
    for (int i = 0; has(i); ++i) {
        if (((i + 1) & 63) == 0) {  // the next request is the first of the next 64
            pages = pages_from(i + 1);
            asm volatile("s_waitcnt vmcnt(0)" : "+v"(pages)::"memory");
        }
        const bool more = has(i + 1);
        if (i == 0 && late_keys) wait_all();
        else wait_but_half();
        const int c0 = (base + block_of(i)) * kBlockKeys;
        const bool edge = c0 + kBlockKeys > kend || c0 < first_key;
        iterate(kAll, true, edge || c0 + kBlockKeys > Pm,
                [&](int key) {
                    const int key0 = c0 + grp * 32 + key;
                    return tree_bits(key0 - Pm) & first_bits(kend - key0) & ~first_bits(first_key - key0);
                },
                [&]() {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    if (more) load_k(i + 1);
                },
                [&]() {
                    if (more) wait_but_half();
                    else wait_all();
                },
                [&](int u) {
                    X8 v = *reinterpret_cast<const X8*>(s.block.v[wave] + direct_off(c, u * 4 + h));
                    if (edge) {  // stale values past the end (or ahead of the window) must not reach the MFMA (0 * NaN)
                        const int k0 = c0 + u * 32 + direct_key_of_row(4 * h);
#pragma unroll
                        for (int j = 0; j < 8; ++j) {
                            const int key = k0 + (j & 3) + 8 * (j >> 2);
                            v[j] = key < kend && key >= first_key ? v[j] : (E)0.f;
                        }
                    }
                    return v;
                });
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (more) load_v(i + 1);
    }
    const bool whole = !SHARES && p.num_splits == 1;
    constexpr int kSc1 = 16;  // past the (per-XCD) L2
    const float L = l[0];
    X4 result;
    {
        const float inv = (L == 0.f || L != L) ? (whole ? 1.f : 0.f) : 1.f / L;
#pragma unroll
        for (int e = 0; e < 4; ++e) result[e] = (E)(o[e] * inv);
    }
    const int my_dim = wave * 16 + h * 4;
    if (whole) {
        const int R = mt * kDirectRows + c;
        if (R <= last_row) *reinterpret_cast<X4*>(p.out + row_at(R) + my_dim) = result;
        return;
    }
    uint32_t* const ctr = p.merge_ctr + kMergeUnitWords * unit;
    if constexpr (SHARES) {
        __shared__ f32x4 s_sums[2][kWaves][8];   // 32 dims
        __shared__ float2 s_sums_ml[2][kWaves];  // their (maximum, sum of the weights)
        __shared__ uint32_t s_abandoned[kDirectItems / 32];
        // The merge in shares, by words that say themselves whether they are there (DirectSlots).  An item is 32 dims of a row, 128 bytes of
        // each slot: a wave reads 16 splits' worth at once, and as many waves as the splits need work on an item, so that a share is
        // one round trip.
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(p.slots->words[unit * p.num_splits], 0, p.num_splits * kSlotBytes, 0x00027000);
        {
            const uint32_t mine = (uint32_t)__builtin_amdgcn_readlane((int)(split < 64 ? fresh[0] : fresh[1]), split & 63);
            const uint64_t bits = bits_as<uint64_t>(result);
            __builtin_amdgcn_raw_buffer_store_b128(u32x4{(uint32_t)bits, mine, (uint32_t)(bits >> 32), mine}, rsrc,
                                                   split * kSlotBytes + (c * 32 + (my_dim >> 2)) * 16, 0, kSc1);
            if (wave == 0 && h == 0)
                __builtin_amdgcn_raw_buffer_store_b128(u32x4{__float_as_uint(M), mine, __float_as_uint(L), mine}, rsrc,
                                                       split * kSlotBytes + (kDirectRows * 32 + c) * 16, 0, kSc1);
        }
        const int item_shift = (p.num_splits > 16) + (p.num_splits > 32) + (p.num_splits > 64);
        const int item_waves = 1 << item_shift, at_once = kWaves >> item_shift;
        const int items = min(kDirectRows, last_row + 1 - mt * kDirectRows) * 4;
        const int slot = wave >> item_shift, part = wave & (item_waves - 1);
        const int my_split = part * 16 + (lane >> 2);  // whose words this lane reads
        const uint32_t my_fresh = (uint32_t)__shfl((int)(part < 4 ? fresh[0] : fresh[1]), my_split & 63);
        int parity = 0;
        // False (in every wave): the wait for the words ran out.
        auto merge_share = [&](int share, uint32_t limit) {
            const unsigned long long t_begin = wall_clock64();
            for (int i0 = share * at_once; i0 < items; i0 += p.merge_shares * at_once) {
                const int item = min(i0 + slot, items - 1), row = item >> 2;
                const int at = my_split * kSlotBytes + item * 128 + (lane & 3) * 32, ml_at = my_split * kSlotBytes + (kDirectRows * 32 + row) * 16;
                u32x4 xa = {0, 0, 0, 0}, xb = xa, ml = xa;
                bool there = my_split >= p.num_splits;
                for (;;) {
                    if (!there) {  // (the lanes that still wait)
                        xa = __builtin_amdgcn_raw_buffer_load_b128(rsrc, at, 0, kSc1);
                        xb = __builtin_amdgcn_raw_buffer_load_b128(rsrc, at + 16, 0, kSc1);
                        ml = __builtin_amdgcn_raw_buffer_load_b128(rsrc, ml_at, 0, kSc1);
                        there = ((xa[1] ^ my_fresh) | (xa[3] ^ my_fresh) | (xb[1] ^ my_fresh) | (xb[3] ^ my_fresh) | (ml[1] ^ my_fresh) | (ml[3] ^ my_fresh)) == 0;
                    }
                    if (__all(there) || wall_clock64() - t_begin >= limit) break;
                    asm volatile("" ::: "memory");  // (loads anew)
                }
                if (!__all(there)) s_late[parity] = 1;
                // Sums over the wave's splits, relative to their own maximum and times kSumScale (exact): a weighted partial is at most its split's own
                // sum, so that all of them together stay finite where each of those was (bfloat16 V of 1e34 and 60000 keys).  Dividing each sum by its
                // weights' instead took 0.2 us a layer.
                const float m = my_split < p.num_splits ? __uint_as_float(ml[0]) : -INFINITY;
                const float top = over_splits<true>(m);
                const float weight = __uint_as_float(ml[2]) * kSumScale * __builtin_amdgcn_exp2f(m - (top == -INFINITY ? 0.f : top));
                const X8 x = bits_as<X8>(u32x4{xa[0], xa[2], xb[0], xb[2]});
                f32x4 lo, hi;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    lo[e] = over_splits<false>(weight * (float)x[e]);
                    hi[e] = over_splits<false>(weight * (float)x[e + 4]);
                }
                const float sum = over_splits<false>(weight);
                if (lane < 4) {
                    s_sums[parity][wave][lane * 2] = lo;
                    s_sums[parity][wave][lane * 2 + 1] = hi;
                    if (lane == 0) s_sums_ml[parity][wave] = make_float2(top, sum);
                }
                __syncthreads();
                if (s_late[parity]) return false;
                if (wave == 0) {
                    // lane (v, quad): four dims of what wave v has summed up; the waves of an item lie 8, 16 and 32 lanes apart
                    const int v = lane >> 3, quad = lane & 7;
                    const float2 v_ml = s_sums_ml[parity][v];
                    f32x4 acc = s_sums[parity][v][quad];
                    float all = v_ml.x;
                    if (item_waves >= 2) all = fmaxf(all, lanes_8(all));
                    if (item_waves >= 4) all = with_lanes_16<true>(all);
                    if (item_waves >= 8) all = with_lanes_32<true>(all);
                    const float scale = __builtin_amdgcn_exp2f(v_ml.x - (all == -INFINITY ? 0.f : all));
                    float den = v_ml.y * scale;
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[e] *= scale;
                    if (item_waves >= 2) {
                        den += lanes_8(den);
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[e] += lanes_8(acc[e]);
                    }
                    if (item_waves >= 4) {
                        den = with_lanes_16<false>(den);
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[e] = with_lanes_16<false>(acc[e]);
                    }
                    if (item_waves >= 8) {
                        den = with_lanes_32<false>(den);
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[e] = with_lanes_32<false>(acc[e]);
                    }
                    const float inv = (den == 0.f || den != den) ? 1.f : 1.f / den;
                    X4 y;
#pragma unroll
                    for (int e = 0; e < 4; ++e) y[e] = (E)(acc[e] * inv);
                    const int t_item = i0 + (v >> item_shift);
                    if (t_item < items && (v & (item_waves - 1)) == 0)
                        *reinterpret_cast<X4*>(p.out + row_at(mt * kDirectRows + (t_item >> 2)) + (t_item & 3) * 32 + quad * 4) = y;
                }
                parity ^= 1;  // (the other one was read ahead of the barrier)
            }
            return true;
        };
        // Everyone has arrived: the words are on their way, and are waited for (the limit has the launch end whatever happens).
        auto merge_what_comes = [&](int share) {
            if (!merge_share(share, 100000000u) && tid == 0) __hip_atomic_fetch_add(&g_attn_report.lost, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        // The arrival stands for nothing but this workgroup's having looked at the generations and sent its words off.
        // (its answer is looked at behind the merge: in front of it would be a round trip)
        __shared__ uint32_t s_before;
        uint32_t before = 0;
        if (tid == 0) before = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool merged = split >= p.merge_shares || merge_share(split, p.merge_wait_ticks);
        if (tid == 0) s_before = before;
        __syncthreads();
        const UnitWord word(ctr, p.num_splits, s_before);
        if (word.last()) {
            // (every workgroup of the unit has read the generations)
            if (wave == 0) {
                uint32_t* gen = p.slots->generation + unit * p.num_splits;
#pragma unroll
                for (int k = 0; k < 2; ++k)
                    if (lane + 64 * k < p.num_splits) __hip_atomic_store(gen + lane + 64 * k, fresh[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if (tid == 0) word.next_generation();
        }
        if (!merged) {
            if (tid == 0) {
                s_arrival.go = word.last() || word.abandon(split);
                s_late[0] = s_late[1] = 0;
            }
            __syncthreads();
            if (s_arrival.go) merge_what_comes(split);
        }
        if (word.last()) {
            if (tid < kDirectItems / 32) s_abandoned[tid] = word.collect_abandoned(tid);
            __syncthreads();
            for (int v = 0; v < kDirectItems / 32; ++v)
                for (uint32_t left = s_abandoned[v]; left != 0; left &= left - 1) merge_what_comes(v * 32 + __builtin_ctz(left));
        }
        return;
    }
    // Merged by the last arrival.  Partials, written through to memory:
    //   o_part [unit][split][16 rows][128],  ml_part [unit][split][16 rows] x (max * scale_log2, sum)
    char* const o_part = reinterpret_cast<char*>(p.o_part) + (size_t)unit * p.num_splits * kPartBytes;
    char* const ml_part = reinterpret_cast<char*>(p.ml_part) + (size_t)unit * p.num_splits * (kDirectRows * 8);
    store_dev64(o_part + split * kPartBytes + (c * kHeadDim + my_dim) * 2, bits_as<uint64_t>(result));
    if (wave == 0 && h == 0)
        store_dev64(ml_part + (split * kDirectRows + c) * 8, (uint64_t)__float_as_uint(M) | ((uint64_t)__float_as_uint(L) << 32));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) s_arrival = arrive_at_unit(p, ctr, p.num_splits, -1);
    __syncthreads();
    const auto o_rsrc = __builtin_amdgcn_make_buffer_rsrc(o_part, 0, p.num_splits * kPartBytes, 0x00027000);
    if (!s_arrival.last) return;

    // The merge: a thread has four dims of a row; the weights of a row's splits are worked out once, by 32 threads.
    // Everything is requested before any of it is used, in groups of four splits that a launch of few skips.  Loads past the last
    // split return zeros, and meet a weight of zero.
    constexpr int kInFlight = 36;
    static_assert(kMaxSplits % 4 == 0, "weights are filled up to a multiple of four");
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < p.num_splits; s0 += kInFlight) {
        X4 x[kInFlight];
#pragma unroll
        for (int u = 0; u < kInFlight; ++u) {
            if (u % 4 == 0 && s0 + u >= p.num_splits) break;
            x[u] = bits_as<X4>(__builtin_amdgcn_raw_buffer_load_b64(o_rsrc, tid * 8, (s0 + u) * kPartBytes, kSc1));
        }
        if (s0 == 0) {
            {
                const int r = tid >> 5;
                constexpr int kMost = kMaxSplits / 32;
                float m[kMost], w[kMost], top = -INFINITY, sum = 0.f;
#pragma unroll
                for (int k = 0; k < kMost; ++k) {
                    const int sp = (tid & 31) + 32 * k;
                    m[k] = -INFINITY;
                    w[k] = 0.f;
                    if (32 * k < p.num_splits && sp < p.num_splits) {
                        const uint64_t ml = load_dev64(ml_part + (sp * kDirectRows + r) * 8);
                        m[k] = __uint_as_float((uint32_t)ml);
                        w[k] = __uint_as_float((uint32_t)(ml >> 32));
                    }
                }
#pragma unroll
                for (int k = 0; k < kMost; ++k) top = fmaxf(top, m[k]);
                top = half_wave<true>(top);
                top = top == -INFINITY ? 0.f : top;
#pragma unroll
                for (int k = 0; k < kMost; ++k) {
                    w[k] *= __builtin_amdgcn_exp2f(m[k] - top);
                    sum += w[k];
                }
                sum = half_wave<false>(sum);
                const float inv = (sum == 0.f || sum != sum) ? 1.f : 1.f / sum;
#pragma unroll
                for (int k = 0; k < kMost; ++k)
                    if (32 * k < p.num_splits) s.weight[(tid & 31) + 32 * k][r] = w[k] * inv;
            }
            __syncthreads();
        }
#pragma unroll
        for (int u = 0; u < kInFlight; ++u) {
            if (u % 4 == 0 && s0 + u >= p.num_splits) break;
            const float w = s.weight[s0 + u][tid >> 5];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(w, (float)x[u][e], acc[e]);
        }
    }
    const int R = mt * kDirectRows + (tid >> 5);
    X4 x;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = (E)acc[e];
    if (R <= last_row) *reinterpret_cast<X4*>(p.out + row_at(R) + (tid & 31) * 4) = x;
}

// (two workgroups per CU)
__global__ __launch_bounds__(kThreads, 4) void tree_attn_direct_kernel(AttnParams p) { tree_attn_direct_body<false, f16>(p); }
__global__ __launch_bounds__(kThreads, 4) void tree_attn_direct_bf16_kernel(AttnParams p) { tree_attn_direct_body<false, bf16>(p); }
__global__ __launch_bounds__(kThreads, 4) void tree_attn_direct_shares_kernel(AttnParams p) { tree_attn_direct_body<true, f16>(p); }
__global__ __launch_bounds__(kThreads, 4) void tree_attn_direct_shares_bf16_kernel(AttnParams p) { tree_attn_direct_body<true, bf16>(p); }
