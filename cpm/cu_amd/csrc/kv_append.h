// One run of rows appended to the paged cache: shared by the stand-alone append and the attention launches that append on the side.
#pragma once
#include "common.h"

namespace cpmcu {

// One rotary pair: (a, b) -> (a cos - b sin, a sin + b cos), every product and sum rounded on its own
// (no fused multiply-add), so the result does not depend on how a compiler contracts the expression.
template <typename E>
__device__ inline void rotate_pair(E& a, E& b, float2 cs) {
#pragma clang fp contract(off)
    const float fa = (float)a, fb = (float)b;
    const float ac = fa * cs.x, bs = fb * cs.y, as = fa * cs.y, bc = fb * cs.x;
    a = (E)(ac - bs);
    b = (E)(as + bc);
}

// copy_to_kvcache, src/model/attn.cuh:14-21: token t of the T new rows goes to position S - T + t.
// A launch is a chain of two round trips (rows beside length -> page ids, then the stores), so the bytes have to be whole
// transactions: kAppendThreads threads take kAppendRows consecutive new rows of one KV head, which they can request before they
// know where they go; K goes straight on as 16-byte pieces, V is transposed through LDS into 16-byte pieces of the page's dim
// rows (eight token slots each).  Only pieces that the run covers in part are written slot by slot.  2048 rows of two heads:
// 7.0 us with one token per workgroup and 2-byte V stores 512 bytes apart, 4.4 with runs of 32 rows (130 workgroups), 3.7 with
// 16 (258).
constexpr int kAppendRows = 16;
constexpr int kAppendThreads = 256;
constexpr int kAppendStride = kHeadDim + 4;  // halves per staged V row: the lanes of a dim read rows 4 or 8 apart
struct AppendStage {
    __attribute__((aligned(8))) uint16_t v[kAppendRows * kAppendStride];
};

// tid: 0 .. kAppendThreads - 1.  n <= 0 rows: only meets the barrier.  length(): the device-side S.  rope (or null): the table of
// (cos, sin) that the K rows of element type E are rotated by on their way.
// ZERO_PAST: the slots past the end in the pieces that hold appended rows become zero (what the attention launches leave there).
template <typename E, bool ZERO_PAST, typename Length>
__device__ inline void kv_append_run(f16* k_pool, f16* v_pool, const int32_t* block_table, const f16* k_new, const f16* v_new,
                                     const float2* rope, int T, int Hkv, int g, int r0, int tid, AppendStage& stage, Length&& length) {
    typedef typename Elem<E>::x8 X8;
    const int n = min(kAppendRows, T - r0);
    const int row = tid >> 4, ch = tid & 15;  // 16 rows x 16 pieces of 16 bytes
    int p0 = 0, lp = 0, page_lo = 0, page_hi = 0;
    const auto page_of = [&](int pos) { return pos / kPage == lp ? page_lo : page_hi; };
    if (n > 0) {
        const int r = r0 + min(row, n - 1);
        const size_t o = ((size_t)r * Hkv + g) * kHeadDim + ch * 8;
        X8 kx = *reinterpret_cast<const X8*>(k_new + o);
        const uint4 vx = *reinterpret_cast<const uint4*>(v_new + o);
        if (rope != nullptr) {
            // the pair (d, d + 64) of a row sits eight lanes apart
            const float2* cs = rope + (size_t)r * (kHeadDim / 2) + (ch & 7) * 8;
            uint4 w = __builtin_bit_cast(uint4, kx);
            w.x = __shfl_xor(w.x, 8);
            w.y = __shfl_xor(w.y, 8);
            w.z = __shfl_xor(w.z, 8);
            w.w = __shfl_xor(w.w, 8);
            const X8 other = __builtin_bit_cast(X8, w);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                E a = ch < 8 ? kx[j] : other[j], b = ch < 8 ? other[j] : kx[j];
                rotate_pair(a, b, cs[j]);
                kx[j] = ch < 8 ? a : b;
            }
        }
        p0 = length() - T + r0;  // position of this run's first row; its rows lie in at most two pages
        lp = p0 / kPage;
        page_lo = block_table[lp];
        page_hi = block_table[(p0 + n - 1) / kPage];
        uint2* staged = reinterpret_cast<uint2*>(stage.v + row * kAppendStride + ch * 8);
        staged[0] = make_uint2(vx.x, vx.y);
        staged[1] = make_uint2(vx.z, vx.w);
        if (row < n) {
            const int pos = p0 + row;
            *reinterpret_cast<X8*>(k_pool + (((size_t)page_of(pos) * Hkv + g) * kPage + pos % kPage) * kHeadDim + ch * 8) = kx;
        }
    }
    __syncthreads();
    if (n <= 0) return;
    // V^T: the one or two 16-slot groups of the run, two pieces each; the pieces of a dim on neighbouring lanes
    const int group0 = p0 & ~15;
    const int npieces = ((p0 + n - 1 - group0) / 16 + 1) * 2;
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const int x = it * kAppendThreads + tid;
        const int d = x >> 2, piece = x & 3;
        if (piece >= npieces) continue;
        const int first = group0 + (piece >> 1) * 16 + (piece & 1) * 4;  // slots 0..3: tokens first .. + 3, slots 4..7: first + 8 ..
        uint32_t v[8], in = 0;
        bool any_new = false;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int r = first + (j & 3) + (j >> 2) * 8 - p0;
            v[j] = stage.v[min(max(r, 0), n - 1) * kAppendStride + d];
            in |= r >= 0 && r < n ? 1u << j : 0u;
            any_new |= r0 + r >= 0 && r0 + r < T;
        }
        if (ZERO_PAST && r0 + n == T && any_new) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (first + (j & 3) + (j >> 2) * 8 - p0 >= n) {
                    v[j] = 0;
                    in |= 1u << j;
                }
        }
        const int slot = (first & ~15) % kPage + (piece & 1) * 8;
        uint16_t* dst = reinterpret_cast<uint16_t*>(v_pool) + (((size_t)page_of(first) * Hkv + g) * kHeadDim + d) * kPage + slot;
        if (in == 0xFFu) {
            *reinterpret_cast<uint4*>(dst) = make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16));
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if ((in >> j) & 1u) dst[j] = (uint16_t)v[j];
        }
    }
}

}  // namespace cpmcu
