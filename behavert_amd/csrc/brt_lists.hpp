// brt_lists.hpp -- walking a neighbour list row (count, then up to K sorted
// indices, padded; stride W = 4(K/4+1) words, 16-byte aligned rows).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "brt_wave.hpp"

namespace brt {

typedef uint32_t vuint4 __attribute__((ext_vector_type(4)));

// Bit k set for the valid entries e = 4q + k of an octet (1 <= e <= count and
// a sorted index below n); invalid lanes of jj are set to i.  Word entry 0 of
// word 0 is the count; the slot of word entry k is e - 1 = 4q + k - 1.
__device__ __forceinline__ uint32_t octet_mask(uint32_t (&jj)[8], uint32_t q, uint32_t count, uint32_t i,
                                               uint32_t n) {
    uint32_t mask = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const uint32_t e = 4u * q + k;
        const bool ok = e >= 1u && e <= count && jj[k] < n;
        mask |= ok ? (1u << k) : 0u;
        jj[k] = ok ? jj[k] : i;
    }
    return mask;
}

// Visits the entries e = 1..count (count capped at K) of agent i's list in
// order, eight at a time: f(base, jj, mask) gets word entries base..base+7
// (list slot base + k - 1), with bit k of mask set for the valid ones.
// Invalid lanes of jj hold i, so gathers through them stay in bounds.
// Each lane reads its own row: the next two 16-byte words loading (AHEAD) while
// the current octet's gathers are in flight, or (WHOLE) rows of W = 36 words
// (K 32..35) all at once.  Words past the count are not loaded: each lane's are an
// access of their own.
template <bool AHEAD = true, bool WHOLE = false, class Fn>
__device__ __forceinline__ uint32_t for_list_octets(const uint32_t* __restrict__ lists, uint32_t W, uint32_t K,
                                                    uint32_t i, uint32_t n, Fn&& f) {
    const vuint4* L = reinterpret_cast<const vuint4*>(lists + (size_t)i * W);
    auto octet = [&](uint32_t q, uint32_t count, vuint4 a, vuint4 b) {
        uint32_t jj[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        const uint32_t mask = octet_mask(jj, q, count, i, n);
        f(4u * q, jj, mask);
    };
    if (WHOLE && W == 36u) {
        vuint4 c[9];
#pragma unroll
        for (uint32_t k = 0; k < 9u; ++k) c[k] = L[k];
        const uint32_t count = c[0].x < K ? c[0].x : K;
#pragma unroll
        for (uint32_t q = 0; q < 9u; q += 2)
            if (4u * q <= count) octet(q, count, c[q], c[q < 8u ? q + 1u : 8u]);
        return count;
    }
    auto word = [&](uint32_t q, uint32_t last) {
        vuint4 v = {0u, 0u, 0u, 0u};
        if (q <= last) v = L[q];
        return v;
    };
    vuint4 a = L[0];
    const uint32_t count = a.x < K ? a.x : K;
    const uint32_t last = count / 4u;  // the word that holds the last entry
    vuint4 b = word(1u, last);
    for (uint32_t q = 0; q <= last; q += 2) {
        vuint4 na, nb;
        if (AHEAD) {
            na = word(q + 2u, last);
            nb = word(q + 3u, last);
        } else if (q != 0u) {
            a = L[q];
            b = word(q + 1u, last);
        }
        octet(q, count, a, b);
        if (AHEAD) {
            a = na;
            b = nb;
        }
    }
    return count;
}

// The same with the rows of a wave's 64 agents loaded by the wave together.
// What bounds most list walks is the number of 64-byte accesses that their loads
// make (about one a clock per CU): a 16-byte word of every lane's own row is 64
// of them, the same bytes in order 16.  Rows of up to kStageWords words (K 35) go
// through LDS whole, longer ones in blocks.  Every lane of the wave takes part:
// row0 is the wave's first agent, i = row0 + lane, and lanes beyond n visit
// nothing.  1M blobs, K 32, whole rows by their own lanes -> staged: a label
// iteration 45.3 -> 37.5 us; with the XCD slices, behaviour forces + features of
// 300,007 agents 57 + 70 -> 46 + 49.
constexpr uint32_t kStageWords = 36u;
constexpr uint32_t kStageChunks = 64u * kStageWords / 4u;  // 16-byte words per wave

// Loads a wave's rows (W <= kStageWords) into LDS, 64 rows of W words.
__device__ __forceinline__ void stage_rows(uint4* stage, const uint32_t* __restrict__ lists, uint32_t W,
                                           uint32_t row0, uint32_t lane, uint32_t n) {
    const uint32_t W4 = W / 4u, rows = row0 < n ? (n - row0 < 64u ? n - row0 : 64u) : 0u, total = rows * W4;
    const vuint4* src = reinterpret_cast<const vuint4*>(lists + (size_t)(rows ? row0 : 0u) * W);
    vuint4* const to = reinterpret_cast<vuint4*>(stage);
    const uint32_t top = total ? total - 1u : 0u;
    if (W4 == 9u) {
        vuint4 c[9];
#pragma unroll
        for (uint32_t k = 0; k < 9u; ++k) c[k] = src[lane + 64u * k < total ? lane + 64u * k : top];
#pragma unroll
        for (uint32_t k = 0; k < 9u; ++k) to[lane + 64u * k] = c[k];
    } else {
#pragma unroll 4
        for (uint32_t k = 0; k < W4; ++k) to[lane + 64u * k] = src[lane + 64u * k < total ? lane + 64u * k : top];
    }
    wave_lds_sync();
}

// Visits the entries of a row in LDS.  Entry e is read before f gets entry e + 1
// (f may overwrite word e - 1 once it has entry e).
template <class Fn>
__device__ __forceinline__ void visit_staged(const uint4* L, uint32_t count, uint32_t i, uint32_t n, Fn&& f) {
    for (uint32_t q = 0; 4u * q <= count; q += 2) {
        const uint4 a = L[q], b = L[4u * (q + 1u) <= count ? q + 1u : q];
        uint32_t jj[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        const uint32_t mask = octet_mask(jj, q, count, i, n);
        f(4u * q, jj, mask);
    }
}

// Rows beyond kStageWords in blocks of their 16-byte words: four of every row, in
// which short lists end, then eight at a time while some list has so many left.
// Blocks of eight from the start are 10 % faster for lists of about 20 entries and
// up to 30 % slower for short ones.  A label iteration of 1,048,576 agents, K 64, at
// 1 / 4 / 12 per cell: each lane its own row 34 / 59 / 157 us, blocks of eight 44 /
// 51 / 98, so 36 / 58 / 101.
constexpr uint32_t kBlockRow = 9u;  // odd: no bank conflicts
constexpr uint32_t kBlockChunks = 64u * kBlockRow;
// words q0 .. q0 + C of every row; those past it and rows past n repeat others
template <uint32_t C>
__device__ __forceinline__ void stage_block(vuint4* to, const vuint4* __restrict__ rows, uint32_t W4, uint32_t row0,
                                            uint32_t lane, uint32_t n, uint32_t q0) {
    vuint4 c[C];
    const uint32_t at = q0 + lane % C < W4 ? q0 + lane % C : W4 - 1u;
#pragma unroll
    for (uint32_t k = 0; k < C; ++k) {
        const uint32_t r = row0 + (64u / C) * k + lane / C;
        c[k] = rows[(size_t)(r < n ? r : n - 1u) * W4 + at];
    }
    wave_lds_sync();  // the previous block has been read
#pragma unroll
    for (uint32_t k = 0; k < C; ++k) to[((64u / C) * k + lane / C) * kBlockRow + lane % C] = c[k];
    wave_lds_sync();
}
template <class Fn>
__device__ __forceinline__ uint32_t wave_list_blocks(uint4* stage, const uint32_t* __restrict__ lists, uint32_t W,
                                                     uint32_t K, uint32_t row0, uint32_t lane, uint32_t n, Fn&& f) {
    const uint32_t i = row0 + lane, W4 = W / 4u;
    const vuint4* const rows = reinterpret_cast<const vuint4*>(lists);
    vuint4* const to = reinterpret_cast<vuint4*>(stage);
    const uint4* const L = stage + lane * kBlockRow;
    uint32_t count = i < n ? 1u : 0u;  // until the first block is there
    for (uint32_t q0 = 0, size; __ballot(4u * q0 <= count) != 0; q0 += size) {
        size = q0 == 0u || __ballot(4u * (q0 + 4u) <= count) == 0 ? 4u : 8u;
        if (size == 4u)
            stage_block<4u>(to, rows, W4, row0, lane, n, q0);
        else
            stage_block<8u>(to, rows, W4, row0, lane, n, q0);
        if (q0 == 0u && i < n) count = L[0].x < K ? L[0].x : K;
        for (uint32_t q = q0; i < n && q < q0 + size && 4u * q <= count; q += 2) {
            const uint4 a = L[q - q0], b = L[4u * (q + 1u) <= count ? q + 1u - q0 : q - q0];
            uint32_t jj[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
            const uint32_t mask = octet_mask(jj, q, count, i, n);
            f(4u * q, jj, mask);
        }
    }
    return i < n ? count : 0u;
}

// How a pass reads the rows of its lists.
enum ListRows : int {
    kRowsOwn = 0,     // each lane its own
    kRowsWhole = 1,   // the wave stages them whole
    kRowsBlocks = 2,  // the wave stages them in blocks
};

// Launches above this many agents stage their rows.  With about one wave per SIMD
// (65,536 agents fill them) a pass is bound by the wave's chain of latencies, which
// LDS lengthens, and in the slices of xcd_block too: up to there each lane reads its
// own row and the workgroups keep their order.  Own -> staged, K 32, 12 per cell,
// us: feature update, 60,000 agents 8.7 -> 9.8, 66,000 8.9 -> 10.9, 78,000 16.6 ->
// 15.6, 100,003 18.0 -> 17.4; cluster steering, 20,000 12.6 -> 14, 100,003 37 -> 32.
constexpr uint32_t kStageAbove = 73728u;
inline ListRows list_rows(uint32_t W, uint32_t n) {
    return n <= kStageAbove ? kRowsOwn : (W <= kStageWords ? kRowsWhole : kRowsBlocks);
}
// 16-byte words of LDS per wave
constexpr uint32_t list_rows_chunks(ListRows rows) {
    return rows == kRowsOwn ? 1u : (rows == kRowsWhole ? kStageChunks : kBlockChunks);
}

template <ListRows ROWS, class Fn>
__device__ __forceinline__ uint32_t walk_list(uint4* stage, const uint32_t* __restrict__ lists, uint32_t W, uint32_t K,
                                              uint32_t row0, uint32_t lane, uint32_t n, Fn&& f) {
    const uint32_t i = row0 + lane;
    if (ROWS == kRowsBlocks) return wave_list_blocks(stage, lists, W, K, row0, lane, n, f);
    if (ROWS == kRowsOwn) return i < n ? for_list_octets<true, true>(lists, W, K, i, n, f) : 0u;
    stage_rows(stage, lists, W, row0, lane, n);
    if (i >= n) return 0u;
    const uint4* L = stage + lane * (W / 4u);
    const uint32_t head = L[0].x, count = head < K ? head : K;
    visit_staged(L, count, i, n, f);
    return count;
}

}  // namespace brt
