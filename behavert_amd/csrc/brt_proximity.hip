// brt_proximity.hip -- Proximity3D on gfx950: capped 27-cell neighbour lists,
// optionally fused with the OpenSteerWrapper steering + integration pass.
//
// Reference semantics (genericCalcNeighgborhoodD, PlugIns/Proximity3D/Proximity3D_kernel.cu:89-125;
// checkForNeighborsInCell / checkForNeighbor, Proximity3D_resources.cu:59-172):
//   * the agent's cell is calcGridPos(pos) WITHOUT clamping;
//   * cells are visited x-offset outermost, then y, then z innermost, each -1..1,
//     skipping cells outside the grid and empty cells;
//   * inside a cell, agents are visited in sorted order, at most
//     maxBodiesPerCell of them, the agent itself skipped;
//   * a candidate is rejected when sqrtf(dx*dx+dy*dy+dz*dz) > r, dx = other - self;
//   * accepted sorted indices are appended until K are held (later ones are
//     ignored; with useKnn the farthest entry is replaced instead).
// Output layout: the reader layout W = 4*(K/4+1) uints per agent
// (Proximity3D_resources.cu:175-198), [0] = count, then the indices, then padding.
//
// Exactness: the distance test is d2 = (dx*dx + dy*dy) + dz*dz (no FMA) against
// T, the largest float with sqrtf(T) <= r; for a correctly rounded, monotone
// sqrtf, "sqrtf(d2) > r" and "d2 > T" agree for every d2, NaN included.
//
// MI355X design.  One lane per sorted agent, 256 lanes per workgroup (64 for
// LDS-list launches of more than 2^17 agents, see prox_block); lists are staged
// in LDS and written out with 16-byte coalesced stores, or gathered in
// registers as 16-byte chunks.  Per wave64:
//   * uniform mode (all lanes in few cells): lanes are grouped by cell; a group
//     walks the shared canonical candidate stream with wave-uniform indices, so
//     candidate positions come through the scalar cache (s_load);
//   * flat mode (LDS lists): each lane walks its own stream of cells with its
//     own cell index, eight (dense waves) or four (sparse waves) candidates
//     per round, their accept bits logged per round;
//   * vector mode (register-chunk lists): each lane walks its own stream, the
//     wave in step cell by cell;
//   * row scan (sparse waves): the cells of a row as one run, nine runs (see
//     scan_rows).
// Small launches take four lanes per agent instead (k_prox_quad).
// Every mode skips a cell whose box lies farther than r from the agent (with
// rounding margins so no candidate that passes the exact test is ever skipped),
// only for interior cells: boundary cells can hold clamped out-of-grid or NaN
// agents whose positions are not inside the cell's box.
#include "brt_device.hpp"
#include "brt_internal.hpp"
#include "brt_steer_common.hpp"
#include "brt_wave.hpp"

// Candidates tested per round of the scan loops (their loads are in flight
// together): per-lane (vector) rounds of dense waves with LDS lists, of sparse
// waves and register-chunk lists, and wave-uniform (scalar) rounds.  Measured
// on gfx950: 8 per round for dense waves with LDS lists (1M-boid blobs, K 32:
// -11 % against 4), 4 for sparse waves (65k boids at ~1 per cell: 8 is 26 %
// slower) and with register-chunk lists (8 spills there).
#ifndef BRT_PROX_GROUP
#define BRT_PROX_GROUP 8
#endif
#ifndef BRT_PROX_GROUP_R
#define BRT_PROX_GROUP_R 4
#endif
#ifndef BRT_PROX_GROUP_U
#define BRT_PROX_GROUP_U 4
#endif
// 1: in dense waves with LDS lists, cells that cannot hold the agent itself run
// rounds without the self test (a second copy of the round code, one ballot
// per cell; elsewhere that measured slower); 0: every round tests for the agent.
#ifndef BRT_PROX_SELF_SPLIT
#define BRT_PROX_SELF_SPLIT 1
#endif
// Neighbours gathered together (positions and headings in flight) by the fused
// steering walk over a finished list.
#ifndef BRT_PROX_STEER_GROUP
#define BRT_PROX_STEER_GROUP 4
#endif
// 1: the loops over the 27 neighbour cells stay loops (one copy of the round
// code per variant; a slab's cell ranges are read from registers by a
// wave-uniform index); 0: they are unrolled, one copy of the round code per cell.
#ifndef BRT_PROX_ROLLED
#define BRT_PROX_ROLLED 1
#endif
// 1: LDS lists are built through a per-round log of accept bits (see
// log_round) when the launch has fewer than 2^24 agents; 0: every accepted
// candidate is appended as it is tested.
#ifndef BRT_PROX_LOG
#define BRT_PROX_LOG 1
#endif
// 1: dense waves with the round log scan in flat mode (see scan_flat).
#ifndef BRT_PROX_FLAT
#define BRT_PROX_FLAT 1
#endif
// 1: sparse waves with the round log scan in flat mode too.
#ifndef BRT_PROX_FLAT_SPARSE
#define BRT_PROX_FLAT_SPARSE 1
#endif
// Workgroup of the single-grid LDS-list neighbour kernels for launches of more
// than 2^17 agents (see prox_block).
#ifndef BRT_PROX_BLOCK_LARGE
#define BRT_PROX_BLOCK_LARGE 64
#endif
// A wave is dense (rounds of BRT_PROX_GROUP candidates) when at least
// BRT_PROX_DENSE_LANES of its lanes sit in cells of BRT_PROX_DENSE_OCC agents
// or more.
#ifndef BRT_PROX_DENSE_OCC
#define BRT_PROX_DENSE_OCC 8
#endif
#ifndef BRT_PROX_DENSE_LANES
#define BRT_PROX_DENSE_LANES 32
#endif
// A wave takes the row scan (scan_rows) unless BRT_PROX_ROW_LANES of its lanes
// have more than BRT_PROX_ROW_OCC agents in their own row's three cells: beyond
// that some run is mostly too long for it, and the lists fill before their last
// cells.  One step of 400,000 uniform agents, per-cell scan -> row scan, at 1 /
// 4 / 6 agents per cell: K 32 152 -> 132 / 185 -> 166 / 204 -> 188 us, K 64
// 190 -> 161 / 268 -> 216 / 307 -> 283 us; with the limit at 15: 4 per cell
// 172 and 247 us; at 8 per cell no wave qualifies (208 us either way).
#ifndef BRT_PROX_ROW_OCC
#define BRT_PROX_ROW_OCC 23
#endif
#ifndef BRT_PROX_ROW_LANES
#define BRT_PROX_ROW_LANES 32
#endif
#if BRT_PROX_ROLLED
#define BRT_CELL_LOOP _Pragma("nounroll")
#else
#define BRT_CELL_LOOP _Pragma("unroll")
#endif

namespace brt {

namespace {

constexpr int kGroupL = BRT_PROX_GROUP;
constexpr int kGroupR = BRT_PROX_GROUP_R;
constexpr int kGroupU = BRT_PROX_GROUP_U;

// Loads through the constant address space: with a wave-uniform index these
// become scalar-cache loads (s_load_dwordx4).  The arrays are not written by
// the kernel that reads them this way.
typedef float vfloat4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) vfloat4* cfloat4_ptr;
typedef const __attribute__((address_space(4))) uint32_t* cuint_ptr;

__device__ __forceinline__ float4 cload(cfloat4_ptr p, uint32_t i) {
    const vfloat4 v = p[i];
    return make_float4(v.x, v.y, v.z, v.w);
}

struct ProxArgs {
    brt_grid_params g;  // single-grid launches
    uint32_t K, W, n;   // n = all agents of the launch (a batch: of every flock)
    uint32_t Ws;        // row stride of the LDS list tile (lds_list_stride(K) >= W)
    float T;            // exact squared-radius threshold
    float Tskip;        // T * (1 + 1e-5): cell-skip threshold on the box distance
    float slack[3];     // per-axis widening of cell boxes for rounding (single grid)
    uint32_t uniform_max_cells;
    uint32_t xcd_remap;
    uint32_t log_rounds;  // LDS lists through the round log (n < 2^24)
    uint32_t together;    // the lanes of a quad visit their cells together (kTogetherK)
    uint32_t cells;       // cells of the launch for the row scan's bounded loads; 0: no row scan
    // agents of its own row beyond which an agent would rather not have its rows
    // scanned, by one lane and by four (row_limit)
    uint32_t row_occ, row_occ_quad;
    const float4* spos;
    const float* pxyz;  // optional: the sorted positions packed as x,y,z (12 bytes each)
    const float4* sfwd;
    const float4* ssa;  // sorted smooth_accel, or NULL: read by agent ID from o.sa_out
    const uint2* hash;
    const uint32_t* cell_start;
    const uint32_t* cell_end;
    uint32_t* lists;
    // fused steering
    brt_steer_params sp;
    SteerCuts cuts;
    float dt;
    uint32_t step;
    AgentOut o;
    // batches: per-flock grids, weights and wave ranges
    BatchView b;
};

// The agents one wave works on and the grid they live in (wave-uniform).
struct Seg {
    brt_grid_params g;
    float slack[3];
    uint32_t cell_base;  // global key of the grid's cell 0
    uint32_t row0;       // sorted index of the wave's lane 0
    uint32_t end;        // one past the segment's last sorted index
    uint32_t id_base;    // agent ID of the segment's first agent
    Weights w;
};

template <bool BATCH>
__device__ __forceinline__ bool wave_segment(const ProxArgs& a, uint32_t gw, Seg& sg) {
    if (!BATCH) {
        sg.g = a.g;
        sg.slack[0] = a.slack[0];
        sg.slack[1] = a.slack[1];
        sg.slack[2] = a.slack[2];
        sg.cell_base = 0;
        sg.row0 = gw * 64u;
        sg.end = a.n;
        sg.id_base = 0;
        sg.w = weights_of(a.sp);
        return sg.row0 < a.n;
    }
    if (gw >= a.b.waves) return false;
    const uint32_t f = __builtin_amdgcn_readfirstlane(a.b.wave_flock[gw]);
    const FlockDev& fd = a.b.flocks[f];
    sg.g = fd.g;
    sg.slack[0] = fd.slack[0];
    sg.slack[1] = fd.slack[1];
    sg.slack[2] = fd.slack[2];
    sg.cell_base = fd.cell_base;
    sg.row0 = fd.offset + (gw - fd.wave_base) * 64u;
    sg.end = fd.offset + fd.n;
    sg.id_base = fd.offset;
    sg.w = Weights{fd.w[0], fd.w[1], fd.w[2]};
    return true;
}

struct Lane {
    float px, py, pz;
    uint32_t i;
    uint32_t cnt;
    uint32_t* row;       // the agent's list row: staged in LDS, or in global memory
    uint32_t* wp;        // LDS lists: the next free entry (row + 1 + cnt) during a round
    uint32_t h0, h1, h2;  // register-chunk lists: entries 0..2 (chunk 0, with the count)
    uint32_t b0, b1, b2;  // register-chunk lists: entries of the pending 16-byte chunk
    // squared distances from the agent to the boxes of the cells one below
    // (lo) and one above (hi) its own on each axis, each gap shrunk by the
    // rounding slack: the box distance of neighbour (dx,dy,dz) is the sum of
    // the three selected terms (offset 0 contributes 0)
    float lo2[3], hi2[3];
};

__device__ __forceinline__ bool interior(int cx, int cy, int cz, const brt_grid_params& g) {
    return cx >= 1 && cy >= 1 && cz >= 1 && cx <= (int)g.grid_size[0] - 2 && cy <= (int)g.grid_size[1] - 2 &&
           cz <= (int)g.grid_size[2] - 2;
}

__device__ __forceinline__ void cell_gaps(const Seg& sg, Lane& L, I3 gp) {
    const float p[3] = {L.px, L.py, L.pz};
    const int c[3] = {gp.x, gp.y, gp.z};
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        const float lo = sg.g.world_origin[ax] + (float)c[ax] * sg.g.cell_size[ax];
        const float f = p[ax] - lo;
        const float gl = fmaxf(f - sg.slack[ax], 0.0f);
        const float gh = fmaxf((sg.g.cell_size[ax] - f) - sg.slack[ax], 0.0f);
        L.lo2[ax] = gl * gl;
        L.hi2[ax] = gh * gh;
    }
}

// The lo or hi term of axis ax for offset d (0 for d = 0), chosen by bit masks
// rather than a select of the two fields, which the compiler may turn into a
// select of their addresses and so keep the lane's state in scratch memory
// when d is not a compile-time constant.
__device__ __forceinline__ float gap2(const Lane& L, int ax, int d) {
    const uint32_t mlo = d < 0 ? 0xFFFFFFFFu : 0u, mhi = d > 0 ? 0xFFFFFFFFu : 0u;
    return __uint_as_float((__float_as_uint(L.lo2[ax]) & mlo) | (__float_as_uint(L.hi2[ax]) & mhi));
}

// Appends sorted index c to the lane's list when take.  LDS lists: one LDS
// word per entry.  Register-chunk lists: the row's 16-byte chunk q holds words
// 4q..4q+3, i.e. entries 4q-1..4q+2; entries are gathered in registers and a
// chunk is stored to global memory when its last entry arrives (chunk 0, which
// holds the count, and the final partial chunk are stored by finish_list).
template <bool LDSL>
__device__ __forceinline__ void append(Lane& L, uint32_t c, bool take) {
    if (LDSL) {
        if (take) L.row[1 + L.cnt] = c;
    } else if (take) {
        const uint32_t k = L.cnt;
        if (k < 3u) {
            L.h0 = k == 0u ? c : L.h0;
            L.h1 = k == 1u ? c : L.h1;
            L.h2 = k == 2u ? c : L.h2;
        } else {
            const uint32_t s = (k - 3u) & 3u;
            if (s == 3u) {
                reinterpret_cast<uint4*>(L.row)[(k - 3u) / 4u + 1u] = make_uint4(L.b0, L.b1, L.b2, c);
            } else {
                L.b0 = s == 0u ? c : L.b0;
                L.b1 = s == 1u ? c : L.b1;
                L.b2 = s == 2u ? c : L.b2;
            }
        }
    }
    L.cnt += take ? 1u : 0u;
}

// Walks the 16-byte chunks of consecutive rows of W4 chunks, 64 apart: the row
// and chunk of lane + 64 k without a division per step.
struct ChunkWalk {
    uint32_t row, chunk, drow, dchunk, w4;
    __device__ __forceinline__ ChunkWalk(uint32_t lane, uint32_t W4) : w4(W4) {
        row = lane / W4;
        chunk = lane - row * W4;
        drow = 64u / W4;
        dchunk = 64u - drow * W4;
    }
    __device__ __forceinline__ void next() {
        row += drow;
        chunk += dchunk;
        if (chunk >= w4) {
            chunk -= w4;
            ++row;
        }
    }
};

// Register-chunk lists: the chunks not yet stored (the pending partial chunk,
// then chunk 0).  Returns the row's first all-padding chunk: those chunks are
// stored by the whole wave together (pad_rows).
__device__ __forceinline__ uint32_t finish_list(Lane& L, uint32_t W) {
    const uint32_t P = BRT_LIST_PAD, k = L.cnt;
    uint4* row = reinterpret_cast<uint4*>(L.row);
    uint32_t q = (k > 3u ? (k - 3u) / 4u : 0u) + 1u;
    const uint32_t rem = k > 3u ? (k - 3u) & 3u : 0u;
    if (4u * q < W) {
        row[q] = make_uint4(rem > 0u ? L.b0 : P, rem > 1u ? L.b1 : P, rem > 2u ? L.b2 : P, P);
        ++q;
    }
    row[0] = make_uint4(k, k > 0u ? L.h0 : P, k > 1u ? L.h1 : P, k > 2u ? L.h2 : P);
    return q;
}

// Register-chunk lists: the all-padding chunks of the wave's rows (consecutive
// rows of W words from sorted index row0; lane l's row starts padding at its
// chunk pad_from), stored by the whole wave with consecutive 16-byte chunks per
// store instead of each lane's own strided row.  The trip count is
// wave-uniform, so every lane takes part in the shuffle.
__device__ __forceinline__ void pad_rows(uint32_t* lists, uint32_t row0, uint32_t rows, uint32_t W, uint32_t lane,
                                         uint32_t pad_from) {
    const uint32_t W4 = W / 4u, total = rows * W4;
    const uint32_t P = BRT_LIST_PAD;
    uint4* dst = reinterpret_cast<uint4*>(lists + (size_t)row0 * W);
    ChunkWalk cw(lane, W4);
    for (uint32_t base = 0; base < total; base += 64u, cw.next()) {
        const uint32_t w = base + lane;
        const uint32_t first = (uint32_t)__shfl((int)pad_from, (int)(cw.row < 64u ? cw.row : 63u));
        if (w < total && cw.chunk >= first) dst[w] = make_uint4(P, P, P, P);
    }
}

// Stores the wave's rows (consecutive, from sorted index row0) out of LDS with
// consecutive 16-byte chunks per store: src holds one row of `stride` words per
// lane, count first; words past the count are padding.  HEADS: src holds only
// the rows' first `stride` words; of the later chunks those that hold entries
// were stored by the row's own lane, the others are padding.
template <bool HEADS>
__device__ __forceinline__ void store_rows(uint32_t* lists, uint32_t row0, uint32_t rows, uint32_t W,
                                           const uint32_t* src, uint32_t stride, uint32_t lane) {
    const uint32_t W4 = W / 4u, total = rows * W4;
    const uint32_t P = BRT_LIST_PAD;
    uint4* dst = reinterpret_cast<uint4*>(lists + (size_t)row0 * W);
    ChunkWalk cw(lane, W4);
    for (uint32_t w = lane; w < total; w += 64u, cw.next()) {
        const uint32_t* row = src + cw.row * stride;
        const uint32_t cnt = row[0], e = 4u * cw.chunk;
        if (!HEADS || e < stride) {
            uint4 v = reinterpret_cast<const uint4*>(row)[cw.chunk];
            v.x = e > cnt ? P : v.x;  // word 0 is the count itself
            v.y = e + 1u > cnt ? P : v.y;
            v.z = e + 2u > cnt ? P : v.z;
            v.w = e + 3u > cnt ? P : v.w;
            dst[w] = v;
        } else if (e > cnt) {
            dst[w] = make_uint4(P, P, P, P);
        }
    }
}

// Tests the candidates j .. j+G-1 (positions q) for lane L and appends
// those that pass, in order, without branching.  rem = lim - j (candidates
// left in the cell), di = i - j (where the agent itself sits in the round).
// SELF: the agent's own index lies in this cell's range, so it is excluded.
// CAP (some lane may reach K inside this round): 1 = every append re-checks
// the count; 2 = the LDS row has room for G - 1 entries past K (stride
// Ws >= K + G, every lane entering the round below K: the last write lands at
// most at row[K + G - 1]), so the round appends freely and the count is
// clamped to K afterwards: entries past K are overwritten by padding.
// LDS lists append through a write pointer: a predicated store and a pointer
// bump per candidate.
template <bool LDSL, int CAP, bool SELF, int G>
__device__ __forceinline__ void test_round(const ProxArgs& a, Lane& L, uint32_t j, uint32_t rem, uint32_t di,
                                           const float4* q) {
    if (LDSL) L.wp = L.row + 1u + L.cnt;
#pragma unroll
    for (int t = 0; t < G; ++t) {
        const float rx = q[t].x - L.px, ry = q[t].y - L.py, rz = q[t].z - L.pz;
        const float xx = rx * rx, yy = ry * ry, zz = rz * rz;
        const float d2 = (xx + yy) + zz;
        bool take = ((uint32_t)t < rem) & !(d2 > a.T);
        if (SELF) take = take & (di != (uint32_t)t);
        if (LDSL) {
            if (CAP == 1) take = take & (L.wp < L.row + 1u + a.K);
            if (take) *L.wp = j + (uint32_t)t;
            L.wp += take ? 1 : 0;
        } else {
            if (CAP) take = take & (L.cnt < a.K);
            append<false>(L, j + (uint32_t)t, take);
        }
    }
    if (LDSL) {
        const uint32_t c = (uint32_t)(L.wp - (L.row + 1u));
        L.cnt = CAP == 2 ? (c < a.K ? c : a.K) : c;
    }
}

// m = 2m + bit in one VALU add-with-carry whose carry-in is the wave's mask of
// the compare that produced bit (the ballot folds into that compare).
__device__ __forceinline__ uint32_t shift_in(uint32_t m, bool bit) {
    const uint64_t c = __builtin_amdgcn_ballot_w64(bit);
    uint32_t r;
    uint64_t carry_out;
    asm("v_addc_co_u32_e64 %0, %1, %2, %2, %3" : "=v"(r), "=s"(carry_out) : "v"(m), "s"(c));
    return r;
}

// Round log (LDS lists, sorted indices below 2^24): the round's accept bits are
// collected with one add-with-carry per candidate (candidate j+t ends in bit
// 7-t), the limit and self tests are applied to the round's bits at once, and a
// round with any bit set appends the word j << 8 | bits to the agent's row.
// The running count includes every accepted bit; a lane stops before a round
// once it holds K, so at most K words are appended (each carries at least one
// bit) and they fit in the row.  expand_log turns the words into the list.
template <int G, bool SELF>
__device__ __forceinline__ void log_round(const ProxArgs& a, Lane& L, uint32_t j, uint32_t rem, uint32_t di,
                                          const float4* q) {
    static_assert(G >= 1 && G <= 8, "a round's bits must fit in 8 bits");
    uint32_t m = 0;
#pragma unroll
    for (int t = 0; t < G; ++t) {
        const float rx = q[t].x - L.px, ry = q[t].y - L.py, rz = q[t].z - L.pz;
        const float xx = rx * rx, yy = ry * ry, zz = rz * rz;
        const float d2 = (xx + yy) + zz;
        m = shift_in(m, !(d2 > a.T));
    }
    // slots t >= rem (rem >= 1) lie past the cell's limit: bits G-1-t below G-rem
    const uint32_t r = rem < (uint32_t)G ? rem : (uint32_t)G;
    m &= ~((1u << ((uint32_t)G - r)) - 1u);
    if (SELF && di < (uint32_t)G) m &= ~(1u << ((uint32_t)G - 1u - di));
    m <<= 8 - G;
    if (m != 0u) {
        *L.wp = (j << 8) | m;
        ++L.wp;
    }
    L.cnt += __popc(m);
}

// Round log of the flat scan: as log_round, with the self test folded into a
// mask the caller selects per round (all ones unless the round holds the
// agent), and the word stored unconditionally, the write pointer advancing only
// when the word carries a bit.  A word is stored only while the lane holds
// fewer than K, so at most K words are kept and the store lands at most at
// row[K] < W; a stored word without bits is overwritten by the next word or
// by the list's padding.
template <int G>
__device__ __forceinline__ void log_round_flat(const ProxArgs& a, Lane& L, uint32_t j, uint32_t rem, uint32_t sm,
                                               const float4* q) {
    static_assert(G >= 1 && G <= 8, "a round's bits must fit in 8 bits");
    uint32_t m = 0;
#pragma unroll
    for (int t = 0; t < G; ++t) {
        const float rx = q[t].x - L.px, ry = q[t].y - L.py, rz = q[t].z - L.pz;
        const float xx = rx * rx, yy = ry * ry, zz = rz * rz;
        const float d2 = (xx + yy) + zz;
        m = shift_in(m, !(d2 > a.T));
    }
    const uint32_t r = rem < (uint32_t)G ? rem : (uint32_t)G;
    m &= ~((1u << ((uint32_t)G - r)) - 1u) & sm;
    m <<= 8 - G;
    *L.wp = (j << 8) | m;
    L.wp += m != 0u ? 1 : 0;
    L.cnt += __popc(m);
}

// Expands the round log into the list, last word first and in place: word e
// sits at row[1+e] and its entries go to row[1+p] for p >= the bits of words
// 0..e-1 >= e, so no unread word is overwritten.  Entries past K are dropped
// and the count is clamped to K.
__device__ __forceinline__ void expand_log(Lane& L, uint32_t K) {
    const uint32_t nlog = (uint32_t)(L.wp - (L.row + 1u));
    uint32_t pos = L.cnt;
    for (uint32_t e = nlog; e-- > 0u;) {
        const uint32_t w = L.row[1u + e];
        uint32_t m = w & 0xFFu;
        const uint32_t j7 = (w >> 8) + 7u;
        pos -= __popc(m);
        uint32_t p = pos;
        while (m != 0u) {
            const uint32_t b = 31u - __clz(m);  // highest bit: the earliest candidate
            if (p < K) L.row[1u + p] = j7 - b;
            m ^= 1u << b;
            ++p;
        }
    }
    L.cnt = L.cnt < K ? L.cnt : K;
}

template <bool LDSL, bool SELF, int G>
__device__ __forceinline__ void test_round_any(const ProxArgs& a, Lane& L, uint32_t j, uint32_t rem, uint32_t di,
                                               const float4* q) {
    if (LDSL && a.log_rounds) {
        log_round<G, SELF>(a, L, j, rem, di, q);
        return;
    }
    if (__ballot(L.cnt + (uint32_t)G > a.K) == 0)
        test_round<LDSL, 0, SELF, G>(a, L, j, rem, di, q);
    else if (LDSL && a.Ws >= a.K + (uint32_t)G)
        test_round<LDSL, 2, SELF, G>(a, L, j, rem, di, q);
    else
        test_round<LDSL, 1, SELF, G>(a, L, j, rem, di, q);
}

// Buffer resource over a float4 array of n elements: 32-bit offsets with an
// immediate part, and reads past the end return zeros instead of faulting.
// Requires n < 2^28.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t float4_rsrc(const float4* p, uint32_t n) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float4*>(p), (short)0, (int)(n * 16u), 0x00020000);
}

__device__ __forceinline__ float4 bload(__amdgpu_buffer_rsrc_t r, uint32_t byte_offset) {
    const vfloat4 v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)byte_offset, 0, 0);
    return make_float4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t xyz_rsrc(const float* p, uint32_t n) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), (short)0, (int)(n * 12u), 0x00020000);
}

// The positions of candidates j .. j+G-1.  PACKED: from the packed x,y,z copy,
// 3G/4 16-byte loads at byte 12j (4-byte aligned; the wave's load count, not
// its bytes, is what the address unit spends its cycles on); else one 16-byte
// load per candidate.  Reads past the end return zeros.
template <int G, bool PACKED>
__device__ __forceinline__ void load_round(__amdgpu_buffer_rsrc_t rpos, __amdgpu_buffer_rsrc_t rxyz, uint32_t j,
                                           float4 (&q)[G]) {
    if (PACKED) {
        static_assert(G % 4 == 0, "packed rounds take multiples of 4 candidates");
        constexpr int NV = 3 * G / 4;
        float f[3 * G];
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const vfloat4 v = __builtin_amdgcn_raw_buffer_load_b128(rxyz, (int)(12u * j + 16u * (uint32_t)k), 0, 0);
            f[4 * k + 0] = v.x;
            f[4 * k + 1] = v.y;
            f[4 * k + 2] = v.z;
            f[4 * k + 3] = v.w;
        }
#pragma unroll
        for (int t = 0; t < G; ++t) q[t] = make_float4(f[3 * t], f[3 * t + 1], f[3 * t + 2], 0.0f);
    } else {
#pragma unroll
        for (int t = 0; t < G; ++t) q[t] = bload(rpos, j * 16u + 16u * (uint32_t)t);
    }
}

// Uniform mode: every active lane shares cell (ux,uy,uz); control flow and
// candidate indices are wave-uniform.
template <bool LDSL>
__device__ __forceinline__ void scan_uniform(const ProxArgs& a, const Seg& sg, Lane& L, int ux, int uy, int uz) {
    const brt_grid_params& g = sg.g;
    cfloat4_ptr cpos = (cfloat4_ptr)a.spos;
    cuint_ptr cstart = (cuint_ptr)a.cell_start;
    cuint_ptr cend = (cuint_ptr)a.cell_end;
    const uint32_t maxBodies = g.max_bodies_per_cell;
    BRT_CELL_LOOP
    for (int dx = -1; dx <= 1; ++dx) {
        BRT_CELL_LOOP
        for (int dy = -1; dy <= 1; ++dy) {
            BRT_CELL_LOOP
            for (int dz = -1; dz <= 1; ++dz) {
                const int cx = ux + dx, cy = uy + dy, cz = uz + dz;
                if (!inGrid(cx, cy, cz, g)) continue;
                const uint32_t key = sg.cell_base + cellKey(cx, cy, cz, g);
                const uint32_t s = cstart[key];
                if (s == BRT_EMPTY_CELL) continue;
                const uint32_t e = cend[key];
                uint32_t lim = (e - s) > maxBodies ? s + maxBodies : e;
                lim = lim < a.n ? lim : a.n;
                if (interior(cx, cy, cz, g)) {
                    const float bd = (gap2(L, 0, dx) + gap2(L, 1, dy)) + gap2(L, 2, dz);
                    const bool need = (L.cnt < a.K) & !(bd > a.Tskip);
                    if (__ballot(need) == 0) continue;
                }
                const bool self_here = s <= L.i && L.i < lim;
                const bool any_self = !(LDSL && BRT_PROX_SELF_SPLIT) || __ballot(self_here) != 0;
                for (uint32_t j = s; j < lim; j += kGroupU) {
                    float4 q[kGroupU];
#pragma unroll
                    for (int t = 0; t < kGroupU; ++t) q[t] = cload(cpos, (j + t < lim) ? j + t : lim - 1);
                    if (L.cnt < a.K) {
                        if (any_self)
                            test_round_any<LDSL, true, kGroupU>(a, L, j, lim - j, L.i - j, q);
                        else
                            test_round_any<LDSL, false, kGroupU>(a, L, j, lim - j, L.i - j, q);
                    }
                    if (__ballot(L.cnt < a.K) == 0) return;
                }
            }
        }
    }
}

// Vector mode: each lane walks its own canonical stream.  The nine cell ranges
// of one x-offset slab are loaded together (one memory latency per slab rather
// than two per cell).
template <bool LDSL, int G, bool SPLIT, bool PACKED>
__device__ __forceinline__ void scan_vector(const ProxArgs& a, const Seg& sg, Lane& L, I3 gp) {
    const brt_grid_params& g = sg.g;
    const uint32_t maxBodies = g.max_bodies_per_cell;
    const __amdgpu_buffer_rsrc_t rpos = float4_rsrc(a.spos, a.n);
    const __amdgpu_buffer_rsrc_t rxyz = xyz_rsrc(PACKED ? a.pxyz : nullptr, PACKED ? a.n : 0u);
    BRT_CELL_LOOP
    for (int dx = -1; dx <= 1; ++dx) {
        const int cx = gp.x + dx;
        uint32_t st[9], en[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            const int cy = gp.y + k / 3 - 1, cz = gp.z + k % 3 - 1;
            const bool ok = inGrid(cx, cy, cz, g);
            const uint32_t key = sg.cell_base + (ok ? cellKey(cx, cy, cz, g) : 0u);
            st[k] = a.cell_start[key];
            en[k] = a.cell_end[key];
            st[k] = ok ? st[k] : BRT_EMPTY_CELL;
        }
        BRT_CELL_LOOP
        for (int k = 0; k < 9; ++k) {
            const int dy = k / 3 - 1, dz = k % 3 - 1;
            const uint32_t s = st[k];
            if (s == BRT_EMPTY_CELL) continue;
            const float bd = (gap2(L, 0, dx) + gap2(L, 1, dy)) + gap2(L, 2, dz);
            if (bd > a.Tskip && interior(cx, gp.y + dy, gp.z + dz, g)) continue;
            const uint32_t e = en[k];
            uint32_t lim = (e - s) > maxBodies ? s + maxBodies : e;
            lim = lim < a.n ? lim : a.n;
            // the agent's own index is in this range only in its own (stored) cell
            const bool any_self = !SPLIT || __ballot(s <= L.i && L.i < lim) != 0;
            for (uint32_t j = s; j < lim; j += G) {
                // candidates past lim are read (zeros past n) and not taken
                float4 q[G];
                load_round<G, PACKED>(rpos, rxyz, j, q);
                if (any_self)
                    test_round_any<LDSL, true, G>(a, L, j, lim - j, L.i - j, q);
                else
                    test_round_any<LDSL, false, G>(a, L, j, lim - j, L.i - j, q);
                if (L.cnt >= a.K) return;
            }
        }
    }
}

// Flat mode (LDS round log): each lane walks its own canonical stream with its
// own cell index, so a lane that finishes a cell goes on to its next cell while
// the others are still in theirs.  The wave then runs about as many rounds as
// its longest stream needs, instead of the sum over the 27 cells of the longest
// stream in each.  The cells to visit (in the grid and not skipped) are a
// 27-bit mask computed up front; the range of a lane's next cell is loaded
// while it scans the current one.
// Bit d+1 set when coordinate c+d (d = -1, 0, 1) lies in [lo, hi].
__device__ __forceinline__ uint32_t offset_bits(int c, int lo, int hi) {
    return ((c - 1 >= lo && c - 1 <= hi) ? 1u : 0u) | ((c >= lo && c <= hi) ? 2u : 0u) |
           ((c + 1 >= lo && c + 1 <= hi) ? 4u : 0u);
}

// 27-bit masks over the cell ordinals c = 9(dx+1) + 3(dy+1) + (dz+1) from the
// per-axis offset bits: the x bits fill blocks of nine, the y bits groups of
// three in every block, the z bits one position in every group.
__device__ __forceinline__ uint32_t cells_of(uint32_t bx, uint32_t by, uint32_t bz) {
    const uint32_t x = ((bx & 1u) | ((bx & 2u) << 8) | ((bx & 4u) << 16)) * 0x1FFu;
    const uint32_t y = (((by & 1u) | ((by & 2u) << 2) | ((by & 4u) << 4)) * 7u) * 0x40201u;
    const uint32_t z = (bz * 0x49u) * 0x40201u;
    return x & y & z;
}

// The cells of the 27-neighbourhood that lie in the grid.
__device__ __forceinline__ uint32_t grid_mask(const brt_grid_params& g, I3 gp) {
    return cells_of(offset_bits(gp.x, 0, (int)g.grid_size[0] - 1), offset_bits(gp.y, 0, (int)g.grid_size[1] - 1),
                    offset_bits(gp.z, 0, (int)g.grid_size[2] - 1));
}

// The cells of the 27-neighbourhood a lane visits: in the grid, and not an
// interior cell whose box lies farther than r (same tests as the cell-by-cell
// scan, without branches).
__device__ __forceinline__ uint32_t visit_mask(const Seg& sg, const Lane& L, I3 gp, float Tskip) {
    const brt_grid_params& g = sg.g;
    const int gx = (int)g.grid_size[0], gy = (int)g.grid_size[1], gz = (int)g.grid_size[2];
    const uint32_t in_grid = grid_mask(g, gp);
    const uint32_t inner = cells_of(offset_bits(gp.x, 1, gx - 2), offset_bits(gp.y, 1, gy - 2),
                                    offset_bits(gp.z, 1, gz - 2));
    uint32_t far = 0;
#pragma unroll
    for (int c = 0; c < 27; ++c) {
        const int dx = c / 9 - 1, dy = (c / 3) % 3 - 1, dz = c % 3 - 1;
        const float bd = (gap2(L, 0, dx) + gap2(L, 1, dy)) + gap2(L, 2, dz);
        far |= bd > Tskip ? (1u << c) : 0u;
    }
    return in_grid & ~(far & inner);
}

// The cells that a lane or, where they lie in its own cell, its quad's other lanes
// visit.  The lanes of a quad then stay in step, until each has its list, and read
// the same candidates in one access, which takes the load off the memory path
// (address unit busy 75 -> 62 % of the fused kernel's time on 1M blobs, 400 -> 393 us)
// for more arithmetic (10.9 -> 12.4 k instructions per wave).  With shorter
// lists the lanes stop too early to gain: a step of 1M agents at 10 / 32 per cell
// and in blobs gains 7 / 2 / 1 % at K 32, 5 / 1 / 0 % at K 28 and loses up to 1 % at K
// 16; of 500,009 agents 7 / 4 / 2 % at K 32, of 300,007 (one wave more than the chip
// holds at once) it loses 1 / 1 / 2 %.  The list pass alone of 1M agents gains 24 / 11 /
// 6 % at K 32.
// Fused steps of long lists lose by it where the cells hold many (the waves in flight
// are fewer then): 1M agents at 10 / 32 per cell and in blobs +8 / -1 / -3 % at K 48,
// +3 / -6 / -5 % at K 64 and +2 / -6 / -5 % at K 80; the list pass alone gains or stays:
// +15 / 1 / 0 % at K 48, +13 / -3 / 0 % at K 64.
constexpr uint32_t kTogetherK = 28u;
constexpr uint32_t kTogetherFusedMax = 56u;
template <int CTRL>
__device__ __forceinline__ uint32_t visit_with(uint32_t todo, I3 gp) {
    const bool same = __builtin_amdgcn_mov_dpp(gp.x, CTRL, 0xF, 0xF, true) == gp.x &&
                      __builtin_amdgcn_mov_dpp(gp.y, CTRL, 0xF, 0xF, true) == gp.y &&
                      __builtin_amdgcn_mov_dpp(gp.z, CTRL, 0xF, 0xF, true) == gp.z;
    // a lane that is not active gives 0
    const uint32_t other = (uint32_t)__builtin_amdgcn_mov_dpp((int)todo, CTRL, 0xF, 0xF, true);
    return todo | (same ? other : 0u);
}
__device__ __forceinline__ uint32_t visit_together(uint32_t todo, I3 gp) {
    todo = visit_with<0xB1>(todo, gp);     // lanes 1,0,3,2
    return visit_with<0x4E>(todo, gp);     // lanes 2,3,0,1
}

// Takes the next cell of the mask todo: its ordinal nc (27 when none is left)
// and its cell range, whose loads are left in flight.
__device__ __forceinline__ void flat_fetch(const ProxArgs& a, const Seg& sg, I3 gp, uint32_t& todo, uint32_t& nc,
                                           uint32_t& ns, uint32_t& ne) {
    const bool any = todo != 0u;
    nc = any ? (uint32_t)__builtin_ctz(todo) : 27u;
    todo &= todo - 1u;
    const uint32_t q3 = (nc * 11u) >> 5;  // nc / 3 for nc < 27
    const uint32_t q9 = (nc * 57u) >> 9;  // nc / 9 for nc < 27
    const int dx = (int)q9 - 1, dy = (int)(q3 - 3u * q9) - 1, dz = (int)(nc - 3u * q3) - 1;
    // with no cell left the loads read cell 0 of the grid and are not used
    const uint32_t key = sg.cell_base + (any ? cellKey(gp.x + dx, gp.y + dy, gp.z + dz, sg.g) : 0u);
    ns = a.cell_start[key];
    ne = a.cell_end[key];
}

// own_start: the first sorted index of the agent's own cell.  Rounds of a cell
// start at its first index and advance by G, so the agent's own index i lies
// in the round j_self = own_start + G * floor((i - own_start) / G), in slot
// (i - own_start) mod G, and in no round of another cell.
template <int G, bool PACKED>
__device__ __forceinline__ void scan_flat(const ProxArgs& a, const Seg& sg, Lane& L, I3 gp, uint32_t own_start) {
    static_assert((G & (G - 1)) == 0, "the self round is found with a mask");
    const brt_grid_params& g = sg.g;
    const uint32_t maxBodies = g.max_bodies_per_cell;
    const __amdgpu_buffer_rsrc_t rpos = float4_rsrc(a.spos, a.n);
    const __amdgpu_buffer_rsrc_t rxyz = xyz_rsrc(PACKED ? a.pxyz : nullptr, PACKED ? a.n : 0u);
    const uint32_t ds = (L.i - own_start) & (uint32_t)(G - 1);
    const uint32_t jself = L.i - ds;
    const uint32_t smask = ~(1u << ((uint32_t)G - 1u - ds));
    uint32_t todo = visit_mask(sg, L, gp, a.Tskip);
    if (a.together) todo = visit_together(todo, gp);
    // the fetched (next) cell: ordinal nc (27: none left) and its range
    uint32_t nc = 27u, ns = BRT_EMPTY_CELL, ne = 0u;
    flat_fetch(a, sg, gp, todo, nc, ns, ne);
    uint32_t j = 0u, lim = 0u;
    bool live = true;
    while (true) {
        if (live && j >= lim) {
            if (nc == 27u) {
                live = false;
            } else {
                if (ns == BRT_EMPTY_CELL) {
                    j = 0u;
                    lim = 0u;
                } else {
                    lim = (ne - ns) > maxBodies ? ns + maxBodies : ne;
                    lim = lim < a.n ? lim : a.n;
                    j = ns;
                }
                // the old range is consumed before the next one is loaded into
                // the same registers (no copy of an in-flight load)
                __builtin_amdgcn_sched_barrier(0);
                flat_fetch(a, sg, gp, todo, nc, ns, ne);
            }
        }
        if (__ballot(live) == 0) break;
        if (live && j < lim) {
            // candidates past lim are read (zeros past n) and not taken
            float4 q[G];
            load_round<G, PACKED>(rpos, rxyz, j, q);
            log_round_flat<G>(a, L, j, lim - j, j == jself ? smask : ~0u, q);
            j += (uint32_t)G;
            if (L.cnt >= a.K) live = false;
        }
    }
}

// Row scan (sparse waves).  What bounds these waves is the VALU work and the
// memory latency spent per cell, 27 cells holding one agent each or none.  x is
// the fastest axis of the cell key, so the cells
// x-1, x, x+1 of one (y, z) row are one contiguous run of sorted agents: nine
// runs replace the 27 cells, and every range of a lane (18 12-byte loads) is in
// flight at once.  The accept bits of a run are kept in a register, candidate c
// in bit 31 - c; the lists want x outermost, so the runs' bits are split at the
// ends of their cells x-1 and x and emitted x offset by x offset.  Runs longer
// than kRowMax candidates do not fit (the wave takes another mode), nor does a
// maxBodiesPerCell limit (it would cut holes into the runs).  Measured: the list
// kernel of 4,194,304 uniform agents (one per cell, K 64) 664 -> 469 us (4,387
// -> 2,795 VALU instructions per wave).
constexpr uint32_t kRowMax = 31;
struct RowRange {
    uint32_t start;  // the run's first sorted index
    uint32_t ends;   // candidates before the end of cell x-1, of cell x, of cell x+1: 8 bits each
    __device__ __forceinline__ uint32_t len() const { return ends >> 16; }
};

typedef uint32_t vuint3 __attribute__((ext_vector_type(3)));

// mask of the first k (0..31) candidates
__device__ __forceinline__ uint32_t first_bits(uint32_t k) { return ~(0xFFFFFFFFu >> k); }

// Where a lane's rows are read: the three cells of a row from x = from (always
// inside the row), shift = how far the wanted x-1 lies beyond from (not zero at
// the grid's faces), and whether any wanted cell exists at all (the test also
// guards the saturated coordinates of far-away agents).  Needs gx >= 3.
struct RowX {
    int from, shift;
    bool any;
};
__device__ __forceinline__ RowX row_x(int x, int gx, bool alive) {
    RowX r;
    r.any = alive && x >= -1 && x <= gx;
    const int want = (r.any ? x : 1) - 1;
    r.from = want < 0 ? 0 : (want > gx - 3 ? gx - 3 : want);
    r.shift = want - r.from;
    return r;
}

// the wanted cells of a row from the three read, absent ones empty
__device__ __forceinline__ vuint3 row_shift(vuint3 v, int shift) {
    const uint32_t none = BRT_EMPTY_CELL;
    vuint3 r;
    r.x = shift == 0 ? v.x : shift == 1 ? v.y : shift == 2 ? v.z : none;
    r.y = shift == 0 ? v.y : shift == 1 ? v.z : shift == -1 ? v.x : none;
    r.z = shift == 0 ? v.z : shift == -1 ? v.y : shift == -2 ? v.x : none;
    return r;
}

__device__ __forceinline__ void load_row(const Seg& sg, I3 gp, RowX x, int dy, int dz, __amdgpu_buffer_rsrc_t rs,
                                         __amdgpu_buffer_rsrc_t re, vuint3& s, vuint3& e) {
    const int gy = (int)sg.g.grid_size[1], gz = (int)sg.g.grid_size[2];
    const bool ok = x.any && gp.y >= -dy && gp.y < gy - dy && gp.z >= -dz && gp.z < gz - dz;
    const uint32_t key = sg.cell_base + (ok ? cellKey(x.from, gp.y + dy, gp.z + dz, sg.g) : 0u);
    s = __builtin_amdgcn_raw_buffer_load_b96(rs, (int)(key * 4u), 0, 0);
    e = __builtin_amdgcn_raw_buffer_load_b96(re, (int)(key * 4u), 0, 0);
    const uint32_t none = ok ? 0u : BRT_EMPTY_CELL;
    s |= none;
    e |= none;
}

// empty cells have start = end = 0xFFFFFFFF: the least start is the run's first
// index, and end + 1 is 0 for an empty cell, so the greatest is the run's end
__device__ __forceinline__ RowRange row_range(vuint3 s, vuint3 e, uint32_t n, uint32_t& len) {
    RowRange r;
    uint32_t m = s.x < s.y ? s.x : s.y;
    r.start = m < s.z ? m : s.z;
    const uint32_t first = r.start + 1u;  // 0: the run is empty
    const uint32_t top = n + 1u;
    uint32_t ea = e.x + 1u, eb = e.y + 1u, ec = e.z + 1u;
    eb = ea > eb ? ea : eb;
    ec = eb > ec ? eb : ec;
    ec = ec < top ? ec : top;
    ea = ea < ec ? ea : ec;
    eb = eb < ec ? eb : ec;
    ea = ea > first ? ea : first;
    eb = eb > first ? eb : first;
    len = ec > first ? ec - first : 0u;
    r.start = len != 0u ? r.start : 0u;
    r.ends = (ea - first) | (eb - first) << 8 | len << 16;  // meant only for len <= kRowMax
    return r;
}

// whether the range of a cell (start, end; both BRT_EMPTY_CELL when empty) holds sorted index i
__device__ __forceinline__ bool holds(uint2 cell, uint32_t i) { return cell.x <= i && i < cell.y; }

// Words of a list's head (count first) that the row scan of a kernel without
// LDS lists stages in LDS; later entries go straight to the row.
constexpr uint32_t kHeadWords = 20u;

// Scans the nine runs of the wave's sparse lanes; put(p, j) gets every accepted
// index j with its place p in visiting order (not in order of p), and their
// number is returned in all; false (nothing done) when some run of some lane is
// too long.  own: the range of the cell the agent lies in, for the other modes.
// Every lane of the wave takes part.  NR: runs whose rounds load together.
// decided(ok): called once, by the whole wave, when it is known whether it scans.
template <bool PACKED, int NR, class Put, class Decided>
__device__ __forceinline__ bool scan_rows(const ProxArgs& a, const Seg& sg, const Lane& L, I3 gp, bool alive,
                                          uint2& own, uint32_t& all, Put&& put, Decided&& decided) {
    constexpr int NL = 4;  // rows whose ranges load together
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(a.cell_start), (short)0,
                                                                        (int)(a.cells * 4u), 0x00020000);
    const __amdgpu_buffer_rsrc_t re = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(a.cell_end), (short)0,
                                                                        (int)(a.cells * 4u), 0x00020000);
    const RowX x = row_x(gp.x, (int)sg.g.grid_size[0], alive);
    const bool any_shift = __ballot(x.shift != 0) != 0;
    vuint3 s[9], e[9];
    RowRange R[9];
    uint32_t most = 0u;
    // the agent's own row first: it tells a crowded wave for two loads
    load_row(sg, gp, x, 0, 0, rs, re, s[4], e[4]);
    if (any_shift) {
        s[4] = row_shift(s[4], x.shift);
        e[4] = row_shift(e[4], x.shift);
    }
    own = make_uint2(s[4].y, e[4].y);
    R[4] = row_range(s[4], e[4], a.n, most);
    if (__popcll(__ballot(most > a.row_occ)) >= BRT_PROX_ROW_LANES) {
        decided(false);
        return false;
    }
    // four rows at a time, to hold no more than their 24 registers
#pragma unroll
    for (int r0 = 0; r0 < 9; r0 += NL + 1) {
#pragma unroll
        for (int r = r0; r < r0 + NL; ++r)
            load_row(sg, gp, x, r / 3 - 1, r % 3 - 1, rs, re, s[r], e[r]);
        if (any_shift) {
#pragma unroll
            for (int r = r0; r < r0 + NL; ++r) {
                s[r] = row_shift(s[r], x.shift);
                e[r] = row_shift(e[r], x.shift);
            }
        }
#pragma unroll
        for (int r = r0; r < r0 + NL; ++r) {
            uint32_t len;
            R[r] = row_range(s[r], e[r], a.n, len);
            most = most > len ? most : len;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    const bool fits = __ballot(most > kRowMax) == 0;
    decided(fits);
    if (!fits) return false;

    const __amdgpu_buffer_rsrc_t rpos = float4_rsrc(a.spos, a.n);
    const __amdgpu_buffer_rsrc_t rxyz = xyz_rsrc(PACKED ? a.pxyz : nullptr, PACKED ? a.n : 0u);
    // an agent that is not sorted into the cell of its position (outside the grid, or
    // moved since the sort) is stored in a cell that any of its runs may hold
    const bool any_out = __ballot(alive && !holds(own, L.i)) != 0;
    uint32_t M[9];
#pragma unroll
    for (int r = 0; r < 9; ++r) M[r] = 0u;
    // rounds of four candidates, the loads of NR runs in flight together; a run
    // that no lane has so many candidates in is passed over
    BRT_CELL_LOOP
    for (uint32_t t0 = 0u; __ballot(most > t0) != 0; t0 += 4u) {
#pragma unroll
        for (int r0 = 0; r0 < 9; r0 += NR) {
            float4 q[NR][4];
            bool on[NR];
#pragma unroll
            for (int k = 0; k < NR; ++k) {
                if (r0 + k >= 9) continue;
                on[k] = __ballot(R[r0 + k].len() > t0) != 0;
                if (on[k]) load_round<4, PACKED>(rpos, rxyz, R[r0 + k].start + t0, q[k]);
            }
#pragma unroll
            for (int k = 0; k < NR; ++k) {
                if (r0 + k >= 9 || !on[k]) continue;
                uint32_t m = 0;
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const float rx = q[k][t].x - L.px, ry = q[k][t].y - L.py, rz = q[k][t].z - L.pz;
                    const float xx = rx * rx, yy = ry * ry, zz = rz * rz;
                    const float d2 = (xx + yy) + zz;
                    m = shift_in(m, !(d2 > a.T));
                }
                M[r0 + k] |= m << (28u - t0);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 9; ++r) {
        uint32_t keep = first_bits(R[r].len());
        if (r == 4 || any_out) {
            const uint32_t d = L.i - R[r].start;
            if (d < 32u) keep &= ~(0x80000000u >> d);
        }
        M[r] &= keep;
    }
    // the lists' order is x offset outermost, then y, then z: the entries of the
    // three x offsets go to places counted up from 0, c0 and c1, run by run
    uint32_t c0 = 0u, c1 = 0u;
    all = 0u;
#pragma unroll
    for (int r = 0; r < 9; ++r) {
        const uint32_t ma = first_bits(R[r].ends & 0xFFu), mb = first_bits((R[r].ends >> 8) & 0xFFu);
        c0 += __popc(M[r] & ma);
        c1 += __popc(M[r] & mb);
        all += __popc(M[r]);
    }
    uint32_t p0 = 0u, p1 = c0, p2 = c1;
#pragma unroll
    for (int r = 0; r < 9; ++r) {
        uint32_t m = M[r];
        const uint32_t ka = R[r].ends & 0xFFu, kb = (R[r].ends >> 8) & 0xFFu;
        while (__ballot(m != 0u) != 0) {
            if (m != 0u) {
                const uint32_t k = (uint32_t)__clz(m);
                m ^= 0x80000000u >> k;
                const bool lo = k < ka, hi = k >= kb;
                const uint32_t p = lo ? p0 : (hi ? p2 : p1);
                p0 += lo ? 1u : 0u;
                p1 += (lo || hi) ? 0u : 1u;
                p2 += hi ? 1u : 0u;
                put(p, R[r].start + k);
            }
        }
    }
    return true;
}

template <bool FUSE, bool BATCH, bool LDSL>
__global__ void __launch_bounds__(256, FUSE || LDSL ? 1 : 5) k_prox(ProxArgs a) {
    // with LDS lists blockDim.x rows of Ws words; the list-only kernel without
    // them blockDim.x heads of kHeadWords; else unused
    alignas(16) extern __shared__ uint32_t s_list[];
    constexpr bool ROWS = LDSL || !FUSE;
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u;
    const uint32_t wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t blk = xcd_block(a.xcd_remap);
    const uint32_t gw = blk * (blockDim.x >> 6) + wid;
    Seg sg;
    const bool wave_live = wave_segment<BATCH>(a, gw, sg);
    Lane L;
    L.i = sg.row0 + lane;
    L.cnt = 0;
    const bool alive = wave_live && L.i < sg.end;
    L.row = LDSL ? s_list + tid * a.Ws : a.lists + (size_t)(alive ? L.i : 0u) * a.W;
    uint32_t* const head = LDSL ? L.row : s_list + tid * kHeadWords;
    L.wp = L.row + 1u;
    L.h0 = L.h1 = L.h2 = L.b0 = L.b1 = L.b2 = BRT_LIST_PAD;
    float4 P = make_float4(0.f, 0.f, 0.f, 0.f);
    if (alive) P = a.spos[L.i];
    L.px = P.x;
    L.py = P.y;
    L.pz = P.z;
    I3 gp = calcGridPos(P.x, P.y, P.z, sg.g);
    cell_gaps(sg, L, gp);

    // fused: the agent's own state (the smoothed acceleration by agent ID when
    // there is no sorted copy), loaded before the list is finished, so that the
    // loads are in flight meanwhile
    uint32_t own_id = 0u;
    float4 own_fwd = make_float4(0.f, 0.f, 0.f, 0.f), own_sa = make_float4(0.f, 0.f, 0.f, 0.f);
    auto load_own = [&]() {
        if (!FUSE || !alive) return;
        own_id = a.hash[L.i].y;
        own_fwd = a.sfwd[L.i];
        if (a.ssa)
            own_sa = a.ssa[L.i];
        else if (own_id < a.n)
            own_sa = a.o.sa_out[own_id];
    };

    // wave-level mode choice: can the wave's lanes be covered by a few cells?
    const uint64_t alive_mask = __ballot(alive);
    uint64_t pending = alive_mask;
    uint32_t groups = 0;
    while (pending != 0 && groups < a.uniform_max_cells) {
        const int leader = __ffsll((unsigned long long)pending) - 1;
        const int ux = __builtin_amdgcn_readlane(gp.x, leader);
        const int uy = __builtin_amdgcn_readlane(gp.y, leader);
        const int uz = __builtin_amdgcn_readlane(gp.z, leader);
        pending &= ~__ballot(alive && gp.x == ux && gp.y == uy && gp.z == uz);
        ++groups;
    }
    const bool uniform = pending == 0;
    bool rows = false, have_own = false;
    uint2 own = make_uint2(0u, 0u);
    if (uniform) {
        pending = alive_mask;
        while (pending != 0) {
            const int leader = __ffsll((unsigned long long)pending) - 1;
            const int ux = __builtin_amdgcn_readlane(gp.x, leader);
            const int uy = __builtin_amdgcn_readlane(gp.y, leader);
            const int uz = __builtin_amdgcn_readlane(gp.z, leader);
            const bool mine = alive && gp.x == ux && gp.y == uy && gp.z == uz;
            pending &= ~__ballot(mine);
            if (mine) scan_uniform<LDSL>(a, sg, L, ux, uy, uz);
        }
    } else {
        const bool can = ROWS && a.cells != 0u && sg.g.max_bodies_per_cell == BRT_UNLIMITED &&
                         sg.g.grid_size[0] >= 3u;
        auto put = [&](uint32_t p, uint32_t j) {
            if (p >= a.K) return;
            // register-chunk kernels hold the head of the list in LDS
            if (LDSL || p < kHeadWords - 1u)
                head[1u + p] = j;
            else
                L.row[1u + p] = j;
        };
        // with LDS lists a third run would cost the fourth wave per SIMD (129 registers),
        // without them a second one the fifth, on which the other scans rely (300,007
        // agents, K 48, three runs and four waves -> one and five: 12 per cell 117 -> 84
        // us, in blobs 416 -> 340, at one per cell 38 -> 34)
        constexpr int NR = LDSL ? 2 : 1;
        uint32_t all = 0u;
        auto any = [](bool) {};
        rows = can && (LDSL && a.pxyz != nullptr ? scan_rows<LDSL, NR>(a, sg, L, gp, alive, own, all, put, any)
                                                 : scan_rows<false, NR>(a, sg, L, gp, alive, own, all, put, any));
        if (rows) L.cnt = all < a.K ? all : a.K;
        have_own = can && __ballot(alive && !holds(own, L.i)) == 0;
    }
    if (!rows && !uniform) {
        // the row scan has read the own cells of agents sorted into them
        // dense waves (most lanes in cells of >= 8 agents) take rounds of
        // kGroupL candidates and skip the self test outside the agent's own
        // cell; sparse waves, dominated by per-cell overhead, take the short
        // rounds of kGroupR with one code path
        bool dense = false;
        uint32_t own_start = 0;
        if (LDSL) {
            if (!have_own && alive) {
                const uint32_t key = a.hash[L.i].x;
                own = make_uint2(a.cell_start[key], a.cell_end[key]);
            }
            own_start = own.x;
            const uint32_t occ = own.y - own.x;
            dense = __popcll(__ballot(alive && occ >= (uint32_t)BRT_PROX_DENSE_OCC)) >= BRT_PROX_DENSE_LANES;
        }
        // with the packed positions a round's loads are 3G/4 instead of G
        const bool packed = a.pxyz != nullptr;
        if (LDSL && BRT_PROX_FLAT && dense && a.log_rounds) {
            if (alive) {
                if (packed)
                    scan_flat<kGroupL, true>(a, sg, L, gp, own_start);
                else
                    scan_flat<kGroupL, false>(a, sg, L, gp, own_start);
            }
        } else if (LDSL && BRT_PROX_FLAT_SPARSE && a.log_rounds) {
            if (alive) {
                if (packed)
                    scan_flat<kGroupR, true>(a, sg, L, gp, own_start);
                else
                    scan_flat<kGroupR, false>(a, sg, L, gp, own_start);
            }
        } else if (alive) {
            if (dense) {
                if (packed)
                    scan_vector<LDSL, kGroupL, BRT_PROX_SELF_SPLIT != 0, true>(a, sg, L, gp);
                else
                    scan_vector<LDSL, kGroupL, BRT_PROX_SELF_SPLIT != 0, false>(a, sg, L, gp);
            } else {
                if (packed)
                    scan_vector<LDSL, kGroupR, false, true>(a, sg, L, gp);
                else
                    scan_vector<LDSL, kGroupR, false, false>(a, sg, L, gp);
            }
        }
    }

    load_own();

    if (LDSL && a.log_rounds && !rows) expand_log(L, a.K);
    const uint32_t wave_rows = wave_live ? ((sg.end - sg.row0) < 64u ? (sg.end - sg.row0) : 64u) : 0u;
    if (LDSL) {
        L.row[0] = L.cnt;
        __syncthreads();
        store_rows<false>(a.lists, sg.row0, wave_rows, a.W, s_list + (size_t)(wid * 64u) * a.Ws, a.Ws, lane);
    } else if (ROWS && rows) {
        head[0] = L.cnt;
        // the lane's own entries past the head: their last chunk's padding
        if (alive && L.cnt >= kHeadWords)
            for (uint32_t q = L.cnt + 1u; (q & 3u) != 0u; ++q) L.row[q] = BRT_LIST_PAD;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        store_rows<true>(a.lists, sg.row0, wave_rows, a.W, s_list + (size_t)(wid * 64u) * kHeadWords, kHeadWords,
                         lane);
    } else {
        uint32_t pad_from = a.W / 4u;
        if (alive) pad_from = finish_list(L, a.W);
        if (wave_live) pad_rows(a.lists, sg.row0, wave_rows, a.W, lane, pad_from);
    }

    // fused steering: walk the finished list (from LDS, or the row this lane
    // just stored), all lanes in step with four neighbour gathers in flight,
    // then integrate.  Same order and operations as k_steer over the written
    // list.
    if (FUSE && alive) {
        const uint32_t id = own_id;
        if (id < a.n) {
            const float4 Fw = own_fwd;
            const float4 SA = own_sa;
            const V3 myPos = v3(P.x, P.y, P.z), myFwd = xyz(Fw);
            SteerAccum acc;
            acc.init();
            const Weights wts = sg.w;
            const float margin = cut_margin(myFwd);
            if (wts.s != 0.0f || wts.a != 0.0f || wts.c != 0.0f) {
                const __amdgpu_buffer_rsrc_t rpos = float4_rsrc(a.spos, a.n);
                const __amdgpu_buffer_rsrc_t rfwd = float4_rsrc(a.sfwd, a.n);
                constexpr int SG = BRT_PROX_STEER_GROUP;
                for (uint32_t t = 0; t < L.cnt; t += SG) {
                    float4 q[SG], f[SG];
#pragma unroll
                    for (int u = 0; u < SG; ++u) {
                        const uint32_t j = (t + u < L.cnt) ? L.row[1 + t + u] : L.i;
                        q[u] = bload(rpos, j * 16u);
                        f[u] = bload(rfwd, j * 16u);
                    }
#pragma unroll
                    for (int u = 0; u < SG; ++u) {
                        if (t + u < L.cnt) {
                            const V3 offset = xyz(q[u]) - myPos;
                            acc.add_cut(a.sp, a.cuts, wts, myFwd, margin, offset, dot(offset, offset), xyz(f[u]));
                        }
                    }
                }
            }
            const uint32_t step = (BATCH && a.b.step) ? *a.b.step : a.step;
            finish_agent(sg.g, a.sp, wts, a.dt, step, L.i, id, id - sg.id_base, myPos, myFwd, Fw.w, xyz(SA), SA.w,
                         acc, a.o);
        }
    }
}

// ---------------------------------------------------------------- four lanes per agent
// Small launches (up to kProxQuadMax agents) leave most SIMDs without a wave, and one wave's chain of
// instructions and memory latencies is their time.  Here a quad of lanes shares
// an agent: 16 agents per wave, 64 per workgroup, rows of W words in LDS.
//   * row scan: lanes 0..2 take the three runs of one y offset each (as
//     scan_rows; the places of a lane's entries follow from the quad's counts);
//   * else a flat scan (as scan_flat) whose rounds test 16 candidates, four per
//     lane, and write what passes straight into the row: the quad's accept bits
//     give every lane its place;
//   * steering: each lane takes every fourth entry, and the sums add the four
//     lanes' terms in list order, the same bits as one lane's; one wave of the
//     workgroup then integrates its 64 agents.

__device__ __forceinline__ V3 quad_add(V3 s, V3 v) {
    return v3(brt::quad_add(s.x, v.x), brt::quad_add(s.y, v.y), brt::quad_add(s.z, v.z));
}

// The row scan of a wave of quads (lane l = 0..3 of each); false: some run is
// too long (nothing done).  Sets L.cnt, the entries in L.row[1..].
template <bool PACKED>
__device__ __forceinline__ bool quad_rows(const ProxArgs& a, const Seg& sg, Lane& L, I3 gp, bool alive, uint32_t l) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(a.cell_start), (short)0,
                                                                        (int)(a.cells * 4u), 0x00020000);
    const __amdgpu_buffer_rsrc_t re = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(a.cell_end), (short)0,
                                                                        (int)(a.cells * 4u), 0x00020000);
    const __amdgpu_buffer_rsrc_t rpos = float4_rsrc(a.spos, a.n);
    const __amdgpu_buffer_rsrc_t rxyz = xyz_rsrc(PACKED ? a.pxyz : nullptr, PACKED ? a.n : 0u);
    const RowX x = row_x(gp.x, (int)sg.g.grid_size[0], alive && l < 3u);
    vuint3 s[3], e[3];
    RowRange R[3];
    uint32_t most = 0u;
#pragma unroll
    for (int k = 0; k < 3; ++k) load_row(sg, gp, x, (int)l - 1, k - 1, rs, re, s[k], e[k]);
    if (__ballot(x.shift != 0) != 0) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            s[k] = row_shift(s[k], x.shift);
            e[k] = row_shift(e[k], x.shift);
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        uint32_t len;
        R[k] = row_range(s[k], e[k], a.n, len);
        most = most > len ? most : len;
    }
    if (__ballot(most > kRowMax) != 0) return false;
    if (__popcll(__ballot(l == 1u && R[1].len() > a.row_occ_quad)) >= 8) return false;
    uint32_t M[3] = {0u, 0u, 0u};
    BRT_CELL_LOOP
    for (uint32_t t0 = 0u; __ballot(most > t0) != 0; t0 += 4u) {
        float4 q[3][4];
#pragma unroll
        for (int k = 0; k < 3; ++k) load_round<4, PACKED>(rpos, rxyz, R[k].start + t0, q[k]);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            uint32_t m = 0;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float rx = q[k][t].x - L.px, ry = q[k][t].y - L.py, rz = q[k][t].z - L.pz;
                const float xx = rx * rx, yy = ry * ry, zz = rz * rz;
                const float d2 = (xx + yy) + zz;
                m = shift_in(m, !(d2 > a.T));
            }
            M[k] |= m << (28u - t0);
        }
    }
    // the lane's entries of the three x offsets, 8 bits each (93 at most)
    uint32_t mine = 0u;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        uint32_t keep = first_bits(R[k].len());
        const uint32_t d = L.i - R[k].start;
        if (d < 32u) keep &= ~(0x80000000u >> d);
        M[k] &= keep;
        const uint32_t lo = first_bits(R[k].ends & 0xFFu), mid = first_bits((R[k].ends >> 8) & 0xFFu);
        mine += __popc(M[k] & lo) | __popc(M[k] & mid & ~lo) << 8 | __popc(M[k] & ~mid) << 16;
    }
    // places: x offset by x offset, in each lane by lane (lane 3 has none)
    const uint32_t c0 = quad_lane<0>(mine), c1 = quad_lane<1>(mine), c2 = quad_lane<2>(mine);
    const uint32_t n0 = (c0 & 0xFFu) + (c1 & 0xFFu) + (c2 & 0xFFu);
    const uint32_t n1 = (c0 >> 8 & 0xFFu) + (c1 >> 8 & 0xFFu) + (c2 >> 8 & 0xFFu);
    const uint32_t n2 = (c0 >> 16) + (c1 >> 16) + (c2 >> 16);
    uint32_t p0 = 0u, p1 = n0, p2 = n0 + n1;
    if (l > 0u) {
        p0 += c0 & 0xFFu;
        p1 += c0 >> 8 & 0xFFu;
        p2 += c0 >> 16;
    }
    if (l > 1u) {
        p0 += c1 & 0xFFu;
        p1 += c1 >> 8 & 0xFFu;
        p2 += c1 >> 16;
    }
    const uint32_t all = n0 + n1 + n2;
    L.cnt = all < a.K ? all : a.K;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        uint32_t m = M[k];
        const uint32_t ka = R[k].ends & 0xFFu, kb = (R[k].ends >> 8) & 0xFFu;
        while (__ballot(m != 0u) != 0) {
            if (m != 0u) {
                const uint32_t b = (uint32_t)__clz(m);
                m ^= 0x80000000u >> b;
                const bool lo = b < ka, hi = b >= kb;
                const uint32_t p = lo ? p0 : (hi ? p2 : p1);
                p0 += lo ? 1u : 0u;
                p1 += (lo || hi) ? 0u : 1u;
                p2 += hi ? 1u : 0u;
                if (p < a.K) L.row[1u + p] = R[k].start + b;
            }
        }
    }
    return true;
}

// The flat scan of quads: as scan_flat, every lane of a quad in the same cell.
template <bool PACKED>
__device__ __forceinline__ void quad_flat(const ProxArgs& a, const Seg& sg, Lane& L, I3 gp, bool alive, uint32_t l) {
    const uint32_t maxBodies = sg.g.max_bodies_per_cell;
    const __amdgpu_buffer_rsrc_t rpos = float4_rsrc(a.spos, a.n);
    const __amdgpu_buffer_rsrc_t rxyz = xyz_rsrc(PACKED ? a.pxyz : nullptr, PACKED ? a.n : 0u);
    uint32_t todo = alive ? visit_mask(sg, L, gp, a.Tskip) : 0u;
    uint32_t nc = 27u, ns = BRT_EMPTY_CELL, ne = 0u;
    flat_fetch(a, sg, gp, todo, nc, ns, ne);
    uint32_t j = 0u, lim = 0u;  // j: the quad's round
    bool live = alive;
    while (true) {
        if (live && j >= lim) {
            if (nc == 27u) {
                live = false;
            } else {
                const bool empty = ns == BRT_EMPTY_CELL;
                lim = (ne - ns) > maxBodies ? ns + maxBodies : ne;
                lim = lim < a.n ? lim : a.n;
                lim = empty ? 0u : lim;
                j = empty ? 0u : ns;
                // the old range is consumed before the next one is loaded into
                // the same registers (no copy of an in-flight load)
                __builtin_amdgcn_sched_barrier(0);
                flat_fetch(a, sg, gp, todo, nc, ns, ne);
            }
        }
        if (__ballot(live) == 0) break;
        if (live && j < lim) {
            // candidates past lim are read (zeros past n) and not taken
            const uint32_t jl = j + 4u * l;
            float4 q[4];
            load_round<4, PACKED>(rpos, rxyz, jl, q);
            uint32_t m = 0;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float rx = q[t].x - L.px, ry = q[t].y - L.py, rz = q[t].z - L.pz;
                const float xx = rx * rx, yy = ry * ry, zz = rz * rz;
                const float d2 = (xx + yy) + zz;
                m = shift_in(m, !(d2 > a.T));
            }
            // slots at or past lim, and the agent itself (candidate jl + t: bit 3 - t)
            const uint32_t left = jl < lim ? lim - jl : 0u;
            m &= left < 4u ? 0xF0u >> left : 0xFu;
            const uint32_t d = L.i - jl;
            if (d < 4u) m &= ~(8u >> d);
            // the quad's 16 bits, candidate j first
            uint32_t w = m << (12u - 4u * l);
            w |= (uint32_t)__builtin_amdgcn_mov_dpp((int)w, 0xB1, 0xF, 0xF, true);  // lanes 1,0,3,2
            w |= (uint32_t)__builtin_amdgcn_mov_dpp((int)w, 0x4E, 0xF, 0xF, true);  // lanes 2,3,0,1
            uint32_t p = L.cnt + __popc(w >> (16u - 4u * l));
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if (m & (8u >> t)) {
                    if (p < a.K) L.row[1u + p] = jl + (uint32_t)t;
                    ++p;
                }
            }
            L.cnt += __popc(w);
            j += 16u;
            if (L.cnt >= a.K) live = false;
        }
    }
    L.cnt = L.cnt < a.K ? L.cnt : a.K;
}

// Lists alone, above kQuadRowsMax agents: the chip has waves enough, and the row scan
// of quads, whose fourth lane idles, takes a third more instructions than one lane
// per agent.  So the workgroup's first wave scans the rows of all 64 agents; only
// where it cannot do the quads go on.  True: this wave is done.  (Every wave meets
// the two barriers, the first wave in scan_rows' decision; the second lets it reuse
// the word that holds the decision.)
// Not beyond K 80, whose list rows would hold a CU's LDS for one wave.
constexpr uint32_t kQuadRowsMax = 49152u;
constexpr uint32_t kQuadRowsMaxK = 80u;
__device__ __forceinline__ bool one_lane_rows(const ProxArgs& a, Seg sg, uint32_t base, uint32_t lane, uint32_t wid,
                                              uint32_t* s_list) {
    if (wid != 0u) {
        __syncthreads();
        const uint32_t rows = s_list[0];
        __syncthreads();
        return rows != 0u;
    }
    sg.row0 = base;
    Lane L;
    L.i = base + lane;
    L.row = s_list + (size_t)lane * a.W;
    const bool alive = L.i < sg.end;
    const float4 P = a.spos[alive ? L.i : a.n - 1u];
    L.px = P.x;
    L.py = P.y;
    L.pz = P.z;
    uint2 own;
    uint32_t all = 0u;
    const bool rows = scan_rows<false, 1>(
        a, sg, L, calcGridPos(P.x, P.y, P.z, sg.g), alive, own, all,
        [&](uint32_t p, uint32_t j) {
            if (p < a.K) L.row[1u + p] = j;
        },
        [&](bool ok) {
            if (lane == 0u) s_list[0] = ok ? 1u : 0u;
            __syncthreads();
            __syncthreads();
        });
    if (!rows) return false;
    L.row[0] = all < a.K ? all : a.K;
    wave_lds_sync();
    store_rows<false>(a.lists, base, sg.end - base < 64u ? sg.end - base : 64u, a.W, s_list, a.W, lane);
    return true;
}

// five waves per SIMD: 100,003 agents 46.3 -> 45.3 us a step, 131,072 in blobs 155 -> 146
// ONE: lists alone above kQuadRowsMax agents (apart, since it takes the sixth wave from
// the others: 12,883 agents, K 64, in a blob 55.2 -> 56.7 us).
template <bool FUSE, bool ONE = false>
__global__ void __launch_bounds__(256, 5) k_prox_quad(ProxArgs a) {
    alignas(16) extern __shared__ uint32_t s_list[];  // 64 rows of W words, then (fused) 64 of kQuadSumWords
    const uint32_t tid = threadIdx.x, lane = tid & 63u, l = tid & 3u;
    const uint32_t wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    Seg sg;
    wave_segment<false>(a, xcd_block(a.xcd_remap), sg);
    const uint32_t base = sg.row0;  // the workgroup's first agent
    sg.row0 += 16u * wid;
    Lane L;
    L.i = sg.row0 + (lane >> 2);
    L.cnt = 0u;
    const bool alive = L.i < sg.end;
    L.row = s_list + (size_t)(tid >> 2) * a.W;
    const float4 P = a.spos[alive ? L.i : a.n - 1u];
    V3 myFwd = v3(0.f, 0.f, 0.f);
    if (FUSE) myFwd = xyz(a.sfwd[alive ? L.i : a.n - 1u]);
    L.px = P.x;
    L.py = P.y;
    L.pz = P.z;
    const I3 gp = calcGridPos(P.x, P.y, P.z, sg.g);
    // the first wave integrates the workgroup's 64 agents, one per lane; their
    // state loads now
    const uint32_t mi = base + lane;
    uint32_t id = a.n;
    float4 mp, mf, ma = make_float4(0.f, 0.f, 0.f, 0.f);
    if (FUSE && wid == 0u && mi < sg.end) {
        id = a.hash[mi].y;
        mp = a.spos[mi];
        mf = a.sfwd[mi];
        if (a.ssa)
            ma = a.ssa[mi];
        else if (id < a.n)
            ma = a.o.sa_out[id];
    }
    const bool can = a.cells != 0u && sg.g.max_bodies_per_cell == BRT_UNLIMITED && sg.g.grid_size[0] >= 3u;
    const bool packed = a.pxyz != nullptr;
    if (ONE && can && one_lane_rows(a, sg, base, lane, wid, s_list)) return;
    const bool rows = can && (packed ? quad_rows<true>(a, sg, L, gp, alive, l)
                                     : quad_rows<false>(a, sg, L, gp, alive, l));
    if (!rows) {
        cell_gaps(sg, L, gp);
        if (packed)
            quad_flat<true>(a, sg, L, gp, alive, l);
        else
            quad_flat<false>(a, sg, L, gp, alive, l);
    }
    if (l == 0u) L.row[0] = L.cnt;
    wave_lds_sync();
    if (sg.row0 < sg.end)
        store_rows<false>(a.lists, sg.row0, sg.end - sg.row0 < 16u ? sg.end - sg.row0 : 16u, a.W,
                          s_list + (size_t)(16u * wid) * a.W, a.W, lane);
    if (!FUSE) return;

    SteerAccum acc;
    acc.init();
    const Weights wts = sg.w;
    uint32_t counts = 0u;  // of the three sums, 10 bits each
    if (alive && (wts.s != 0.0f || wts.a != 0.0f || wts.c != 0.0f)) {
        const V3 myPos = v3(P.x, P.y, P.z);
        const float margin = cut_margin(myFwd);
        const __amdgpu_buffer_rsrc_t rpos = float4_rsrc(a.spos, a.n);
        const __amdgpu_buffer_rsrc_t rfwd = float4_rsrc(a.sfwd, a.n);
        constexpr uint32_t U = 2;  // entries of a lane in flight
        for (uint32_t t = 0u; t < L.cnt; t += 4u * U) {
            float4 q[U], f[U];
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) {
                const uint32_t e = t + 4u * u + l;
                const uint32_t j = e < L.cnt ? L.row[1u + e] : L.i;
                q[u] = bload(rpos, j * 16u);
                f[u] = bload(rfwd, j * 16u);
            }
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) {
                if (__ballot(t + 4u * u < L.cnt) == 0) continue;
                SteerAccum one;
                one.init();
                if (t + 4u * u + l < L.cnt) {
                    const V3 offset = xyz(q[u]) - myPos;
                    one.add_cut(a.sp, a.cuts, wts, myFwd, margin, offset, dot(offset, offset), xyz(f[u]));
                }
                acc.sSep = quad_add(acc.sSep, one.sSep);
                acc.sAli = quad_add(acc.sAli, one.sAli);
                acc.sCoh = quad_add(acc.sCoh, one.sCoh);
                counts += one.nSep | one.nAli << 10 | one.nCoh << 20;
            }
        }
        counts = quad_lane<0>(counts) + quad_lane<1>(counts) + quad_lane<2>(counts) + quad_lane<3>(counts);
    }
    float* const sums = reinterpret_cast<float*>(s_list + 64u * a.W);
    if (l == 0u) {
        float* const d = sums + (tid >> 2) * kQuadSumWords;
        d[0] = acc.sSep.x;
        d[1] = acc.sSep.y;
        d[2] = acc.sSep.z;
        d[3] = acc.sAli.x;
        d[4] = acc.sAli.y;
        d[5] = acc.sAli.z;
        d[6] = acc.sCoh.x;
        d[7] = acc.sCoh.y;
        d[8] = acc.sCoh.z;
        d[9] = __uint_as_float(counts);
    }
    __syncthreads();
    if (wid != 0u || id >= a.n) return;
    const float* const d = sums + lane * kQuadSumWords;
    acc.sSep = v3(d[0], d[1], d[2]);
    acc.sAli = v3(d[3], d[4], d[5]);
    acc.sCoh = v3(d[6], d[7], d[8]);
    const uint32_t c = __float_as_uint(d[9]);
    acc.nSep = c & 0x3FFu;
    acc.nAli = c >> 10 & 0x3FFu;
    acc.nCoh = c >> 20;
    finish_agent(sg.g, a.sp, wts, a.dt, a.step, mi, id, id, xyz(mp), xyz(mf), mf.w, xyz(ma), ma.w, acc, a.o);
}

// KNN mode (useKnn): what a candidate does depends on every accepted one before
// it, so the accepted candidates are taken one by one, in visiting order.  Taken
// as they are found, the search for the farthest entry (K reads) ran for every
// candidate for which some lane needed it, behind one load in flight.  Here the
// accepted indices are gathered first and each lane goes through its own, the
// e-th of every lane at a time, the next one's position loading meanwhile:
//   * sparse waves: the row scan puts them in order (knn_rows), if no lane has
//     more than K + kKnnLog;
//   * else the flat scan logs accept bits, and when some lane's log is full all
//     lanes work theirs off (knn_scan); a full list's greatest distance then
//     bounds what is logged further.
// The lists, the log and the distances lie in LDS word by word across the lanes
// (no bank conflicts).  K 16, one kernel: 200,003 agents at 2 / 4 / 8 per cell
// (100,003, 200,003, 400,007) 56 -> 29 / 120 -> 73 / 430 -> 225 us, 200,003 in
// 12 blobs (up to hundreds per cell) 1.70 -> 1.03 ms.  A log of 16 or 32 words:
// 79 or 74 us at 4 per cell (below K + 24 too few waves take the rows).
// Agents per cell from which a KNN wave's rounds take 8 candidates instead of 4
// (200,003 agents at 4 per cell without the row scan: 81 -> 87 us at 8).
#ifndef BRT_KNN_DENSE_OCC
#define BRT_KNN_DENSE_OCC 3
#endif
constexpr uint32_t kKnnLog = 24u;

// What an accepted candidate does to agent L's list (k words and distances
// apart by B): appended while there is room, else it takes the place of the
// farthest entry if it is nearer than the farthest was at the last replacement.
struct KnnList {
    uint32_t* list;
    float* md;
    uint32_t B, K, cnt;
    float mx;
    // all lanes of the wave; have: this lane has candidate j at q
    __device__ __forceinline__ void add(const Lane& L, bool have, uint32_t j, float4 q) {
        const float rx = q.x - L.px, ry = q.y - L.py, rz = q.z - L.pz;
        const float xx = rx * rx, yy = ry * ry, zz = rz * rz;
        const float dist = sqrtf((xx + yy) + zz);
        bool replace = false;
        if (have) {
            if (cnt < K) {
                list[cnt * B] = j;
                md[cnt * B] = dist;
                mx = fmaxf(mx, dist);
                ++cnt;
            } else {
                replace = dist < mx;
            }
        }
        if (__ballot(replace) != 0 && replace) {
            float far = md[0];
            uint32_t at = 0u;
#pragma unroll 4
            for (uint32_t t = 1u; t < K; ++t) {
                const float d = md[t * B];
                at = far < d ? t : at;
                far = far < d ? d : far;
            }
            list[at * B] = j;
            md[at * B] = dist;
            mx = far;
        }
    }
};

// Sparse waves: the row scan puts the accepted indices into list[0..room) in
// visiting order, and each lane goes through its own, two loads ahead.  The
// first K stay where they are.  false: some run or some lane's candidates are
// too many.
__device__ __forceinline__ bool knn_rows(const ProxArgs& a, const Seg& sg, const Lane& L, I3 gp, bool alive,
                                         uint32_t room, KnnList& kl) {
    uint2 own;
    uint32_t all = 0u;
    const uint32_t B = kl.B;
    const bool can = a.cells != 0u && sg.g.max_bodies_per_cell == BRT_UNLIMITED && sg.g.grid_size[0] >= 3u;
    if (!can || !scan_rows<false, 3>(a, sg, L, gp, alive, own, all, [&](uint32_t p, uint32_t j) {
            if (p < room) kl.list[p * B] = j;
        }, [](bool) {}))
        return false;
    if (__ballot(all > room) != 0) return false;
    const __amdgpu_buffer_rsrc_t rpos = float4_rsrc(a.spos, a.n);
    auto index = [&](uint32_t e) { return e < all ? kl.list[e * B] : L.i; };
    uint32_t j = index(0u), jn = index(1u);
    float4 q = bload(rpos, j * 16u);
    for (uint32_t e = 0u; __ballot(e < all) != 0; ++e) {
        const float4 qn = bload(rpos, jn * 16u);
        const uint32_t jnn = index(e + 2u);
        kl.add(L, e < all, j, q);
        j = jn;
        jn = jnn;
        q = qn;
    }
    return true;
}

template <int G>
__device__ __forceinline__ void knn_scan(const ProxArgs& a, const Seg& sg, const Lane& L, I3 gp, bool alive,
                                         uint32_t* log, KnnList& kl) {
    const uint32_t B = kl.B;
    const uint32_t maxBodies = sg.g.max_bodies_per_cell;
    const __amdgpu_buffer_rsrc_t rpos = float4_rsrc(a.spos, a.n);
    uint32_t nw = 0u;
    float cut = a.T;  // squared distance beyond which candidates are left out
    // words of the log: first index << 8 | accept bits, or (2^24 agents and
    // more) one index each
    const bool packed = a.log_rounds != 0u;
    const uint32_t room = packed ? kKnnLog : kKnnLog - (uint32_t)G + 1u;

    auto work_off = [&]() {
        uint32_t e = 0u, m = 0u, jb = 0u;
        auto next = [&](uint32_t& j) {
            if (m == 0u && e < nw) {
                const uint32_t w = log[e * B];
                ++e;
                jb = packed ? w >> 8 : w;
                m = packed ? w & 0xFFu : 0x80u;
            }
            const bool any = m != 0u;
            const uint32_t b = 31u - __clz(any ? m : 1u);
            m = any ? m ^ (1u << b) : 0u;
            j = any ? jb + 7u - b : L.i;
            return any;
        };
        uint32_t j;
        bool have = next(j);
        float4 q = bload(rpos, j * 16u);
        while (__ballot(have) != 0) {
            uint32_t jn;
            const bool have_n = next(jn);
            const float4 qn = bload(rpos, jn * 16u);
            kl.add(L, have, j, q);
            j = jn;
            have = have_n;
            q = qn;
        }
        nw = 0u;
        // Once the list is full, an entry is only ever replaced by a nearer
        // candidate than mx, and mx is then set to one of the distances, so none
        // of these values exceeds the greatest of them now: a candidate that is
        // farther away can do nothing any more and is not logged (the margin is
        // far above the rounding of sqrtf and of the square).
        if (__ballot(kl.cnt == a.K) != 0 && kl.cnt == a.K) {
            float far = kl.mx;
#pragma unroll 4
            for (uint32_t t = 0u; t < a.K; ++t) far = fmaxf(far, kl.md[t * B]);
            cut = fminf(a.T, far * far * 1.00001f);
        }
    };

    // every cell in the grid: with positions that have moved since the sort, a
    // cell's agents can lie outside its box
    uint32_t todo = alive ? grid_mask(sg.g, gp) : 0u;
    uint32_t nc = 27u, ns = BRT_EMPTY_CELL, ne = 0u;
    flat_fetch(a, sg, gp, todo, nc, ns, ne);
    uint32_t j = 0u, lim = 0u;
    bool live = alive;
    while (true) {
        if (live && j >= lim) {
            if (nc == 27u) {
                live = false;
            } else {
                if (ns == BRT_EMPTY_CELL) {
                    j = 0u;
                    lim = 0u;
                } else {
                    lim = (ne - ns) > maxBodies ? ns + maxBodies : ne;
                    lim = lim < a.n ? lim : a.n;
                    j = ns;
                }
                __builtin_amdgcn_sched_barrier(0);  // as in scan_flat
                flat_fetch(a, sg, gp, todo, nc, ns, ne);
            }
        }
        if (__ballot(live) == 0) break;
        if (live && j < lim) {
            float4 q[G];
            load_round<G, false>(rpos, rpos, j, q);
            uint32_t m = 0u;
#pragma unroll
            for (int t = 0; t < G; ++t) {
                const float rx = q[t].x - L.px, ry = q[t].y - L.py, rz = q[t].z - L.pz;
                const float xx = rx * rx, yy = ry * ry, zz = rz * rz;
                const float d2 = (xx + yy) + zz;
                m = shift_in(m, !(d2 > cut));
            }
            const uint32_t rem = lim - j, r = rem < (uint32_t)G ? rem : (uint32_t)G, di = L.i - j;
            m &= ~((1u << ((uint32_t)G - r)) - 1u);
            if (di < (uint32_t)G) m &= ~(1u << ((uint32_t)G - 1u - di));
            m <<= 8 - G;
            if (packed) {
                if (m != 0u) {
                    log[nw * B] = (j << 8) | m;
                    ++nw;
                }
            } else {
                while (m != 0u) {
                    const uint32_t b = 31u - __clz(m);
                    m ^= 1u << b;
                    log[nw * B] = j + 7u - b;
                    ++nw;
                }
            }
            j += (uint32_t)G;
        }
        if (__ballot(nw >= room) != 0) work_off();
    }
    work_off();
}

__global__ void __launch_bounds__(64) k_neighbors_knn(ProxArgs a) {
    extern __shared__ uint32_t s_mem[];
    const uint32_t B = blockDim.x, lane = threadIdx.x;
    const uint32_t blk = xcd_block(a.xcd_remap);
    Seg sg;
    sg.g = a.g;
    sg.slack[0] = a.slack[0];
    sg.slack[1] = a.slack[1];
    sg.slack[2] = a.slack[2];
    sg.cell_base = 0;
    sg.row0 = blk * B;
    sg.end = a.n;
    uint32_t* s_log = s_mem + a.K * B;
    Lane L;
    L.i = sg.row0 + lane;
    const bool alive = L.i < a.n;
    const float4 P = a.spos[alive ? L.i : a.n - 1u];
    L.px = P.x;
    L.py = P.y;
    L.pz = P.z;
    const I3 gp = calcGridPos(P.x, P.y, P.z, sg.g);
    KnnList kl{s_mem + lane, reinterpret_cast<float*>(s_mem + (a.K + kKnnLog) * B) + lane, B, a.K, 0u, 0.0f};
    // the row scan's indices run on from the list into the log
    if (!knn_rows(a, sg, L, gp, alive, a.K + kKnnLog, kl)) {
        // rounds of 8 candidates in crowded waves, else of 4
        uint32_t occ = 0u;
        if (alive && inGrid(gp.x, gp.y, gp.z, sg.g)) {
            const uint32_t key = cellKey(gp.x, gp.y, gp.z, sg.g);
            occ = a.cell_end[key] - a.cell_start[key];
        }
        if (2 * __popcll(__ballot(occ >= (uint32_t)BRT_KNN_DENSE_OCC)) >= (int)B)
            knn_scan<8>(a, sg, L, gp, alive, s_log + lane, kl);
        else
            knn_scan<4>(a, sg, L, gp, alive, s_log + lane, kl);
    }
    const uint32_t cnt = kl.cnt;
    __syncthreads();
    s_log[lane] = cnt;
    __syncthreads();
    // 16 bytes per lane per store, consecutive across the lanes
    const uint32_t W4 = a.W / 4u, rows = (a.n - sg.row0) < B ? (a.n - sg.row0) : B;
    uint4* dst = reinterpret_cast<uint4*>(a.lists + (size_t)sg.row0 * a.W);
    for (uint32_t w = lane; w < rows * W4; w += B) {
        const uint32_t r = w / W4, c = w - r * W4, k = s_log[r];
        uint32_t v[4];
#pragma unroll
        for (uint32_t x = 0; x < 4u; ++x) {
            const uint32_t e = 4u * c + x;  // word e: entry e - 1; word 0: the count
            v[x] = e == 0u ? k : e <= k ? s_mem[(e - 1u) * B + r] : BRT_LIST_PAD;
        }
        dst[w] = make_uint4(v[0], v[1], v[2], v[3]);
    }
}

// Workgroup of the single-grid LDS-list neighbour kernels: one wave for launches
// above the four-lane kernels', so that a wave that finishes early releases its LDS
// tile at once instead of waiting for the slowest wave of a larger workgroup
// (1M-boid blob flock: 64 lanes 4-5 % faster than 256; a step of 200,003 agents at
// 1 / 16 per cell / in blobs, K 20, 90 / 118 / 204 -> 87 / 109 / 199 us); 256 lanes
// for smaller ones, halved while the tile exceeds 40 KB.
uint32_t prox_block(uint32_t W, uint32_t n) {
    uint32_t B = n > kProxQuadMax ? BRT_PROX_BLOCK_LARGE : 256u;
    while (B > 64 && (size_t)B * W * 4u > 40u * 1024u) B /= 2;
    return B;
}

// ProxArgs::row_occ: a list that fills in its first cells needs no row scan, which
// tests the candidates of all 27.  Agents of the own row (three per one in a cell) at
// which the two cost the same: 1.6 K with one lane per agent, 2 K but no fewer than
// 14 with four.  One lane, 131,072 agents at 1 / 3 / 6 per cell, cell by cell -> row
// scan, us: K 4 20 -> 16 / 20 -> 23 / 20 -> 32, K 8 22 -> 16 / 24 -> 23 / 26 -> 32, K
// 16 23 -> 17 / 30 -> 24 / 36 -> 34.  KNN lists, whose row scan holds K + 24 accepted
// candidates: about half of that.
uint32_t row_limit(const brt_prox_params& p) {
    const uint32_t K = p.max_neighbors, k = p.use_knn ? (K + kKnnLog) / 2u : K * 8u / 5u;
    return k < BRT_PROX_ROW_OCC ? k : BRT_PROX_ROW_OCC;
}
// With four lanes no limit in flocks of up to four per cell on average or 16,384
// agents, whose slowest wave sets the time: there the few waves over the limit take
// longer than the others save.  A step, no limit -> limit, us: 12,883 agents, K 8, at 3 /
// 6 per cell 23 -> 29 / 27 -> 29; 100,003 agents 52 -> 56 / 62 -> 57, K 4 51 -> 53 / 61 -> 52.
uint32_t quad_row_limit(uint32_t K, uint32_t n, uint32_t cells) {
    if (n <= 16384u || n / 4u <= cells) return 0xFFFFFFFFu;
    return 2u * K > 14u ? 2u * K : 14u;
}

template <bool FUSE>
bool launch_quad(ProxArgs a, uint32_t cells, hipStream_t s) {
    if (!prox_quad_fits(a.K, a.n, FUSE)) return false;
    a.row_occ_quad = quad_row_limit(a.K, a.n, cells);
    const auto kernel =
        !FUSE && a.n > kQuadRowsMax && a.K <= kQuadRowsMaxK ? k_prox_quad<false, true> : k_prox_quad<FUSE, false>;
    BRT_LAUNCH(kernel, dim3((a.n + 63u) / 64u), dim3(256), prox_quad_lds(a.K, FUSE), s, a);
    return true;
}

ProxArgs make_args(const brt_grid_params& g, const brt_prox_params& p, float threshold, const float4* spos,
                   const uint2* hash, const uint32_t* cell_start, const uint32_t* cell_end, uint32_t n,
                   uint32_t* lists, uint32_t uniform_max_cells, uint32_t xcd_remap, uint32_t cells, bool fused) {
    ProxArgs a{};
    a.cells = cells < (1u << 30) ? cells : 0u;  // 32-bit byte offsets
    a.row_occ = row_limit(p);
    a.g = g;
    a.K = p.max_neighbors;
    a.W = list_stride(p.max_neighbors);
    a.Ws = lds_list_stride(p.max_neighbors);
    a.n = n;
    a.T = threshold;
    // the skip threshold errs toward scanning: 1e-5 relative on d2 and a
    // per-axis widening of 1e-5 of the grid's coordinate range, both far above
    // the few-ulp rounding of positions, cell bounds and d2
    a.Tskip = threshold * 1.00001f;
    cell_slack(g, a.slack);
    a.uniform_max_cells = uniform_max_cells;
    a.xcd_remap = xcd_remap;
    a.log_rounds = n < (1u << 24) ? BRT_PROX_LOG : 0u;
    a.together = p.max_neighbors >= kTogetherK && (!fused || p.max_neighbors <= kTogetherFusedMax) ? 1u : 0u;
    a.spos = spos;
    a.hash = hash;
    a.cell_start = cell_start;
    a.cell_end = cell_end;
    a.lists = lists;
    return a;
}

}  // namespace

hipError_t launch_neighbors(const brt_grid_params& g, const brt_prox_params& p, float threshold,
                            const float4* spos, const uint2* hash, const uint32_t* cell_start,
                            const uint32_t* cell_end, uint32_t n, uint32_t* lists, uint32_t uniform_max_cells,
                            uint32_t xcd_remap, uint32_t lds_lists, bool quads, hipStream_t s, const float* pxyz) {
    const uint32_t K = p.max_neighbors;
    ProxArgs a = make_args(g, p, threshold, spos, hash, cell_start, cell_end, n, lists, uniform_max_cells, xcd_remap,
                           g.num_cells, false);
    if (p.use_knn) {
        // one wave per workgroup, fewer lanes of it where the lists need the LDS
        uint32_t B = 64;
        while (B > 8 && (size_t)B * (2u * K + kKnnLog) * 4u > 40u * 1024u) B /= 2;
        BRT_LAUNCH(k_neighbors_knn, dim3((n + B - 1) / B), dim3(B), (size_t)B * (2u * K + kKnnLog) * 4u, s, a);
        return hipGetLastError();
    }
    a.pxyz = pxyz;
    const uint32_t B = prox_block(a.Ws, n);
    if (quads && launch_quad<false>(a, g.num_cells, s)) return hipGetLastError();
    if (lds_lists)
        BRT_LAUNCH((k_prox<false, false, true>), dim3((n + B - 1) / B), dim3(B), (size_t)B * a.Ws * 4u, s, a);
    else {
        if (n >= kXcdRunMin && a.xcd_remap) a.xcd_remap = 2u;
        BRT_LAUNCH((k_prox<false, false, false>), dim3((n + 255) / 256), dim3(256), 256u * kHeadWords * 4u, s, a);
    }
    return hipGetLastError();
}

hipError_t launch_neighbors_steer(const brt_grid_params& g, const brt_prox_params& p, float threshold,
                                  const brt_steer_params& sp, float dt, uint32_t step, const float4* spos,
                                  const float4* sfwd, const float4* ssa, const uint2* hash,
                                  const uint32_t* cell_start, const uint32_t* cell_end, uint32_t n, uint32_t* lists,
                                  float2* wander, float4* pos_out, float4* fwd_out, float4* sa_out,
                                  uint32_t uniform_max_cells, uint32_t xcd_remap, uint32_t lds_lists, bool quads,
                                  hipStream_t s, const float* pxyz) {
    ProxArgs a = make_args(g, p, threshold, spos, hash, cell_start, cell_end, n, lists, uniform_max_cells, xcd_remap,
                           g.num_cells, true);
    a.pxyz = pxyz;
    a.sfwd = sfwd;
    a.ssa = ssa;
    a.sp = sp;
    a.cuts = steer_cuts(sp);
    a.dt = dt;
    a.step = step;
    a.o = AgentOut{pos_out, fwd_out, sa_out, nullptr, wander};
    const uint32_t B = prox_block(a.Ws, n);
    if (quads && launch_quad<true>(a, g.num_cells, s)) return hipGetLastError();
    if (lds_lists)
        BRT_LAUNCH((k_prox<true, false, true>), dim3((n + B - 1) / B), dim3(B), (size_t)B * a.Ws * 4u, s, a);
    else
        BRT_LAUNCH((k_prox<true, false, false>), dim3((n + 255) / 256), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_batch_neighbors_steer(const BatchView& b, uint32_t n, const brt_prox_params& p, float threshold,
                                        const brt_steer_params& sp, float dt, const float4* spos, const float4* sfwd,
                                        const float4* ssa, const uint2* hash, const uint32_t* cell_start,
                                        const uint32_t* cell_end, uint32_t* lists, float2* wander, float4* pos_out,
                                        float4* fwd_out, float4* sa_out, uint32_t block, uint32_t uniform_max_cells,
                                        uint32_t xcd_remap, uint32_t lds_lists, hipStream_t s, const float* pxyz) {
    brt_grid_params g0{};
    ProxArgs a = make_args(g0, p, threshold, spos, hash, cell_start, cell_end, n, lists, uniform_max_cells, xcd_remap,
                           b.cells, true);
    a.pxyz = pxyz;
    a.sfwd = sfwd;
    a.ssa = ssa;
    a.sp = sp;
    a.cuts = steer_cuts(sp);
    a.dt = dt;
    a.step = 0;
    a.o = AgentOut{pos_out, fwd_out, sa_out, nullptr, wander};
    a.b = b;
    const uint32_t B = block ? block : prox_block(a.Ws, 0u);
    const uint32_t wpb = B / 64u;
    if (lds_lists)
        hipLaunchKernelGGL((k_prox<true, true, true>), dim3((b.waves + wpb - 1) / wpb), dim3(B), (size_t)B * a.Ws * 4u,
                           s, a);
    else
        hipLaunchKernelGGL((k_prox<true, true, false>), dim3((b.waves + wpb - 1) / wpb), dim3(B), 0, s, a);
    return hipGetLastError();
}

}  // namespace brt
