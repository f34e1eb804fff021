// brt_envgrid.hip -- EnvGrid3D on gfx950: cell hash, stable key/ID radix sort,
// reorder of the per-agent float4 features and the cell ranges.
//
// Reference semantics:
//   genCalcHashD ........... PlugIns/EnvGrid3D/envgrid3d_kernel.cu:55-68
//   RadixSort (stable) ..... PlugIns/EnvGrid3D/radixsort.cu:50-80 (4 x 8-bit LSD passes,
//                            values = agent IDs in order, so the result is the
//                            (key, ID) lexicographic order)
//   reorderDataFloat4 ...... PlugIns/EnvGrid3D/envgrid3d_kernel.cu:110-122
//   genericFindCellStartD .. PlugIns/Proximity3D/Proximity3D_kernel.cu:54-84
//
// Design (MI355X): the sort is a onesweep LSD radix sort.  The hash kernel also
// builds the digit histograms of every pass; each pass is then ONE kernel: a tile
// of 4096 pairs ranks its keys per wave64 with 64-bit ballots (a digit "match"
// mask per lane), combines the four waves' counts in LDS, publishes its per-digit
// count and finds its global offset by decoupled look-back over the preceding
// tiles' status words, then scatters through LDS so each digit's run is written
// with consecutive addresses.  Only ceil(log2(cells)/8) passes run: keys are
// < cells, so the higher digits are all zero and cannot change a stable order.
#include "brt_device.hpp"
#include "brt_internal.hpp"
#include "brt_wave.hpp"

namespace brt {

namespace {

constexpr uint32_t kFlagAgg = 1u << 30;
constexpr uint32_t kFlagInc = 2u << 30;
constexpr uint32_t kValueMask = (1u << 30) - 1u;
// Predecessor statuses loaded together per look-back step (onesweep pass at
// 1M keys: 19.4 us with 1, 18.3 with 4, 18.4 with 8, 19.3 with 16; at 4M keys
// 46.3, 43.5, 44.6 and 48.7 us).
#ifndef BRT_SORT_LOOKBACK
#define BRT_SORT_LOOKBACK 4
#endif
constexpr int kLookback = BRT_SORT_LOOKBACK;

__device__ __forceinline__ uint32_t block_excl_scan_256(uint32_t v, uint32_t* s_tmp) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) s_tmp[wave] = x;
    __syncthreads();
    uint32_t wo = 0;
    for (int w = 0; w < wave; ++w) wo += s_tmp[w];
    __syncthreads();
    return wo + x - v;
}

// Every cell empty (start = end = BRT_EMPTY_CELL) before the reorder writes
// the occupied ones; four cells per thread with 16-byte stores where aligned.
__device__ __forceinline__ void fill_empty_cells(uint32_t* __restrict__ cell_start, uint32_t* __restrict__ cell_end,
                                                 uint32_t num_cells) {
    const uint32_t stride = gridDim.x * blockDim.x;
    const uint32_t n4 = num_cells / 4u;
    const uint4 e = make_uint4(BRT_EMPTY_CELL, BRT_EMPTY_CELL, BRT_EMPTY_CELL, BRT_EMPTY_CELL);
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride) {
        reinterpret_cast<uint4*>(cell_start)[i] = e;
        reinterpret_cast<uint4*>(cell_end)[i] = e;
    }
    for (uint32_t i = n4 * 4u + blockIdx.x * blockDim.x + threadIdx.x; i < num_cells; i += stride) {
        cell_start[i] = BRT_EMPTY_CELL;
        cell_end[i] = BRT_EMPTY_CELL;
    }
}

__global__ void __launch_bounds__(256) k_prepare(uint32_t* __restrict__ meta, uint32_t meta_words,
                                                 uint32_t* __restrict__ cell_start,
                                                 uint32_t* __restrict__ cell_end, uint32_t num_cells) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < meta_words; i += stride) meta[i] = 0u;
    if (cell_start) fill_empty_cells(cell_start, cell_end, num_cells);
}

// genCalcHashD fused with the per-pass digit histograms (and, when cell_start
// is given, the empty-cell fill).
__global__ void __launch_bounds__(256) k_hash_hist(brt_grid_params g, const float4* __restrict__ pos,
                                                   uint32_t n, uint2* __restrict__ out,
                                                   uint32_t* __restrict__ hist, SortPlan plan,
                                                   uint32_t* __restrict__ cell_start,
                                                   uint32_t* __restrict__ cell_end) {
    __shared__ uint32_t s_hist[kMaxPasses * kRadix];
    if (cell_start) fill_empty_cells(cell_start, cell_end, g.num_cells);
    for (uint32_t t = threadIdx.x; t < plan.passes * kRadix; t += blockDim.x) s_hist[t] = 0u;
    __syncthreads();
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        float4 p = pos[i];
        uint32_t key = calcGridHash(calcGridPos(p.x, p.y, p.z, g), g);
        out[i] = make_uint2(key, i);
        for (uint32_t q = 0; q < plan.passes; ++q)
            atomicAdd(&s_hist[q * kRadix + ((key >> plan.shift[q]) & ((1u << plan.nbits[q]) - 1u))], 1u);
    }
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < plan.passes * kRadix; t += blockDim.x) {
        uint32_t v = s_hist[t];
        if (v) atomicAdd(&hist[(blockIdx.x % kHistCopies) * kHistWords + t], v);
    }
}

// genCalcHashD over a batch of flocks: each wave hashes up to 64 agents of one
// flock with that flock's grid, the key offset by the flock's first global
// cell, so one stable sort orders every flock and keeps each in its own range.
__global__ void __launch_bounds__(256) k_batch_hash_hist(BatchView b, const float4* __restrict__ pos,
                                                         uint2* __restrict__ out, uint32_t* __restrict__ hist,
                                                         SortPlan plan, uint32_t* __restrict__ cell_start,
                                                         uint32_t* __restrict__ cell_end, uint32_t num_cells) {
    __shared__ uint32_t s_hist[kMaxPasses * kRadix];
    if (cell_start) fill_empty_cells(cell_start, cell_end, num_cells);
    for (uint32_t t = threadIdx.x; t < plan.passes * kRadix; t += blockDim.x) s_hist[t] = 0u;
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wstride = gridDim.x * (blockDim.x >> 6);
    for (uint32_t gw = blockIdx.x * (blockDim.x >> 6) + wid; gw < b.waves; gw += wstride) {
        const uint32_t f = __builtin_amdgcn_readfirstlane(b.wave_flock[gw]);
        const FlockDev& fd = b.flocks[f];
        const uint32_t i = fd.offset + (gw - fd.wave_base) * 64u + lane;
        if (i < fd.offset + fd.n) {
            const float4 p = pos[i];
            const uint32_t key = fd.cell_base + calcGridHash(calcGridPos(p.x, p.y, p.z, fd.g), fd.g);
            out[i] = make_uint2(key, i);
            for (uint32_t q = 0; q < plan.passes; ++q)
                atomicAdd(&s_hist[q * kRadix + ((key >> plan.shift[q]) & ((1u << plan.nbits[q]) - 1u))], 1u);
        }
    }
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < plan.passes * kRadix; t += blockDim.x) {
        uint32_t v = s_hist[t];
        if (v) atomicAdd(&hist[(blockIdx.x % kHistCopies) * kHistWords + t], v);
    }
}

__global__ void k_set_word(uint32_t* p, uint32_t v) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *p = v;
}

// Histograms of existing pairs (standalone sort); optionally copies the pairs.
__global__ void __launch_bounds__(256) k_hist(const uint2* __restrict__ in, uint2* __restrict__ copy_out,
                                              uint32_t n, uint32_t* __restrict__ hist, SortPlan plan) {
    __shared__ uint32_t s_hist[kMaxPasses * kRadix];
    for (uint32_t t = threadIdx.x; t < plan.passes * kRadix; t += blockDim.x) s_hist[t] = 0u;
    __syncthreads();
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        uint2 v = in[i];
        if (copy_out) copy_out[i] = v;
        for (uint32_t q = 0; q < plan.passes; ++q)
            atomicAdd(&s_hist[q * kRadix + ((v.x >> plan.shift[q]) & ((1u << plan.nbits[q]) - 1u))], 1u);
    }
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < plan.passes * kRadix; t += blockDim.x) {
        uint32_t v = s_hist[t];
        if (v) atomicAdd(&hist[(blockIdx.x % kHistCopies) * kHistWords + t], v);
    }
}

// One onesweep pass.  Items are held warp-striped: item k of lane l of wave w is
// element tile_base + w*64*ITEMS + k*64 + l, so (w, k, l) order is input order and
// ranking in that order keeps the sort stable.
template <int ITEMS>
__global__ void __launch_bounds__(kSortThreads) k_onesweep(const uint2* __restrict__ in, uint2* __restrict__ out,
                                                            uint32_t n, uint32_t shift, uint32_t nbits,
                                                            const uint32_t* __restrict__ ghist,
                                                            uint32_t* __restrict__ status,
                                                            uint32_t* __restrict__ tile_counter,
                                                            uint32_t* __restrict__ dev_flags,
                                                            uint32_t* __restrict__ prev_hist,
                                                            uint32_t* __restrict__ prev_counter,
                                                            uint32_t* __restrict__ prev_status) {
    constexpr int TILE = kSortThreads * ITEMS;
    __shared__ uint32_t s_tile;
    __shared__ uint32_t s_whist[4][kRadix];
    __shared__ uint32_t s_digit_start[kRadix];
    __shared__ uint32_t s_base[kRadix];
    __shared__ uint32_t s_gcount[kRadix];
    __shared__ uint32_t s_tmp[4];
    __shared__ uint2 s_items[TILE];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const uint32_t mask = (1u << nbits) - 1u;

    if (tid == 0) s_tile = atomicAdd(tile_counter, 1u);
#pragma unroll
    for (int w = 0; w < 4; ++w) s_whist[w][tid] = 0u;
    __syncthreads();
    const uint32_t tile = s_tile;
    const uint32_t wbase = tile * TILE + wave * (64 * ITEMS);
    // A tile ID past the grid means the counter did not start at zero (the
    // metadata a step relies on was not returned to zero): no tile is
    // processed out of bounds; the flag reports the wrong sort.
    if (tile >= gridDim.x) {
        if (tid == 0)
            __hip_atomic_fetch_or(dev_flags, BRT_DEVFLAG_SORT_LOOKBACK, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        return;
    }
    // the previous pass's metadata back to zero (its tiles use the same IDs)
    if (prev_status) {
        prev_status[(size_t)tile * kRadix + tid] = 0u;
        if (tile == 0u) {
#pragma unroll
            for (uint32_t c = 0; c < kHistCopies; ++c) prev_hist[c * kHistWords + tid] = 0u;
            if (tid == 0) *prev_counter = 0u;
        }
    }

    uint2 it[ITEMS];
    uint32_t rank[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        uint32_t idx = wbase + k * 64 + lane;
        it[k] = idx < n ? in[idx] : make_uint2(0u, 0u);
    }
    // this pass's global count of digit tid, summed over the histogram copies
    // while the items load, and parked in LDS (not in registers) over the
    // ranking
    {
        uint32_t gc = 0u;
#pragma unroll
        for (uint32_t c = 0; c < kHistCopies; ++c) gc += ghist[c * kHistWords + tid];
        s_gcount[tid] = gc;
    }
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const bool valid = (wbase + k * 64 + lane) < n;
        const uint32_t d = (it[k].x >> shift) & mask;
        const uint64_t vm = __ballot(valid);
        // lanes whose digit equals this lane's: the AND over the eight bits of
        // (ballot of bit b) XNOR (this lane's bit b replicated), on the two
        // 32-bit halves (bits above nbits are zero in every lane and leave the
        // mask unchanged)
        uint32_t m_lo = (uint32_t)vm, m_hi = (uint32_t)(vm >> 32);
#pragma unroll
        for (uint32_t b = 0; b < 8u; ++b) {
            const uint32_t rep = (uint32_t)((int32_t)(d << (31u - b)) >> 31);  // bit b: 0 or ~0
            const uint64_t bal = __ballot(rep != 0u);
            m_lo &= ~((uint32_t)bal ^ rep);
            m_hi &= ~((uint32_t)(bal >> 32) ^ rep);
        }
        const uint64_t m = ((uint64_t)m_hi << 32) | m_lo;
        const uint32_t cnt = __popcll(m);
        const uint32_t below = __popcll(m & lt);
        const int leader = __ffsll((unsigned long long)m) - 1;
        uint32_t prev = 0;
        if (valid) prev = s_whist[wave][d];
        __builtin_amdgcn_wave_barrier();
        if (valid && lane == leader) s_whist[wave][d] = prev + cnt;
        __builtin_amdgcn_wave_barrier();
        rank[k] = prev + below;
    }
    __syncthreads();

    // digit = tid: per-wave exclusive offsets and the tile's count
    const uint32_t c0 = s_whist[0][tid], c1 = s_whist[1][tid], c2 = s_whist[2][tid], c3 = s_whist[3][tid];
    const uint32_t tcount = c0 + c1 + c2 + c3;
    s_whist[0][tid] = 0u;
    s_whist[1][tid] = c0;
    s_whist[2][tid] = c0 + c1;
    s_whist[3][tid] = c0 + c1 + c2;
    uint32_t* my_status = status + (size_t)tile * kRadix + tid;
    if (tile == 0)
        __hip_atomic_store(my_status, kFlagInc | tcount, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
        __hip_atomic_store(my_status, kFlagAgg | tcount, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

    const uint32_t digit_start = block_excl_scan_256(tcount, s_tmp);
    const uint32_t gex = block_excl_scan_256(s_gcount[tid], s_tmp);
    s_digit_start[tid] = digit_start;

    // decoupled look-back over the preceding tiles for digit tid, kLookback
    // tiles per step: the statuses of tiles p, p-1, ..., p-kLookback+1 are
    // loaded together and taken nearest first (aggregates summed up to the
    // first inclusive prefix), so a walk over m tiles waits for about
    // m / kLookback memory latencies instead of m
    uint32_t excl = 0u;
    if (tile > 0) {
        int32_t p = (int32_t)tile - 1;
        uint32_t spins = 0;
        while (p >= 0) {
            uint32_t v[kLookback];
#pragma unroll
            for (int k = 0; k < kLookback; ++k)
                v[k] = (p - k >= 0) ? __hip_atomic_load(status + (size_t)(p - k) * kRadix + tid, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT)
                                    : kFlagInc;  // before tile 0: never reached (tile 0 is inclusive)
            uint32_t add = 0u, used = 0u;
            bool inc = false, stall = false;
#pragma unroll
            for (int k = 0; k < kLookback; ++k) {
                const uint32_t flag = v[k] & ~kValueMask;
                if (!inc && !stall) {
                    if (flag == 0u) {
                        stall = true;
                    } else {
                        add += v[k] & kValueMask;
                        used = (uint32_t)k + 1u;
                        inc = flag == kFlagInc;
                    }
                }
            }
            excl += add;
            if (inc) break;
            p -= (int32_t)used;
            if (stall) {
                // A predecessor tile has started (tile IDs are taken in start
                // order) and publishes without waiting, so this wait ends; the
                // bound only turns an impossible stall into a flagged wrong
                // result instead of a hang: the sticky device flag is raised
                // for the host to report.
                if (++spins > (1u << 24)) {
                    __hip_atomic_fetch_or(dev_flags, BRT_DEVFLAG_SORT_LOOKBACK, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_SYSTEM);
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
        }
        __hip_atomic_store(my_status, kFlagInc | (excl + tcount), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    s_base[tid] = gex + excl;
    __syncthreads();

    // local scatter into digit order, then coalesced write-out
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const bool valid = (wbase + k * 64 + lane) < n;
        if (valid) {
            const uint32_t d = (it[k].x >> shift) & mask;
            s_items[s_digit_start[d] + s_whist[wave][d] + rank[k]] = it[k];
        }
    }
    __syncthreads();
    const uint32_t tile_begin = tile * TILE;
    const uint32_t tile_n = (n - tile_begin) < (uint32_t)TILE ? (n - tile_begin) : (uint32_t)TILE;
    if (tile_n == (uint32_t)TILE) {
        // full tile: the ITEMS slots of a thread are independent, so their LDS
        // reads overlap
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            const uint32_t j = (uint32_t)(k * kSortThreads + tid);
            const uint2 v = s_items[j];
            const uint32_t d = (v.x >> shift) & mask;
            const uint32_t g = s_base[d] + (j - s_digit_start[d]);
            if (g < n) out[g] = v;
        }
    } else {
        for (uint32_t j = tid; j < tile_n; j += kSortThreads) {
            const uint2 v = s_items[j];
            const uint32_t d = (v.x >> shift) & mask;
            const uint32_t g = s_base[d] + (j - s_digit_start[d]);
            if (g < n) out[g] = v;
        }
    }
}

// ------------------------------------------------------------------ small flocks
// A sort of up to 2^17 agents is not bound by its bytes but by its chain of
// launches and latencies: a onesweep pass takes 8.3 us for one tile and 11 us
// for 25, and a flock of 100,003 needs three besides the hash and the reorder.
// Here the cells are split over up to 256 workgroups instead of the agents over
// tiles: each workgroup reads every key (4 bytes each, from its L2), takes the
// agents of its own cells into LDS, sorts them there by (cell, ID) and writes
// its part of the sorted pairs, the gathered state and the cell ranges, empty
// ones included.  Nothing passes between workgroups.  Hash + sort + reorder of
// 4,096 / 65,536 / 100,003 agents: 24.3 -> 9.6 / 31.8 -> 18.2 / 45 -> 21.8 us.
// A flock gathered in few cells would fall to few workgroups.  So a range with more
// agents than one workgroup sorts well (crowded) is cut into chunks of up to 2,047
// agents by their IDs, and workgroups whose own range is light take chunks of it too:
// which of them help with which range follows from a sample of the keys (CellShare),
// the same in every workgroup.  131,072 agents in 1 / 27 / 2,197 cells of 64^3, sorted
// pairs alone: 251 / 1170 / 192 us by the ranges' own workgroups, 61 / 72 / 80 us so
// (the radix sort: 40); the whole step 539 / 3200 / 315 -> 99 / 1172 / 155 us, with
// the radix sort and its separate passes 84 / 4828 / 151.  The sample costs up to
// 0.5 us at 130,200 evenly spread agents (17.9 -> 18.4).
// The kernel keeps no array in scratch (see emit): with 20 bytes per lane there some
// builds of it took 13 us more at every size.
constexpr uint32_t kCellThreads = 1024;
constexpr uint32_t kCellGroups = 256;   // workgroups at most, one per CU
constexpr uint32_t kCellIdBits = 17;    // agents below 2^17
constexpr uint32_t kCellsPerGroup = 4096;
constexpr uint32_t kCellCap = 4096;     // agents a workgroup sorts at a time
constexpr uint32_t kCellRankMax = 512;  // agents ranked by counting up to here, else bitonic
constexpr uint32_t kNoKey = 0x7FFFFFFFu;  // beside every key (below 2^20)
constexpr uint32_t kCellDense = 64;     // agents of a cell ranked within it up to here
// Agents that a workgroup sorts by itself if some cell holds more than kCellDense; in
// larger flocks all that it holds, since every chunk reads the keys again.  One sort of
// the range -> chunks, pairs alone: ranges of 2,214 in 16,384 agents 39 -> 36 us, 3,000
// in 3,000 40 -> 29; 2,423 in 33,194 42 -> 72, 2,877 in 65,536 44 -> 50.
__device__ __forceinline__ uint32_t cell_alone(uint32_t n) { return n <= 16384u ? 2048u : kCellCap; }
// IDs of a block; a chunk ends with the block in which it reaches as many agents
constexpr uint32_t kCellBlock = 1024;
constexpr uint32_t kCellBlocks = (1u << kCellIdBits) / kCellBlock;
constexpr uint32_t kCellSample = 1024;  // keys from which the helpers are spread,
constexpr uint32_t kCellRun = 8;        // in runs of so many
constexpr uint32_t kCellGather = 4;     // float4 arrays gathered (position, heading, acceleration, features)

__global__ void __launch_bounds__(256) k_hash_keys(brt_grid_params g, const float4* __restrict__ pos, uint32_t n,
                                                   uint32_t* __restrict__ keys) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 p = pos[i];
    keys[i] = calcGridHash(calcGridPos(p.x, p.y, p.z, g), g);
}

__global__ void __launch_bounds__(256) k_batch_hash_keys(BatchView b, const float4* __restrict__ pos,
                                                         uint32_t* __restrict__ keys) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t gw = blockIdx.x * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (gw >= b.waves) return;
    const uint32_t f = __builtin_amdgcn_readfirstlane(b.wave_flock[gw]);
    const FlockDev& fd = b.flocks[f];
    const uint32_t i = fd.offset + (gw - fd.wave_base) * 64u + lane;
    if (i >= fd.offset + fd.n) return;
    const float4 p = pos[i];
    keys[i] = fd.cell_base + calcGridHash(calcGridPos(p.x, p.y, p.z, fd.g), fd.g);
}

// Exclusive scan of one value per thread over the workgroup; total to all.
__device__ __forceinline__ uint32_t cell_group_scan(uint32_t v, uint32_t* s_wave, uint32_t& total) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o);
        if (lane >= (uint32_t)o) x += y;
    }
    __syncthreads();  // the previous use of s_wave is over
    if (lane == 63u) s_wave[wave] = x;
    __syncthreads();
    uint32_t before = 0u, all = 0u;
#pragma unroll
    for (uint32_t w = 0; w < kCellThreads / 64u; ++w) {
        const uint32_t c = s_wave[w];
        before += w < wave ? c : 0u;
        all += c;
    }
    total = all;
    return before + x - v;
}

// Sorts s_list[0..m), whose values are all different, ascending (m <= kCellCap).
// Up to kCellRankMax by counting the smaller ones, the list split between
// 1024 / m threads per value; above by a bitonic network, in which the steps
// of distance <= 64 stay within a wave and need no barrier.
__device__ __forceinline__ void cell_group_sort(uint32_t* s_list, uint32_t* s_rank, uint32_t m) {
    const uint32_t tid = threadIdx.x;
    if (m <= kCellRankMax) {
        const uint32_t m64 = (m + 63u) / 64u * 64u, parts = kCellThreads / m64;
        const uint32_t m4 = (m + 3u) / 4u, seg = (m4 + parts - 1u) / parts;
        if (tid < 4u * m4 - m) s_list[m + tid] = 0xFFFFFFFFu;
        if (tid < m64) s_rank[tid] = 0u;
        __syncthreads();
        const uint32_t part = tid / m64, e = tid - part * m64;
        if (part < parts && e < m) {
            const uint32_t mine = s_list[e];
            const uint32_t to = (part + 1u) * seg < m4 ? (part + 1u) * seg : m4;
            uint32_t c = 0u;
#pragma unroll 4
            for (uint32_t j = part * seg; j < to; ++j) {
                const uint4 v = reinterpret_cast<const uint4*>(s_list)[j];
                c += (v.x < mine ? 1u : 0u) + (v.y < mine ? 1u : 0u) + (v.z < mine ? 1u : 0u) +
                     (v.w < mine ? 1u : 0u);
            }
            if (c) atomicAdd(&s_rank[e], c);
        }
        __syncthreads();
        uint32_t v = 0u, r = 0u;
        if (tid < m) {
            v = s_list[tid];
            r = s_rank[tid];
        }
        __syncthreads();
        if (tid < m) s_list[r] = v;
        __syncthreads();
        return;
    }
    uint32_t P = 2u * kCellRankMax;
    while (P < m) P *= 2u;
    for (uint32_t t = m + tid; t < P; t += kCellThreads) s_list[t] = 0xFFFFFFFFu;
    __syncthreads();
    for (uint32_t k = 2u; k <= P; k *= 2u) {
        for (uint32_t j = k / 2u; j > 0u; j /= 2u) {
            for (uint32_t t = tid; t < P / 2u; t += kCellThreads) {
                const uint32_t i = 2u * t - (t & (j - 1u));
                const uint32_t a = s_list[i], b = s_list[i + j];
                if ((a > b) == ((i & k) == 0u)) {
                    s_list[i] = b;
                    s_list[i + j] = a;
                }
            }
            // the next step's pairs are this wave's own while its distance is <= 64
            if (j > 64u || j == 1u)
                __syncthreads();
            else
                wave_lds_sync();
        }
    }
}

// The quad of keys from i on, kNoKey from n on.
__device__ __forceinline__ uint4 key_quad(const uint32_t* __restrict__ keys, uint32_t i, uint32_t n) {
    if (i + 4u <= n) return *reinterpret_cast<const uint4*>(keys + i);
    return make_uint4(i < n ? keys[i] : kNoKey, i + 1u < n ? keys[i + 1u] : kNoKey,
                      i + 2u < n ? keys[i + 2u] : kNoKey, i + 3u < n ? keys[i + 3u] : kNoKey);
}

// f(i, rel) for every quad of keys from i on, [from, to): rel = key - c0, beyond every
// cell of the workgroup for the others.  All lanes of a wave, whose 64 quads follow
// each other; four quads of a lane load together.  from: a multiple of 4.
template <class Fn>
__device__ __forceinline__ void for_quads(const uint32_t* __restrict__ keys, uint32_t from, uint32_t to, uint32_t c0,
                                          Fn&& f) {
    for (uint32_t i0 = from + 4u * threadIdx.x; i0 - 4u * threadIdx.x < to; i0 += 16u * kCellThreads) {
        const uint4 k0 = key_quad(keys, i0, to), k1 = key_quad(keys, i0 + 4u * kCellThreads, to);
        const uint4 k2 = key_quad(keys, i0 + 8u * kCellThreads, to), k3 = key_quad(keys, i0 + 12u * kCellThreads, to);
        f(i0, make_uint4(k0.x - c0, k0.y - c0, k0.z - c0, k0.w - c0));
        f(i0 + 4u * kCellThreads, make_uint4(k1.x - c0, k1.y - c0, k1.z - c0, k1.w - c0));
        f(i0 + 8u * kCellThreads, make_uint4(k2.x - c0, k2.y - c0, k2.z - c0, k2.w - c0));
        f(i0 + 12u * kCellThreads, make_uint4(k3.x - c0, k3.y - c0, k3.z - c0, k3.w - c0));
    }
}

// ++count[r] for every r < nc of the wave's rel.  Where most are the same, those in one
// go (atomics of many lanes to one cell follow each other); the four most frequent ones
// so, at each wave, took 120 instead of 67 us for 131,072 agents in 216 cells.
__device__ __forceinline__ void wave_count(uint32_t* count, uint4 rel, uint32_t nc) {
    const uint32_t r = __builtin_amdgcn_readfirstlane(rel.x);
    if (r < nc && __popcll(__ballot(rel.x == r)) >= 32) {
        const uint32_t hits = (uint32_t)(__popcll(__ballot(rel.x == r)) + __popcll(__ballot(rel.y == r)) +
                                         __popcll(__ballot(rel.z == r)) + __popcll(__ballot(rel.w == r)));
        if ((threadIdx.x & 63u) == 0u) atomicAdd(&count[r], hits);
        rel.x = rel.x == r ? kNoKey : rel.x;
        rel.y = rel.y == r ? kNoKey : rel.y;
        rel.z = rel.z == r ? kNoKey : rel.z;
        rel.w = rel.w == r ? kNoKey : rel.w;
    }
    if (rel.x < nc) atomicAdd(&count[rel.x], 1u);
    if (rel.y < nc) atomicAdd(&count[rel.y], 1u);
    if (rel.z < nc) atomicAdd(&count[rel.z], 1u);
    if (rel.w < nc) atomicAdd(&count[rel.w], 1u);
}

// A place of *next for every lane that hits.
__device__ __forceinline__ uint32_t wave_place(uint32_t* next, bool hit) {
    const uint64_t m = __ballot(hit);
    uint32_t at = 0u;
    if (m == 0) return at;
    const int first = __ffsll((unsigned long long)m) - 1;
    if ((int)(threadIdx.x & 63u) == first) at = atomicAdd(next, (uint32_t)__popcll(m));
    at = __builtin_amdgcn_readlane(at, first);
    return at + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Who helps with the crowded ranges.  s_cnt[g] of the kCellSample sampled keys lie in
// range g; a range that seems to hold more than half of cell_alone(n) wants one helper
// per kCellBlock agents (17 samples or more, where even spreading gives 4 or fewer; so
// that few crowded ranges are left to their own workgroup by chance).
// The ranges that want none are light; the h-th light range's workgroup is the h-th
// helper, if there are so many.  One wave (lane l has the ranges 4 l .. 4 l + 3); the
// same in every workgroup.
struct CellShare {
    static constexpr uint32_t kOwn = kCellGroups / 64u;
    uint32_t wants[kOwn], wanted;  // helpers, and those of the ranges before
    uint32_t light;                // light ranges before, of 4 l on
    uint32_t lights;               // all
    __device__ __forceinline__ CellShare(const uint32_t* s_cnt, uint32_t n, uint32_t groups, uint32_t lane) {
        uint32_t sum = 0u;  // wanted helpers << 16 | light ranges
#pragma unroll
        for (uint32_t g = 0; g < kOwn; ++g) {
            const uint32_t agents = (uint32_t)((uint64_t)s_cnt[kOwn * lane + g] * n / kCellSample);
            wants[g] = agents > cell_alone(n) / 2u ? agents / kCellBlock : 0u;
            sum += wants[g] << 16 | (wants[g] == 0u && kOwn * lane + g < groups ? 1u : 0u);
        }
        uint32_t x = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o);
            if (lane >= (uint32_t)o) x += y;
        }
        lights = __builtin_amdgcn_readlane(x, 63) & 0xFFFFu;
        wanted = (x - sum) >> 16;
        light = (x - sum) & 0xFFFFu;
    }
    // of the helpers before + 0 .. before + want, those that there are
    __device__ __forceinline__ uint32_t have(uint32_t before, uint32_t want) const {
        const uint32_t end = before + want < lights ? before + want : lights;
        return end > before ? end - before : 0u;
    }
    // To one lane: the workgroups that share range g.
    __device__ __forceinline__ void shared(uint32_t g, uint32_t lane, uint32_t* s_slices) const {
        uint32_t before = wanted;
#pragma unroll
        for (uint32_t k = 0; k < kOwn; ++k) {
            if (kOwn * lane + k == g) *s_slices = 1u + have(before, wants[k]);
            before += wants[k];
        }
    }
    // To one lane, if the workgroup of range b helps: with which range, as which of
    // how many.
    __device__ __forceinline__ void help(uint32_t b, uint32_t lane, uint32_t* s_group, uint32_t* s_slice,
                                         uint32_t* s_slices) const {
        uint32_t h = light;
        bool is_light = false;
#pragma unroll
        for (uint32_t k = 0; k < kOwn; ++k) {
            if (kOwn * lane + k < b && wants[k] == 0u) ++h;
            if (kOwn * lane + k == b) is_light = wants[k] == 0u;
        }
        is_light = __ballot(is_light) != 0;
        h = __builtin_amdgcn_readlane(h, b / kOwn);
        uint32_t before = wanted;
#pragma unroll
        for (uint32_t k = 0; k < kOwn; ++k) {
            if (is_light && before <= h && h < before + wants[k]) {
                *s_group = kOwn * lane + k;
                *s_slice = 1u + h - before;
                *s_slices = 1u + have(before, wants[k]);
            }
            before += wants[k];
        }
    }
};

// Offsets of the cells c0 .. c0 + nc - 1 from their counts s_off, and, with cell_start,
// their ranges, four consecutive cells per thread at most.  The largest count of the
// thread's cells.
__device__ __forceinline__ uint32_t cell_group_offsets(uint32_t* s_off, uint32_t* s_wave, uint32_t c0, uint32_t nc,
                                                       uint32_t base, uint32_t* __restrict__ cell_start,
                                                       uint32_t* __restrict__ cell_end) {
    constexpr uint32_t E = kCellsPerGroup / kCellThreads;
    uint32_t cnt[E], sum = 0u, total, most = 0u;
#pragma unroll
    for (uint32_t k = 0; k < E; ++k) {
        const uint32_t c = threadIdx.x * E + k;
        cnt[k] = c < nc ? s_off[c] : 0u;
        sum += cnt[k];
        most = most > cnt[k] ? most : cnt[k];
    }
    uint32_t off = cell_group_scan(sum, s_wave, total);
#pragma unroll
    for (uint32_t k = 0; k < E; ++k) {
        const uint32_t c = threadIdx.x * E + k;
        if (c < nc) {
            s_off[c] = off;
            if (cell_start) {
                cell_start[c0 + c] = cnt[k] ? base + off : BRT_EMPTY_CELL;
                cell_end[c0 + c] = cnt[k] ? base + off + cnt[k] : BRT_EMPTY_CELL;
            }
        }
        off += cnt[k];
    }
    return most;
}

__global__ void __launch_bounds__(kCellThreads) k_cell_sort(const uint32_t* __restrict__ keys, uint32_t n,
                                                            uint32_t num_cells, uint32_t cells_per_group,
                                                            uint2* __restrict__ hash, ReorderArgs f,
                                                            uint32_t* __restrict__ cell_start,
                                                            uint32_t* __restrict__ cell_end) {
    // 16-byte aligned: the sort reads four values at once
    __shared__ alignas(16) uint32_t s_list[kCellCap];
    __shared__ alignas(16) uint32_t s_slot[kCellCap];
    __shared__ uint32_t s_off[kCellsPerGroup];
    __shared__ uint32_t s_rank[kCellRankMax];
    __shared__ uint32_t s_wave[kCellThreads / 64];
    __shared__ uint32_t s_cnt[kCellGroups], s_block[kCellBlocks];
    __shared__ uint32_t s_count, s_agents, s_below, s_most, s_wanted, s_group, s_slice, s_slices, s_lo, s_hi;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t alone = cell_alone(n);
    const bool spread = n > alone;  // some range may be crowded
    // this thread's key of the sample: in short runs, since IDs may be in order of place
    const uint32_t sampled = spread ? keys[tid / kCellRun * (n / (kCellSample / kCellRun)) + tid % kCellRun] : 0u;
    static_assert(kCellSample == kCellThreads, "one sampled key per thread");
    uint32_t c0 = blockIdx.x * cells_per_group;
    uint32_t nc = num_cells - c0 < cells_per_group ? num_cells - c0 : cells_per_group;

    // agent id of cell c0 + rel to sorted index g; the gathers in flight together
    // (of the compiler's own vector type: float4 structs that are loaded under a
    // condition end up in memory, 16 bytes per lane in LDS and 20 in scratch)
    auto emit = [&](uint32_t g, uint32_t rel, uint32_t id) {
        typedef float f32x4 __attribute__((ext_vector_type(4)));
        f32x4 v[kCellGather];
#pragma unroll
        for (uint32_t q = 0; q < kCellGather; ++q)
            if (q < f.count) v[q] = reinterpret_cast<const f32x4*>(f.in[q])[id];
        hash[g] = make_uint2(c0 + rel, id);
#pragma unroll
        for (uint32_t q = 0; q < kCellGather; ++q)
            if (q < f.count) reinterpret_cast<f32x4*>(f.out[q])[g] = v[q];
        if (f.xyz0) {
            float* d = f.xyz0 + 3u * (size_t)g;
            d[0] = v[0].x;
            d[1] = v[0].y;
            d[2] = v[0].z;
        }
    };
    for (uint32_t c = tid; c < nc; c += kCellThreads) s_off[c] = 0u;
    if (tid < kCellGroups) s_cnt[tid] = 0u;
    if (tid == 0u) {
        s_count = 0u;
        s_agents = 0u;
        s_below = 0u;
        s_most = 0u;
        s_wanted = 0u;
    }
    __syncthreads();

    // Every key: the number below c0, and the quads of keys that hold one of
    // this workgroup's cells (about one in n / (4 m)) into s_list, in any order.
    // Bound by the VALU work per key, so a quad's hits are sorted out later; a
    // lane has two quads loading while it tests two.
    {
        constexpr int U = 2;
        constexpr uint32_t kStep = kCellThreads * 4u * U;
        int32_t above = 0;  // minus the number of keys below c0
        bool full = false;
        auto load = [&](uint32_t i0, uint4 (&k)[U]) {
            if (i0 + 256u * U <= n) {  // the same for the whole wave
#pragma unroll
                for (int u = 0; u < U; ++u)
                    k[u] = *reinterpret_cast<const uint4*>(keys + i0 + 256u * u + 4u * lane);
                return;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t i = i0 + 256u * u + 4u * lane;
                k[u].x = i < n ? keys[i] : kNoKey;
                k[u].y = i + 1u < n ? keys[i + 1u] : kNoKey;
                k[u].z = i + 2u < n ? keys[i + 2u] : kNoKey;
                k[u].w = i + 3u < n ? keys[i + 3u] : kNoKey;
            }
        };
        auto test = [&](uint32_t i0, const uint4 (&k)[U]) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int32_t r[4] = {(int32_t)(k[u].x - c0), (int32_t)(k[u].y - c0), (int32_t)(k[u].z - c0),
                                      (int32_t)(k[u].w - c0)};
                uint32_t least = 0xFFFFFFFFu;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int32_t below = r[c] < -1 ? -1 : (r[c] > 0 ? 0 : r[c]);
                    above += below;
                    least = least < (uint32_t)r[c] ? least : (uint32_t)r[c];
                }
                // (the list is full: the range is crowded, and its keys are read again)
                if (least < nc && !full) {
                    const uint32_t at = atomicAdd(&s_count, 1u);
                    if (at < kCellCap) s_list[at] = i0 / 4u + 64u * u + lane;
                    full = at >= kCellCap;
                }
            }
        };
        uint4 k0[U], k1[U];
        uint32_t i0 = wave * (256u * U);
        load(i0, k0);
        while (i0 < n) {
            load(i0 + kStep, k1);
            test(i0, k0);
            i0 += kStep;
            if (i0 >= n) break;
            load(i0 + kStep, k0);
            test(i0, k1);
            i0 += kStep;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) above += __shfl_down(above, o);
        if (lane == 0u) atomicAdd(&s_below, (uint32_t)-above);
    }
    if (spread) {
        const uint32_t g = sampled / cells_per_group;
        if (g < kCellGroups) atomicAdd(&s_cnt[g], 1u);
    }
    __syncthreads();

    // the quads' agents into s_slot, as cell | ID, and their number per cell
    const uint32_t quads = s_count;
    if (spread && tid < kCellGroups && s_cnt[tid] > alone / 2u * kCellSample / n) s_wanted = 1u;
    if (quads <= kCellCap) {
        for (uint32_t t = tid; t < quads; t += kCellThreads) {
            const uint32_t i = 4u * s_list[t];
#pragma unroll
            for (uint32_t c = 0; c < 4u; ++c) {
                const uint32_t rel = (i + c < n ? keys[i + c] : kNoKey) - c0;
                if (rel < nc) {
                    atomicAdd(&s_off[rel], 1u);
                    const uint32_t at = atomicAdd(&s_agents, 1u);
                    if (at < kCellCap) s_slot[at] = rel << kCellIdBits | (i + c);
                }
            }
        }
    }
    __syncthreads();
    uint32_t m = s_agents, base = s_below;
    bool crowded = quads > kCellCap || m > kCellCap;
    if (!crowded) {
        const uint32_t most = cell_group_offsets(s_off, s_wave, c0, nc, base, cell_start, cell_end);
        if (most > kCellDense) s_most = 1u;  // some cell is crowded
        __syncthreads();
        if (s_most == 0u) {
            // no crowded cell: each agent to a place of its cell, then ranked among
            // the cell's agents; s_off[c] becomes the end of cell c
            for (uint32_t i = tid; i < m; i += kCellThreads) {
                const uint32_t v = s_slot[i];
                s_list[atomicAdd(&s_off[v >> kCellIdBits], 1u)] = v;
            }
            __syncthreads();
            for (uint32_t i = tid; i < m; i += kCellThreads) {
                const uint32_t v = s_list[i], rel = v >> kCellIdBits;
                const uint32_t from = rel ? s_off[rel - 1u] : 0u, to = s_off[rel];
                uint32_t r = from;
                for (uint32_t j = from; j < to; ++j) r += s_list[j] < v ? 1u : 0u;
                emit(base + r, rel, v & ((1u << kCellIdBits) - 1u));
            }
        } else if (m <= alone) {
            cell_group_sort(s_slot, s_rank, m);
            for (uint32_t i = tid; i < m; i += kCellThreads) {
                const uint32_t v = s_slot[i];
                emit(base + i, v >> kCellIdBits, v & ((1u << kCellIdBits) - 1u));
            }
        } else {
            crowded = true;
        }
    }
    if (!crowded && s_wanted == 0u) return;

    // The crowded range of this workgroup (own = 1), or a share of another's (0).
    auto work = [&](uint32_t own) __attribute__((always_inline)) {
        __syncthreads();
        if (tid == 0u) {
            s_group = blockIdx.x;
            s_slice = 0u;
            s_slices = own;
        }
        __syncthreads();
        if (wave == 0u && s_wanted != 0u) {
            const CellShare share(s_cnt, n, (num_cells + cells_per_group - 1u) / cells_per_group, lane);
            if (own != 0u)
                share.shared(blockIdx.x, lane, &s_slices);
            else
                share.help(blockIdx.x, lane, &s_group, &s_slice, &s_slices);
        }
        __syncthreads();
        const uint32_t slice = s_slice, slices = s_slices;
        if (slices == 0u) return;
        c0 = s_group * cells_per_group;
        nc = num_cells - c0 < cells_per_group ? num_cells - c0 : cells_per_group;
        for (uint32_t c = tid; c < nc; c += kCellThreads) s_off[c] = 0u;
        if (tid < kCellBlocks) s_block[tid] = 0u;
        if (tid == 0u) {
            s_agents = 0u;
            s_below = 0u;
            s_most = 0u;
        }
        __syncthreads();
        {
            uint32_t agents = 0u, below = 0u;  // of the wave
            for_quads(keys, 0u, n, c0, [&](uint32_t i, const uint4& rel) {
                wave_count(s_off, rel, nc);
                const uint32_t hits = (uint32_t)(__popcll(__ballot(rel.x < nc)) + __popcll(__ballot(rel.y < nc)) +
                                                 __popcll(__ballot(rel.z < nc)) + __popcll(__ballot(rel.w < nc)));
                below += (uint32_t)(__popcll(__ballot((int32_t)rel.x < 0)) + __popcll(__ballot((int32_t)rel.y < 0)) +
                                    __popcll(__ballot((int32_t)rel.z < 0)) + __popcll(__ballot((int32_t)rel.w < 0)));
                agents += hits;
                // a wave's quads lie in one block
                if (hits != 0u && lane == 0u) atomicAdd(&s_block[i / kCellBlock], hits);
            });
            if (lane == 0u) {
                atomicAdd(&s_agents, agents);
                atomicAdd(&s_below, below);
            }
        }
        __syncthreads();
        m = s_agents;
        base = s_below;
        const uint32_t most =
            cell_group_offsets(s_off, s_wave, c0, nc, base, slice == 0u ? cell_start : nullptr, cell_end);
        if (most > kCellDense) s_most = 1u;
        __syncthreads();
        // (the range's own workgroup has sorted it)
        if (m <= alone || (m <= kCellCap && s_most == 0u)) return;  // a helper: own ranges are crowded

        // chunks of consecutive IDs, each of at most 2 kCellBlock - 1 agents, in turn by
        // the workgroups that share the range
        // a block's chunk: the agents of the blocks before it / kCellBlock
        const uint32_t in_block = tid < kCellBlocks ? s_block[tid] : 0u;
        uint32_t sum_blocks;
        const uint32_t before_block = cell_group_scan(in_block, s_wave, sum_blocks);
        const uint32_t my_chunk = before_block / kCellBlock, chunks = (m - 1u) / kCellBlock + 1u;
        uint32_t* const s_before = s_slot;  // by cell: its agents before the chunk
        static_assert(kCellCap >= kCellsPerGroup && kCellCap >= 2u * kCellBlock, "LDS of the crowded path");
        for (uint32_t chunk = slice; chunk < chunks; chunk += slices) {
            __syncthreads();  // the chunk before is done
            for (uint32_t c = tid; c < nc; c += kCellThreads) s_before[c] = 0u;
            if (tid == 0u) {
                s_count = 0u;
                s_lo = kCellBlocks;
                s_hi = 0u;
            }
            __syncthreads();
            if (in_block != 0u && my_chunk == chunk) {
                atomicMin(&s_lo, tid);
                atomicMax(&s_hi, tid + 1u);
            }
            __syncthreads();
            const uint32_t lo = s_lo * kCellBlock, end = s_hi * kCellBlock, hi = end < n ? end : n;
            if (lo >= hi) continue;  // no block ends up in this one
            for_quads(keys, 0u, lo, c0, [&](uint32_t, const uint4& rel) { wave_count(s_before, rel, nc); });
            auto take = [&](uint32_t i, uint32_t rel) {
                const uint32_t at = wave_place(&s_count, rel < nc);
                if (rel < nc) s_list[at] = rel << kCellIdBits | i;
            };
            for_quads(keys, lo, hi, c0, [&](uint32_t i, const uint4& rel) {
                take(i, rel.x);
                take(i + 1u, rel.y);
                take(i + 2u, rel.z);
                take(i + 3u, rel.w);
            });
            __syncthreads();
            const uint32_t mm = s_count;
            cell_group_sort(s_list, s_rank, mm);
            // s_before[c]: the place of the chunk's first agent of cell c, less its index
            for (uint32_t i = tid; i < mm; i += kCellThreads) {
                const uint32_t rel = s_list[i] >> kCellIdBits;
                if (i == 0u || s_list[i - 1u] >> kCellIdBits != rel) s_before[rel] += s_off[rel] - i;
            }
            __syncthreads();
            for (uint32_t i = tid; i < mm; i += kCellThreads) {
                const uint32_t v = s_list[i], rel = v >> kCellIdBits;
                emit(base + s_before[rel] + i, rel, v & ((1u << kCellIdBits) - 1u));
            }
        }
    };
    // Both where a range is crowded that the sample shows light: its workgroup is
    // counted on as a helper.  (Twice in the code and not in a loop: what the compiler
    // moves before the loop takes 0.4 us of the flocks without crowded ranges.)
    if (crowded) work(1u);
    if (s_wanted != 0u) work(0u);
}

// reorderDataFloat4 for every feature + cell start/end of the sorted keys.
// With cleanup, the sort's last pass's metadata goes back to zero as well.
__global__ void __launch_bounds__(256) k_reorder_ranges(const uint2* __restrict__ hash, uint32_t n, ReorderArgs f,
                                                        uint32_t num_cells, uint32_t* __restrict__ cell_start,
                                                        uint32_t* __restrict__ cell_end, SortCleanup cleanup) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (cleanup.hist) {
        const uint32_t stride = gridDim.x * blockDim.x;
        for (uint32_t w = i; w < cleanup.status_words; w += stride) cleanup.status[w] = 0u;
        for (uint32_t w = i; w < kHistCopies * kRadix; w += stride)
            cleanup.hist[(w / kRadix) * kHistWords + (w % kRadix)] = 0u;
        if (i == 0) *cleanup.counter = 0u;
    }
    if (i >= n) return;
    const uint2 h = hash[i];
    if (h.y < n) {
        for (uint32_t q = 0; q < f.count; ++q) {
            const float4 v = f.in[q][h.y];
            f.out[q][i] = v;
            if (q == 0 && f.xyz0) {
                float* d = f.xyz0 + 3u * (size_t)i;
                d[0] = v.x;
                d[1] = v.y;
                d[2] = v.z;
            }
        }
    }
    if (cell_start && h.x < num_cells) {
        if (i == 0 || hash[i - 1].x != h.x) cell_start[h.x] = i;
        if (i == n - 1 || hash[i + 1].x != h.x) cell_end[h.x] = i + 1;
    }
}

// k_reorder_ranges from records of four float4 by ID (k_pack's), one lane per
// part: the four lanes of an agent read its 64 bytes together.
__global__ void __launch_bounds__(256) k_reorder_records(const uint2* __restrict__ hash, uint32_t n,
                                                         const float4* __restrict__ rec, ReorderArgs f,
                                                         uint32_t num_cells, uint32_t* __restrict__ cell_start,
                                                         uint32_t* __restrict__ cell_end, SortCleanup cleanup) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, i = t >> 2, p = t & 3u;
    if (cleanup.hist) {
        const uint32_t stride = gridDim.x * blockDim.x;
        for (uint32_t w = t; w < cleanup.status_words; w += stride) cleanup.status[w] = 0u;
        for (uint32_t w = t; w < kHistCopies * kRadix; w += stride)
            cleanup.hist[(w / kRadix) * kHistWords + (w % kRadix)] = 0u;
        if (t == 0) *cleanup.counter = 0u;
    }
    if (i >= n) return;
    const uint2 h = hash[i];
    if (p < f.count && h.y < n) {
        const float4 v = rec[4u * (size_t)h.y + p];
        float4* const out = p == 0u ? f.out[0] : (p == 1u ? f.out[1] : (p == 2u ? f.out[2] : f.out[3]));
        out[i] = v;
        if (p == 0u && f.xyz0) {
            float* d = f.xyz0 + 3u * (size_t)i;
            d[0] = v.x;
            d[1] = v.y;
            d[2] = v.z;
        }
    }
    if (p == 3u && h.x < num_cells) {
        if (i == 0 || hash[i - 1].x != h.x) cell_start[h.x] = i;
        if (i == n - 1 || hash[i + 1].x != h.x) cell_end[h.x] = i + 1;
    }
}

// Workgroups of the histogram kernels: each adds its per-workgroup histograms
// of every pass into one of the kHistCopies global copies, one atomic per
// nonzero bin.  With a single copy the contended atomics set the kernel's time
// (1M agents: 12.5 us with 256 workgroups against 24.6 us with 1024); spread
// over 8 copies they no longer do, and 1024 workgroups (capped at one per
// 256 keys) measured fastest (1M agents: 8.6 us; 4M: 24.8 us, from 38.7).
#ifndef BRT_HIST_BLOCKS
#define BRT_HIST_BLOCKS 1024u
#endif
inline uint32_t hist_blocks(uint32_t) { return BRT_HIST_BLOCKS; }

inline uint32_t grid_for(uint32_t n, uint32_t block, uint32_t cap) {
    uint32_t g = (n + block - 1) / block;
    if (g < 1) g = 1;
    return g < cap ? g : cap;
}

}  // namespace

SortPlan make_sort_plan(uint32_t n, uint32_t num_cells, uint32_t items) {
    SortPlan p{};
    p.items = items == 8u ? 8u : 16u;
    uint32_t bits = 0;
    while (bits < 32 && ((num_cells - 1u) >> bits)) ++bits;
    p.passes = (bits + 7u) / 8u;
    for (uint32_t q = 0; q < p.passes; ++q) {
        p.shift[q] = 8u * q;
        p.nbits[q] = (bits - 8u * q) < 8u ? (bits - 8u * q) : 8u;
    }
    const uint32_t tile = kSortThreads * p.items;
    p.tiles = (n + tile - 1) / tile;
    return p;
}

size_t sort_meta_words(const SortPlan& p) {
    return (size_t)kMetaStatus + (size_t)p.passes * p.tiles * kRadix;
}

SortCleanup sort_cleanup(uint32_t* meta, const SortPlan& plan) {
    SortCleanup c{};
    if (!meta || plan.passes == 0u) return c;
    const uint32_t last = plan.passes - 1u;
    c.hist = meta + kMetaHist + last * kRadix;
    c.counter = meta + kMetaCounters + last;
    c.status = meta + kMetaStatus + (size_t)last * plan.tiles * kRadix;
    c.status_words = plan.tiles * kRadix;
    return c;
}

LaunchMark& launch_mark() {
    static thread_local LaunchMark m;
    return m;
}

hipError_t launch_prepare(uint32_t* meta, size_t meta_words, uint32_t* cell_start, uint32_t* cell_end,
                          uint32_t num_cells, hipStream_t s) {
    size_t work = meta_words > (size_t)num_cells / 4 ? meta_words : (size_t)num_cells / 4;
    uint32_t grid = grid_for((uint32_t)(work > 0xFFFFFFFFull ? 0xFFFFFFFFu : work), 256, 2048);
    BRT_LAUNCH(k_prepare, dim3(grid), dim3(256), 0, s, meta, (uint32_t)meta_words, cell_start, cell_end, num_cells);
    return hipGetLastError();
}

hipError_t launch_hash_hist(const brt_grid_params& g, const float4* pos, uint32_t n, uint2* out, uint32_t* meta,
                            const SortPlan& plan, hipStream_t s, uint32_t* cell_start, uint32_t* cell_end) {
    uint32_t grid = grid_for(n, 256, hist_blocks(n));
    BRT_LAUNCH(k_hash_hist, dim3(grid), dim3(256), 0, s, g, pos, n, out, meta + kMetaHist, plan, cell_start,
               cell_start ? cell_end : nullptr);
    return hipGetLastError();
}

hipError_t launch_batch_hash_hist(const BatchView& b, const float4* pos, uint2* out, uint32_t* meta,
                                  const SortPlan& plan, hipStream_t s, uint32_t* cell_start, uint32_t* cell_end,
                                  uint32_t num_cells) {
    uint32_t grid = grid_for(b.waves, 4, hist_blocks(b.waves * 64u));
    hipLaunchKernelGGL(k_batch_hash_hist, dim3(grid), dim3(256), 0, s, b, pos, out, meta + kMetaHist, plan,
                       cell_start, cell_start ? cell_end : nullptr, num_cells);
    return hipGetLastError();
}

hipError_t launch_set_word(uint32_t* p, uint32_t v, hipStream_t s) {
    hipLaunchKernelGGL(k_set_word, dim3(1), dim3(64), 0, s, p, v);
    return hipGetLastError();
}

hipError_t launch_hist(const uint2* in, uint2* copy_out, uint32_t n, uint32_t* meta, const SortPlan& plan,
                       hipStream_t s) {
    uint32_t grid = grid_for(n, 256, hist_blocks(n));
    hipLaunchKernelGGL(k_hist, dim3(grid), dim3(256), 0, s, in, copy_out, n, meta + kMetaHist, plan);
    return hipGetLastError();
}

// Cells per workgroup of the small-flock sort; 0: the radix sort takes the flock.
// The limits: IDs of 17 bits beside the cell, 4,096 cells per workgroup, and an
// average of at most 1,024 agents per workgroup (few cells leave few workgroups).
uint32_t cell_sort_cells(uint32_t n, uint32_t num_cells) {
    if (n == 0u || n > (1u << kCellIdBits) || num_cells > kCellGroups * kCellsPerGroup) return 0u;
    const uint32_t per = (num_cells + kCellGroups - 1u) / kCellGroups;
    const uint32_t groups = (num_cells + per - 1u) / per;
    return n <= 1024u * groups ? per : 0u;
}

hipError_t launch_hash_keys(const brt_grid_params& g, const float4* pos, uint32_t n, uint32_t* keys, hipStream_t s) {
    BRT_LAUNCH(k_hash_keys, dim3((n + 255) / 256), dim3(256), 0, s, g, pos, n, keys);
    return hipGetLastError();
}

hipError_t launch_batch_hash_keys(const BatchView& b, const float4* pos, uint32_t* keys, hipStream_t s) {
    hipLaunchKernelGGL(k_batch_hash_keys, dim3((b.waves + 3) / 4), dim3(256), 0, s, b, pos, keys);
    return hipGetLastError();
}

hipError_t launch_cell_sort(const uint32_t* keys, uint32_t n, uint32_t num_cells, uint2* hash, const ReorderArgs& f,
                            uint32_t* cell_start, uint32_t* cell_end, hipStream_t s) {
    const uint32_t per = cell_sort_cells(n, num_cells);
    if (per == 0u || f.count > kCellGather || (f.xyz0 && f.count == 0u)) return hipErrorInvalidValue;
    const uint32_t groups = (num_cells + per - 1u) / per;
    BRT_LAUNCH(k_cell_sort, dim3(groups), dim3(kCellThreads), 0, s, keys, n, num_cells, per, hash, f, cell_start,
               cell_end);
    return hipGetLastError();
}

hipError_t launch_onesweep(const uint2* in, uint2* out, uint32_t n, uint32_t pass, const SortPlan& plan,
                           uint32_t* meta, uint32_t* dev_flags, hipStream_t s) {
    uint32_t* status = meta + kMetaStatus + (size_t)pass * plan.tiles * kRadix;
    uint32_t* prev_hist = pass ? meta + kMetaHist + (pass - 1u) * kRadix : nullptr;
    uint32_t* prev_counter = pass ? meta + kMetaCounters + (pass - 1u) : nullptr;
    uint32_t* prev_status = pass ? status - (size_t)plan.tiles * kRadix : nullptr;
    if (plan.items == 8u)
        BRT_LAUNCH(k_onesweep<8>, dim3(plan.tiles), dim3(kSortThreads), 0, s, in, out, n, plan.shift[pass],
                   plan.nbits[pass], meta + kMetaHist + pass * kRadix, status, meta + kMetaCounters + pass, dev_flags,
                   prev_hist, prev_counter, prev_status);
    else
        BRT_LAUNCH(k_onesweep<16>, dim3(plan.tiles), dim3(kSortThreads), 0, s, in, out, n, plan.shift[pass],
                   plan.nbits[pass], meta + kMetaHist + pass * kRadix, status, meta + kMetaCounters + pass, dev_flags,
                   prev_hist, prev_counter, prev_status);
    return hipGetLastError();
}

hipError_t launch_reorder_ranges(const uint2* hash, uint32_t n, const ReorderArgs& f, uint32_t num_cells,
                                 uint32_t* cell_start, uint32_t* cell_end, hipStream_t s, const SortCleanup* cleanup) {
    const SortCleanup c = cleanup ? *cleanup : SortCleanup{};
    uint32_t work = n;
    if (c.hist && work < c.status_words) work = c.status_words;
    if (c.hist && work < kHistCopies * kRadix) work = kHistCopies * kRadix;
    uint32_t grid = (work + 255) / 256;
    if (grid == 0) return hipSuccess;
    if (f.records) {
        BRT_LAUNCH(k_reorder_records, dim3((unsigned)(((size_t)n * 4u + 255u) / 256u)), dim3(256), 0, s, hash, n,
                   f.records, f, num_cells, cell_start, cell_end, c);
        return hipGetLastError();
    }
    BRT_LAUNCH(k_reorder_ranges, dim3(grid), dim3(256), 0, s, hash, n, f, num_cells, cell_start, cell_end, c);
    return hipGetLastError();
}

}  // namespace brt
