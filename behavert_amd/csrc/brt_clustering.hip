// brt_clustering.hip -- BehaviorClustering's similarity and cluster-steering
// kernels on gfx950.
//
// Reference semantics:
//   computeSimilarity(FromTex) ....... PlugIns/BehaviorClustering/BehaviorClustering_resources.cu:156-198
//   updateSimilarityStats ............ BehaviorClustering_resources.cu:84-150
//   interpolateSimilarity ............ BehaviorClustering_resources.cu:61-80
//   computeNeighNaiveSimilarities .... BehaviorClustering_kernel.cu:306-353
//   computeAdaptiveSimilarities ...... BehaviorClustering_kernel.cu:438-497
//   steerForClusterCohesion/Alignment  BehaviorClustering_resources.cu:282-384
//   xxxsteerForSeek/Flee ............. PlugIns/OpenSteerWrapper/OpenSteerWrapper_resources.cu:294-322
// The reference's pipeline (BehaviorClusteringPlugIn::steerForClustering,
// BehaviorClusteringPlugIn.h:737-817) runs the naive similarities, then the
// adaptive pass over them, then the two steering kernels.  Here the naive and
// adaptive passes are one kernel: the adaptive pass consumes each naive value
// once, in list order, so fusing them changes no bit.
//
// One lane per sorted agent.  The agent's own feature vector is held in
// registers; a neighbour's is gathered by ID.  Sums run in the reference's
// order (k = 0..F-1 for the dot products, list order for the forces), with
// one rounding per operation (-ffp-contract=off).
#include "brt_device.hpp"
#include "brt_internal.hpp"
#include "brt_lists.hpp"

namespace brt {

namespace {

// cutil_math clamp(f, a, b) = fmaxf(a, fminf(f, b))
__device__ __forceinline__ float cclamp(float f, float a, float b) { return fmaxf(a, fminf(f, b)); }

__device__ __forceinline__ float linear_interp(float x, float xa, float ya, float xb, float yb) {
    return ya * ((x - xb) / (xa - xb)) + yb * ((x - xa) / (xb - xa));
}

// the line through (avg, 0.5) and (mx, 1) above avg, through (mn, 0) and (avg,
// 0.5) below, evaluated once on selected operands
__device__ __forceinline__ float interpolate_similarity(float v, float mn, float avg, float mx) {
    const bool up = v > avg;
    return cclamp(linear_interp(v, up ? avg : mn, up ? 0.5f : 0.0f, up ? mx : avg, up ? 1.0f : 0.5f), 0.0f, 1.0f);
}

__device__ __forceinline__ float4 update_similarity_stats(float sim, float4 st, const brt_bc_params& bc) {
    float mn = st.x, avg = st.y, mx = st.z;
    const float ctrl = bc.avg_similarity_controller;
    const float blend = sim * ctrl + ((mx + mn) / 2.0f) * (1.0f - ctrl);
    avg = avg + (blend - st.y) * bc.stats_params[0];
    avg = cclamp(avg, 0.0f, 1.0f);
    if (sim < mn) {
        mn = mn + (sim - mn) * bc.stats_params[1];
        if (mn > avg) mn = cclamp(mn, 0.0f, sim);
    } else if (mn < avg) {
        mn = mn + bc.stats_params[2];
    }
    if (sim > mx) {
        mx = mx + (sim - mx) * bc.stats_params[1];
        if (mx < avg) mx = cclamp(mx, sim, 1.0f);
    } else if (mx > avg) {
        mx = mx - bc.stats_params[2];
    }
    st.x = mn;
    st.y = avg;
    st.z = mx;
    return st;
}

// Features gathered from agent-ID order into sorted order, padded with zeros
// to FQ float4 per agent, and each agent's feature norm sqrtf(sum_k f_k^2)
// (k ascending, as the reference's computeSimilarity accumulates it,
// BehaviorClustering_resources.cu:156-198).  Neighbours are near each other in
// sorted order, so the similarity pass then reads them with L2 locality and
// without the sorted->ID indirection.
// vec: F is a multiple of 4 and `features` 16-byte aligned, so each row is
// read as float4s.
__global__ void __launch_bounds__(256) k_bc_sort_features(uint32_t F, uint32_t FQ, uint32_t n, uint32_t vec,
                                                          const uint2* __restrict__ hash,
                                                          const float* __restrict__ features,
                                                          float4* __restrict__ sfeat, float* __restrict__ norms) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t id = hash[i].y;
    float4* out = sfeat + (size_t)i * FQ;
    if (id >= n) {
        for (uint32_t q = 0; q < FQ; ++q) out[q] = make_float4(0.f, 0.f, 0.f, 0.f);
        norms[i] = 0.0f;
        return;
    }
    const float* f = features + (size_t)id * F;
    float acc = 0.0f;
    for (uint32_t q = 0; q < FQ; ++q) {
        float v[4];
        if (vec) {
            const float4 x = reinterpret_cast<const float4*>(f)[q];
            v[0] = x.x;
            v[1] = x.y;
            v[2] = x.z;
            v[3] = x.w;
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = 4u * q + c < F ? f[4u * q + c] : 0.0f;
        }
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (4u * q + c < F) acc = acc + v[c] * v[c];
        out[q] = make_float4(v[0], v[1], v[2], v[3]);
    }
    norms[i] = sqrtf(acc);
}

// The similarity of agent i (own features `mine`, norm n1) to a gathered
// neighbour: (d / (n1 * n2) + 1) / 2 with d summed over k < F in order.
template <int FQ>
__device__ __forceinline__ float naive_similarity(const float4 (&mine)[FQ], const float4 (&other)[FQ], uint32_t F,
                                                  float n1, float n2) {
    float d = 0.0f;
#pragma unroll
    for (int q = 0; q < FQ; ++q) {
        const float a[4] = {mine[q].x, mine[q].y, mine[q].z, mine[q].w};
        const float b[4] = {other[q].x, other[q].y, other[q].z, other[q].w};
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if ((uint32_t)(4 * q + c) < F) d = d + a[c] * b[c];
    }
    return (d / (n1 * n2) + 1.0f) / 2.0f;
}

// Cluster cohesion + alignment accumulators (steerForClusterCohesion/Alignment,
// BehaviorClustering_resources.cu:282-384).  seek and flee share the truncated
// offset: myPos - p = -(p - myPos) and truncateLength(-v) = -truncateLength(v)
// exactly, so flee = (-t) - v is the reference's flee to the bit.
struct ClusterAccum {
    V3 coh, ali;
    __device__ __forceinline__ void init() {
        coh = v3(0.f, 0.f, 0.f);
        ali = coh;
    }
    __device__ __forceinline__ void add(V3 myPos, V3 vel, float maxSpeed, V3 op, V3 of, float sim) {
        const V3 t = truncateLength(op - myPos, maxSpeed);
        const V3 seek = t - vel;
        const V3 flee = v3(-t.x, -t.y, -t.z) - vel;
        coh = coh + (seek * sim + flee * (1.0f - sim));
        ali = ali + of * sim;
    }
    // force_out = a + (c + force_in), the blend order of the two kernels
    __device__ __forceinline__ float4 finish(uint32_t count, V3 myFwd, const brt_bc_params& bc, float4 f0) const {
        V3 c = coh, a = ali;
        if (count > 0) {
            c = normalize(c / (float)count) * bc.cluster_weight;
            a = normalize(a / (float)count - myFwd) * bc.alignment_weight;
        }
        const V3 f1 = c + xyz(f0);
        const V3 f2 = a + f1;
        return make_float4(f2.x, f2.y, f2.z, 0.0f);
    }
};

// LDS of a wave: the list rows, overwritten in place by the similarities (slot t
// at word t, entry t + 1's word once it is read), for rows of up to kStageWords
// words, else only the similarities; and, with the cluster steering, the tile that
// the records' parts change lanes in.
constexpr uint32_t kTileChunks = 4u * 65u;  // float4; the 65: no bank conflicts
inline __host__ __device__ uint32_t similarity_row_words(uint32_t K, uint32_t W) {
    return W <= kStageWords ? W : K + 1u;
}
inline uint32_t similarity_wave_bytes(uint32_t K, uint32_t W) {
    return ((64u * similarity_row_words(K, W) * 4u + 15u) / 16u + kTileChunks) * 16u;
}

// Stores the similarities of a wave's agents out of LDS: rows of RW words, K + 1
// of them contiguous in sims.  vec: sims is 16-byte aligned, and so is the wave's
// first row; then 16 bytes per lane per store (similarities alone of 100,003 agents, F 8,
// short lists: K 32 16.6 -> 15.6, K 128 38 -> 28, K 252 99 -> 57 us).
__device__ __forceinline__ void store_similarities(float* __restrict__ sims, uint32_t row0, uint32_t n, uint32_t K,
                                                   uint32_t RW, const float* src, uint32_t lane, uint32_t vec) {
    const uint32_t S = K + 1u, total = (n - row0 < 64u ? n - row0 : 64u) * S;
    float* const dst = sims + (size_t)row0 * S;
    uint32_t x = 0u;  // the words stored so far
    if (vec) {
        const uint32_t total4 = total / 4u;
        x = 4u * total4;
        if (RW == S) {
            for (uint32_t t = lane; t < total4; t += 64u)
                reinterpret_cast<float4*>(dst)[t] = reinterpret_cast<const float4*>(src)[t];
        } else {
            const uint32_t dr = 256u / S, dc = 256u - dr * S;
            uint32_t r = 4u * lane / S, c = 4u * lane - r * S;
            for (uint32_t t = lane; t < total4; t += 64u) {
                float v[4];
                uint32_t at = r * RW + c, cc = c;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    v[k] = src[at];
                    const bool wrap = ++cc == S;
                    at += wrap ? RW - S + 1u : 1u;
                    cc = wrap ? 0u : cc;
                }
                reinterpret_cast<float4*>(dst)[t] = make_float4(v[0], v[1], v[2], v[3]);
                r += dr;
                c += dc;
                if (c >= S) {
                    c -= S;
                    ++r;
                }
            }
        }
    }
    const uint32_t dr = 64u / S, dc = 64u - dr * S;
    x += lane;
    uint32_t r = x / S, c = x - r * S;
    for (; x < total; x += 64u) {
        dst[x] = src[r * RW + c];
        r += dr;
        c += dc;
        if (c >= S) {
            c -= S;
            ++r;
        }
    }
}

// computeNeighNaiveSimilarities (+ computeAdaptiveSimilarities) over sorted
// features; with STEER also steerForClusterCohesion + Alignment on the fly (the
// whole of BehaviorClusteringPlugIn::steerForClustering).  One lane per sorted
// agent; neighbours in groups of G (8 gathers of FQ float4 in flight at FQ <= 2).
// Each lane writes its similarity row into LDS, in the place of its staged list row
// where there is one (not with STEER, whose lanes read their own rows), and the
// wave then stores the rows with coalesced writes.
extern __shared__ float4 bc_rows[];

// What the steering of STEER reads and writes.
struct SteerIo {
    brt_steer_params sp;
    const float4* spos;
    const float4* sfwd;
    const float4* force_in;
    float4* force_out;
};

template <bool ADAPTIVE, bool STEER, int FQ>
__device__ __forceinline__ void similarity_agent(uint32_t i, uint32_t K, uint32_t W, const brt_bc_params& bc,
                                                 uint32_t n, const uint2* __restrict__ hash,
                                                 const uint32_t* __restrict__ lists,
                                                 const float4* __restrict__ sfeat, const float* __restrict__ norms,
                                                 const float4* __restrict__ stats_in, float4* __restrict__ stats_out,
                                                 uint32_t* row, bool staged, const SteerIo& io) {
    float* const out = reinterpret_cast<float*>(row);
    constexpr int G = FQ <= 2 ? 8 : (FQ <= 4 ? 4 : 2);
    const uint32_t F = bc.feature_count;
    const uint32_t id = hash[i].y;
    float4 mine[FQ];
#pragma unroll
    for (int q = 0; q < FQ; ++q) mine[q] = sfeat[(size_t)i * FQ + q];
    const float n1 = norms[i];
    const bool valid = id < n;
    float4 st = ADAPTIVE && valid ? stats_in[id] : make_float4(0.f, 0.f, 0.f, 0.f);
    V3 myPos = v3(0.f, 0.f, 0.f), myFwd = myPos, vel = myPos;
    if (STEER) {
        const float4 P = io.spos[i], Fw = io.sfwd[i];
        myPos = xyz(P);
        myFwd = xyz(Fw);
        vel = myFwd * Fw.w;
    }
    ClusterAccum acc;
    acc.init();
    auto visit = [&](uint32_t base, const uint32_t(&jj)[8], uint32_t mask) {
#pragma unroll
        for (int g0 = 0; g0 < 8; g0 += G) {
            float4 other[G][FQ], op[G], of[G];
            float n2[G];
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const uint32_t j = jj[g0 + g];
#pragma unroll
                for (int q = 0; q < FQ; ++q) other[g][q] = sfeat[(size_t)j * FQ + q];
                n2[g] = norms[j];
                if (STEER) {
                    op[g] = io.spos[j];
                    of[g] = io.sfwd[j];
                }
            }
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const int k = g0 + g;
                if (!(mask & (1u << k))) continue;
                float sim = 0.0f;
                if (valid) {
                    sim = naive_similarity<FQ>(mine, other[g], F, n1, n2[g]);
                    if (ADAPTIVE) {
                        st = update_similarity_stats(sim, st, bc);
                        sim = interpolate_similarity(sim, st.x, st.y, st.z);
                    }
                }
                out[base + k - 1u] = sim;
                if (STEER) acc.add(myPos, vel, io.sp.max_speed, xyz(op[g]), xyz(of[g]), sim);
            }
        }
    };
    uint32_t count;
    if (!STEER && staged) {
        count = row[0] < K ? row[0] : K;
        visit_staged(reinterpret_cast<const uint4*>(row), count, i, n, visit);
    } else {
        count = for_list_octets(lists, W, K, i, n, visit);
    }
    for (uint32_t t = count; t <= K; ++t) out[t] = 0.0f;
    if (ADAPTIVE && valid) stats_out[id] = st;
    if (STEER) io.force_out[i] = acc.finish(count, myFwd, bc, io.force_in[i]);
}

template <bool ADAPTIVE, bool STEER, int FQ>
__global__ void __launch_bounds__(256) k_bc_similarities(uint32_t K, uint32_t W, brt_bc_params bc, uint32_t n,
                                                         const uint2* __restrict__ hash,
                                                         const uint32_t* __restrict__ lists,
                                                         const float4* __restrict__ sfeat,
                                                         const float* __restrict__ norms,
                                                         const float4* __restrict__ stats_in,
                                                         float4* __restrict__ stats_out, float* __restrict__ sims,
                                                         uint32_t sims_vec, SteerIo io, uint32_t xcd_remap) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t row0 = xcd_block(xcd_remap) * blockDim.x + wave * 64u, i = row0 + lane;
    if (row0 >= n) return;
    const bool staged = !STEER && W <= kStageWords;
    const uint32_t RW = STEER ? K + 1u : similarity_row_words(K, W);
    uint32_t* const mem = reinterpret_cast<uint32_t*>(bc_rows) + (size_t)wave * 64u * RW;
    if (staged) stage_rows(reinterpret_cast<uint4*>(mem), lists, W, row0, lane, n);
    if (i < n)
        similarity_agent<ADAPTIVE, STEER, FQ>(i, K, W, bc, n, hash, lists, sfeat, norms, stats_in, stats_out,
                                              mem + lane * RW, staged, io);
    wave_lds_sync();
    store_similarities(sims, row0, n, K, RW, reinterpret_cast<const float*>(mem), lane, sims_vec);
}

// ---- similarities and cluster steering in one pass
// (the whole of BehaviorClusteringPlugIn::steerForClustering).  The pass reads
// position, heading, norm and features of every listed neighbour: five gathers
// per entry, each touching up to 64 cache lines of which the L1 takes about one
// a clock (10,032 per wave at K 32 and 8 features: 267 of the kernel's 357 us).
// So a neighbour's values are one record of 64 bytes (a multiple, with more
// features) in sorted order, and the four lanes of a quad load it together, one
// line instead of four; the parts change lanes through LDS.  2,854 accesses per
// wave and 237 us: bound by the arithmetic (6,890 VALU instructions per wave).
// Record parts: (pos, norm), (heading, 0), the features; 4 * kRounds float4.
typedef float vfloat4 __attribute__((ext_vector_type(4)));

template <int FQ>
constexpr int record_rounds() {
    return (2 + FQ + 3) / 4;
}

template <int FQ>
__global__ void __launch_bounds__(256) k_bc_records(uint32_t F, uint32_t n, uint32_t vec,
                                                    const uint2* __restrict__ hash,
                                                    const float* __restrict__ features,
                                                    const float4* __restrict__ spos,
                                                    const float4* __restrict__ sfwd, float4* __restrict__ rec) {
    constexpr uint32_t RP = 4u * record_rounds<FQ>();
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t i = t / RP, p = t % RP;  // one lane per part
    if (i >= n) return;
    const uint32_t id = hash[i].y;
    const float* f = features + (size_t)(id < n ? id : 0u) * F;
    auto part = [&](uint32_t q) {
        float v[4];
        if (vec) {
            const float4 x = reinterpret_cast<const float4*>(f)[q];
            v[0] = x.x;
            v[1] = x.y;
            v[2] = x.z;
            v[3] = x.w;
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = 4u * q + c < F ? f[4u * q + c] : 0.0f;
        }
        return make_float4(v[0], v[1], v[2], v[3]);
    };
    float4 r = make_float4(0.f, 0.f, 0.f, 0.f);
    if (p == 0u) {
        const float4 P = spos[i];
        float acc = 0.0f;
        if (id < n) {
#pragma unroll
            for (uint32_t q = 0; q < (uint32_t)FQ; ++q) {
                const float4 x = part(q);
                const float v[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (4u * q + c < F) acc = acc + v[c] * v[c];
            }
        }
        r = make_float4(P.x, P.y, P.z, sqrtf(acc));
    } else if (p == 1u) {
        const float4 Fw = sfwd[i];
        r = make_float4(Fw.x, Fw.y, Fw.z, 0.0f);
    } else if (p < 2u + (uint32_t)FQ && id < n) {
        r = part(p - 2u);
    }
    rec[t] = r;
}

// STAGED: the list rows in LDS (W <= kStageWords); else in memory, read ahead, which
// takes the registers of the fourth wave per SIMD with up to 8 features (staged rows
// too, when both were one kernel: 200,003 agents, K 16, F 8 44 -> 48 us).
template <bool ADAPTIVE, int FQ, bool STAGED>
__global__ void __launch_bounds__(256) k_bc_similarities_steer(
    uint32_t K, uint32_t W, brt_bc_params bc, uint32_t n, const uint2* __restrict__ hash,
    const uint32_t* __restrict__ lists, const float4* __restrict__ rec, const float4* __restrict__ stats_in,
    float4* __restrict__ stats_out, float* __restrict__ sims, brt_steer_params sp, const float4* __restrict__ sfwd,
    const float4* force_in, float4* force_out, uint32_t wave_bytes, uint32_t sims_vec, uint32_t xcd_remap) {
    constexpr int NR = record_rounds<FQ>();
    constexpr uint32_t RP = 4u * NR;
    constexpr int G = NR == 1 ? 4 : (NR == 2 ? 2 : 1);  // entries in flight
    const uint32_t lane = threadIdx.x & 63u, l = lane & 3u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t row0 = xcd_block(xcd_remap) * blockDim.x + wave * 64u;
    if (row0 >= n) return;
    const uint32_t i = row0 + lane, at = i < n ? i : n - 1u;
    char* const mem = reinterpret_cast<char*>(bc_rows) + (size_t)wave * wave_bytes;
    const uint32_t RW = similarity_row_words(K, W);
    uint32_t* const row = reinterpret_cast<uint32_t*>(mem) + lane * RW;
    vfloat4* const tile = reinterpret_cast<vfloat4*>(mem + wave_bytes - kTileChunks * 16u);
    if (STAGED) stage_rows(reinterpret_cast<uint4*>(mem), lists, W, row0, lane, n);
    const vuint4* const L = reinterpret_cast<const vuint4*>(lists + (size_t)at * W);
    // word q of the row, if it holds an entry (else any value)
    auto word = [&](uint32_t q, uint32_t last) {
        if (STAGED) return reinterpret_cast<const vuint4*>(row)[q < last ? q : last];
        vuint4 v = {0u, 0u, 0u, 0u};
        if (q <= last) v = L[q];
        return v;
    };

    const uint32_t F = bc.feature_count;
    const uint32_t id = hash[at].y;
    const bool valid = id < n && i < n;
    float4 own[RP];
#pragma unroll
    for (uint32_t p = 0; p < RP; ++p)
        if (p != 1u && p < 2u + (uint32_t)FQ) own[p] = rec[(size_t)at * RP + p];
    float4 mine[FQ];
#pragma unroll
    for (int q = 0; q < FQ; ++q) mine[q] = own[2 + q];
    const float n1 = own[0].w;
    const float4 Fw = sfwd[at];
    const V3 myPos = xyz(own[0]), myFwd = xyz(Fw), vel = myFwd * Fw.w;
    float4 st = ADAPTIVE && valid ? stats_in[id] : make_float4(0.f, 0.f, 0.f, 0.f);
    ClusterAccum acc;
    acc.init();

    vuint4 a = word(0u, 0u);
    const uint32_t count = i < n ? (a.x < K ? a.x : K) : 0u, last = count / 4u;
    float* const out = reinterpret_cast<float*>(row);
    vuint4 b, na, nb;
    if (!STAGED) b = word(1u, last);
    // all lanes of the wave stay in step: those past their list load their own record
    for (uint32_t q = 0; __ballot(q <= last) != 0; q += 2) {
        // rows in memory: the next words load during this octet's gathers; staged
        // ones are read when they are used (this octet overwrites the row up to word
        // 4 q + 6)
        if (!STAGED) {
            na = word(q + 2u, last);
            nb = word(q + 3u, last);
        } else {
            if (q != 0u) a = word(q, last);
            b = word(q + 1u, last);
        }
        uint32_t jj[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        const uint32_t mask = octet_mask(jj, q, count, at, n);
#pragma unroll
        for (int g0 = 0; g0 < 8; g0 += G) {
            if (__ballot((mask >> g0 & ((1u << G) - 1u)) != 0u) == 0) continue;
            // part 4 r + l of the quad's lane k's record
            vfloat4 in[G][NR][4];
#pragma unroll
            for (int g = 0; g < G; ++g) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t x = jj[g0 + g];
                    const uint32_t j = k == 0   ? quad_lane<0>(x)
                                       : k == 1 ? quad_lane<1>(x)
                                       : k == 2 ? quad_lane<2>(x)
                                                : quad_lane<3>(x);
                    const vfloat4* const src = reinterpret_cast<const vfloat4*>(rec) + (size_t)j * RP + l;
#pragma unroll
                    for (int r = 0; r < NR; ++r) in[g][r][k] = src[4 * r];
                }
            }
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const int k = g0 + g;
                vfloat4 got[RP];
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    // LDS operations of a wave take effect in order
#pragma unroll
                    for (int c = 0; c < 4; ++c) tile[65 * c + lane] = in[g][r][c];
                    wave_lds_sync();
#pragma unroll
                    for (int c = 0; c < 4; ++c) got[4 * r + c] = tile[65u * l + (lane - l) + c];
                    wave_lds_sync();
                }
                if (!(mask & (1u << k))) continue;
                float4 other[FQ];
#pragma unroll
                for (int f = 0; f < FQ; ++f)
                    other[f] = make_float4(got[2 + f].x, got[2 + f].y, got[2 + f].z, got[2 + f].w);
                float sim = 0.0f;
                if (valid) {
                    sim = naive_similarity<FQ>(mine, other, F, n1, got[0].w);
                    if (ADAPTIVE) {
                        st = update_similarity_stats(sim, st, bc);
                        sim = interpolate_similarity(sim, st.x, st.y, st.z);
                    }
                }
                out[4u * q + (uint32_t)k - 1u] = sim;
                acc.add(myPos, vel, sp.max_speed, v3(got[0].x, got[0].y, got[0].z), v3(got[1].x, got[1].y, got[1].z),
                        sim);
            }
        }
        if (!STAGED) {
            a = na;
            b = nb;
        }
    }
    if (i < n) {
        for (uint32_t t = count; t <= K; ++t) out[t] = 0.0f;
        if (ADAPTIVE && valid) stats_out[id] = st;
        force_out[i] = acc.finish(count, myFwd, bc, force_in[i]);
    }
    wave_lds_sync();
    store_similarities(sims, row0, n, K, RW, reinterpret_cast<const float*>(mem), lane, sims_vec);
}

// steerForClusterCohesion + Alignment from stored similarities.
template <ListRows ROWS>
__global__ void __launch_bounds__(256) k_bc_cluster_steer(uint32_t K, uint32_t W, brt_steer_params sp,
                                                          brt_bc_params bc, uint32_t n,
                                                          const float4* __restrict__ spos,
                                                          const float4* __restrict__ sfwd,
                                                          const uint32_t* __restrict__ lists,
                                                          const float* __restrict__ sims,
                                                          const float4* force_in, float4* force_out,
                                                          uint32_t xcd_remap) {
    __shared__ uint4 s_stage[4][list_rows_chunks(ROWS)];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t i = xcd_block(ROWS == kRowsOwn ? 0u : xcd_remap) * blockDim.x + threadIdx.x;
    const uint32_t at = i < n ? i : n - 1u;
    const float4 P = spos[at], Fw = sfwd[at];
    const V3 myPos = xyz(P), myFwd = xyz(Fw);
    const V3 vel = myFwd * Fw.w;
    const float* s = sims + (size_t)at * (K + 1u);
    ClusterAccum acc;
    acc.init();
    const uint32_t count = walk_list<ROWS>(s_stage[wave], lists, W, K, i - lane, lane, n, [&](uint32_t base, const uint32_t(&jj)[8], uint32_t mask) {
        float4 op[8], of[8];
        float sv[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            op[k] = spos[jj[k]];
            of[k] = sfwd[jj[k]];
            sv[k] = (mask & (1u << k)) ? s[base + k - 1u] : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (mask & (1u << k)) acc.add(myPos, vel, sp.max_speed, xyz(op[k]), xyz(of[k]), sv[k]);
    });
    if (i < n) force_out[i] = acc.finish(count, myFwd, bc, force_in[i]);
}

// ---------------------------------------------------------------- cluster membership
// Local propagation (BehaviorClusteringPlugIn::computeClusterMembership,
// BehaviorClusteringPlugIn.h:823-865): every agent's label starts as its sorted
// index (resetClusterMembership, BehaviorClustering_kernel.cu:632-652), then T
// Jacobi iterations replace it by the least label among itself and its listed
// neighbours (computeClusterMembership_kernel, :583-625), then the connector
// pairs each agent's position with its label's (CMConnection_kernel, :657-689).
// The reference keeps the labels in float3.x by agent ID and gathers a
// neighbour's through the sorted->ID map; here they live in sorted order during
// the iterations (a neighbour's label is then lbl[j], next to the agent's own
// in memory), so each iteration reads the list row and one float per entry.
// The first iteration reads no labels (they are the indices themselves) and
// the last writes the float3 by ID and the connector.  Same values: a min of
// the same operands, the same T, no rounding.
// SCAN: false without iterations (the labels are the indices).
template <bool FIRST, bool LAST, ListRows ROWS, bool SCAN = true>
__global__ void __launch_bounds__(256) k_lp_iterate(uint32_t K, uint32_t W, uint32_t n, const uint2* __restrict__ hash,
                                                    const uint32_t* __restrict__ lists,
                                                    const float* __restrict__ lbl_in, float* __restrict__ lbl_out,
                                                    const float* m_in, float* m_out,
                                                    const float4* __restrict__ spos, float4* __restrict__ conn,
                                                    uint32_t xcd_remap) {
    __shared__ uint4 s_stage[4][list_rows_chunks(ROWS)];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t i = xcd_block(ROWS == kRowsOwn ? 0u : xcd_remap) * blockDim.x + threadIdx.x, at = i < n ? i : n - 1u;
    float mn = FIRST ? (float)i : lbl_in[at];
    // the last iteration's reads by ID load during the walk
    uint32_t id = n;
    float y = 0.0f, z = 0.0f;
    float4 P = make_float4(0.f, 0.f, 0.f, 0.f);
    if (LAST) {
        id = hash[at].y;
        if (id < n) {
            y = m_in[(size_t)id * 3u + 1u];
            z = m_in[(size_t)id * 3u + 2u];
        }
        if (conn) P = spos[at];
    }
    if (SCAN) {
        walk_list<ROWS>(s_stage[wave], lists, W, K, i - lane, lane, n, [&](uint32_t, const uint32_t(&jj)[8], uint32_t mask) {
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = FIRST ? (float)jj[k] : lbl_in[jj[k]];
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if ((mask & (1u << k)) && mn > v[k]) mn = v[k];
        });
    }
    if (i >= n) return;
    if (!LAST) {
        lbl_out[i] = mn;
        return;
    }
    if (id >= n) return;
    const size_t o = (size_t)id * 3u;
    m_out[o] = mn;
    m_out[o + 1] = y;
    m_out[o + 2] = z;
    if (conn) {
        conn[2u * (size_t)id] = P;
        conn[2u * (size_t)id + 1u] = spos[(uint32_t)mn];
    }
}

// Labels from float3 by agent ID into sorted order beside the position (one
// gather per agent), so the hit-rate pass reads a neighbour's both in one load.
__global__ void __launch_bounds__(256) k_gather_labels(uint32_t n, const uint2* __restrict__ hash,
                                                       const float* __restrict__ m_in,
                                                       const float4* __restrict__ spos, float4* __restrict__ lbl) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t id = hash[i].y;
    const float4 p = spos[i];
    lbl[i] = make_float4(p.x, p.y, p.z, id < n ? m_in[(size_t)id * 3u] : 0.0f);
}

// analyzeClusterHitRate's kernel (BehaviorClustering_kernel.cu:502-578): among
// the listed neighbours within sameClusterMaxRadius, the fraction sharing the
// agent's label and the mean of their labels (-1 with none); float3 by ID.
// T: the greatest squared length within the radius (length(o) > radius exactly
// when dot(o, o) > T, the square root being correctly rounded).  1M blobs, K 32,
// with the labels gathered beside the positions: 114.8 -> 65 us.
template <ListRows ROWS>
__global__ void __launch_bounds__(256) k_hit_rate(uint32_t K, uint32_t W, float T, uint32_t n,
                                                  const uint2* __restrict__ hash, const uint32_t* __restrict__ lists,
                                                  const float4* __restrict__ lbl, float* __restrict__ m_out,
                                                  uint32_t xcd_remap) {
    __shared__ uint4 s_stage[4][list_rows_chunks(ROWS)];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t i = xcd_block(ROWS == kRowsOwn ? 0u : xcd_remap) * blockDim.x + threadIdx.x;
    const uint32_t id = i < n ? hash[i].y : n;
    const float4 own = lbl[i < n ? i : n - 1u];
    const float my = own.w;
    const V3 myPos = xyz(own);
    int close = 0;
    float real = 0.0f, hit = 0.0f;
    walk_list<ROWS>(s_stage[wave], lists, W, K, i - lane, lane, n, [&](uint32_t, const uint32_t(&jj)[8], uint32_t mask) {
        float4 op[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) op[k] = lbl[jj[k]];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (!(mask & (1u << k))) continue;
            const V3 offset = xyz(op[k]) - myPos;
            if (dot(offset, offset) > T) continue;
            ++close;
            real = real + op[k].w;
            if (my == op[k].w) hit = hit + 1.0f;
        }
    });
    if (id >= n) return;
    if (close > 0) {
        hit = hit / (float)close;
        real = real / (float)close;
    } else {
        real = -1.0f;
    }
    const size_t o = (size_t)id * 3u;
    m_out[o] = my;
    m_out[o + 1] = hit;
    m_out[o + 2] = real;
}

}  // namespace

namespace {

template <ListRows ROWS>
hipError_t launch_label_iterations(uint32_t K, uint32_t n, uint32_t iterations, const uint2* hash,
                                   const uint32_t* lists, const float4* spos, const float* m_in, float* m_out,
                                   float4* conn, float* lbl_a, float* lbl_b, uint32_t xcd_remap, hipStream_t s) {
    const uint32_t W = list_stride(K);
    const dim3 grid((n + 255) / 256), block(256);
    if (iterations == 1) {
        hipLaunchKernelGGL((k_lp_iterate<true, true, ROWS>), grid, block, 0, s, K, W, n, hash, lists, nullptr,
                           nullptr, m_in, m_out, spos, conn, xcd_remap);
        return hipGetLastError();
    }
    hipLaunchKernelGGL((k_lp_iterate<true, false, ROWS>), grid, block, 0, s, K, W, n, hash, lists, nullptr, lbl_a,
                       m_in, m_out, spos, conn, xcd_remap);
    float* src = lbl_a;
    float* dst = lbl_b;
    for (uint32_t t = 1; t + 1 < iterations; ++t) {
        hipLaunchKernelGGL((k_lp_iterate<false, false, ROWS>), grid, block, 0, s, K, W, n, hash, lists, src, dst,
                           m_in, m_out, spos, conn, xcd_remap);
        float* x = src;
        src = dst;
        dst = x;
    }
    hipLaunchKernelGGL((k_lp_iterate<false, true, ROWS>), grid, block, 0, s, K, W, n, hash, lists, src, nullptr,
                       m_in, m_out, spos, conn, xcd_remap);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_cluster_membership(uint32_t K, uint32_t n, uint32_t iterations, const uint2* hash,
                                     const uint32_t* lists, const float4* spos, const float* m_in, float* m_out,
                                     float4* conn, float* lbl_a, float* lbl_b, uint32_t xcd_remap, hipStream_t s) {
    if (iterations == 0) {
        hipLaunchKernelGGL((k_lp_iterate<true, true, kRowsOwn, false>), dim3((n + 255) / 256), dim3(256), 0, s, K,
                           list_stride(K), n, hash, lists, nullptr, nullptr, m_in, m_out, spos, conn, xcd_remap);
        return hipGetLastError();
    }
    const ListRows rows = list_rows(list_stride(K), n);
    const auto launch = rows == kRowsOwn     ? launch_label_iterations<kRowsOwn>
                        : rows == kRowsWhole ? launch_label_iterations<kRowsWhole>
                                             : launch_label_iterations<kRowsBlocks>;
    return launch(K, n, iterations, hash, lists, spos, m_in, m_out, conn, lbl_a, lbl_b, xcd_remap, s);
}

hipError_t launch_hit_rate(uint32_t K, float radius, uint32_t n, const uint2* hash, const uint32_t* lists,
                           const float4* spos, const float* m_in, float* m_out, float4* lbl, uint32_t xcd_remap,
                           hipStream_t s) {
    const dim3 grid((n + 255) / 256), block(256);
    hipLaunchKernelGGL(k_gather_labels, grid, block, 0, s, n, hash, m_in, spos, lbl);
    const auto kernel = list_stride(K) <= kStageWords ? k_hit_rate<kRowsWhole> : k_hit_rate<kRowsBlocks>;
    hipLaunchKernelGGL(kernel, grid, block, 0, s, K, list_stride(K), brt_radius_threshold(radius), n, hash, lists, lbl,
                       m_out, xcd_remap);
    return hipGetLastError();
}

namespace {

template <int FQ>
hipError_t launch_sims(uint32_t K, const brt_bc_params& bc, uint32_t n, const uint2* hash, const uint32_t* lists,
                       const float* features, uint32_t vec, const float4* stats_in, float4* stats_out, float* sims,
                       void* scratch, void* records, const brt_steer_params* sp, const float4* spos,
                       const float4* sfwd, const float4* force_in, float4* force_out, uint32_t xcd_remap,
                       hipStream_t s) {
    const uint32_t F = bc.feature_count, W = list_stride(K);
    const uint32_t sims_vec = ((uintptr_t)sims & 15u) == 0 ? 1u : 0u;
    if (sp && records) {
        constexpr uint32_t RP = 4u * record_rounds<FQ>();
        float4* rec = reinterpret_cast<float4*>(records);
        hipLaunchKernelGGL((k_bc_records<FQ>), dim3((unsigned)(((size_t)n * RP + 255u) / 256u)), dim3(256), 0, s, F, n,
                           vec, hash, features, spos, sfwd, rec);
        // four waves per workgroup while three workgroups fit a CU's LDS, else one
        const uint32_t bytes = similarity_wave_bytes(K, W), B = 4u * bytes <= 160u * 1024u / 3u ? 256u : 64u;
        const auto kernel = W <= kStageWords ? (bc.adaptive ? k_bc_similarities_steer<true, FQ, true>
                                                            : k_bc_similarities_steer<false, FQ, true>)
                                             : (bc.adaptive ? k_bc_similarities_steer<true, FQ, false>
                                                            : k_bc_similarities_steer<false, FQ, false>);
        hipLaunchKernelGGL(kernel, dim3((n + B - 1) / B), dim3(B), B / 64u * bytes, s, K, W, bc, n, hash, lists, rec,
                           stats_in, stats_out, sims, *sp, sfwd, force_in, force_out, bytes, sims_vec, xcd_remap);
        return hipGetLastError();
    }
    float4* sfeat = reinterpret_cast<float4*>(scratch);
    float* norms = reinterpret_cast<float*>(sfeat + (size_t)n * FQ);
    hipLaunchKernelGGL(k_bc_sort_features, dim3((n + 255) / 256), dim3(256), 0, s, F, (uint32_t)FQ, n, vec, hash,
                       features, sfeat, norms);
    // the LDS rows: 256 agents while they stay within 40 KB, else one wave
    const size_t bytes = (size_t)64u * (sp ? K + 1u : similarity_row_words(K, W)) * 4u;
    const uint32_t B = 4u * bytes <= 40u * 1024u ? 256u : 64u;
    const size_t lds = B / 64u * bytes;
    const dim3 grid((n + B - 1) / B), block(B);
    const SteerIo io = sp ? SteerIo{*sp, spos, sfwd, force_in, force_out} : SteerIo{};
    const auto kernel = sp ? (bc.adaptive ? k_bc_similarities<true, true, FQ> : k_bc_similarities<false, true, FQ>)
                           : (bc.adaptive ? k_bc_similarities<true, false, FQ> : k_bc_similarities<false, false, FQ>);
    hipLaunchKernelGGL(kernel, grid, block, lds, s, K, W, bc, n, hash, lists, sfeat, norms, stats_in, stats_out, sims,
                       sims_vec, io, sp ? 0u : xcd_remap);
    return hipGetLastError();
}

}  // namespace

size_t bc_scratch_bytes(uint32_t feature_count, uint32_t n) {
    const size_t FQ = (feature_count + 3u) / 4u;
    return (size_t)n * FQ * 16u + ((size_t)n * 4u + 15u) / 16u * 16u;
}

// Where the accesses of the gathers set the pace: below, each agent's own gathers have
// the shorter chain and leave room for more waves (K 32, F 8: 1,000 agents 13.4 us, from
// records 15.5; 60,000 20 and 22).  Lists of one density or another lie on either side;
// the lines are where the records win over flocks of 1, 4 and 12 per cell and blobs
// taken together.  Own gathers -> records, us, at these four:
//   * from 98,304 agents with 5 features or more, K >= 24 (from 9 on, every K): 100,003
//     agents, K 32, F 8 27 -> 29, 42 -> 42, 51 -> 44, 49 -> 44; F 16 31 -> 37, 56 -> 54,
//     76 -> 56, 74 -> 56; K 16, F 16 30 -> 35, 44 -> 39, 46 -> 39, 44 -> 38;
//   * from 147,456 below K 24: 131,072 agents, K 16, F 8 27 -> 30, 31 -> 34, 32 -> 33,
//     33 -> 34;
//   * from 196,608 with up to 4 features, where a record saves one access in four, and
//     from K 49 on: 131,072 agents, K 24, F 4 25 -> 29, 34 -> 39, 38 -> 39, 39 -> 39;
//     and there for K 16 to 48 (K 16, F 4, 200,003 agents 33 -> 35, 48 -> 43, 50 -> 42,
//     47 -> 42), up to 786,432 agents for the short ones (1,048,576 agents 132 -> 156,
//     186 -> 190, 212 -> 190, 196 -> 185).
// Lists beyond K 64 (80 from 9 features on) leave the records' tile too few waves:
// 1,048,576 agents at 1 / 4 / 12 per cell, F 8, K 80 238 -> 260, 373 -> 383, 661 -> 675;
// F 16, K 80 344 -> 341, 525 -> 501, 990 -> 885.
size_t bc_record_bytes(uint32_t K, uint32_t feature_count, uint32_t n) {
    const size_t FQ = (feature_count + 3u) / 4u;
    const bool pays = FQ == 1u ? K >= (n < (3u << 18) ? 16u : 24u) && K <= 48u : K <= (FQ == 2u ? 64u : 80u);
    const uint32_t least = FQ == 1u || K > 48u ? 3u << 16 : FQ == 2u && K < 24u ? 9u << 14 : 3u << 15;
    return n >= least && pays ? (size_t)n * ((FQ + 5u) / 4u) * 64u : 0u;
}

hipError_t launch_bc_similarities(uint32_t K, const brt_bc_params& bc, uint32_t n, const uint2* hash,
                                  const uint32_t* lists, const float* features, const float4* stats_in,
                                  float4* stats_out, float* sims, void* scratch, void* records,
                                  const brt_steer_params* sp, const float4* spos, const float4* sfwd,
                                  const float4* force_in, float4* force_out, uint32_t xcd_remap, hipStream_t s) {
    const uint32_t F = bc.feature_count;
    const uint32_t vec = (F % 4u == 0 && ((uintptr_t)features & 15u) == 0) ? 1u : 0u;
#define BRT_SIMS_CASE(Q)                                                                                             \
    case Q:                                                                                                          \
        return launch_sims<Q>(K, bc, n, hash, lists, features, vec, stats_in, stats_out, sims, scratch, records, sp, \
                              spos, sfwd, force_in, force_out, xcd_remap, s);
    switch ((F + 3u) / 4u) {
        BRT_SIMS_CASE(1)
        BRT_SIMS_CASE(2)
        BRT_SIMS_CASE(3)
        BRT_SIMS_CASE(4)
        BRT_SIMS_CASE(5)
        BRT_SIMS_CASE(6)
        BRT_SIMS_CASE(7)
        BRT_SIMS_CASE(8)
        default:
            return hipErrorInvalidValue;
    }
#undef BRT_SIMS_CASE
}

hipError_t launch_bc_cluster_steer(uint32_t K, const brt_steer_params& sp, const brt_bc_params& bc, uint32_t n,
                                   const float4* spos, const float4* sfwd, const uint32_t* lists, const float* sims,
                                   const float4* force_in, float4* force_out, uint32_t xcd_remap, hipStream_t s) {
    const ListRows rows = list_rows(list_stride(K), n);
    const auto kernel = rows == kRowsOwn     ? k_bc_cluster_steer<kRowsOwn>
                        : rows == kRowsWhole ? k_bc_cluster_steer<kRowsWhole>
                                             : k_bc_cluster_steer<kRowsBlocks>;
    hipLaunchKernelGGL(kernel, dim3((n + 255) / 256), dim3(256), 0, s, K, list_stride(K), sp, bc, n, spos, sfwd, lists,
                       sims, force_in, force_out, xcd_remap);
    return hipGetLastError();
}

}  // namespace brt
