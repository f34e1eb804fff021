// brt_opensteer.hip -- OpenSteerWrapper + Body on gfx950: one fused pass per step.
//
// The reference runs, per step, resetSteerForce + one kernel per behaviour
// (each re-reading the neighbour list and re-gathering neighbour state and
// read-modify-writing a double-buffered float4 force) + the integrator
// (PlugIns/OpenSteerWrapper/include/OpenSteerWrapperPlugIn.h:288-426,
//  OpenSteerWrapper_kernel.cu:62-333).  Here one lane per sorted agent walks its
// list once and keeps the three behaviour sums in registers.  The sums are still
// formed in list order and combined into the force in the reference's order
//   force = (((0 + sep*w_s) + align*w_a) + coh*w_c) [+ seek*w_t] [+ wander*w_w] [+ worldSeek]
// so the result equals the unfused sequence bit for bit.  The new state is
// written by agent ID (newX[hash[i].y] = ..., OpenSteerWrapper_kernel.cu:324-331).
//
// BehaviorClustering feature update (build-defined, no GPU counterpart in the
// reference): f'[id(i)] = f[id(i)] + rate * (mean_j f[id(j)] - f[id(i)]), the list
// walked in order with the sorted->ID map hash[j].y as in
// BehaviorClustering_computeNeighNaiveSimilarities (BehaviorClustering_kernel.cu:306-353).
#include "brt_device.hpp"
#include "brt_internal.hpp"
#include "brt_lists.hpp"
#include "brt_steer_common.hpp"

namespace brt {

namespace {

// The feature update of the agent at sorted index i (ID id):
// f + (mean of the listed neighbours' features - f) * rate, the mean over the
// list's count; the entries are visited eight at a time with their ID and
// feature gathers in flight together and summed in list order.
// walk(fn) visits the agent's list.
template <class Walk>
__device__ __forceinline__ float4 feature_update(float rate, uint32_t n, const uint2* __restrict__ hash,
                                                 const float4* __restrict__ fin, uint32_t id, Walk&& walk) {
    const float4 f = fin[id];
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    const uint32_t count = walk([&](uint32_t, const uint32_t(&jj)[8], uint32_t mask) {
        uint32_t jid[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) jid[k] = hash[jj[k]].y;
        float4 q[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) q[k] = fin[jid[k] < n ? jid[k] : id];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (((mask >> k) & 1u) == 0u || jid[k] >= n) continue;
            s.x = s.x + q[k].x;
            s.y = s.y + q[k].y;
            s.z = s.z + q[k].z;
            s.w = s.w + q[k].w;
        }
    });
    if (count == 0) return f;
    const float inv = 1.0f / (float)count;  // cutil float4 / float
    float4 r;
    r.x = f.x + (s.x * inv - f.x) * rate;
    r.y = f.y + (s.y * inv - f.y) * rate;
    r.z = f.z + (s.z * inv - f.z) * rate;
    r.w = f.w + (s.w * inv - f.w) * rate;
    return r;
}

template <ListRows ROWS>
__global__ void __launch_bounds__(256) k_features(uint32_t W, float rate, uint32_t n, const uint2* __restrict__ hash,
                                                  const uint32_t* __restrict__ lists,
                                                  const float4* __restrict__ fin, float4* __restrict__ fout,
                                                  uint32_t xcd_remap) {
    __shared__ uint4 s_stage[4][list_rows_chunks(ROWS)];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t i = xcd_block(ROWS == kRowsOwn ? 0u : xcd_remap) * blockDim.x + threadIdx.x;
    const uint32_t id = i < n ? hash[i].y : n;
    const float4 f = feature_update(rate, n, hash, fin, id < n ? id : 0u, [&](auto&& fn) {
        return walk_list<ROWS>(s_stage[wave], lists, W, W - 1u, i - lane, lane, n, fn);
    });
    if (id < n) fout[id] = f;
}

// One lane per sorted agent: walk the list in order (8 entries per round, their
// gathers issued together), accumulate the behaviour sums, then assemble the
// force and integrate (APPLY), or only store the behaviour force in sorted
// order (the steer-force accumulator of the decomposed sequence).
// FEAT: the same pass also writes the agent's feature update (the result of
// feature_update), summing the neighbours' features in the same list walk as
// the steering sums; with all steering weights zero it calls feature_update.
// The neighbours' features are read from sfeat, the features in sorted order
// (sfeat[j] = fin[hash[j].y], gathered with the state), so the walk reads them
// next to their positions instead of at random agent IDs.
// REC: the new state (and feature) goes to one 64-byte record by ID instead of
// to the arrays: a write to a random ID costs the same whatever its size (about
// 45 G a second), and k_unpack moves the records to the arrays in order.
// With FEAT each lane reads its own row.
template <bool APPLY, ListRows ROWS, bool FEAT = false, bool REC = false>
__global__ void __launch_bounds__(256, ROWS == kRowsOwn ? 1 : 4)
    k_steer(brt_grid_params g, uint32_t W, brt_steer_params sp, SteerCuts cuts, float dt,
                                               uint32_t step, uint32_t n, const float4* __restrict__ spos,
                                               const float4* __restrict__ sfwd, const float4* __restrict__ ssa,
                                               const uint2* __restrict__ hash,
                                               const uint32_t* __restrict__ lists, AgentOut o, uint32_t xcd_remap,
                                               float feature_rate = 0.0f, const float4* __restrict__ fin = nullptr,
                                               float4* __restrict__ fout = nullptr,
                                               const float4* __restrict__ sfeat = nullptr) {
    __shared__ uint4 s_stage[4][list_rows_chunks(ROWS)];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t i = xcd_block(ROWS == kRowsOwn ? 0u : xcd_remap) * blockDim.x + threadIdx.x;
    const uint32_t at = i < n ? i : n - 1u;
    const uint32_t id = i < n ? hash[i].y : n;
    if (FEAT && id >= n) return;
    const float4 P = spos[at];
    const float4 Fw = sfwd[at];
    // no sorted copy of the smoothed acceleration: the agent's own, by ID
    float4 SA = make_float4(0.f, 0.f, 0.f, 0.f);
    if (APPLY && id < n) SA = ssa ? ssa[at] : o.sa_out[id];
    const V3 myPos = xyz(P);
    const V3 myFwd = xyz(Fw);

    const Weights wts = weights_of(sp);
    const bool any = wts.s != 0.0f || wts.a != 0.0f || wts.c != 0.0f;
    const float margin = cut_margin(myFwd);

    SteerAccum acc;
    acc.init();
    // FEAT: the feature sum of the same entries, in the same order as
    // feature_update (their IDs load with the positions and headings)
    float4 fsum = make_float4(0.f, 0.f, 0.f, 0.f);
    uint32_t count = 0;
    if (any) {
        // the list in order, eight entries at a time with their gathers in flight;
        // the feature variants hold four more gathers per entry and load the
        // next words after them (K 64: 3 % faster than ahead)
        auto visit = [&](uint32_t, const uint32_t(&jj)[8], uint32_t mask) {
            float4 qp[8], qf[8], fq[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                qp[t] = spos[jj[t]];
                qf[t] = sfwd[jj[t]];
                if (FEAT) fq[t] = sfeat[jj[t]];
            }
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                if ((mask >> t) & 1u) {
                    const V3 offset = xyz(qp[t]) - myPos;
                    acc.add_cut(sp, cuts, wts, myFwd, margin, offset, dot(offset, offset), xyz(qf[t]));
                }
            }
            if (FEAT) {
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    if (((mask >> t) & 1u) == 0u) continue;
                    fsum.x = fsum.x + fq[t].x;
                    fsum.y = fsum.y + fq[t].y;
                    fsum.z = fsum.z + fq[t].z;
                    fsum.w = fsum.w + fq[t].w;
                }
            }
        };
        if (FEAT)
            count = for_list_octets<false>(lists, W, W - 1u, i, n, visit);
        else
            count = walk_list<ROWS>(s_stage[wave], lists, W, W - 1u, i - lane, lane, n, visit);
    }
    float4 feature = make_float4(0.f, 0.f, 0.f, 0.f);
    if (FEAT) {
        if (!any) {
            feature = feature_update(feature_rate, n, hash, fin, id,
                                      [&](auto&& fn) { return for_list_octets(lists, W, W - 1u, i, n, fn); });
        } else {
            const float4 f = sfeat[i];
            float4 r = f;
            if (count != 0) {
                const float inv = 1.0f / (float)count;  // cutil float4 / float
                r.x = f.x + (fsum.x * inv - f.x) * feature_rate;
                r.y = f.y + (fsum.y * inv - f.y) * feature_rate;
                r.z = f.z + (fsum.z * inv - f.z) * feature_rate;
                r.w = f.w + (fsum.w * inv - f.w) * feature_rate;
            }
            feature = r;
        }
        if (!REC) fout[id] = feature;
    }
    if (id >= n) return;
    if (APPLY && REC) {
        float2 wander = make_float2(0.f, 0.f);
        const V3 f = behaviour_force(sp, wts, dt, step, id, id, myPos, myFwd, Fw.w, acc, o.wander, &wander);
        const NewState s = integrate(g, sp, dt, i, f, myPos, myFwd, Fw.w, xyz(SA), nullptr);
        float4* const rec = o.rec + 4u * (size_t)id;
        rec[0] = make_float4(s.pos.x, s.pos.y, s.pos.z, wander.x);
        rec[1] = make_float4(s.fwd.x, s.fwd.y, s.fwd.z, s.speed);
        rec[2] = make_float4(s.sa.x, s.sa.y, s.sa.z, wander.y);
        rec[3] = feature;  // without features too: whole 64 bytes
        return;
    }
    if (APPLY) {
        finish_agent(g, sp, wts, dt, step, i, id, id, myPos, myFwd, Fw.w, xyz(SA), SA.w, acc, o);
    } else {
        const V3 f = behaviour_force(sp, wts, dt, step, id, id, myPos, myFwd, Fw.w, acc, o.wander, o.wander + id);
        o.force_out[i] = make_float4(f.x, f.y, f.z, 0.0f);
    }
}

// Four state arrays (float4 by ID) into one 64-byte record per agent, so that a
// gather by ID reads one of them: one lane per part.
__global__ void __launch_bounds__(256) k_pack(uint32_t n, const float4* __restrict__ a, const float4* __restrict__ b,
                                              const float4* __restrict__ c, const float4* __restrict__ d,
                                              float4* __restrict__ rec) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, i = t >> 2, p = t & 3u;
    if (i >= n) return;
    const float4* const src = p == 0u ? a : (p == 1u ? b : (p == 2u ? c : d));
    if (src) rec[t] = src[i];
}

// k_steer's records to the arrays (feature and wander optional; the smoothed
// acceleration keeps its fourth component).
__global__ void __launch_bounds__(256) k_unpack(uint32_t n, const float4* __restrict__ rec, AgentOut o,
                                                float4* __restrict__ feature) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, i = t >> 2, p = t & 3u;
    if (i >= n) return;
    if (p == 3u && !feature) return;
    float4 v = rec[t];
    const float extra = v.w;
    if (p == 0u) v.w = 1.0f;
    if (p == 2u) v.w = o.sa_out[i].w;
    float4* const dst = p == 0u ? o.pos_out : (p == 1u ? o.fwd_out : (p == 2u ? o.sa_out : feature));
    dst[i] = v;
    if (o.wander && (p & 1u) == 0u) reinterpret_cast<float*>(o.wander)[2u * (size_t)i + (p >> 1)] = extra;
}

// applySteeringForces from an accumulated force (sorted float4): the world-centre
// seek and the integrator of the fused pass, on a force built by other passes.
__global__ void __launch_bounds__(256) k_apply(brt_grid_params g, brt_steer_params sp, float dt, uint32_t n,
                                               const float4* __restrict__ spos, const float4* __restrict__ sfwd,
                                               const float4* __restrict__ ssa, const uint2* __restrict__ hash,
                                               const float4* __restrict__ force_in, AgentOut o) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t id = hash[i].y;
    if (id >= n) return;
    const float4 Fw = sfwd[i], SA = ssa[i];
    apply_force(g, sp, dt, i, id, xyz(force_in[i]), xyz(spos[i]), xyz(Fw), Fw.w, xyz(SA), SA.w, o);
}


}  // namespace

namespace {

// The smallest float t >= 0 with sqrtf(t) >= m, so that sqrtf(d2) < m <=> d2 < t
// for every float d2 (NaN included: both false).
float below_cut(float m) {
    if (m != m) return -INFINITY;
    if (m <= 0.0f) return 0.0f;
    if (m == INFINITY) return INFINITY;
    float t = m * m;
    if (t == INFINITY) t = 3.40282347e38f;
    while (t > 0.0f && sqrtf(nextafterf(t, -INFINITY)) >= m) t = nextafterf(t, -INFINITY);
    while (sqrtf(t) < m) t = nextafterf(t, INFINITY);
    return t;
}

}  // namespace

SteerCuts steer_cuts(const brt_steer_params& sp) {
    SteerCuts c{};
    c.tmin = below_cut(sp.sensing_min_radius);
    const float* b[3] = {sp.separation, sp.alignment, sp.cohesion};
    for (int k = 0; k < 3; ++k) {
        c.tmax[k] = brt_radius_threshold(b[k][1]);
        c.cmax[k] = b[k][2];
    }
    c.same = (c.tmax[0] == c.tmax[1] && c.tmax[0] == c.tmax[2] && c.cmax[0] == c.cmax[1] && c.cmax[0] == c.cmax[2])
                 ? 1u
                 : 0u;
    return c;
}

hipError_t launch_steer(const brt_grid_params& g, uint32_t K, const brt_steer_params& sp, float dt, uint32_t step,
                        uint32_t n, const float4* spos, const float4* sfwd, const float4* ssa, const uint2* hash,
                        const uint32_t* lists, float2* wander, float4* pos_out, float4* fwd_out, float4* sa_out,
                        float4* force_out, uint32_t xcd_remap, hipStream_t s, float feature_rate,
                        const float4* features_in, float4* features_out, const float4* sorted_features,
                        float4* records) {
    AgentOut o{pos_out, fwd_out, sa_out, force_out, wander};
    const SteerCuts cuts = steer_cuts(sp);
    const uint32_t W = list_stride(K);
    const dim3 grid((n + 255) / 256);
    const ListRows rows = list_rows(W, n);  // records: from 2^19 agents, never kRowsOwn
    if (features_in && !sorted_features) return hipErrorInvalidValue;
    if (K > 32u && n >= kXcdRunMin && xcd_remap) xcd_remap = 2u;  // as the list pass before it
    if (records) {
        o.rec = records;
        // the phase's events: the first kernel's start, the second's end
        const hipEvent_t stop = launch_mark().stop;
        launch_mark().stop = nullptr;
        if (features_in)
            BRT_LAUNCH((k_steer<true, kRowsOwn, true, true>), grid, dim3(256), 0, s, g, W, sp, cuts, dt, step, n, spos,
                       sfwd, ssa, hash, lists, o, xcd_remap, feature_rate, features_in, features_out, sorted_features);
        else
            BRT_LAUNCH((rows == kRowsWhole ? k_steer<true, kRowsWhole, false, true>
                                           : k_steer<true, kRowsBlocks, false, true>),
                       grid, dim3(256), 0, s, g, W, sp, cuts, dt, step, n, spos, sfwd, ssa, hash, lists, o, xcd_remap,
                       0.0f, nullptr, nullptr, nullptr);
        o.wander = sp.wander_weight != 0.0f ? wander : nullptr;
        launch_mark().stop = stop;
        BRT_LAUNCH(k_unpack, dim3((unsigned)(((size_t)n * 4u + 255u) / 256u)), dim3(256), 0, s, n, records, o,
                   features_in ? features_out : nullptr);
        return hipGetLastError();
    }
    if (features_in)
        BRT_LAUNCH((k_steer<true, kRowsOwn, true>), grid, dim3(256), 0, s, g, W, sp, cuts, dt, step, n, spos, sfwd, ssa,
                   hash, lists, o, xcd_remap, feature_rate, features_in, features_out, sorted_features);
    else
        BRT_LAUNCH((rows == kRowsOwn     ? k_steer<true, kRowsOwn>
                    : rows == kRowsWhole ? k_steer<true, kRowsWhole>
                                         : k_steer<true, kRowsBlocks>),
                   grid, dim3(256), 0, s, g, W, sp, cuts, dt, step, n, spos, sfwd, ssa, hash, lists, o, xcd_remap, 0.0f,
                   nullptr, nullptr, nullptr);
    return hipGetLastError();
}

hipError_t launch_pack(uint32_t n, const float4* a, const float4* b, const float4* c, const float4* d, float4* rec,
                       hipStream_t s) {
    BRT_LAUNCH(k_pack, dim3((unsigned)(((size_t)n * 4u + 255u) / 256u)), dim3(256), 0, s, n, a, b, c, d, rec);
    return hipGetLastError();
}

hipError_t launch_steer_forces(uint32_t K, const brt_steer_params& sp, float dt, uint32_t step, uint32_t n,
                               const float4* spos, const float4* sfwd, const uint2* hash, const uint32_t* lists,
                               float2* wander, float4* force_out, uint32_t xcd_remap, hipStream_t s) {
    AgentOut o{nullptr, nullptr, nullptr, force_out, wander};
    brt_grid_params g{};
    const ListRows rows = list_rows(list_stride(K), n);
    const auto kernel = rows == kRowsOwn     ? k_steer<false, kRowsOwn>
                        : rows == kRowsWhole ? k_steer<false, kRowsWhole>
                                             : k_steer<false, kRowsBlocks>;
    hipLaunchKernelGGL(kernel, dim3((n + 255) / 256), dim3(256), 0, s, g, list_stride(K), sp, steer_cuts(sp), dt, step,
                       n, spos, sfwd, sfwd, hash, lists, o, xcd_remap, 0.0f, nullptr, nullptr, nullptr);
    return hipGetLastError();
}

hipError_t launch_apply(const brt_grid_params& g, const brt_steer_params& sp, float dt, uint32_t n, const float4* spos,
                        const float4* sfwd, const float4* ssa, const uint2* hash, const float4* force_in,
                        float4* pos_out, float4* fwd_out, float4* sa_out, float4* force_out, hipStream_t s) {
    AgentOut o{pos_out, fwd_out, sa_out, force_out, nullptr};
    hipLaunchKernelGGL(k_apply, dim3((n + 255) / 256), dim3(256), 0, s, g, sp, dt, n, spos, sfwd, ssa, hash, force_in,
                       o);
    return hipGetLastError();
}

hipError_t launch_features(uint32_t K, float rate, uint32_t n, const uint2* hash, const uint32_t* lists,
                           const float4* fin, float4* fout, uint32_t xcd_remap, hipStream_t s) {
    const ListRows rows = list_rows(list_stride(K), n);
    BRT_LAUNCH((rows == kRowsOwn     ? k_features<kRowsOwn>
                : rows == kRowsWhole ? k_features<kRowsWhole>
                                     : k_features<kRowsBlocks>), dim3((n + 255) / 256), dim3(256), 0, s,
               list_stride(K), rate, n, hash, lists, fin, fout, xcd_remap);
    return hipGetLastError();
}

}  // namespace brt
