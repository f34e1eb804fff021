// brt_adjoint.hip -- reverse-mode adjoint of one steering + integration step.
//
// Forward (one agent i, lists fixed as the forward step built them):
//   u_s = normalize(mean_j -(p_j-p_i)/|p_j-p_i|^2), u_a = normalize(mean_j f_j - f_i),
//   u_c = normalize(mean_j (p_j-p_i)), F = w_s u_s + w_a u_a + w_c u_c [+ seeks],
//   then applySteeringForceSingle (PlugIns/OpenSteerWrapper/OpenSteerWrapper_resources.cu:326-379):
//   F' = adjustRawSteeringForce(F, s, f), c = truncate(F', maxF), acc = c / m,
//   a1 = a + (acc - a) r, v0 = f s + a1 dt, v = truncate(v0, maxS),
//   s1 = |v|, p1 = p + v dt, f1 = normalize(v).
// Given dL/d(p1, f1, s1, a1) by agent ID, two kernels produce dL/d(p, f, s, a)
// by agent ID, with no atomics, so the same inputs always give the same bits:
//   k_adjoint_own (one lane per sorted agent i) or k_adjoint_own_quad (four)
//     recomputes agent i's forward values with the forward kernels' arithmetic,
//     back-propagates through the integrator and its own behaviour sums, and
//     stores by sorted index its own terms and a record of what its neighbours'
//     terms are made of (position, heading, the separation, cohesion and
//     alignment sums' adjoints, flags);
//   k_adjoint_gather (several lanes per sorted agent j) finds every agent i
//     whose list holds j -- j's own list when that list can stand in for them
//     (and the cells where agents below the grid are kept, for j on a low face),
//     else the agents of the 27 cells around j's cell -- by repeating the list
//     test (radius, cell range, and, for a full list, j's place in i's
//     visiting order against i's last entry), adds i's terms for p_j and f_j
//     in a fixed order, and writes the sums by ID.
// The radius/angle predicates, the list membership and the world-box test are
// piecewise constant and carry no gradient.  dL/dw for the three behaviour
// weights is reduced per workgroup and then in a fixed order.
// The reference has no adjoint; the forward it differentiates is the one
// restated in brt_steer_common.hpp.
#include "brt_device.hpp"
#include "brt_internal.hpp"
#include "brt_steer_common.hpp"
#include "brt_wave.hpp"

namespace brt {

namespace {

__device__ __forceinline__ V3 normalize_bwd(V3 x, V3 ybar) {
    const float len = length(x);
    const V3 y = x * (1.0f / len);
    return (ybar - y * dot(y, ybar)) * (1.0f / len);
}

__device__ __forceinline__ V3 truncate_bwd(V3 x, float maxLength, V3 ybar) {
    const float len = length(x);
    if (len <= maxLength) return ybar;
    const V3 u = x * (1.0f / len);
    return (ybar - u * dot(u, ybar)) * (maxLength / len);
}

// Flags of an agent's neighbour-term vectors: which of its behaviour sums have
// neighbour terms, whether its own cell (calcGridPos) lies in the grid, and
// whether its list is full (count == K), and whether that cell is on a low
// face of the grid (a coordinate 0: agents below the grid are keyed at the
// far face, so lists there are not symmetric).
constexpr uint32_t kAdjSep = 1u, kAdjAli = 2u, kAdjCoh = 4u, kAdjInGrid = 8u, kAdjFull = 16u, kAdjLowFace = 32u;

struct AdjArgs {
    brt_grid_params g;
    brt_steer_params sp;
    float dt;
    uint32_t K, W, n;
    const float4* spos;
    const float4* sfwd;
    const float4* ssa;
    const uint2* hash;
    const uint32_t* lists;
    const float4* gpos_out;
    const float4* gfwd_out;
    const float4* gsa_out;
    // by sorted index: 3 float4 of own terms (dL/dp, (dL/df, dL/ds), dL/da) and
    // the record of 4 float4, 64 bytes, that the neighbours' terms are made of:
    // (p.xyz f.x | f.yz S.xy | S.z C.xyz | A.xyz flags)
    float4* own;
    float4* rec;
    float* partials;  // per workgroup: 3 floats
    uint32_t xcd_remap;
};

// Sums the per-workgroup partials in a fixed order (strided per-thread sums,
// then a fixed LDS tree) and adds the result to weight_grad; the same inputs
// always give the same bits.
// (256 threads)
__device__ void reduce_partials(const float* __restrict__ partials, uint32_t blocks, float* __restrict__ weight_grad) {
    __shared__ float s_sum[3][256];
    const uint32_t tid = threadIdx.x;
    float v0 = 0.0f, v1 = 0.0f, v2 = 0.0f;
    for (uint32_t b = tid; b < blocks; b += 256u) {
        v0 += partials[(size_t)b * 3 + 0];
        v1 += partials[(size_t)b * 3 + 1];
        v2 += partials[(size_t)b * 3 + 2];
    }
    s_sum[0][tid] = v0;
    s_sum[1][tid] = v1;
    s_sum[2][tid] = v2;
    __syncthreads();
    for (uint32_t o = 128; o > 0; o >>= 1) {
        if (tid < o) {
            s_sum[0][tid] += s_sum[0][tid + o];
            s_sum[1][tid] += s_sum[1][tid + o];
            s_sum[2][tid] += s_sum[2][tid + o];
        }
        __syncthreads();
    }
    if (tid < 3) weight_grad[tid] = weight_grad[tid] + s_sum[tid][0];
}

// The terms one pair (i, j) of agent i's list contributes to dL/d(off),
// off = p_j - p_i, from i's separation and cohesion sums (anyP: one of them
// holds the pair), and whether i's alignment sum holds it; the forward's
// predicates, recomputed with the forward's arithmetic.
__device__ __forceinline__ V3 pair_terms(const brt_steer_params& sp, uint32_t flags, V3 f, V3 off, V3 Sbar, V3 Cbar,
                                         bool& anyP, bool& ali) {
    const float d2 = dot(off, off);
    const float dist = sqrtf(d2);
    const float cosA = dot(f, off * (1.0f / dist));
    const float minR = sp.sensing_min_radius;
    V3 offbar = v3(0.f, 0.f, 0.f);
    anyP = false;
    if ((flags & kAdjSep) && inBoid(dist, cosA, minR, sp.separation[1], sp.separation[2])) {
        // d/d(off) of -off/|off|^2
        const float inv = 1.0f / d2;
        offbar = offbar - Sbar * inv + off * (2.0f * dot(off, Sbar) * inv * inv);
        anyP = true;
    }
    if ((flags & kAdjCoh) && inBoid(dist, cosA, minR, sp.cohesion[1], sp.cohesion[2])) {
        offbar = offbar + Cbar;
        anyP = true;
    }
    ali = (flags & kAdjAli) && inBoid(dist, cosA, minR, sp.alignment[1], sp.alignment[2]);
    return offbar;
}

// The value that lane k of this lane's quad holds (NL == 4: four lanes of one
// agent, all active), or the lane's own (NL == 1).
template <int NL>
__device__ __forceinline__ float quad_get(float v, int k) {
    if (NL == 1) return v;
    return k == 0 ? quad_lane<0>(v) : k == 1 ? quad_lane<1>(v) : k == 2 ? quad_lane<2>(v) : quad_lane<3>(v);
}

// s + v of the quad's lanes in order: entry by entry as one lane would add them.
template <int NL>
__device__ __forceinline__ V3 quad_add(V3 s, V3 v) {
#pragma unroll
    for (int k = 0; k < NL; ++k) s = s + v3(quad_get<NL>(v.x, k), quad_get<NL>(v.y, k), quad_get<NL>(v.z, k));
    return s;
}

template <int NL>
__device__ __forceinline__ uint32_t quad_count(uint32_t v) {
    if (NL == 1) return v;
    v += (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true);  // lanes 1,0,3,2
    v += (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true);  // lanes 2,3,0,1
    return v;
}

__device__ __forceinline__ V3 keep(V3 v, bool on) { return on ? v : v3(0.f, 0.f, 0.f); }

// An agent's adjoints before its neighbours' share, and the record's vectors.
struct OwnBack {
    V3 p, f, a, S, A, C;
    float s;
    uint32_t flags;
    float wg[3];
};

// From the behaviour sums through the integrator and back to them; full: the
// agent's list is full.
__device__ __forceinline__ OwnBack own_backward(const AdjArgs& a, uint32_t id, float4 P, float4 Fw, float4 SA,
                                                float4 gP, float4 gF, float4 gA, const SteerAccum& acc, bool full) {
    const brt_steer_params& sp = a.sp;
    const V3 p = xyz(P), f = xyz(Fw), sa = xyz(SA);
    const float s = Fw.w;
    OwnBack r;
    r.wg[0] = r.wg[1] = r.wg[2] = 0.0f;
    V3 xs = v3(0.f, 0.f, 0.f), xa = xs, xc = xs, us = xs, ua = xs, uc = xs;
    V3 F = v3(0.f, 0.f, 0.f);
    if (sp.separation[0] != 0.0f) {
        if (acc.nSep > 0) {
            xs = acc.sSep / (float)acc.nSep;
            us = normalize(xs);
        }
        F = us * sp.separation[0] + F;
    }
    if (sp.alignment[0] != 0.0f) {
        if (acc.nAli > 0) {
            xa = acc.sAli / (float)acc.nAli - f;
            ua = normalize(xa);
        }
        F = ua * sp.alignment[0] + F;
    }
    if (sp.cohesion[0] != 0.0f) {
        if (acc.nCoh > 0) {
            xc = acc.sCoh / (float)acc.nCoh;
            uc = normalize(xc);
        }
        F = uc * sp.cohesion[0] + F;
    }
    V3 tgt = v3(0.f, 0.f, 0.f), seekOff = tgt;
    const bool doTarget = sp.num_targets > 0 && sp.target_weight != 0.0f;
    if (doTarget) {
        const float* t = sp.targets[id % sp.num_targets];
        tgt = v3(t[0], t[1], t[2]);
        seekOff = tgt - p;
        F = steerForSeek(p, s, f, tgt, sp.max_speed) * sp.target_weight + F;
    }
    bool doCenter = false;
    V3 centerOff = v3(0.f, 0.f, 0.f);
    if (sp.seek_world_center) {
        const brt_grid_params& g = a.g;
        const bool inside = (p.x > g.world_center[0] - g.world_radius[0]) &&
                            (p.x < g.world_center[0] + g.world_radius[0]) &&
                            (p.y > g.world_center[1] - g.world_radius[1]) &&
                            (p.y < g.world_center[1] + g.world_radius[1]) &&
                            (p.z > g.world_center[2] - g.world_radius[2]) &&
                            (p.z < g.world_center[2] + g.world_radius[2]);
        const V3 c = v3(g.world_center[0], g.world_center[1], g.world_center[2]);
        doCenter = !inside;
        centerOff = c - p;
        F = (inside ? v3(0.f, 0.f, 0.f) : steerForSeek(p, s, f, c, sp.max_speed)) + F;
    }

    // ---- forward recompute: integrator ------------------------------------
    const V3 adjF = adjustRawSteeringForce(F, s, f, sp.max_speed);
    const V3 clipped = truncateLength(adjF, sp.max_force);
    const V3 accel = clipped / sp.mass;
    float rate = 0.0f;
    V3 a1 = sa;
    if (a.dt > 0.0f) {
        rate = clampf(clampf(9.0f * a.dt, 0.15f, 0.4f), 0.0f, 1.0f);
        a1 = sa + (accel - sa) * rate;
    }
    const V3 v0 = f * s + a1 * a.dt;
    const V3 v = truncateLength(v0, sp.max_speed);

    // ---- backward: integrator -------------------------------------------
    const V3 gp1 = xyz(gP), gf1 = xyz(gF), ga1 = xyz(gA);
    const float gs1 = gF.w;
    const float vlen = length(v);
    const V3 f1 = v * (1.0f / vlen);
    V3 vbar = gp1 * a.dt + normalize_bwd(v, gf1) + f1 * gs1;
    const V3 v0bar = truncate_bwd(v0, sp.max_speed, vbar);
    V3 pbar = gp1;
    V3 fbar = v0bar * s;
    float sbar = dot(v0bar, f);
    V3 a1bar = ga1 + v0bar * a.dt;
    V3 abar = a1bar;
    V3 accbar = v3(0.f, 0.f, 0.f);
    if (a.dt > 0.0f) {
        abar = a1bar * (1.0f - rate);
        accbar = a1bar * rate;
    }
    const V3 clipbar = accbar / sp.mass;
    V3 Fbar = truncate_bwd(adjF, sp.max_force, clipbar);
    // adjustRawSteeringForce: identity unless slow and F != 0 and outside the cone
    const float maxAdj = 0.2f * sp.max_speed;
    const bool zeroF = F.x == 0.0f && F.y == 0.0f && F.z == 0.0f;
    if (!(s > maxAdj || zeroF)) {
        const float range = s / maxAdj;
        const float c = 1.0f + (-2.0f * pow20(range));
        const float L = length(F);
        const V3 d = F / L;
        if (dot(d, f) < c) {
            const V3 o = Fbar;  // dL/d(output of the cone limit)
            const float proj = dot(F, f);
            const V3 perp = F - f * proj;
            const float pl = length(perp);
            const V3 u = perp * (1.0f / pl);
            const float pd = sqrtf(1.0f - c * c);
            const V3 inner = f * c + u * pd;
            const float Lbar = dot(o, inner);
            const V3 gi = o * L;
            fbar = fbar + gi * c;
            const V3 ubar = gi * pd;
            const V3 perpbar = (ubar - u * dot(u, ubar)) * (1.0f / pl);
            Fbar = perpbar - f * dot(f, perpbar) + F * (Lbar / L);
            fbar = fbar - perpbar * proj - F * dot(f, perpbar);
            // c = 1 - 2x, x = (s/maxAdj)^20, and pd = sqrt(1 - c^2) = 2 r^10 sqrt(1 - x):
            // dc/ds = -40 r^19 / maxAdj and dpd/ds = 20 c r^9 / (maxAdj sqrt(1 - x)), finite
            // where the FP32 pd itself rounds to 0 (c rounds to 1 for small r)
            float r9 = 1.0f;
            for (int k = 0; k < 9; ++k) r9 = r9 * range;
            const float r10 = r9 * range;
            const float r19 = r9 * r10;
            const float om = 1.0f - r10 * r10;
            const float dc_ds = -40.0f * r19 / maxAdj;
            const float dpd_ds = om > 0.0f ? 20.0f * c * r9 / (maxAdj * sqrtf(om)) : 0.0f;
            sbar = sbar + dot(gi, f) * dc_ds + dot(gi, u) * dpd_ds;
        }
    }
    // seeks: d/d(p, f, s) of truncate(target - p, maxS) - f s
    if (doTarget) {
        const V3 g = Fbar * sp.target_weight;
        pbar = pbar - truncate_bwd(seekOff, sp.max_speed, g);
        fbar = fbar - g * s;
        sbar = sbar - dot(g, f);
    }
    if (doCenter) {
        pbar = pbar - truncate_bwd(centerOff, sp.max_speed, Fbar);
        fbar = fbar - Fbar * s;
        sbar = sbar - dot(Fbar, f);
    }

    // ---- backward: behaviour sums -------------------------------------------
    V3 Sbar = v3(0.f, 0.f, 0.f), Abar = Sbar, Cbar = Sbar;
    uint32_t flags = full ? kAdjFull : 0u;
    {
        const I3 gpi = calcGridPos(p.x, p.y, p.z, a.g);
        if (inGrid(gpi.x, gpi.y, gpi.z, a.g)) flags |= kAdjInGrid;
        if (gpi.x == 0 || gpi.y == 0 || gpi.z == 0) flags |= kAdjLowFace;
    }
    if (sp.separation[0] != 0.0f && acc.nSep > 0) {
        flags |= kAdjSep;
        r.wg[0] = dot(Fbar, us);
        Sbar = normalize_bwd(xs, Fbar * sp.separation[0]) * (1.0f / (float)acc.nSep);
    }
    if (sp.alignment[0] != 0.0f && acc.nAli > 0) {
        flags |= kAdjAli;
        r.wg[1] = dot(Fbar, ua);
        const V3 xbar = normalize_bwd(xa, Fbar * sp.alignment[0]);
        fbar = fbar - xbar;
        Abar = xbar * (1.0f / (float)acc.nAli);
    }
    if (sp.cohesion[0] != 0.0f && acc.nCoh > 0) {
        flags |= kAdjCoh;
        r.wg[2] = dot(Fbar, uc);
        Cbar = normalize_bwd(xc, Fbar * sp.cohesion[0]) * (1.0f / (float)acc.nCoh);
    }
    r.p = pbar;
    r.f = fbar;
    r.a = abar;
    r.S = Sbar;
    r.A = Abar;
    r.C = Cbar;
    r.s = sbar;
    r.flags = flags;
    return r;
}

// The list entries one lane takes of an agent's list, NL lanes to the agent:
// U of them from entry t on, a.n where there is none, with their positions.
template <int NL, int U>
__device__ __forceinline__ void load_entries(const AdjArgs& a, uint32_t i, uint32_t l, const uint32_t* row,
                                             uint32_t count, uint32_t t, uint32_t (&jj)[U], float4 (&q)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint32_t e = t + (uint32_t)(NL * u) + l;
        const uint32_t j = row[e < a.W - 1u ? 1u + e : 0u];
        jj[u] = e < count && j < a.n ? j : a.n;
        q[u] = a.spos[jj[u] < a.n ? jj[u] : i];
    }
}

// The agent's behaviour sums, in list order; jf, qf: the first trip's entries and
// positions, kept for own_share.
template <int NL, int U>
__device__ __forceinline__ SteerAccum own_sums(const AdjArgs& a, uint32_t i, uint32_t l, const uint32_t* row,
                                               uint32_t count, V3 p, V3 f, uint32_t (&jf)[U], float4 (&qf)[U]) {
    const brt_steer_params& sp = a.sp;
    SteerAccum acc;
    acc.init();
    load_entries<NL, U>(a, i, l, row, count, 0u, jf, qf);
    for (uint32_t t = 0; t < count; t += (uint32_t)(NL * U)) {
        uint32_t jj[U];
        float4 q[U], fq[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            jj[u] = jf[u];
            q[u] = qf[u];
        }
        if (t != 0u) load_entries<NL, U>(a, i, l, row, count, t, jj, q);
#pragma unroll
        for (int u = 0; u < U; ++u) fq[u] = a.sfwd[jj[u] < a.n ? jj[u] : i];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            SteerAccum one;
            one.init();
            const V3 off = xyz(q[u]) - p;
            if (jj[u] < a.n) one.add(sp, weights_of(sp), f, off, dot(off, off), xyz(fq[u]));
            acc.sSep = quad_add<NL>(acc.sSep, one.sSep);
            acc.sAli = quad_add<NL>(acc.sAli, one.sAli);
            acc.sCoh = quad_add<NL>(acc.sCoh, one.sCoh);
            acc.nSep += one.nSep;
            acc.nAli += one.nAli;
            acc.nCoh += one.nCoh;
        }
    }
    acc.nSep = quad_count<NL>(acc.nSep);
    acc.nAli = quad_count<NL>(acc.nAli);
    acc.nCoh = quad_count<NL>(acc.nCoh);
    return acc;
}

// The agent's share of the neighbour terms: p_i appears in every offset p_j - p_i
// of its own sums (the same per-pair terms k_adjoint_gather adds to p_j).
template <int NL, int U>
__device__ __forceinline__ V3 own_share(const AdjArgs& a, uint32_t i, uint32_t l, const uint32_t* row, uint32_t count,
                                        V3 p, V3 f, uint32_t flags, V3 S, V3 C, V3 pbar, uint32_t (&jf)[U],
                                        float4 (&qf)[U]) {
    for (uint32_t t = 0; t < count; t += (uint32_t)(NL * U)) {
        if (t != 0u) load_entries<NL, U>(a, i, l, row, count, t, jf, qf);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const V3 off = xyz(qf[u]) - p;
            bool anyP = false, ali;
            V3 o = v3(0.f, 0.f, 0.f);
            if (jf[u] < a.n) o = pair_terms(a.sp, flags, f, off, S, C, anyP, ali);
            pbar = quad_add<NL>(pbar, keep(v3(-o.x, -o.y, -o.z), anyP));
        }
    }
    return pbar;
}

__device__ __forceinline__ void store_record(const AdjArgs& a, uint32_t i, V3 p, V3 f, const OwnBack& r) {
    float4* const rec = a.rec + 4u * (size_t)i;
    rec[0] = make_float4(p.x, p.y, p.z, f.x);
    rec[1] = make_float4(f.y, f.z, r.S.x, r.S.y);
    rec[2] = make_float4(r.S.z, r.C.x, r.C.y, r.C.z);
    rec[3] = make_float4(r.A.x, r.A.y, r.A.z, __uint_as_float(r.flags));
}

// a hash entry without a valid ID: no terms
__device__ __forceinline__ void store_nothing(const AdjArgs& a, uint32_t i) {
    const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (uint32_t k = 0; k < 3u; ++k) a.own[3u * (size_t)i + k] = z;
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) a.rec[4u * (size_t)i + k] = z;
}

// sum over the wave in a fixed order, to lane 0
__device__ __forceinline__ float wave_sum(float v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o);
    return v;
}

__device__ __forceinline__ bool has_behaviours(const brt_steer_params& sp) {
    return sp.separation[0] != 0.0f || sp.alignment[0] != 0.0f || sp.cohesion[0] != 0.0f;
}

// One lane per agent.
__global__ void __launch_bounds__(256) k_adjoint_own(AdjArgs a) {
    constexpr int U = 4;
    __shared__ float s_red[3][4];
    const uint32_t i = xcd_block(a.xcd_remap) * blockDim.x + threadIdx.x;
    float wg[3] = {0.f, 0.f, 0.f};
    if (i < a.n && a.hash[i].y < a.n) {
        const uint32_t id = a.hash[i].y;
        const float4 P = a.spos[i], Fw = a.sfwd[i], SA = a.ssa[i];
        const float4 gP = a.gpos_out[id], gF = a.gfwd_out[id], gA = a.gsa_out[id];
        const V3 p = xyz(P), f = xyz(Fw);
        const uint32_t* row = a.lists + (size_t)i * a.W;
        const uint32_t count = has_behaviours(a.sp) ? (row[0] < a.W - 1u ? row[0] : a.W - 1u) : 0u;
        uint32_t jf[U];
        float4 qf[U];
        const SteerAccum acc = own_sums<1, U>(a, i, 0u, row, count, p, f, jf, qf);
        const OwnBack r = own_backward(a, id, P, Fw, SA, gP, gF, gA, acc, row[0] >= a.K);
        const V3 pbar = own_share<1, U>(a, i, 0u, row, count, p, f, r.flags, r.S, r.C, r.p, jf, qf);
        a.own[3u * (size_t)i + 0u] = make_float4(pbar.x, pbar.y, pbar.z, 0.0f);
        a.own[3u * (size_t)i + 1u] = make_float4(r.f.x, r.f.y, r.f.z, r.s);
        a.own[3u * (size_t)i + 2u] = make_float4(r.a.x, r.a.y, r.a.z, 0.0f);
        store_record(a, i, p, f, r);
        wg[0] = r.wg[0];
        wg[1] = r.wg[1];
        wg[2] = r.wg[2];
    } else if (i < a.n) {
        store_nothing(a, i);
    }
    // workgroup reduction of dL/dw in a fixed order
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float v = wave_sum(wg[k]);
        if (lane == 0) s_red[k][wave] = v;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const uint32_t nw = blockDim.x / 64u;
        float v = 0.0f;
        for (uint32_t w = 0; w < nw; ++w) v += s_red[threadIdx.x][w];
        a.partials[(size_t)blockIdx.x * 3 + threadIdx.x] = v;
    }
}

// Four lanes per agent, 64 agents per workgroup (small flocks): lane l takes the
// list entries l, l + 4, ..., and the sums add the four lanes' terms in list
// order (the same bits as one lane).  The integrator between the two walks, some
// 1,500 instructions, runs on the first wave, one lane per agent.  Bound by a
// wave's chain of list and neighbour loads, which four lanes shorten (65,536
// agents are one wave per SIMD with one lane each): 65,536 agents 23.4 us with one
// lane, 19.9 with the integrator on all four, 16.5 so.
constexpr uint32_t kOwnWords = 13u;  // LDS words per agent: odd, no bank conflicts
__global__ void __launch_bounds__(256) k_adjoint_own_quad(AdjArgs a) {
    constexpr int U = 2;
    __shared__ float s_own[64u * kOwnWords];
    const uint32_t tid = threadIdx.x, l = tid & 3u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t base = xcd_block(a.xcd_remap) * 64u;
    const uint32_t i = base + (tid >> 2), at = i < a.n ? i : a.n - 1u;
    const bool walk = i < a.n && has_behaviours(a.sp);
    const V3 p = xyz(a.spos[at]), f = xyz(a.sfwd[at]);
    const uint32_t* row = a.lists + (size_t)at * a.W;
    const uint32_t count = walk ? (row[0] < a.W - 1u ? row[0] : a.W - 1u) : 0u;
    // the first wave's agents: their own loads start now
    const uint32_t mi = base + tid;
    uint32_t id = a.n;
    float4 P, Fw, SA, gP, gF, gA;
    bool full = false;
    if (wave == 0u && mi < a.n) {
        id = a.hash[mi].y;
        P = a.spos[mi];
        Fw = a.sfwd[mi];
        SA = a.ssa[mi];
        full = a.lists[(size_t)mi * a.W] >= a.K;
        if (id < a.n) {
            gP = a.gpos_out[id];
            gF = a.gfwd_out[id];
            gA = a.gsa_out[id];
        }
    }
    uint32_t jf[U];
    float4 qf[U];
    const SteerAccum acc = own_sums<4, U>(a, at, l, row, count, p, f, jf, qf);
    float* const d = s_own + (tid >> 2) * kOwnWords;
    if (l == 0u) {
        d[0] = acc.sSep.x;
        d[1] = acc.sSep.y;
        d[2] = acc.sSep.z;
        d[3] = acc.sAli.x;
        d[4] = acc.sAli.y;
        d[5] = acc.sAli.z;
        d[6] = acc.sCoh.x;
        d[7] = acc.sCoh.y;
        d[8] = acc.sCoh.z;
        d[9] = __uint_as_float(acc.nSep | acc.nAli << 10 | acc.nCoh << 20);
    }
    __syncthreads();
    if (wave == 0u) {
        float wg[3] = {0.f, 0.f, 0.f};
        float* const m = s_own + tid * kOwnWords;
        if (id < a.n) {
            SteerAccum sum;
            sum.sSep = v3(m[0], m[1], m[2]);
            sum.sAli = v3(m[3], m[4], m[5]);
            sum.sCoh = v3(m[6], m[7], m[8]);
            const uint32_t c = __float_as_uint(m[9]);
            sum.nSep = c & 0x3FFu;
            sum.nAli = c >> 10 & 0x3FFu;
            sum.nCoh = c >> 20;
            const OwnBack r = own_backward(a, id, P, Fw, SA, gP, gF, gA, sum, full);
            m[0] = r.S.x;
            m[1] = r.S.y;
            m[2] = r.S.z;
            m[3] = r.C.x;
            m[4] = r.C.y;
            m[5] = r.C.z;
            m[6] = r.p.x;
            m[7] = r.p.y;
            m[8] = r.p.z;
            m[9] = __uint_as_float(r.flags);
            a.own[3u * (size_t)mi + 1u] = make_float4(r.f.x, r.f.y, r.f.z, r.s);
            a.own[3u * (size_t)mi + 2u] = make_float4(r.a.x, r.a.y, r.a.z, 0.0f);
            store_record(a, mi, xyz(P), xyz(Fw), r);
            wg[0] = r.wg[0];
            wg[1] = r.wg[1];
            wg[2] = r.wg[2];
        } else if (mi < a.n) {
#pragma unroll
            for (uint32_t k = 0; k < 10u; ++k) m[k] = 0.0f;  // no flags: no share
            store_nothing(a, mi);
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float v = wave_sum(wg[k]);
            if (tid == 0u) a.partials[(size_t)blockIdx.x * 3 + k] = v;
        }
    }
    __syncthreads();
    const V3 pbar = own_share<4, U>(a, at, l, row, count, p, f, __float_as_uint(d[9]), v3(d[0], d[1], d[2]),
                                    v3(d[3], d[4], d[5]), v3(d[6], d[7], d[8]), jf, qf);
    if (l == 0u && i < a.n) a.own[3u * (size_t)i] = make_float4(pbar.x, pbar.y, pbar.z, 0.0f);
}

// Lanes per agent of k_adjoint_gather: lane l takes entries l, l+L, ... of the
// agent's own list (or neighbour cells l, l+L, ... of the 27 when the list
// cannot stand in for them).
#ifndef BRT_ADJ_GATHER_LANES
#define BRT_ADJ_GATHER_LANES 4
#endif
constexpr uint32_t kGatherLanes = BRT_ADJ_GATHER_LANES;
static_assert(kGatherLanes >= 4 && kGatherLanes <= 64 && (kGatherLanes & (kGatherLanes - 1)) == 0, "lanes per agent: a power of 2, at least the three output vectors");

struct GatherArgs {
    brt_grid_params g;
    brt_steer_params sp;
    uint32_t K, W, n;
    float T;        // the list test's squared-radius threshold
    uint32_t knn;   // lists built by replacement (useKnn)
    const float4* spos;
    const uint2* hash;
    const uint32_t* lists;
    const uint32_t* cell_start;
    const uint32_t* cell_end;
    const float4* own;
    const float4* rec;
    float4* gpos_in;
    float4* gfwd_in;
    float4* gsa_in;
    const float* partials;
    uint32_t partial_blocks;
    float* weight_grad;
};

__device__ __forceinline__ I3 key_cell(uint32_t key, const brt_grid_params& g) {
    const uint32_t gx = g.grid_size[0], gy = g.grid_size[1];
    const uint32_t xy = key % (gx * gy);
    return I3{(int)(xy % gx), (int)(xy / gx), (int)(key / (gx * gy))};
}

// The ordinal of neighbour cell c of an agent in cell gi, in the visiting
// order (x offset outermost, z innermost).
__device__ __forceinline__ int cell_ordinal(I3 c, I3 gi) {
    return 9 * (c.x - gi.x + 1) + 3 * (c.y - gi.y + 1) + (c.z - gi.z + 1);
}

// Whether sorted agent j (key cell cj) is in agent i's list, given that j is
// visible to list tests, is not i and passes the radius test against i: j must
// lie in one of i's 27 cells (known when i lies inside the grid and was found
// in a cell next to j's: near); then it is in the list when the list is not
// full (every candidate that passed is), or, for a full list, when j comes no
// later than the last entry in i's visiting order (cell ordinal, then sorted
// index: the list is the first K that passed), or, for KNN lists
// (replacement), when the row holds j.
// (cj: j's key cell; for j inside the grid it is j's own cell, which from_pos
// computes from Pj only when needed.)
__device__ __forceinline__ bool in_list(const GatherArgs& a, uint32_t i, uint32_t flags_i, float4 Pi, uint32_t j,
                                        I3 cj, bool from_pos, float4 Pj, bool near) {
    const bool full = (flags_i & kAdjFull) != 0u;
    if (near && (flags_i & kAdjInGrid) && !full) return true;
    if (from_pos) cj = calcGridPos(Pj.x, Pj.y, Pj.z, a.g);
    const I3 gi = calcGridPos(Pi.x, Pi.y, Pi.z, a.g);
    if (abs(cj.x - gi.x) > 1 || abs(cj.y - gi.y) > 1 || abs(cj.z - gi.z) > 1) return false;
    if (!full) return true;
    const uint32_t* row = a.lists + (size_t)i * a.W;
    if (a.knn) {
        for (uint32_t t = 1; t <= a.K; ++t)
            if (row[t] == j) return true;
        return false;
    }
    const uint32_t last = row[a.K];
    if (last >= a.n) return false;
    const int oj = cell_ordinal(cj, gi), ol = cell_ordinal(key_cell(a.hash[last].x, a.g), gi);
    return oj < ol || (oj == ol && j <= last);
}

// The record k_adjoint_own left for an agent.
struct Rec {
    float4 r[4];
    __device__ __forceinline__ void load(const float4* rec, uint32_t i) {
#pragma unroll
        for (int k = 0; k < 4; ++k) r[k] = rec[4u * (size_t)i + k];
    }
    __device__ __forceinline__ uint32_t flags() const { return __float_as_uint(r[3].w); }
    // adds the terms the agent's list holds for p_j and f_j (off = p_j - p_i)
    __device__ __forceinline__ void add_pair(const brt_steer_params& sp, V3 off, V3& accP, V3& accF) const {
        bool anyP, ali;
        const V3 offbar = pair_terms(sp, flags(), v3(r[0].w, r[1].x, r[1].y), off, v3(r[1].z, r[1].w, r[2].x),
                                     v3(r[2].y, r[2].z, r[2].w), anyP, ali);
        if (anyP) accP = accP + offbar;
        if (ali) accF = accF + xyz(r[3]);
    }
};

// The key coordinate, on one axis, of the cells whose agents can hold in their
// lists an agent of key coordinate c: c + d for d = -1, 0, 1 inside the grid,
// except that for c = 0 the offset -1 stands for coordinate G-1, where the
// hash keys agents whose coordinate lies below the grid (calcGridHash's
// unsigned clamp); -1: no such cell.
__device__ __forceinline__ int gather_axis(int c, int d, uint32_t G) {
    if (d < 0 && c == 0) return (int)G - 1 > 1 ? (int)G - 1 : -1;
    const int k = c + d;
    return (k >= 0 && k < (int)G) ? k : -1;
}

// dL/d(p_j, f_j, s_j, a_j) by agent ID: agent j's own terms plus the terms of
// every agent i whose list holds j.  When j lies in the grid, its list is not
// full and maxBodiesPerCell cuts no cell, those agents are all in j's own list
// (the radius test is symmetric: d2 has the same bits both ways), so the lanes
// walk that list; for j on a low face of the grid they also scan the far
// face's cells in which agents below the grid are kept (j's list does not reach
// those).  Otherwise they scan the 27 cells around j's cell.
// Each lane sums its part in order and the lanes' sums are combined by a fixed
// butterfly.  Bound by the slowest lane's chain of loads, so all of an agent's own
// are in flight together, then two entries' 64-byte records, and agents on a low
// face (7 % of a 40^3 grid's, nearly every wave has one) walk their list too
// instead of 27 cells: 65,536 agents, one per cell, 33.0 -> 16.0 us.  The last workgroup adds the weight-gradient partials of
// k_adjoint_own in a fixed order and does nothing else.
__global__ void __launch_bounds__(256) k_adjoint_gather(GatherArgs a) {
    if (blockIdx.x == gridDim.x - 1u) {
        reduce_partials(a.partials, a.partial_blocks, a.weight_grad);
        return;
    }
    constexpr uint32_t L = kGatherLanes;
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t j = t / L, l = t % L;
    const brt_steer_params& sp = a.sp;
    const brt_grid_params& g = a.g;
    V3 accP = v3(0.f, 0.f, 0.f), accF = accP;
    uint32_t id = a.n;
    float4 own = make_float4(0.f, 0.f, 0.f, 0.f);
    if (j < a.n) {
        // all of the agent's own loads in flight together
        const uint2 hj = a.hash[j];
        const float4 Pj = a.spos[j];
        const uint32_t fj = __float_as_uint(a.rec[4u * (size_t)j + 3u].w);
        const uint32_t* row = a.lists + (size_t)j * a.W;
        const uint32_t cnt = row[0] < a.W - 1u ? row[0] : a.W - 1u;
        constexpr uint32_t kAhead = 2u;  // entries of a lane in flight
        uint32_t ii[kAhead];
#pragma unroll
        for (uint32_t u = 0; u < kAhead; ++u) ii[u] = row[l + u * L < a.W - 1u ? 1u + l + u * L : 0u];
        own = a.own[3u * (size_t)j + (l < 3u ? l : 0u)];
        id = hj.y;
        const uint32_t key = hj.x;
        const bool behaviours = sp.separation[0] != 0.0f || sp.alignment[0] != 0.0f || sp.cohesion[0] != 0.0f;
        const bool unlimited = g.max_bodies_per_cell == 0xFFFFFFFFu;
        // maxBodiesPerCell hides agents past the first ones of their cell from
        // every list test
        const bool visible = key < g.num_cells && (unlimited || j - a.cell_start[key] < g.max_bodies_per_cell);
        if (behaviours && id < a.n && visible) {
            const V3 pj = xyz(Pj);
            const bool by_list = unlimited && (fj & kAdjInGrid) && !(fj & kAdjFull);
            if (by_list) {
                for (uint32_t e = l; e < cnt; e += kAhead * L) {
                    if (e != l) {
#pragma unroll
                        for (uint32_t u = 0; u < kAhead; ++u)
                            ii[u] = row[e + u * L < a.W - 1u ? 1u + e + u * L : 0u];
                    }
                    Rec R[kAhead];
#pragma unroll
                    for (uint32_t u = 0; u < kAhead; ++u) {
                        if (e + u * L >= cnt || ii[u] >= a.n) ii[u] = a.n;
                        R[u].load(a.rec, ii[u] < a.n ? ii[u] : j);
                    }
#pragma unroll
                    for (uint32_t u = 0; u < kAhead; ++u) {
                        const uint32_t i = ii[u];
                        if (i >= a.n) continue;
                        if (!in_list(a, i, R[u].flags(), R[u].r[0], j, I3{0, 0, 0}, true, Pj, true)) continue;
                        R[u].add_pair(sp, pj - xyz(R[u].r[0]), accP, accF);
                    }
                }
            }
            if (!by_list || (fj & kAdjLowFace)) {
                // the lane's cells: their ranges load together, then the first
                // agent of each (a chain of three loads instead of three per cell)
                constexpr uint32_t kCells = (27u + L - 1u) / L;
                const I3 cj = key_cell(key, g);
                uint32_t cs[kCells], ce[kCells], nearby = 0u;
#pragma unroll
                for (uint32_t k = 0; k < kCells; ++k) {
                    const uint32_t c = l + k * L;
                    const int dx = (int)(c / 9u) - 1, dy = (int)((c / 3u) % 3u) - 1, dz = (int)(c % 3u) - 1;
                    const int nx = gather_axis(cj.x, dx, g.grid_size[0]);
                    const int ny = gather_axis(cj.y, dy, g.grid_size[1]);
                    const int nz = gather_axis(cj.z, dz, g.grid_size[2]);
                    const bool near = nx == cj.x + dx && ny == cj.y + dy && nz == cj.z + dz;
                    const bool take = c < 27u && nx >= 0 && ny >= 0 && nz >= 0 && !(by_list && near);
                    cs[k] = BRT_EMPTY_CELL;
                    ce[k] = 0u;
                    if (take) {
                        const uint32_t nk = cellKey(nx, ny, nz, g);
                        cs[k] = a.cell_start[nk];
                        ce[k] = a.cell_end[nk];
                    }
                    nearby |= near ? 1u << k : 0u;
                }
                float4 first[kCells];
#pragma unroll
                for (uint32_t k = 0; k < kCells; ++k) {
                    first[k] = Pj;
                    if (cs[k] != BRT_EMPTY_CELL) first[k] = a.spos[cs[k]];
                }
#pragma unroll
                for (uint32_t k = 0; k < kCells; ++k) {
                    if (cs[k] == BRT_EMPTY_CELL) continue;
                    float4 Pi = first[k];
                    for (uint32_t i = cs[k]; i < ce[k];) {
                        const uint32_t here = i++;
                        const float4 Ph = Pi;
                        if (i < ce[k]) Pi = a.spos[i];
                        if (here == j) continue;
                        // the list test of agent `here` for candidate j (d2 as k_prox forms it)
                        const V3 off = pj - xyz(Ph);
                        if (dot(off, off) > a.T) continue;
                        Rec R;
                        R.load(a.rec, here);
                        if (!in_list(a, here, R.flags(), Ph, j, cj, false, Pj, (nearby >> k & 1u) != 0u)) continue;
                        R.add_pair(sp, off, accP, accF);
                    }
                }
            }
        }
    }
#pragma unroll
    for (uint32_t o = 1; o < L; o <<= 1) {
        accP.x += __shfl_xor(accP.x, (int)o);
        accP.y += __shfl_xor(accP.y, (int)o);
        accP.z += __shfl_xor(accP.z, (int)o);
        accF.x += __shfl_xor(accF.x, (int)o);
        accF.y += __shfl_xor(accF.y, (int)o);
        accF.z += __shfl_xor(accF.z, (int)o);
    }
    // lane 0 stores dL/dp, lane 1 dL/d(f, s), lane 2 dL/da
    if (j < a.n && l < 3u && id < a.n) {
        const V3 more = l == 0u ? accP : accF;
        float4 r = own;
        if (l < 2u) r = make_float4(own.x + more.x, own.y + more.y, own.z + more.z, l == 0u ? 0.0f : own.w);
        float4* const out = l == 0u ? a.gpos_in : (l == 1u ? a.gfwd_in : a.gsa_in);
        out[id] = r;
    }
}

// Agents up to which k_adjoint_own takes four lanes per agent.
constexpr uint32_t kOwnQuadMax = 1u << 17;

}  // namespace

hipError_t launch_adjoint(const brt_grid_params& g, const brt_prox_params& p, float threshold,
                          const brt_steer_params& sp, float dt, uint32_t n, const float4* spos, const float4* sfwd,
                          const float4* ssa, const uint2* hash, const uint32_t* lists, const uint32_t* cell_start,
                          const uint32_t* cell_end, const float4* gpos_out, const float4* gfwd_out,
                          const float4* gsa_out, float4* gpos_in, float4* gfwd_in, float4* gsa_in, float4* scratch,
                          float* partials, float* weight_grad, uint32_t xcd_remap, hipStream_t s) {
    AdjArgs a{};
    a.g = g;
    a.sp = sp;
    a.dt = dt;
    a.K = p.max_neighbors;
    a.W = list_stride(p.max_neighbors);
    a.n = n;
    a.spos = spos;
    a.sfwd = sfwd;
    a.ssa = ssa;
    a.hash = hash;
    a.lists = lists;
    a.gpos_out = gpos_out;
    a.gfwd_out = gfwd_out;
    a.gsa_out = gsa_out;
    a.rec = scratch;  // 64-byte aligned
    a.own = scratch + 4u * (size_t)n;
    a.partials = partials;
    a.xcd_remap = xcd_remap;
    const bool quads = n <= kOwnQuadMax;
    const uint32_t blocks = quads ? (n + 63u) / 64u : (n + 255u) / 256u;
    if (quads)
        hipLaunchKernelGGL(k_adjoint_own_quad, dim3(blocks), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL(k_adjoint_own, dim3(blocks), dim3(256), 0, s, a);
    GatherArgs b{};
    b.g = g;
    b.sp = sp;
    b.K = p.max_neighbors;
    b.W = a.W;
    b.n = n;
    b.T = threshold;
    b.knn = p.use_knn ? 1u : 0u;
    b.spos = spos;
    b.hash = hash;
    b.lists = lists;
    b.cell_start = cell_start;
    b.cell_end = cell_end;
    b.own = a.own;
    b.rec = a.rec;
    b.gpos_in = gpos_in;
    b.gfwd_in = gfwd_in;
    b.gsa_in = gsa_in;
    b.partials = partials;
    b.partial_blocks = blocks;
    b.weight_grad = weight_grad;
    const size_t threads = (size_t)n * kGatherLanes;
    hipLaunchKernelGGL(k_adjoint_gather, dim3((unsigned)((threads + 255) / 256) + 1u), dim3(256), 0, s, b);
    return hipGetLastError();
}

}  // namespace brt
