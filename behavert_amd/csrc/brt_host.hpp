// brt_host.hpp -- the library context and the host-side helpers shared by the
// C ABI translation units (status codes, validation, scratch management).
#pragma once

#include <hip/hip_runtime.h>

#include <array>
#include <string>
#include <vector>

#include "../../include/behavert_amd.h"
#include "brt_internal.hpp"

struct brt_context {
    int device = 0;
    std::string err;
    void* tmp = nullptr;        // sort ping-pong buffer (uint2[n]); label ping-pong (float[2n])
    size_t tmp_bytes = 0;
    uint32_t* meta = nullptr;   // histograms, tile counters, look-back status
    size_t meta_bytes = 0;
    // every word of meta is zero once the work enqueued so far has run: the
    // last sort on it was a step's, whose passes and reorder return what they
    // used to zero; then the next step's sort needs no clearing launch
    bool meta_clean = false;
    float* partials = nullptr;  // adjoint: per-workgroup weight-gradient partials
    size_t partials_bytes = 0;
    void* xyz = nullptr;        // brt_step: the sorted positions packed as x,y,z
    size_t xyz_bytes = 0;
    // brt_step: the state by ID as records (step_record_bytes); brt_bc_similarities_steer:
    // the neighbours' (bc_record_bytes)
    void* records = nullptr;
    size_t records_bytes = 0;
    uint32_t* dev_flags = nullptr;  // sticky device-side failure flags (BRT_DEVFLAG_*)
    void* scratch = nullptr;        // this device's no-allocation step scratch (a static device array)
    bool timing = false;
    // per timed step: a start and a stop event per phase (bound to the
    // phase's first and last kernel) and the mask of the phases that ran
    std::vector<std::array<hipEvent_t, 2 * BRT_NUM_PHASES>> events;
    std::vector<uint32_t> events_mask;
    size_t events_used = 0;
    double phase_ms[BRT_NUM_PHASES] = {0, 0, 0, 0, 0};
    uint32_t phase_steps = 0;
    int fused_step = -1;        // -1: automatic (resolve_fused)
    uint32_t uniform_max_cells = 1;
    uint32_t xcd_remap = 1;
    int lds_lists = -1;         // -1: automatic (resolve_lds_lists)
    // brt_step's captured graphs (BRT_OPT_STEP_GRAPH), most recently used last,
    // and the key of the last call (a graph is captured on the second call
    // with a key)
    int step_graph = 0;
    hipStream_t cap_stream = nullptr;
    struct StepGraph {
        std::vector<unsigned char> key;
        void* tmp = nullptr;  // the scratch the graph was captured with
        uint32_t* meta = nullptr;
        void* xyz = nullptr;
        void* records = nullptr;
        hipGraph_t graph = nullptr;
        hipGraphExec_t exec = nullptr;
    };
    std::vector<StepGraph> graphs;
    std::vector<unsigned char> last_key;
};

// Automatic launch shapes, from the K = 32 and K = 64 workloads measured on
// gfx950: at K = 32 the fused neighbour + steering kernel and LDS-staged lists
// are fastest; beyond, two passes with register-chunk lists unless the flock's
// size and grid say otherwise (resolve_step).
inline bool resolve_fused(const brt_context* ctx, const brt_prox_params* p) {
    return ctx->fused_step >= 0 ? ctx->fused_step != 0 : p->max_neighbors <= 32u;
}
inline uint32_t resolve_lds_lists(const brt_context* ctx, const brt_prox_params* p) {
    return ctx->lds_lists >= 0 ? (uint32_t)(ctx->lds_lists != 0) : (p->max_neighbors <= 32u ? 1u : 0u);
}
// Whether the neighbour search of n agents takes four lanes per agent (lists
// automatic), and so packs their positions.
inline bool resolve_quads(const brt_context* ctx, const brt_prox_params* p, uint32_t n, bool fused) {
    return ctx->lds_lists < 0 && !p->use_knn && brt::prox_quad_fits(p->max_neighbors, n, fused);
}
// Lists beyond K = 32, automatic: from K 81 on the LDS rows leave too few waves.
inline bool wide_lists(const brt_context* ctx, const brt_prox_params* p) {
    return ctx->lds_lists < 0 && !p->use_knn && p->max_neighbors > 32u && p->max_neighbors <= 80u;
}
// Whether a list pass alone stages such lists in LDS: in crowded grids, whose
// waves then scan in flat mode.  A two-pass step with features, 1,048,576 agents,
// K 40, registers -> LDS at 1 / 4 / 16 per cell: 386 -> 402, 513 -> 536, 975 ->
// 767 us; K 64 419 -> 460, 547 -> 612, 1271 -> 1120.
inline uint32_t resolve_list_lds(const brt_context* ctx, const brt_prox_params* p, uint32_t n, uint32_t cells) {
    return wide_lists(ctx, p) ? (n / 8u >= cells ? 1u : 0u) : resolve_lds_lists(ctx, p);
}

// The shape of a step of n agents in a grid of `cells`.  Beyond K = 32:
//   * fused where the quads take the whole step in one launch (K 64, one per cell,
//     1,000 / 65,536 agents: 26 / 44 us in two passes, 21 / 36 in one);
//   * fused with LDS lists up to K 80, two passes with register lists -> fused at
//     1 / 4 / 16 per cell / in blobs: 1,048,576 agents, K 48, 353 -> 320, 471 ->
//     408, 972 -> 607, 1108 -> 701 us, K 64 377 -> 369, 494 -> 462, 1146 -> 805,
//     1274 -> 889, K 80 402 -> 402, 513 -> 514, 1213 -> 949, 1410 -> 1083 (K 100
//     420 -> 469, 1230 -> 1251); but from 2^21 agents only where the grid is
//     crowded: 2,097,152 agents, K 64, 729 -> 802, 936 -> 984, 2267 -> 1651;
//   * two passes with the feature update, whose steering pass does it (fused and
//     the features apart: 433 us against 386 at K 40 and one per cell, 823
//     against 767 at 16).
struct StepShape {
    bool fused;
    uint32_t lds;
};
inline StepShape resolve_step(const brt_context* ctx, const brt_prox_params* p, uint32_t n, uint32_t cells,
                              bool features) {
    if (p->use_knn) return StepShape{false, resolve_lds_lists(ctx, p)};
    bool fused = resolve_fused(ctx, p);
    if (ctx->fused_step < 0 && !features)
        fused = fused || resolve_quads(ctx, p, n, true) ||
                (wide_lists(ctx, p) && (n < (1u << 21) || n / 8u >= cells));
    return StepShape{fused, fused && wide_lists(ctx, p) ? 1u : resolve_list_lds(ctx, p, n, cells)};
}

namespace brt {
namespace host {

int set_err(brt_context* ctx, int code, const char* fmt, ...);
int hip_err(brt_context* ctx, hipError_t e, const char* what);
int use_device(brt_context* ctx);
int check_grid(brt_context* ctx, const brt_grid_params* g);
int check_n(brt_context* ctx, uint32_t n);
// the neighbour kernels address positions with 32-bit byte offsets
int check_n_lists(brt_context* ctx, uint32_t n);
int check_prox(brt_context* ctx, const brt_prox_params* p);
int check_steer(brt_context* ctx, const brt_steer_params* s);
int ensure_tmp(brt_context* ctx, size_t bytes);
int ensure_scratch(brt_context* ctx, uint32_t n, const brt::SortPlan& plan);
// Scratch that its callers can do without and that does not grow while s is being
// captured: whether the records hold `need` bytes; the packed positions of n
// agents, or NULL (the neighbour search then reads the float4 ones).
bool ensure_records(brt_context* ctx, size_t need, hipStream_t s);
float* step_xyz(brt_context* ctx, uint32_t n, hipStream_t s);
// synchronises the device, reads and clears the sticky flags; BRT_ERR_HIP with
// a message when one was raised
int check_dev_flags(brt_context* ctx);

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace host
}  // namespace brt

#define BRT_HIP(call, what)                              \
    do {                                                 \
        hipError_t e_ = (call);                          \
        if (e_ != hipSuccess) return hip_err(ctx, e_, what); \
    } while (0)

#define BRT_REQUIRE(cond, ...)                                              \
    do {                                                                    \
        if (!(cond)) return set_err(ctx, BRT_ERR_INVALID_ARGUMENT, __VA_ARGS__); \
    } while (0)

