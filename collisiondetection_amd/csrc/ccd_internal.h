// Internal declarations shared by the HIP translation units of libccd_amd.so.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <string>
#include <unordered_map>

#include "../../include/ccd_amd.h"

// Launch shape of the narrowphase (tuned by ccd_autotune).  Both forms use the tile; block and waves_per_cu shape
// the persistent grid of the one-pass form.
struct QueueShape {
    int block = 256;       // threads per block: 64, 128 or 256
    int tile = 1024;       // stencils a wavefront takes at a time (fewer on short lists)
    int waves_per_cu = 8;  // resident wavefronts per compute unit in the persistent grid (two per SIMD)
    int group = 0;         // accepted and reported, without effect (0 or 1)
};

struct ccd_ctx {
    int device = 0;
    int num_cus = 256;
    bool ee_split = true;         // edge-edge narrowphase screened, else in one pass
    QueueShape vf_shape;
    QueueShape ee_shape;
    hipStream_t own_stream = nullptr;
    hipStream_t stream = nullptr;
    std::string err;
    struct Buf {
        void *ptr = nullptr;
        size_t bytes = 0;
        bool external = false;   // memory owned by someone else (a server's pool): never freed here
    };
    std::unordered_map<std::string, Buf> bufs;   // named grow-only device buffers
    int64_t device_bytes = 0;
    int64_t *h_counts = nullptr;                  // pinned host mailbox for device counters
    int64_t *d_counts = nullptr;                  // device counters (CCD_NCOUNTERS int64)
    // Stage timing with HIP events on the context's stream (ccd_set_profiling).
    bool profiling = false;
    hipEvent_t ev[2 * CCD_NTIMERS] = {};
    bool pending[CCD_NTIMERS] = {};
    double stage_ms[CCD_NTIMERS] = {};
    int64_t stage_calls[CCD_NTIMERS] = {};
    // Grow-only capacities of the broadphase outputs (tiles of the related-face rows, stencils).
    int64_t cap_rows = 0, cap_vf = 0, cap_ee = 0;
    bool count_pairs = false;   // whether C_PAIRS is computed (a server reports it)
    // Sorted face order of the last full broadphase build (kept for refits).
    const int32_t *tree_order = nullptr;
    // Captured detection pipeline (ccd_batch_detect with CCD_GRAPH): replayed while its arguments match.
    bool capturing = false;
    bool graph_valid = false;
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    unsigned char graph_key[256] = {};
    int64_t graph_replays = 0;
    // The candidates of the last broadphase (ccd_last_candidates).
    const int32_t *last_vf = nullptr, *last_ee = nullptr;
    int64_t last_nvf = 0, last_nee = 0;
};

namespace ccdi {

constexpr int NCOUNTERS = 16;

// Counter slots in ctx->d_counts.
enum Counter {
    C_PAIRS = 0,    // overlapping non-neighbouring face pairs (where count_pairs is set)
    C_VF = 1,       // unique vertex-face stencils
    C_EE = 2,       // unique edge-edge stencils
    C_VF_HITS = 3,  // colliding vertex-face stencils
    C_EE_HITS = 4,  // colliding edge-edge stencils
    C_BAD = 5,      // validation failures
    C_ROWS = 6,     // tiles of the related-face rows
};

int set_error(ccd_ctx *ctx, int code, const char *fmt, ...);
// Stage timers: no-ops unless profiling is on.  prof_collect needs the stream to be synchronised.
void prof_begin(ccd_ctx *ctx, int timer);
void prof_end(ccd_ctx *ctx, int timer);
void prof_collect(ccd_ctx *ctx);
// Grow-only named device buffer.  Returns nullptr (and sets the context error) on failure.
void *buffer(ccd_ctx *ctx, const char *name, size_t bytes);

}   // namespace ccdi

#define CCD_HIP_CHECK(ctx, call)                                                                          \
    do {                                                                                                  \
        hipError_t _e = (call);                                                                           \
        if (_e != hipSuccess)                                                                             \
            return ccdi::set_error((ctx), CCD_E_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(_e), \
                                   __FILE__, __LINE__);                                                   \
    } while (0)

#define CCD_LAUNCH_CHECK(ctx) CCD_HIP_CHECK(ctx, hipGetLastError())

// ----------------------------------------------------------------------------------------------
// Narrowphase launchers (narrowphase.hip)
// ----------------------------------------------------------------------------------------------
namespace ccdi {
// The context's counters that a narrowphase works with, one buffer size for every caller (a request to grow it
// frees and allocates, and so stalls the device): [0..1] the one-pass form's queues, [2..3] a server's checksums
// of the hits.  Null without memory.
constexpr int QUEUE_WORK = 4;
inline unsigned long long *queue_work(ccd_ctx *ctx) { return (unsigned long long *)buffer(ctx, "queue_work", QUEUE_WORK * 8); }
int launch_primitives(ccd_ctx *ctx, int kind, const double *q, const double *eta, double eta_s, int64_t n,
                      uint8_t *hit, double *t);
// Where a narrowphase's results go: appended to a hit list (PER_STENCIL false), or at each stencil's own
// index, with a thickness per stencil (PER_STENCIL true).
struct NarrowOut {
    int4 *out_keys = nullptr;
    double *out_toi = nullptr;
    int64_t cap = 0;
    unsigned long long *counter = nullptr;
    const double *eta = nullptr;   // per stencil, or null
    uint8_t *hit = nullptr;
    double *t = nullptr;
    uint8_t *sub = nullptr;
};
// The screening narrowphase (screened.hip) over n stencils (or the device count n_dev, if smaller), n < 2^31.
// list: open_list_bytes of device memory for at least n stencils, uninitialised; tile: stencils that a
// wavefront takes at a time on long lists.  open_list: the context's buffer, or null for n >= 2^31.
int launch_screened(ccd_ctx *ctx, bool vf, bool per_stencil, const double *qs, const double *qe, const int32_t *keys,
                    const int64_t *n_dev, int64_t n, double eta, const NarrowOut &o, int tile, void *list);
// Windows of multi-entry histories that a kernel gathers for the screening narrowphase, in shards with a
// counter each (claims on one counter take about 10 ns each, one after another).
struct WindowPool {
    static constexpr int SHARDS = 64, STRIDE = 8;   // (a counter per 64 bytes)
    double *pos;        // [24 * capacity] four vertices at the window's start, four at its end
    double *eta;
    int32_t *owner;     // the stencil, -1: nothing here
    uint32_t *place;    // the window among the stencil's
    uint8_t *hit;       // results, as launch_narrow2's
    uint8_t *sub;
    double *t;
    unsigned long long *claimed;   // [SHARDS * STRIDE]; may exceed per_shard
    int64_t per_shard;             // a multiple of 64; at most 65,536 for all shards' regions of 64
    __device__ __forceinline__ int64_t filled(int64_t shard) const
    {
        const int64_t c = (int64_t)claimed[shard * STRIDE];
        return c < per_shard ? c : per_shard;
    }
};
int launch_screened_pool(ccd_ctx *ctx, bool vf, const WindowPool &pool, void *list);
int64_t open_list_bytes(int64_t n);
void *open_list(ccd_ctx *ctx, int64_t n);
// One result per stencil.  list: the caller's, for these n stencils, else the context's own.
int launch_narrow2(ccd_ctx *ctx, bool vf, const double *qs, const double *qe, const int32_t *keys,
                   const double *eta, double eta_s, int64_t n, uint8_t *hit, double *t, uint8_t *sub,
                   void *list = nullptr);
// entries: history entries per vertex on average.
int launch_narrow_hist(ccd_ctx *ctx, bool vf, const int64_t *off, const double *ht, const double *hp,
                       const int32_t *keys, const double *eta, double eta_s, int64_t n, uint8_t *hit, double *t,
                       uint8_t *sub, int32_t *win, int64_t entries);
// Narrowphase over a stencil list, appending the colliding stencils (keys and times) to out_keys / out_toi
// with a device counter; at most cap are written.  Screened when `list` (for at least n_max stencils) is
// given, else the whole cascade on a persistent work queue, whose counter *work must be zero.
int launch_narrow2_queue(ccd_ctx *ctx, bool vf, const double *qs, const double *qe, const int32_t *keys,
                         const int64_t *n_dev, int64_t n_max, double eta, int32_t *out_keys, double *out_toi,
                         int64_t cap, int64_t *counter, unsigned long long *work, const QueueShape &shape,
                         void *list = nullptr);
// Work accounting: per-stage execution counts (ccd::Stage order) summed over the stencils into counts.
int launch_narrow2_count(ccd_ctx *ctx, bool vf, const double *qs, const double *qe, const int32_t *keys,
                         int64_t n, double eta, unsigned long long *counts);
// Validation: counts keys outside [0, nverts) into *bad.
// Separating-plane narrowphase over a CSR history: launch_min_gap writes History::computeMinimumGap's
// value (as bits) to *gap_bits on the device; launch_separating_plane reads it (eps = gap / 4).
int launch_min_gap(ccd_ctx *ctx, const int64_t *off, const double *ht, int64_t nverts, uint64_t *gap_bits);
// entries: history entries per vertex on average.
int launch_separating_plane(ccd_ctx *ctx, bool vf, const int64_t *off, const double *ht, const double *hp,
                            const int32_t *keys, const double *eta, double eta_s, int64_t n, const uint64_t *gap_bits,
                            uint8_t *status, int64_t *undecided, int64_t entries);
int launch_validate_keys(ccd_ctx *ctx, const int32_t *keys, int64_t n4, int64_t nverts, int64_t *bad);
int launch_validate_history(ccd_ctx *ctx, const int64_t *off, const double *ht, int64_t nverts, int64_t nentries,
                            int64_t *bad);

// ----------------------------------------------------------------------------------------------
// Broadphase (broadphase.hip).  Produces the unique candidate stencils in device buffers owned by
// the context; *vf / *ee receive their device addresses and the counts are left in ctx->d_counts.
// ----------------------------------------------------------------------------------------------
struct Candidates {
    int32_t *vf = nullptr;
    int32_t *ee = nullptr;
    int64_t nvf = 0, nee = 0;
    int64_t vf_cap = 0, ee_cap = 0;
};
// aabb selects AABBBroadPhase's 3-axis bounds (used by the mesh self-distance), else the 13-axis k-DOP.
// inst_off (device, ninst+1 face offsets) runs independent instances in one pass: no pair crosses
// instances.  Synchronous: checks capacities and reruns after growing them.
int broadphase(ccd_ctx *ctx, const int32_t *faces, int64_t F, const double *qs, const double *qe,
               const int64_t *hist_off, const double *hist_pos, int64_t V, double eta, const uint8_t *fixed,
               Candidates &out, bool aabb = false, const int64_t *inst_off = nullptr, int ninst = 1);
// The same pipeline as launches only (no host synchronisation, no allocation once prepared): it can be
// captured in a HIP graph.  Counts land in ctx->d_counts; buffers must come from broadphase_prepare.
int broadphase_prepare(ccd_ctx *ctx, int64_t F, int64_t V, bool batched);
int broadphase_launch(ccd_ctx *ctx, const int32_t *faces, int64_t F, const double *qs, const double *qe,
                      const int64_t *hist_off, const double *hist_pos, int64_t V, double eta, const uint8_t *fixed,
                      bool aabb, const int64_t *inst_off, int ninst);
int build_vertex_face_table_buffers(ccd_ctx *ctx, int64_t F, int64_t V);
// Refit of the last full build's tree with new positions (launches only; see broadphase.hip).
int broadphase_refit_launch(ccd_ctx *ctx, const int32_t *faces, int64_t F, const double *qs, const double *qe,
                            int64_t V, double eta, const uint8_t *fixed, const int64_t *inst_off, int ninst);
// Vertex -> face CSR table (device buffers "vf_off" / "vf_list"), and its current addresses.
int build_vertex_face_table(ccd_ctx *ctx, const int32_t *faces, int64_t F, int64_t V);
void vertex_face_table(ccd_ctx *ctx, const int32_t **off, const int32_t **list);
int sort_stencils(ccd_ctx *ctx, int32_t *keys, int64_t n);

// Device-wide primitives (devprims.hip): plain launches, safe inside a captured graph.
int fill_u32(ccd_ctx *ctx, uint32_t *p, int64_t n, uint32_t v);
int fill_u64(ccd_ctx *ctx, uint64_t *p, int64_t n, uint64_t v);
size_t scan_temp_bytes(int64_t n);
int exclusive_scan_i32(ccd_ctx *ctx, const int32_t *in, int32_t *out, int64_t n, void *temp, int64_t *total);
int exclusive_scan_i64(ccd_ctx *ctx, const int64_t *in, int64_t *out, int64_t n, void *temp, int64_t *total);
size_t radix_sort_temp_bytes(int64_t n);
// Sorts by the low `bits` bits of the keys; the result is in (keys_alt, vals_alt) when result_in_alt.
int radix_sort_pairs(ccd_ctx *ctx, uint64_t *keys, int32_t *vals, uint64_t *keys_alt, int32_t *vals_alt, int64_t n,
                     int bits, void *temp, bool &result_in_alt);

// Proximity (distance.hip)
int launch_distance_primitives(ccd_ctx *ctx, int kind, const double *q, double eta, int64_t n, uint8_t *flag,
                               double *vec, double *bary);
int mesh_self_distance(ccd_ctx *ctx, const double *verts, int64_t V, const int32_t *faces, int64_t F,
                       const uint8_t *fixed, double *out, int64_t *nvf, int64_t *nee);
}   // namespace ccdi
