// fs_host.cpp -- C ABI of libflexshell: contexts, models, CSR pattern and
// scatter-plan construction, and the launch sequences of the hot path.
//
// Nothing here computes element or matrix values on the host: the host only
// builds integer structure (node adjacency, CSR pattern, pair tables) and
// small per-material factors; all floating-point work of stiffness, mass,
// normals and the time loop runs in the kernels of fs_kernels.hip.
#include <hip/hip_runtime.h>

#include <fcntl.h>
#include <sys/file.h>
#include <sys/stat.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <cerrno>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <new>
#include <string>
#include <thread>
#include <type_traits>
#include <vector>

#include "../../include/flexshell.h"
#include "fs_device.h"
#include "fs_threads.h"

namespace fs {
hipError_t launch_element_blocks(const ElemParams &p, const double *x, const double *y, const double *z,
                                 const int32_t *conn, const double *nx, const double *ny, const double *nz,
                                 const uint8_t *valid, double *Kb, int *status, hipStream_t st, int variant);
int element_variants(int nen);
void element_variant_shape(int nen, int variant, int *ne, int *wg);
hipError_t launch_scatter(const ScatterPlan &sp, const double *Kb, double *vals, hipStream_t st);
int64_t scan_tiles(int64_t n);
hipError_t launch_neighbours(bool fill, int64_t N, int nen, int64_t E, const int32_t *conn, const int32_t *ne_ptr,
                             const int32_t *ne_list, int32_t *nbr_ptr, int32_t *nbr, int64_t *sums, hipStream_t st);
hipError_t launch_plan_rows(const PlanArgs &a, hipStream_t st);
hipError_t launch_plan_pairs(const PlanArgs &a, hipStream_t st);
hipError_t launch_tile_place(int64_t n, const int32_t *pairs, const ScatterPlan &sp, const int4 *node_rec, int4 *rec,
                             hipStream_t st);
hipError_t launch_pattern_rows(int64_t n, const int32_t *rowptr, int base, int64_t *out, hipStream_t st);
hipError_t launch_pattern_cols(const ScatterPlan &sp, const int64_t *node_dof, int base, int64_t w0, int64_t w1,
                               int64_t *col, hipStream_t st);
int fused_tile_elems(int nen);
hipError_t launch_element_fused(const ElemParams &p, const double *x, const double *y, const double *z,
                                const int32_t *conn, const double *nx, const double *ny, const double *nz,
                                const uint8_t *valid, int *status, const ScatterPlan &sp, const TilePlan &tp,
                                double *vals, hipStream_t st);
hipError_t launch_pair_finalize(const ScatterPlan &sp, const TilePlan &tp, double *vals, hipStream_t st);
hipError_t launch_normals(int nen, int64_t N, int E, const double *x, const double *y, const double *z,
                          const int32_t *conn, const int32_t *ne_ptr, const int32_t *ne_list, double ntol,
                          const double *gnrm, const int32_t *egroup, double *nx, double *ny, double *nz,
                          uint8_t *valid, hipStream_t st);
hipError_t launch_number_dofs(int64_t n, const uint8_t *fixed, int64_t *tile_free, int64_t *total, int64_t *dof,
                              hipStream_t st);
int64_t number_dofs_tiles(int64_t n);
hipError_t launch_surface_load(int nen, int npts, int64_t N, int E, const double *x, const double *y,
                               const double *z, const int32_t *conn, const int32_t *ne_ptr, const int32_t *ne_list,
                               int per_point, const double *force, const int64_t *node_dof, int64_t nrows, double *F,
                               hipStream_t st);
hipError_t launch_load_points(int nen, int npts, int E, const double *x, const double *y, const double *z,
                              const int32_t *conn, double *out, hipStream_t st);
hipError_t launch_resultants(int nen, int composite, const ResParams &rp, const double *x, const double *y,
                             const double *z, const int32_t *conn, const double *nx, const double *ny,
                             const double *nz, const uint8_t *valid, hipStream_t st);
hipError_t launch_mass(int nen, int64_t N, int E, int composite, const double *g_rho_t, const double *g_inertia,
                       const int32_t *elem_group, const double *x, const double *y, const double *z,
                       const int32_t *conn, const int32_t *ne_ptr, const int32_t *ne_list, const int64_t *node_dof,
                       int64_t nrows, double *diag, hipStream_t st);
hipError_t launch_cd_mass(int64_t nv, int64_t n, const int64_t *map, const double *mdiag, double dt, double cdamp,
                          const int32_t *row_group, const double *group_dt, const double *group_cdamp, double *Cd,
                          double *invMC, hipStream_t st);
hipError_t launch_cd_place(int64_t nv, int64_t n, const int64_t *map, const double *src, double *dst, hipStream_t st);
hipError_t launch_cd_place(int64_t nv, int64_t n, const int64_t *map, const int32_t *src, int32_t *dst, int32_t rest,
                           hipStream_t st);
hipError_t launch_cd_probe(int64_t n, int nprobes, const int64_t *plist, int32_t *probe, hipStream_t st);
hipError_t launch_cd_collect(int64_t nv, int64_t n, const int64_t *map, const double *src, double *dst,
                             hipStream_t st);
hipError_t launch_cd_init(int64_t n, double dt, double g0, const double *invMC, const double *Fmag, const double *U0,
                          const double *V, double *A, double *U1, const int32_t *row_group, const double *group_dt,
                          const double *gtab, hipStream_t st);
hipError_t launch_cd_step(int tpr, const RunRows &rows, const double *kval,
                          const double *Ucur, double *Unext, double *V, double *A, const double *invMC,
                          const double *Cd, const double *Fmag, double gstep, double dt, int damped,
                          const int32_t *probe_slot, double *probe_dst, const int32_t *row_group,
                          const double *group_dt, const double *gtab, hipStream_t st);
hipError_t launch_spmv(const RunRows &rows, const double *kval, const double *x, double *y, hipStream_t st);
hipError_t launch_spmv_node(int nl, int pj, const NodeRows &nrw, const int2 *slotrec, const double *kval,
                            const double *x, double *y, hipStream_t st);
hipError_t launch_cd_node_step(int nl, int pj, const NodeRows &nrw, const int2 *slotrec, const double *kval,
                               const double *Ucur, double *Unext, double *V, double *A, const double *invMC,
                               const double *Cd, const double *Fmag, double gstep, double dt, int damped,
                               const int32_t *probe_slot, double *probe_dst, const int32_t *row_group,
                               const double *group_dt, const double *gtab, hipStream_t st);
hipError_t launch_patch_cut(int64_t nsegs, int most, const int4 *segs, const float4 *src, float4 *dst, hipStream_t st);
hipError_t launch_patch_count(int64_t np, const float4 *points, const int32_t *pstart, const int32_t *nbr_ptr,
                              const int32_t *nbr_node, int32_t *pnode, int32_t *slot, int4 *rec, uint16_t *nptr,
                              int64_t *tot, hipStream_t st);
hipError_t launch_patch_fill(int64_t np, const int32_t *nbr_ptr, const int32_t *nbr_node, const int32_t *pnode,
                             const int32_t *slot, const int4 *rec, const uint16_t *nptr, int64_t over, uint2 *ent,
                             int32_t *entk, int32_t *hpos, int64_t *tot, hipStream_t st);
hipError_t launch_patch_map(const PatchOp &op, const int64_t *node_dof, int64_t *map, hipStream_t st);
hipError_t launch_patch_build(const PatchOp &op, int kind, const ScatterPlan &sp, const double *kval,
                              const MixedOp &mixed, const int32_t *conn, int nen, int nsr, hipStream_t st);
hipError_t launch_patch_init(const PatchOp &op, double dt, double g0, const double *invMC, const double *Fmag,
                             const double *U0, double *W, double *U1, const int32_t *row_group,
                             const double *group_dt, const double *gtab, unsigned long long *pub, hipStream_t st);
hipError_t patch_loop_occupancy(const PatchOp &op, int f32, int *per_cu);
hipError_t launch_cd_patch_loop(const PatchLoop &a, int f32, hipStream_t st);
hipError_t launch_cd_patch_step(const PatchOp &op, int f32, const double *Ucur, double *Unext, double *W, const double *invMC,
                                const double *Cd, const double *Fmag, double gstep, double dt, int damped, int forced,
                                int last, const int32_t *probe_slot, double *probe_dst,
                                const int32_t *row_group, const double *group_dt, const double *gtab, hipStream_t st);
hipError_t launch_dot(int64_t n, const double *x, const double *y, const double *d, double *part, double *out,
                      hipStream_t st);
hipError_t launch_pwr(const RunRows &rows, const double *kval, const double *x, double *y, const double *mdiag,
                      const double *scale, double *part, double *ss, hipStream_t st);
hipError_t launch_pwr_node(int nl, int pj, const NodeRows &nrw, const int2 *slotrec, const double *kval,
                           const double *x, double *y, const double *mdiag, const double *scale, double *part,
                           double *ss, hipStream_t st);
hipError_t noalloc_workspace(int device, double **out);
hipError_t launch_mixed_build(const ScatterPlan &sp, const double *Kb, const int64_t *goff, float2 *kmb, short2 *kml,
                              hipStream_t st);
hipError_t launch_mixed_drill(int nen, int64_t N, int E, const int32_t *ne_ptr, const int32_t *ne_list,
                              const int32_t *conn, const double *dre, double *dr, hipStream_t st);
hipError_t launch_coo_reduce(int64_t nnz, const int64_t *cptr, const int64_t *clist, const double *mats,
                             double *out, hipStream_t st);
hipError_t launch_cd_mixed_step(int nen, int nsr, const MixedOp &op, const double *Ucur, double *Unext,
                                double *V, double *A, const double *invMC, const double *Cd, const double *Fmag,
                                double gstep, double dt, int damped, int forced, const int32_t *probe_slot,
                                double *probe_dst, const int32_t *row_group, const double *group_dt,
                                const double *gtab, hipStream_t st);
}  // namespace fs

namespace {
// Device buffers released by the models of a context are kept for reuse by
// the same context instead of being returned with hipFree, which waits for
// the whole device (every other context's work included).  Reuse is safe
// because every ABI call ends with its stream synchronised, so a released
// buffer has no pending work.  Shared by the context and every live buffer
// allocated through it; outlives the context until the last buffer is gone.
struct BufCache {
    std::mutex mu;
    std::multimap<size_t, void *> spare;  // bytes -> block
    size_t spare_bytes = 0;
    size_t cap = size_t(4) << 30;         // bytes kept per context at most
    int refs = 1;                         // the context + live buffers
    bool alive = true;                    // false once the context is destroyed
};
}  // namespace

// Slots and threads of a device-to-host copy (d2h).
constexpr int STAGE_SLOTS = 16, STAGE_THREADS = 8;

struct fs_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    // the caller's handle plus one per live model: fs_ctx_destroy drops the
    // caller's reference, the last release tears the context down, so a
    // model may outlive fs_ctx_destroy (it may then only be destroyed)
    std::atomic<int> refs{1};
    std::string err;
    BufCache *cache = nullptr;
    // element-kernel launch shape per (family T3/Q4, shear formulation):
    // -1 = not tuned yet (the autotuner times every shape on the first
    // stiffness evaluation of that kind and keeps the fastest)
    int elem_variant[2][2] = {{-1, -1}, {-1, -1}};
    bool autotune = true;
    // assembly pipeline: the element kernels run in asm_chunks element
    // ranges on `stream`; the scatter of the node pairs completed by each
    // range runs on `stream2` (default priority) while the next range computes
    hipStream_t stream2 = nullptr;
    int asm_chunks = 1;
    std::vector<hipEvent_t> ev;  // ordering events of the pipeline (no timing)
    // pinned staging slots of the device-to-host copies (64 MB at most, grown
    // by the copies that use them) and their completion events
    char *stage = nullptr;
    size_t stage_bytes = 0;
    hipEvent_t stage_ev[STAGE_SLOTS] = {};
    // row products of the FP64 explicit step: 0 = lanes per row
    // (cd_step_kernel), 8/16 = lanes per node (cd_node_step_kernel) with
    // cd_pj positions per lane (0: from the block's longest row)
    int cd_lanes = 8;
    int cd_pj = 0;
    // the device's workspace of the allocation-free entry points (address of
    // its copy of the file-scope array, taken at context creation), and the
    // status of that lookup
    double *scratch = nullptr;
    hipError_t scratch_status = hipSuccess;
    // one-launch loop: longest wait of a lane in polls (0: the default, negative:
    // the loop runs step by step), the word its waits run out into (pinned
    // host memory, allocated on first use), and whether one has
    int64_t loop_polls = 0;
    int *loop_stop = nullptr;
    bool loop_gave_up = false;
    // stiffness assembly: 1 = fused element tiles (element kernel writes the
    // CSR values of the pairs it completes, boundary pairs finalised after);
    // 0 = element blocks to HBM, then the pair scatter
    int assembly = 1;
};

namespace {

struct DevBuf {
    void *p = nullptr;
    size_t bytes = 0;          // size of the block (may exceed the request)
    BufCache *cache = nullptr; // owner's cache, or nullptr
    DevBuf() = default;
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    ~DevBuf() { release(); }
    void release() {
        if (p) {
            if (cache) {
                int left;
                {
                    std::lock_guard<std::mutex> lk(cache->mu);
                    if (cache->alive && cache->spare_bytes + bytes <= cache->cap) {
                        cache->spare.insert({bytes, p});
                        cache->spare_bytes += bytes;
                    } else {
                        (void)hipFree(p);
                    }
                    left = --cache->refs;
                }
                if (left == 0) delete cache;
            } else {
                (void)hipFree(p);
            }
        }
        p = nullptr;
        bytes = 0;
        cache = nullptr;
    }
    template <class T>
    T *as() const { return static_cast<T *>(p); }
};

// Fused-assembly plan of a block (fs::TilePlan): the element tiles, their
// pair entries and the boundary pairs; built on the first fused stiffness.
struct TileStore {
    int ne = 0;  // elements per tile it was built for (0: not built)
    int64_t ntiles = 0, nent = 0, nbnd = 0, nslots = 0;
    DevBuf tile_elem, tile_conn, tp_ptr, trec, tcontrib, tslot, brec, bp_ptr, partial;
    void reset() {
        ne = 0;
        ntiles = nent = nbnd = nslots = 0;
        for (DevBuf *b : {&tile_elem, &tile_conn, &tp_ptr, &trec, &tcontrib, &tslot, &brec, &bp_ptr, &partial})
            b->release();
    }
};

// Patch form of the free-free stiffness (fs::PatchOp): the plan, built on
// the first loop that takes it, and the values it holds.
struct PatchStore {
    bool planned = false, usable = false;
    int64_t npatch = 0, nent = 0;
    int slots = 0;
    bool loops = false;        // the one-launch loop takes the plan (hpos is there)
    // its launches: bounds of sets of whole components, and the largest set
    std::vector<int32_t> sets;
    int32_t largest_set = 0;
    int loop_per_cu[2] = {0, 0};  // its workgroups per CU, FP64 and F32 (0: not asked yet)
    // what it is filled with (FS_PREC_*, -1 nothing) and the generations of the
    // values (Block::vgen, MixedStore::kgen) that came from
    int kind = -1;
    uint64_t vgen = 0, kgen = 0;
    DevBuf rec, ent, entk, hpos, dpnode, nptr, map, k2, kh, kl, dg;
    void reset() {
        planned = usable = false;
        npatch = nent = 0;
        slots = 0;
        loops = false;
        sets.clear();
        largest_set = 0;
        loop_per_cu[0] = loop_per_cu[1] = 0;
        kind = -1;
        for (DevBuf *b : {&rec, &ent, &entk, &hpos, &dpnode, &nptr, &map, &k2, &kh, &kl, &dg}) b->release();
    }
};

struct Block {
    bool built = false;
    int64_t nrows = 0;
    int64_t nnz = 0;
    int64_t nnodes = 0;
    // scatter plan (device)
    int64_t npairs = 0;
    // running maximum over the pairs, in pair order, of the last element
    // contributing to a pair: the pairs [0, k) with pair_emax[k-1] < e are
    // complete once the elements [0, e) are (host)
    std::vector<int32_t> pair_emax;
    int64_t nnb = 0, ncontrib = 0;  // neighbour slots, contributions
    const int32_t *nbr_ptr = nullptr, *nbr_node = nullptr;  // the model's lists (device)
    DevBuf rowptr, nbr_pair, nbr_off, node_code, node_rowstart, node_rec, contrib_ptr, contrib,
        pair_node, pair_slot;
    // device values (CSR order) and, for the free-free block, the run records
    // of the row products of the time loop (fs::RunRows)
    DevBuf rowrec, slotrec, kval, mdiag;
    // free-free block: node records of the node-grouped step (fs::NodeRows)
    DevBuf noderec, nodeinfo;
    int64_t nrownodes = 0;
    int32_t max_rowlen = 0;
    bool k_ready = false, m_ready = false;
    uint64_t vgen = 0;  // raised before each launch that writes kval
    PatchStore patch;
    // host copies for the planner of the fused assembly (host_plan): neighbour
    // slot -> (pair << 1 | side), pair nodes, starts of the pairs' contributions;
    // per node {first free row's CSR position, first fixed row's (-1), row length,
    // 4-bit comp codes}
    std::unique_ptr<int32_t[]> h_nb_pair, h_pnode, h_cptr, h_node_rec;
    TileStore tiles;
    void reset() {
        built = k_ready = m_ready = false;
        h_nb_pair.reset();
        h_pnode.reset();
        h_cptr.reset();
        h_node_rec.reset();
        tiles.reset();
        patch.reset();
        nrows = nnz = npairs = nrownodes = nnb = ncontrib = 0;
        max_rowlen = 0;
        pair_emax.clear();
        for (DevBuf *b : {&rowptr, &nbr_pair, &nbr_off, &node_code, &node_rowstart, &node_rec,
                          &contrib_ptr, &contrib, &pair_node, &pair_slot, &rowrec, &slotrec, &kval, &mdiag, &noderec, &nodeinfo})
            b->release();
    }
};

}  // namespace

// Mixed-precision operator resident for the explicit loop (see fs::MixedOp).
struct MixedStore {
    bool built = false;
    uint64_t kgen = 0;   // element-parameter generation it was built from
    bool shear_fp32 = false;  // transverse shear in the FP32 slices (no factor rows)
    int nsr = 0;
    int64_t nslices = 0;
    int64_t kmb_pairs = 0;  // float2 values
    DevBuf goff, kmb, kml, cs, dr, ne_pack;
    float build_ms = 0.f;
    void reset() {
        built = false;
        for (DevBuf *b : {&goff, &kmb, &kml, &cs, &dr, &ne_pack}) b->release();
    }
};

// Device state of the explicit loop, kept with its step graph between
// calls: a call whose launch parameters (sizes, scalars, load factors,
// buffer addresses and the operator's records) equal those of the graph
// uploads its initial state into the same buffers and replays the graph,
// instead of capturing and instantiating its nsteps launches again.
struct StepCache {
    DevBuf dPub, dForced;  // one-launch loop
    DevBuf dU[2], dV, dA, dF, dInv, dC, dSlot, dProbe, dRG, dGdt, dGcd, dG, dPlist;
    std::vector<uint64_t> key;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    int64_t replays = 0;  // launches of a graph taken from the cache
    void drop_graph() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        exec = nullptr;
        graph = nullptr;
        key.clear();
    }
    ~StepCache() { drop_graph(); }
    void release() {
        for (DevBuf *b : {&dPub, &dForced, &dU[0], &dU[1], &dV, &dA, &dF, &dInv, &dC, &dSlot, &dProbe, &dRG, &dGdt, &dGcd,
                          &dG, &dPlist})
            b->release();
    }
};

struct fs_model {
    fs_ctx *ctx = nullptr;
    int nen = 0;
    int64_t N = 0, E = 0;
    std::vector<int32_t> conn;       // E x nen row-major, 0-based (host)
    std::vector<int32_t> ne_ptr, ne_list;  // node -> elements (ascending)
    // node -> neighbour nodes, itself among them (sorted): on the device, and on
    // the host once a host planner has asked for them (host_lists)
    int64_t nnb = 0;
    std::unique_ptr<int32_t[]> nbr_ptr, nbr_list;
    DevBuf x, y, z, dconn, dne_ptr, dne_list, dnbr_ptr, dnbr_list, nx, ny, nz, valid, node_dof, Kb, status;
    bool hubs = false;  // a node has more elements than node_neighbours_kernel takes
    bool normals_ready = false;
    bool dofs_ready = false;
    std::vector<int64_t> dof;  // N x 6 row-major, 0-based
    int64_t nall = 0, nfree = 0;
    Block blk[2];
    // group data for the last stiffness/mass call
    DevBuf g_Labd, g_Lh, g_csys, g_t, g_group, g_inertia, m_group, g_homog, g_rho_t;
    double timing[7] = {0, 0, 0, 0, 0, 0, 0};
    int32_t cd_form = -1;  // FS_CD_* of the last loop
    // parameters of the last element-stiffness launch (device pointers into
    // the group buffers above) and their generation
    fs::ElemParams last_ep{};
    uint64_t kgen = 0;
    MixedStore mixed;
    StepCache step;
};

// Buffered element matrices of a FEMM with no element kernel here, reduced
// into CSR on the device (fs_coo_*): the pattern and, per stored entry, the
// positions of its contributions in the element-matrix buffer.
struct fs_coo {
    fs_ctx *ctx = nullptr;
    int64_t nrows = 0, ncols = 0, nmat = 0;
    int32_t kr = 0, kc = 0;
    int64_t nnz = 0;
    std::vector<int64_t> rowptr, colval;  // 0-based
    DevBuf cptr, clist, mats, vals;
};

namespace {

// Host array whose elements are not initialised: for large arrays that
// threads fill, so that one thread does not touch all their pages first.
template <class T>
using HostArray = std::unique_ptr<T[]>;
template <class T>
HostArray<T> host_array(int64_t n) {
    return HostArray<T>(new T[(size_t)std::max<int64_t>(n, 1)]);
}

// Records the message of a failing call and waits for the work the call
// had already queued on the context's streams, so that the device buffers
// the call releases on its way out (returned to the context's spare list)
// have no pending kernels or copies.  Every ABI call therefore ends with its
// streams synchronised, on the error paths too.
int fail(fs_ctx *c, int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (c) {
        c->err = buf;
        if (c->stream) (void)hipStreamSynchronize(c->stream);
        if (c->stream2) (void)hipStreamSynchronize(c->stream2);
    }
    // the error is reported: clear the runtime's last-error state, which the
    // launch checks (hipGetLastError) of later calls would otherwise read
    (void)hipGetLastError();
    return code;
}

#define FS_HIP(ctx, call)                                                                           \
    do {                                                                                            \
        hipError_t e_ = (call);                                                                     \
        if (e_ != hipSuccess) return fail((ctx), FS_ERR_DEVICE, "%s: %s", #call, hipGetErrorString(e_)); \
    } while (0)

int dalloc(fs_ctx *c, DevBuf &b, size_t bytes) {
    b.release();
    if (bytes == 0) bytes = 8;
    BufCache *cache = c->cache;
    {
        // best fit among the spare blocks, at most 25 % + 1 MiB larger
        std::lock_guard<std::mutex> lk(cache->mu);
        auto it = cache->spare.lower_bound(bytes);
        if (it != cache->spare.end() && it->first <= bytes + bytes / 4 + (size_t(1) << 20)) {
            b.p = it->second;
            b.bytes = it->first;
            cache->spare_bytes -= it->first;
            cache->spare.erase(it);
            b.cache = cache;
            ++cache->refs;
            return FS_OK;
        }
    }
    hipError_t e = hipMalloc(&b.p, bytes);
    if (e == hipErrorOutOfMemory) {
        // give the spare blocks back and try once more
        {
            std::lock_guard<std::mutex> lk(cache->mu);
            for (auto &kv : cache->spare) (void)hipFree(kv.second);
            cache->spare.clear();
            cache->spare_bytes = 0;
        }
        e = hipMalloc(&b.p, bytes);
    }
    if (e != hipSuccess) {
        b.p = nullptr;
        return fail(c, FS_ERR_NOMEM, "hipMalloc(%zu bytes): %s", bytes, hipGetErrorString(e));
    }
    b.bytes = bytes;
    std::lock_guard<std::mutex> lk(cache->mu);
    b.cache = cache;
    ++cache->refs;
    return FS_OK;
}

template <class T>
int upload(fs_ctx *c, DevBuf &b, const T *src, size_t n) {
    int s = dalloc(c, b, n * sizeof(T));
    if (s) return s;
    if (n) FS_HIP(c, hipMemcpyAsync(b.p, src, n * sizeof(T), hipMemcpyHostToDevice, c->stream));
    return FS_OK;
}

// dalloc that keeps the buffer when it is already large enough (its
// address then stays the same from call to call).
int ensure(fs_ctx *c, DevBuf &b, size_t bytes) {
    if (b.p && b.bytes >= std::max<size_t>(bytes, 8)) return FS_OK;
    return dalloc(c, b, bytes);
}

template <class T>
int put(fs_ctx *c, DevBuf &b, const T *src, size_t n) {
    int s = ensure(c, b, n * sizeof(T));
    if (s) return s;
    if (n) FS_HIP(c, hipMemcpyAsync(b.p, src, n * sizeof(T), hipMemcpyHostToDevice, c->stream));
    return FS_OK;
}

// Appends the bytes of a trivially copyable value to a cache key.
template <class T>
void key_add(std::vector<uint64_t> &k, const T &v) {
    static_assert(std::is_trivially_copyable<T>::value, "key values are plain data");
    uint64_t w[(sizeof(T) + 7) / 8] = {};
    std::memcpy(w, &v, sizeof(T));
    k.insert(k.end(), w, w + (sizeof(T) + 7) / 8);
}

// Device-to-host copy ordered on the context's own stream, so that contexts
// sharing a device never serialise on the null stream.  The bytes go through
// pinned chunks: while the DMA of later chunks runs, up to STAGE_THREADS
// threads copy the arrived ones into `dst`, which spreads the first-touch page
// faults of a fresh destination over them.  A thread that has emptied a chunk's
// slot queues the copy that uses the slot next.  Into fresh pages, direct copy
// (pinned by the runtime) against this: 2 MB 1.2 -> 0.4 ms, 28 MB 2.8 -> 0.9,
// 100 MB 10 -> 2.6, 680 MB 68 -> 15.5 (18 through two 32 MB chunks in turn); into
// touched pages 256 KB 120 -> 25 us, 1 MB 440 -> 74, 28 MB 1.7 -> 0.9 ms.  More
// threads than 8, or more slots than 16, gain nothing; chunks of 1 MB cost 30 %
// on the largest copies, of 4 MB idle threads on those below 64 MB.
// Memory that the runtime knows (pinned, managed) takes the copy directly, as it
// takes the DMA itself: values of 6, 21, 62 and 170 MB, with their kernels, in 0.18,
// 0.47, 1.24 and 3.2 ms, where the way through the chunks takes 0.29, 0.70, 1.73
// and 3.9.
int d2h(fs_ctx *c, void *dst, const void *src, size_t bytes) {
    if (bytes == 0) return FS_OK;
    hipPointerAttribute_t attr{};
    if (hipPointerGetAttributes(&attr, dst) != hipSuccess) {
        (void)hipGetLastError();  // ordinary host memory
    } else if (attr.type != hipMemoryTypeUnregistered) {
        FS_HIP(c, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, c->stream));
        FS_HIP(c, hipStreamSynchronize(c->stream));
        return FS_OK;
    }
    const size_t MB = size_t(1) << 20;
    const size_t ch = bytes <= 4 * MB ? MB : bytes <= 64 * MB ? 2 * MB : 4 * MB;
    const size_t n = (bytes + ch - 1) / ch, ns = std::min(n, (size_t)STAGE_SLOTS);
    if (c->stage_bytes < std::min(bytes, ns * ch)) {
        if (c->stage) (void)hipHostFree(c->stage);
        c->stage = nullptr;
        c->stage_bytes = 0;
        size_t want = MB;
        while (want < std::min(bytes, ns * ch)) want *= 2;
        if (hipHostMalloc((void **)&c->stage, want, hipHostMallocDefault) == hipSuccess) {
            c->stage_bytes = want;
        } else {  // no pinned memory to be had: the direct copy
            (void)hipGetLastError();
            c->stage = nullptr;
            FS_HIP(c, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, c->stream));
            FS_HIP(c, hipStreamSynchronize(c->stream));
            return FS_OK;
        }
    }
    if (n == 1) {
        FS_HIP(c, hipMemcpyAsync(c->stage, src, bytes, hipMemcpyDeviceToHost, c->stream));
        FS_HIP(c, hipStreamSynchronize(c->stream));
        std::memcpy(dst, c->stage, bytes);
        return FS_OK;
    }
    for (size_t i = 0; i < ns; ++i)
        if (!c->stage_ev[i]) FS_HIP(c, hipEventCreateWithFlags(&c->stage_ev[i], hipEventDisableTiming));
    std::atomic<size_t> queued[STAGE_SLOTS], next{0};  // queued[i % ns]: chunk i + 1 once i is on its way
    std::atomic<int> err{hipSuccess};
    for (auto &q : queued) q = 0;
    auto enqueue = [&](size_t i) {
        hipError_t e = hipMemcpyAsync(c->stage + (i % ns) * ch, (const char *)src + i * ch, std::min(ch, bytes - i * ch),
                                      hipMemcpyDeviceToHost, c->stream);
        if (e == hipSuccess) e = hipEventRecord(c->stage_ev[i % ns], c->stream);
        if (e != hipSuccess) err = e;
        queued[i % ns].store(i + 1, std::memory_order_release);
    };
    for (size_t i = 0; i < ns; ++i) enqueue(i);
    auto work = [&] {
        hipError_t e = hipSetDevice(c->device);
        if (e != hipSuccess) err = e;
        for (size_t i; err == hipSuccess && (i = next++) < n;) {
            // chunk i is queued by the thread that empties its slot of chunk i - ns
            while (queued[i % ns].load(std::memory_order_acquire) != i + 1) {
                if (err != hipSuccess) return;
                std::this_thread::yield();
            }
            if ((e = hipEventSynchronize(c->stage_ev[i % ns])) != hipSuccess) {
                err = e;
                return;
            }
            std::memcpy((char *)dst + i * ch, c->stage + (i % ns) * ch, std::min(ch, bytes - i * ch));
            if (i + ns < n) enqueue(i + ns);
        }
    };
    {
        const size_t nt = std::min({(size_t)fs::host_threads(), (size_t)STAGE_THREADS, bytes / (2 * MB) + 1});
        fs::Threads th;
        for (size_t t = 1; t < nt && th.start(work); ++t) {
        }
        work();
    }
    FS_HIP(c, (hipError_t)err.load());
    return FS_OK;
}

// Upper Cholesky factor of a symmetric n x n matrix (row-major): M = L' L.
bool chol_upper(int n, const double *M, double *L) {
    for (int i = 0; i < n * n; ++i) L[i] = 0.0;
    for (int i = 0; i < n; ++i) {
        double d = M[i * n + i];
        for (int k = 0; k < i; ++k) d -= L[k * n + i] * L[k * n + i];
        if (!(d > 0.0)) return false;
        const double lii = std::sqrt(d);
        L[i * n + i] = lii;
        for (int j = i + 1; j < n; ++j) {
            double s = M[i * n + j];
            for (int k = 0; k < i; ++k) s -= L[k * n + i] * L[k * n + j];
            L[i * n + j] = s / lii;
        }
    }
    return true;
}

// column-major n x n -> row-major
void cm2rm(int n, const double *cm, double *rm) {
    for (int i = 0; i < n; ++i)
        for (int j = 0; j < n; ++j) rm[i * n + j] = cm[j * n + i];
}

// A device array of a plan, copied to the host once; not zeroed first,
// so that the threads of the copy touch its pages.
template <class T>
int host_copy(fs_ctx *c, HostArray<T> &v, const DevBuf &b, int64_t n) {
    if (v) return FS_OK;
    v = host_array<T>(n);
    const int s = d2h(c, v.get(), b.p, n * sizeof(T));
    if (s) v.reset();
    return s;
}

// Host copies of the neighbour lists.
int host_lists(fs_model *m) {
    const int s = host_copy(m->ctx, m->nbr_ptr, m->dnbr_ptr, m->N + 1);
    return s ? s : host_copy(m->ctx, m->nbr_list, m->dnbr_list, m->nnb);
}

// Node -> neighbour lists (sorted, including the node itself); a node in no
// element has none: its rows stay empty, as in the COO assembly.  Made by a kernel
// unless a node has more elements than NBR_MAX neighbours can come from; then on
// the host, in two passes over the nodes (sizes, then lists).
int make_neighbours(fs_model *m) {
    fs_ctx *c = m->ctx;
    const int nen = m->nen;
    const int64_t N = m->N;
    int s;
    int32_t most = 0, nnb = 0;
    for (int64_t n = 0; n < N; ++n) most = std::max(most, m->ne_ptr[n + 1] - m->ne_ptr[n]);
    m->hubs = (int64_t)most * (nen - 1) + 1 > fs::NBR_MAX;
    if (!m->hubs) {
        DevBuf sums;
        if ((s = dalloc(c, m->dnbr_ptr, (N + 1) * 4)) || (s = dalloc(c, sums, (fs::scan_tiles(N) + 1) * 8))) return s;
        auto launch = [&](bool fill) {
            return fs::launch_neighbours(fill, N, nen, m->E, m->dconn.as<int32_t>(), m->dne_ptr.as<int32_t>(),
                                         m->dne_list.as<int32_t>(), m->dnbr_ptr.as<int32_t>(),
                                         m->dnbr_list.as<int32_t>(), sums.as<int64_t>(), c->stream);
        };
        FS_HIP(c, launch(false));
        if ((s = d2h(c, &nnb, m->dnbr_ptr.as<int32_t>() + N, 4)) || (s = dalloc(c, m->dnbr_list, (size_t)nnb * 4)))
            return s;
        m->nnb = nnb;
        FS_HIP(c, launch(true));
        FS_HIP(c, hipStreamSynchronize(c->stream));
        return FS_OK;
    }
    m->nbr_ptr = host_array<int32_t>(N + 1);
    auto neighbours = [&](int64_t n, std::vector<int32_t> &tmp) {
        tmp.clear();
        for (int k = m->ne_ptr[n]; k < m->ne_ptr[n + 1]; ++k) {
            const int e = m->ne_list[k];
            for (int a = 0; a < nen; ++a) tmp.push_back(m->conn[(int64_t)e * nen + a]);
        }
        std::sort(tmp.begin(), tmp.end());
        tmp.erase(std::unique(tmp.begin(), tmp.end()), tmp.end());
    };
    m->nbr_ptr[0] = 0;
    fs::parallel_chunks(N, [&](int64_t n0, int64_t n1) {
        std::vector<int32_t> tmp;
        for (int64_t n = n0; n < n1; ++n) {
            neighbours(n, tmp);
            m->nbr_ptr[n + 1] = (int32_t)tmp.size();
        }
    });
    for (int64_t n = 0; n < N; ++n) m->nbr_ptr[n + 1] += m->nbr_ptr[n];
    m->nnb = m->nbr_ptr[N];
    m->nbr_list = host_array<int32_t>(m->nnb);
    fs::parallel_chunks(N, [&](int64_t n0, int64_t n1) {
        std::vector<int32_t> tmp;
        for (int64_t n = n0; n < n1; ++n) {
            neighbours(n, tmp);
            std::copy(tmp.begin(), tmp.end(), m->nbr_list.get() + m->nbr_ptr[n]);
        }
    });
    if ((s = upload(c, m->dnbr_ptr, m->nbr_ptr.get(), N + 1)) || (s = upload(c, m->dnbr_list, m->nbr_list.get(), m->nnb)))
        return s;
    FS_HIP(c, hipStreamSynchronize(c->stream));
    return FS_OK;
}

// Pattern, scatter plan and records of the row products of a block, planned on
// the device from the node lists and the dof numbers (fs::PlanArgs); the
// host reads the totals between the two parts, and copies of the plan only where
// a host planner asks for them (host_plan).
int build_block(fs_model *m, int which) {
    fs_ctx *c = m->ctx;
    Block &B = m->blk[which];
    if (B.built) return FS_OK;
    if (!m->dofs_ready) return fail(c, FS_ERR_STATE, "pattern: equation numbers not set (fs_model_set_dofs)");
    const int64_t N = m->N, E = m->E;
    const bool ff = which == FS_BLOCK_FF;
    const int nblk = m->nen * (m->nen + 1) / 2;
    fs::PlanArgs a{};
    a.N = N;
    a.E = E;
    a.nen = m->nen;
    a.nrows = ff ? m->nfree : m->nall;
    a.nfree = m->nfree;
    a.nnb = m->nnb;
    // every node in an element is its own neighbour, and neighbours are mutual
    int64_t used = 0;
    for (int64_t I = 0; I < N; ++I) used += m->ne_ptr[I + 1] > m->ne_ptr[I];
    a.npairs = (a.nnb + used) / 2;
    DevBuf tot, sums, first, count, rowlen, diag, base, isfree;
    fs::PlanTotals t{UINT64_MAX, 0, 0, 0};
    const int64_t longest = std::max({a.nrows, N, a.npairs});
    int s;
    if ((s = dalloc(c, tot, sizeof t)) || (s = dalloc(c, sums, (fs::scan_tiles(longest) + 1) * 8)) ||
        (s = dalloc(c, first, 2 * N * 8)) || (s = dalloc(c, count, N * 4)) || (s = dalloc(c, rowlen, N * 4)) ||
        (s = dalloc(c, B.node_code, N * 6)) || (s = dalloc(c, B.nbr_off, 2 * a.nnb * 4)) ||
        (s = dalloc(c, B.rowptr, (a.nrows + 1) * 4)))
        return s;
    a.dof = m->node_dof.as<int64_t>();
    a.conn = m->dconn.as<int32_t>();
    a.ne_ptr = m->dne_ptr.as<int32_t>();
    a.ne_list = m->dne_list.as<int32_t>();
    a.nbr_ptr = B.nbr_ptr = m->dnbr_ptr.as<int32_t>();
    a.nbr = B.nbr_node = m->dnbr_list.as<int32_t>();
    a.tot = tot.as<fs::PlanTotals>();
    a.sums = sums.as<int64_t>();
    a.code = B.node_code.as<int8_t>();
    a.first = first.as<int64_t>();
    a.count = count.as<int32_t>();
    a.off = B.nbr_off.as<int32_t>();
    a.rowlen = rowlen.as<int32_t>();
    a.rowptr = B.rowptr.as<int32_t>();
    // the rows of nodes with long lists, which would take a lane of the kernel
    // the square of the length
    std::vector<std::vector<int32_t>> hubs;  // row length, then offsets
    for (int64_t I = 0; I < (m->hubs ? N : 0); ++I) {
        const int k0 = m->nbr_ptr[I], n = m->nbr_ptr[I + 1] - k0;
        if (n <= fs::PLAN_HUB) continue;
        hubs.emplace_back(1 + 2 * (size_t)n, -1);
        std::vector<int32_t> &h = hubs.back();
        std::vector<std::pair<int64_t, int>> runs;  // first dof, 2 slot + kind
        for (int k = 0; k < n; ++k) {
            int64_t lo[2] = {INT64_MAX, INT64_MAX};
            for (int cc = 0; cc < 6; ++cc) {
                const int64_t d = m->dof[(int64_t)m->nbr_list[k0 + k] * 6 + cc];
                if (d < a.nrows) lo[d >= a.nfree] = std::min(lo[d >= a.nfree], d);
            }
            for (int q = 0; q < 2; ++q)
                if (lo[q] != INT64_MAX) runs.push_back({lo[q], 2 * k + q});
        }
        std::sort(runs.begin(), runs.end());
        int32_t pos = 0;
        for (const auto &run : runs) {
            h[1 + run.second] = pos;
            const int64_t J = m->nbr_list[k0 + run.second / 2];
            for (int cc = 0; cc < 6; ++cc) {
                const int64_t d = m->dof[J * 6 + cc];
                pos += d < a.nrows && (d >= a.nfree) == (run.second % 2 == 1);
            }
        }
        h[0] = pos;
        t.max_any = std::max(t.max_any, pos);
        for (int cc = 0; cc < 6; ++cc)
            if (m->dof[I * 6 + cc] < a.nfree) t.max_free = std::max(t.max_free, pos);
        FS_HIP(c, hipMemcpyAsync(a.rowlen + I, &h[0], 4, hipMemcpyHostToDevice, c->stream));
        FS_HIP(c, hipMemcpyAsync(a.off + 2 * (int64_t)k0, &h[1], 8 * (size_t)n, hipMemcpyHostToDevice, c->stream));
    }
    FS_HIP(c, hipMemcpyAsync(tot.p, &t, sizeof t, hipMemcpyHostToDevice, c->stream));
    FS_HIP(c, fs::launch_plan_rows(a, c->stream));
    if ((s = d2h(c, &t, tot.p, sizeof t))) return s;
    if (t.bad != UINT64_MAX)
        return fail(c, FS_ERR_UNSUPPORTED, "node %lld: %s dofs are not consecutive numbers", (long long)(t.bad / 2),
                    t.bad % 2 ? "fixed" : "free");
    if (t.nnz >= (int64_t(1) << 31))
        return fail(c, FS_ERR_UNSUPPORTED, "block with %lld stored entries exceeds 32-bit positions", (long long)t.nnz);
    if (a.npairs >= (int64_t(1) << 27))
        return fail(c, FS_ERR_UNSUPPORTED, "too many node pairs (%lld)", (long long)a.npairs);
    if (E * nblk >= (int64_t(1) << 30))
        return fail(c, FS_ERR_UNSUPPORTED, "too many element blocks (%lld)", (long long)(E * nblk));
    if (ff && t.max_any >= (1 << 27)) return fail(c, FS_ERR_UNSUPPORTED, "row of more than 2^27 entries");
    if ((s = dalloc(c, B.node_rowstart, N * 6 * 4)) || (s = dalloc(c, B.node_rec, N * 16)) ||
        (s = dalloc(c, diag, N * 4)) || (s = dalloc(c, base, (N + 1) * 4)) || (s = dalloc(c, B.nbr_pair, a.nnb * 4)) ||
        (s = dalloc(c, B.pair_node, 2 * a.npairs * 4)) || (s = dalloc(c, B.pair_slot, 2 * a.npairs * 4)) ||
        (s = dalloc(c, B.contrib_ptr, (a.npairs + 1) * 4)) || (s = dalloc(c, B.contrib, E * nblk * 4)))
        return s;
    a.rowstart = B.node_rowstart.as<int32_t>();
    a.node_rec = B.node_rec.as<int4>();
    a.diag = diag.as<int32_t>();
    a.base = base.as<int32_t>();
    a.nbr_pair = B.nbr_pair.as<int32_t>();
    a.pair_node = B.pair_node.as<int32_t>();
    a.pair_slot = B.pair_slot.as<int32_t>();
    a.contrib_ptr = B.contrib_ptr.as<int32_t>();
    a.contrib = B.contrib.as<int32_t>();
    int32_t nodes = 0;
    if (ff) {
        if ((s = dalloc(c, isfree, (N + 1) * 4)) || (s = dalloc(c, B.rowrec, a.nrows * 16)) ||
            (s = dalloc(c, B.slotrec, a.nnb * 8)) || (s = dalloc(c, B.noderec, N * 16)) ||
            (s = dalloc(c, B.nodeinfo, N * 4)))
            return s;
        a.isfree = isfree.as<int32_t>();
        a.rowrec = B.rowrec.as<int4>();
        a.slotrec = B.slotrec.as<int2>();
        a.noderec = B.noderec.as<int4>();
        a.nodeinfo = B.nodeinfo.as<int32_t>();
    }
    if ((s = dalloc(c, B.kval, (size_t)t.nnz * sizeof(double)))) return s;
    if ((s = dalloc(c, B.mdiag, (size_t)a.nrows * sizeof(double)))) return s;
    FS_HIP(c, fs::launch_plan_pairs(a, c->stream));
    if (ff && (s = d2h(c, &nodes, isfree.as<int32_t>() + N, 4))) return s;
    FS_HIP(c, hipStreamSynchronize(c->stream));
    B.nrownodes = nodes;
    B.max_rowlen = ff ? t.max_free : 0;
    B.nnb = a.nnb;
    B.ncontrib = E * nblk;
    B.npairs = a.npairs;
    B.nnodes = N;
    B.nrows = a.nrows;
    B.nnz = t.nnz;
    B.built = true;
    B.k_ready = B.m_ready = false;
    return FS_OK;
}

// Host copies of the plan for the planner of the fused assembly.
int host_plan(fs_ctx *c, Block &B) {
    int s;
    if ((s = host_copy(c, B.h_nb_pair, B.nbr_pair, B.nnb)) || (s = host_copy(c, B.h_pnode, B.pair_node, 2 * B.npairs)) ||
        (s = host_copy(c, B.h_cptr, B.contrib_ptr, B.npairs + 1)) ||
        (s = host_copy(c, B.h_node_rec, B.node_rec, 4 * B.nnodes)))
        return s;
    return FS_OK;
}

// pair_emax, for the pipelined assembly.
int pair_order(fs_model *m, Block &B) {
    if ((int64_t)B.pair_emax.size() == B.npairs) return FS_OK;
    const int nblk = m->nen * (m->nen + 1) / 2;
    HostArray<int32_t> list;
    int s;
    if ((s = host_copy(m->ctx, B.h_cptr, B.contrib_ptr, B.npairs + 1)) ||
        (s = host_copy(m->ctx, list, B.contrib, B.ncontrib)))
        return s;
    B.pair_emax.assign(B.npairs, -1);
    for (int64_t p = 0; p < B.npairs; ++p) {
        if (B.h_cptr[p + 1] > B.h_cptr[p]) B.pair_emax[p] = (list[B.h_cptr[p + 1] - 1] >> 1) / nblk;  // its last element
        if (p) B.pair_emax[p] = std::max(B.pair_emax[p], B.pair_emax[p - 1]);
    }
    return FS_OK;
}

fs::RunRows runrows_of(const Block &B) {
    fs::RunRows r;
    r.n = B.nrows;
    r.rowrec = B.rowrec.as<int4>();
    r.slotrec = B.slotrec.as<int2>();
    return r;
}

fs::NodeRows noderows_of(const Block &B) {
    fs::NodeRows r;
    r.n = B.nrownodes;
    r.rec = B.noderec.as<int4>();
    r.info = B.nodeinfo.as<int32_t>();
    return r;
}

// Positions per lane of the node-grouped row products: the context's setting,
// or enough for one pass over the longest row of the block where the
// register budget allows (8 lanes: 4..8, 16 lanes: 2..4).
int node_pj(const fs_ctx *c, const Block &B) {
    if (c->cd_lanes == 0 || c->cd_pj != 0) return c->cd_pj;
    const int lo = c->cd_lanes == 8 ? 4 : 2, hi = c->cd_lanes == 8 ? 8 : 4;
    return std::min(hi, std::max(lo, (B.max_rowlen + c->cd_lanes - 1) / c->cd_lanes));
}

fs::ScatterPlan plan_of(const Block &B) {
    fs::ScatterPlan sp;
    sp.nnodes = B.nnodes;
    sp.nbr_ptr = B.nbr_ptr;
    sp.nbr_node = B.nbr_node;
    sp.nbr_pair = B.nbr_pair.as<int32_t>();
    sp.nbr_off = B.nbr_off.as<int32_t>();
    sp.node_code = B.node_code.as<int8_t>();
    sp.node_rowstart = B.node_rowstart.as<int32_t>();
    sp.contrib_ptr = B.contrib_ptr.as<int32_t>();
    sp.contrib = B.contrib.as<int32_t>();
    sp.npairs = B.npairs;
    sp.pbegin = 0;
    sp.pend = B.npairs;
    sp.pair_node = B.pair_node.as<int32_t>();
    sp.pair_slot = B.pair_slot.as<int32_t>();
    return sp;
}

fs::TilePlan tileplan_of(const Block &B) {
    fs::TilePlan tp;
    tp.ntiles = B.tiles.ntiles;
    tp.nbnd = B.tiles.nbnd;
    tp.tp_ptr = B.tiles.tp_ptr.as<int32_t>();
    tp.trec = B.tiles.trec.as<int4>();
    tp.tcontrib = B.tiles.tcontrib.as<uint64_t>();
    tp.tslot = B.tiles.tslot.as<int32_t>();
    tp.brec = B.tiles.brec.as<int4>();
    tp.bp_ptr = B.tiles.bp_ptr.as<int32_t>();
    tp.partial = B.tiles.partial.as<double>();
    return tp;
}

fs::PatchOp patchop_of(const PatchStore &P) {
    fs::PatchOp op;
    op.npatch = (int32_t)P.npatch;
    op.slots = P.slots;
    op.over = P.npatch * fs::PATCH_WG;
    op.rec = P.rec.as<int4>();
    op.ent = P.ent.as<uint2>();
    op.entk = P.entk.as<int32_t>();
    op.hpos = P.hpos.as<int32_t>();
    op.pnode = P.dpnode.as<int32_t>();
    op.nptr = P.nptr.as<uint16_t>();
    op.k2 = P.k2.as<double2>();
    op.kh = P.kh.as<float4>();
    op.kl = P.kl.as<short4>();
    op.dg = P.dg.as<double>();
    return op;
}

// Patches of one launch of the one-launch loop at most, so of one component too:
// two a CU of 256 CUs.
constexpr int64_t PATCH_LOOP_MAX = 512;

// Partial slots a patch may have: 6 doubles each in LDS (48 KB), so that two
// workgroups fit a CU.
constexpr int PATCH_MAX_SLOTS = 1024;

// Patch plan of the free-free block (fs::PatchOp).  The nodes with free dofs
// are grouped by connected component, and each component is cut by
// recursive coordinate bisection into patches of at most PATCH_NODES nodes of
// nearly equal size: a set that needs k patches is cut across its longest
// extent, ties by node number, into shares of floor(k/2) and the rest.  The
// cuts depend on a component's own nodes only, so a model is cut alike alone and
// in a batch; components that need no cut share patches.  A mesh with a node of more neighbours than a
// patch may have partial slots keeps the row forms (usable false).
int build_patches(fs_model *m) {
    fs_ctx *c = m->ctx;
    Block &B = m->blk[FS_BLOCK_FF];
    PatchStore &P = B.patch;
    P.reset();
    P.planned = true;
    const int64_t N = m->N;
    constexpr int PN = fs::PATCH_NODES;
    if (N >= (int64_t(1) << 27)) return FS_OK;
    if (const int e = host_lists(m)) return e;
    std::vector<uint8_t> act(N);
    fs::parallel_chunks(N, [&](int64_t I0, int64_t I1) {
        for (int64_t I = I0; I < I1; ++I) {
            act[I] = 0;
            for (int cc = 0; cc < 6; ++cc) act[I] |= m->dof[I * 6 + cc] < m->nfree;
        }
    }, 262144);
    auto active = [&](int64_t I) { return act[I] != 0; };  // node with free dofs
    auto degree = [&](int64_t I) { return m->nbr_ptr[I + 1] - m->nbr_ptr[I]; };
    // coordinates, copied while the components are found
    HostArray<double> xyz = host_array<double>(3 * N);
    FS_HIP(c, hipMemcpyAsync(xyz.get(), m->x.p, N * 8, hipMemcpyDeviceToHost, c->stream));
    FS_HIP(c, hipMemcpyAsync(xyz.get() + N, m->y.p, N * 8, hipMemcpyDeviceToHost, c->stream));
    FS_HIP(c, hipMemcpyAsync(xyz.get() + 2 * N, m->z.p, N * 8, hipMemcpyDeviceToHost, c->stream));
    // components: union-find, the smaller number of two roots stays one
    HostArray<int32_t> par = host_array<int32_t>(N);
    for (int64_t i = 0; i < N; ++i) par[i] = (int32_t)i;
    auto find = [&](int32_t x) {
        for (;;) {
            const int32_t px = __atomic_load_n(&par[x], __ATOMIC_RELAXED);
            if (px == x) return x;
            const int32_t g = __atomic_load_n(&par[px], __ATOMIC_RELAXED);
            if (g != px) __atomic_store_n(&par[x], g, __ATOMIC_RELAXED);
            x = g;
        }
    };
    fs::parallel_chunks(N, [&](int64_t I0, int64_t I1) {
        for (int64_t I = I0; I < I1; ++I)
            for (int k = m->nbr_ptr[I]; k < m->nbr_ptr[I + 1] && m->nbr_list[k] < I; ++k) {
                int32_t a = (int32_t)I, b = m->nbr_list[k];
                for (;;) {
                    a = find(a);
                    b = find(b);
                    if (a == b) break;
                    if (a < b) std::swap(a, b);
                    int32_t want = a;
                    if (__atomic_compare_exchange_n(&par[a], &want, b, false, __ATOMIC_RELAXED, __ATOMIC_RELAXED)) break;
                }
            }
    }, 262144);
    // active nodes by component (components by their smallest node), in node
    // order within one; a mesh of one component is laid out in parallel
    struct Pt {
        float x[3];  // from the component's first node
        int32_t id;
    };
    FS_HIP(c, hipStreamSynchronize(c->stream));
    auto point = [&](int64_t I, int64_t I0) {
        Pt q{{0.f, 0.f, 0.f}, (int32_t)I};
        for (int d = 0; d < 3; ++d) {
            const float v = (float)(xyz[d * N + I] - xyz[d * N + I0]);
            if (std::isfinite(v)) q.x[d] = v;  // an order needs numbers
        }
        return q;
    };
    std::atomic<int64_t> roots{0};
    std::atomic<bool> hub{false}, wide{false};
    constexpr int64_t CH = 8192;  // nodes counted together
    const int64_t nch = (N + CH - 1) / CH;
    std::vector<int64_t> at(nch + 1, 0);
    fs::parallel_chunks(nch, [&](int64_t k0, int64_t k1) {
        int64_t nr = 0;
        for (int64_t k = k0; k < k1; ++k)
            for (int64_t I = k * CH; I < std::min(N, (k + 1) * CH); ++I) {
                nr += find((int32_t)I) == I;
                at[k + 1] += active(I);
                if (active(I) && degree(I) > PATCH_MAX_SLOTS) hub = true;
                if (active(I) && degree(I) * PN > PATCH_MAX_SLOTS) wide = true;
            }
        roots += nr;
    }, 16);
    for (int64_t k = 0; k < nch; ++k) at[k + 1] += at[k];
    const int64_t npt = at[nch];
    if (hub || npt == 0) return FS_OK;
    HostArray<Pt> pt = host_array<Pt>(npt);
    std::vector<int64_t> cptr(2, 0);
    if (roots == 1) {
        cptr[1] = npt;
        fs::parallel_chunks(nch, [&](int64_t k0, int64_t k1) {
            int64_t to = at[k0];
            for (int64_t I = k0 * CH; I < std::min(N, k1 * CH); ++I)
                if (active(I)) pt[to++] = point(I, 0);
        }, 16);
    } else {
        cptr.assign(1, 0);
        std::vector<int32_t> cid(N, -1), cfirst;
        for (int64_t I = 0; I < N; ++I) {
            const int32_t r = find((int32_t)I);  // the component's first node
            if (cid[r] < 0) {
                cid[r] = (int32_t)cptr.size() - 1;
                cptr.push_back(0);
                cfirst.push_back(r);
            }
            cid[I] = cid[r];
            if (active(I)) ++cptr[cid[I] + 1];
        }
        for (size_t k = 0; k + 1 < cptr.size(); ++k) cptr[k + 1] += cptr[k];
        std::vector<int64_t> fill(cptr.begin(), cptr.end() - 1);
        for (int64_t I = 0; I < N; ++I)
            if (active(I)) pt[fill[cid[I]]++] = point(I, cfirst[cid[I]]);
    }
    // Small components (tiny models of a batch, nodes in no element) share a patch as
    // long as they fit it whole.  A node's sums go by its own list, so that its results
    // are bitwise those of a patch of its own.  4,000 models of 4 nodes take 1.1 us
    // a step that way, 7.8 with a patch each and 5.2 with the row products; models
    // of 9 nodes 2.3, 8.5 and 12.7.
    std::vector<int64_t> units(1, 0);
    int64_t open_nodes = PN + 1, open_slots = 0;  // of the patch that the next small one may share
    for (size_t k = 0; k + 1 < cptr.size(); ++k) {
        const int64_t n = cptr[k + 1] - cptr[k];
        if (n == 0) continue;
        int64_t slots = 0;
        for (int64_t i = cptr[k]; n <= PN && i < cptr[k + 1]; ++i) slots += degree(pt[i].id);
        const bool small = n <= PN && slots <= PATCH_MAX_SLOTS;
        if (small && open_nodes + n <= PN && open_slots + slots <= PATCH_MAX_SLOTS) {
            units.back() = cptr[k + 1];
            open_nodes += n;
            open_slots += slots;
        } else {
            units.push_back(cptr[k + 1]);
            open_nodes = small ? n : PN + 1;
            open_slots = slots;
        }
    }
    cptr.swap(units);
    const int64_t nc = (int64_t)cptr.size() - 1;
    // Where no patch of PN nodes can have too many slots, the sizes of the cuts are
    // known beforehand and kernels make them, a launch a level; else the host cuts
    // (a patch with too many slots is cut again).  The host also cuts small meshes:
    // a loop's first call takes 0.46 ms that way and 0.50 with the launches on 56
    // nodes, 0.81 and 0.77 on 2,928, 4.2 and 2.8 on 26,000, 16.7 and 12.5 on 131,000.
    // Both make the same patches.
    if (npt >= INT32_MAX) return FS_OK;
    const bool kernel_cuts = !wide && npt >= 2048;
    std::vector<std::vector<int4>> levels;
    std::vector<uint8_t> head(npt + 1, 0);  // 1 where a patch begins
    if (kernel_cuts) {
        std::vector<int4> segs;
        for (int64_t k = 0; k < nc; ++k)
            if (cptr[k + 1] > cptr[k]) segs.push_back({(int)cptr[k], (int)(cptr[k + 1] - cptr[k]), 0, 0});
        for (bool cut = true; cut;) {
            cut = false;
            std::vector<int4> next;
            for (int4 &q : segs) {
                const int64_t k = (q.y + PN - 1) / PN;
                q.z = (int)((int64_t)q.y * (k / 2) / k);  // 0: a patch
                if (q.z) next.push_back({q.x, q.z, 0, 0});
                next.push_back({q.x + q.z, q.y - q.z, 0, 0});
                cut |= q.z != 0;
            }
            if (cut) levels.push_back(std::move(segs));
            segs = std::move(next);
        }
        for (const int4 &q : segs) head[q.x] = 1;
    }
    std::function<void(int64_t, int64_t)> bisect = [&](int64_t b, int64_t n) {
        Pt *q = pt.get() + b;
        int64_t k = (n + PN - 1) / PN;
        if (k == 1) {
            int64_t slots = 0;
            for (int64_t i = 0; i < n; ++i) slots += degree(q[i].id);
            if (slots <= PATCH_MAX_SLOTS) {
                head[b] = 1;
                return;
            }
            k = 2;
        }
        const int64_t n1 = n * (k / 2) / k;
        float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (int64_t i = 0; i < n; ++i)
            for (int d = 0; d < 3; ++d) {
                lo[d] = std::min(lo[d], q[i].x[d]);
                hi[d] = std::max(hi[d], q[i].x[d]);
            }
        int ax = 0;
        for (int d = 1; d < 3; ++d)
            if (hi[d] - lo[d] > hi[ax] - lo[ax]) ax = d;
        std::nth_element(q, q + n1, q + n, [ax](const Pt &u, const Pt &v) {
            return u.x[ax] != v.x[ax] ? u.x[ax] < v.x[ax] : u.id < v.id;
        });
        if (n > 65536) {  // creating a thread can take as long as cutting 50,000 nodes (3 ms)
            fs::run_shares(2, [&](int64_t t) { t ? bisect(b + n1, n - n1) : bisect(b, n1); });
        } else {
            bisect(b, n1);
            bisect(b + n1, n - n1);
        }
    };
    fs::parallel_chunks(kernel_cuts ? 0 : nc, [&](int64_t k0, int64_t k1) {
        for (int64_t k = k0; k < k1; ++k)
            if (cptr[k + 1] > cptr[k]) bisect(cptr[k], cptr[k + 1] - cptr[k]);
    }, 16);
    std::vector<int32_t> pstart;
    for (int64_t i = 0; i < npt; ++i)
        if (head[i]) pstart.push_back((int32_t)i);
    const int64_t np = (int64_t)pstart.size();
    pstart.push_back((int32_t)npt);
    if (np * PN >= (int64_t(1) << 26)) return FS_OK;  // slots are 26-bit numbers
    // sets of consecutive components for the one-launch loop (a component, or the
    // small ones that share its patch, is a set of its own unless it fits the current one)
    P.sets.assign(1, 0);
    bool halos = true;
    for (int64_t k = 0; k < nc && halos; ++k) {
        auto patch_at = [&](int64_t i) { return (int32_t)(std::lower_bound(pstart.begin(), pstart.end(), (int32_t)i) - pstart.begin()); };
        const int32_t b = patch_at(cptr[k]), e = patch_at(cptr[k + 1]);
        halos = e - b <= PATCH_LOOP_MAX;
        if (e - P.sets.back() > PATCH_LOOP_MAX) P.sets.push_back(b);
    }
    P.sets.push_back((int32_t)np);
    for (size_t k = 0; k + 1 < P.sets.size(); ++k) P.largest_set = std::max(P.largest_set, P.sets[k + 1] - P.sets[k]);
    // the lists on the device
    int s;
    DevBuf dpt[2], dsegs, dstart, dslot, dtot;
    const int32_t *nbp = B.nbr_ptr, *nbn = B.nbr_node;
    if ((s = upload(c, dpt[0], pt.get(), npt)) || (s = upload(c, dstart, pstart.data(), pstart.size())) ||
        (s = dalloc(c, dslot, N * 4)) || (s = dalloc(c, dtot, 32)) || (s = dalloc(c, P.dpnode, (size_t)np * PN * 4)) ||
        (s = dalloc(c, P.rec, (size_t)np * 16)) || (s = dalloc(c, P.nptr, (size_t)np * (PN + 1) * 2)))
        return s;
    std::vector<int4> all;
    for (const std::vector<int4> &l : levels) all.insert(all.end(), l.begin(), l.end());
    if (!all.empty() && ((s = upload(c, dsegs, all.data(), all.size())) || (s = dalloc(c, dpt[1], npt * sizeof(Pt)))))
        return s;
    int at0 = 0, cur = 0;
    for (const std::vector<int4> &l : levels) {
        int most = 0;
        for (const int4 &q : l) most = std::max(most, q.y);
        FS_HIP(c, fs::launch_patch_cut((int64_t)l.size(), most, dsegs.as<int4>() + at0, dpt[cur].as<float4>(),
                                       dpt[1 - cur].as<float4>(), c->stream));
        at0 += (int)l.size();
        cur = 1 - cur;
    }
    FS_HIP(c, hipMemsetAsync(dslot.p, 0xff, N * 4, c->stream));
    FS_HIP(c, fs::launch_patch_count(np, dpt[cur].as<float4>(), dstart.as<int32_t>(), nbp, nbn, P.dpnode.as<int32_t>(),
                                     dslot.as<int32_t>(), P.rec.as<int4>(), P.nptr.as<uint16_t>(),
                                     dtot.as<int64_t>(), c->stream));
    int64_t tot[4];
    if ((s = d2h(c, tot, dtot.p, 32))) return s;
    const int64_t nent = tot[0], over = np * fs::PATCH_WG, ntab = over + tot[2];
    if (nent >= (int64_t(1) << 30)) return FS_OK;
    if ((s = dalloc(c, P.ent, (size_t)ntab * 8)) || (s = dalloc(c, P.entk, (size_t)ntab * 4)) ||
        (halos && (s = dalloc(c, P.hpos, (size_t)np * fs::PATCH_HALO * 4))) ||
        (s = dalloc(c, P.map, (size_t)np * PN * 6 * 8)) || (s = dalloc(c, P.dg, (size_t)np * PN * fs::PATCH_TRI * 8)))
        return s;
    FS_HIP(c, fs::launch_patch_fill(np, nbp, nbn, P.dpnode.as<int32_t>(), dslot.as<int32_t>(), P.rec.as<int4>(),
                                    P.nptr.as<uint16_t>(), over, P.ent.as<uint2>(), P.entk.as<int32_t>(),
                                    halos ? P.hpos.as<int32_t>() : nullptr, dtot.as<int64_t>(), c->stream));
    P.npatch = np;
    P.nent = nent;
    P.slots = (int)tot[1];
    FS_HIP(c, fs::launch_patch_map(patchop_of(P), m->node_dof.as<int64_t>(), P.map.as<int64_t>(), c->stream));
    if ((s = d2h(c, tot, dtot.p, 32))) return s;  // and the host lists end here
    P.loops = halos && tot[3] != 0;
    P.usable = true;
    return FS_OK;
}

// Steps from which a loop takes the patch form.  Its plan costs a model's first
// such loop once.  A first loop of 100 steps takes, row form against patch form with
// its plan, 0.67 | 0.74 ms (1,271 nodes), 0.99 | 1.06 (6,076), 1.47 | 1.27 (12,221),
// 3.7 | 3.3 (36,381), 6.2 | 4.6 (51,657), and a later one 0.65 | 0.43, 0.81 | 0.43,
// 1.21 | 0.57, 2.9 | 1.6, 4.9 | 2.3: at 100 steps the first loop breaks even on the
// small meshes, below that it would lose.
constexpr int64_t PATCH_MIN_STEPS = 100;

// 3 x 21-bit Morton code of a point scaled into [0, 1)^3.
uint64_t morton3(double x, double y, double z) {
    auto spread = [](uint64_t v) {
        v &= 0x1fffff;
        v = (v | v << 32) & 0x1f00000000ffffULL;
        v = (v | v << 16) & 0x1f0000ff0000ffULL;
        v = (v | v << 8) & 0x100f00f00f00f00fULL;
        v = (v | v << 4) & 0x10c30c30c30c30c3ULL;
        v = (v | v << 2) & 0x1249249249249249ULL;
        return v;
    };
    auto q = [](double t) {
        const double u = t * 2097152.0;
        return (uint64_t)(u < 0.0 ? 0.0 : (u > 2097151.0 ? 2097151.0 : u));
    };
    return spread(q(x)) | spread(q(y)) << 1 | spread(q(z)) << 2;
}

// Fused-assembly plan of a block.  Elements are grouped into tiles of NE:
// per connected component (components in the order of their first
// element), elements sorted along a Morton curve of their centroids scaled
// by the component's bounding box, then cut into consecutive runs of NE, so
// a tile is a compact patch and never spans two components (a model gives
// the same tiles alone and inside a batch).  A tile's elements are kept in
// ascending order.  For every upper node pair a tile touches, its
// contributions within the tile are listed in element order; the pair is
// completed in the tile when they are all its contributions, otherwise (or
// when more than six fall in one tile, in runs of six) it leaves partial
// sums, added up afterwards in tile order.
int build_tiles(fs_model *m, int which, int NE) {
    fs_ctx *c = m->ctx;
    Block &B = m->blk[which];
    TileStore &T = B.tiles;
    T.reset();
    const int nen = m->nen;
    const int nblk = nen * (nen + 1) / 2;
    const int64_t E = m->E, N = m->N;
    if (NE > 32 || nblk > 16) return fail(c, FS_ERR_UNSUPPORTED, "fused assembly: tile of %d elements", NE);
    int s;
    if ((s = host_plan(c, B)) || (s = host_lists(m))) return s;
    // components: union-find over the nodes of each element
    std::vector<int32_t> par(N);
    for (int64_t i = 0; i < N; ++i) par[i] = (int32_t)i;
    auto find = [&](int32_t x) {
        while (par[x] != x) {
            par[x] = par[par[x]];
            x = par[x];
        }
        return x;
    };
    for (int64_t e = 0; e < E; ++e)
        for (int a = 1; a < nen; ++a) {
            const int32_t r0 = find(m->conn[e * nen]), r1 = find(m->conn[e * nen + a]);
            if (r0 != r1) par[std::max(r0, r1)] = std::min(r0, r1);
        }
    std::vector<int32_t> comp(E), cid(N, -1);
    int32_t ncomp = 0;
    for (int64_t e = 0; e < E; ++e) {
        const int32_t r = find(m->conn[e * nen]);
        if (cid[r] < 0) cid[r] = ncomp++;
        comp[e] = cid[r];
    }
    // centroids, component boxes, Morton keys
    std::vector<double> cen(3 * E), lo(3 * ncomp, 1e300), hi(3 * ncomp, -1e300);
    std::vector<double> X(3 * N);
    {
        std::vector<double> x(N), y(N), z(N);
        FS_HIP(c, hipMemcpyAsync(x.data(), m->x.p, N * 8, hipMemcpyDeviceToHost, c->stream));
        FS_HIP(c, hipMemcpyAsync(y.data(), m->y.p, N * 8, hipMemcpyDeviceToHost, c->stream));
        FS_HIP(c, hipMemcpyAsync(z.data(), m->z.p, N * 8, hipMemcpyDeviceToHost, c->stream));
        FS_HIP(c, hipStreamSynchronize(c->stream));
        for (int64_t i = 0; i < N; ++i) {
            X[3 * i] = x[i];
            X[3 * i + 1] = y[i];
            X[3 * i + 2] = z[i];
        }
    }
    for (int64_t e = 0; e < E; ++e) {
        for (int k = 0; k < 3; ++k) {
            double v = 0.0;
            for (int a = 0; a < nen; ++a) v += X[3 * (int64_t)m->conn[e * nen + a] + k];
            v /= nen;
            cen[3 * e + k] = v;
            lo[3 * comp[e] + k] = std::min(lo[3 * comp[e] + k], v);
            hi[3 * comp[e] + k] = std::max(hi[3 * comp[e] + k], v);
        }
    }
    std::vector<uint64_t> key(E);
    fs::parallel_chunks(E, [&](int64_t e0, int64_t e1) {
        for (int64_t e = e0; e < e1; ++e) {
            const int g = comp[e];
            double ext = 0.0;
            for (int k = 0; k < 3; ++k) ext = std::max(ext, hi[3 * g + k] - lo[3 * g + k]);
            const double sc = ext > 0.0 ? 1.0 / (ext * (1.0 + 1e-9)) : 0.0;
            key[e] = morton3((cen[3 * e] - lo[3 * g]) * sc, (cen[3 * e + 1] - lo[3 * g + 1]) * sc,
                             (cen[3 * e + 2] - lo[3 * g + 2]) * sc);
        }
    });
    std::vector<int32_t> order(E);
    for (int64_t e = 0; e < E; ++e) order[e] = (int32_t)e;
    std::sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
        if (comp[a] != comp[b]) return comp[a] < comp[b];
        if (key[a] != key[b]) return key[a] < key[b];
        return a < b;
    });
    // tiles by recursive coordinate bisection of each component's element
    // centroids: a set of n > NE elements is cut across its longest extent
    // into ceil(k / 2) NE elements and the rest (k = ceil(n / NE), ties by
    // element number), so that every tile but the last of a set holds NE
    // elements and tiles are compact patches visited in a space-filling
    // order.  Against runs of NE elements along the Morton curve of the
    // centroids this cuts the node pairs that straddle tiles from 421,805 to
    // 389,058 and their partial slots from 912,990 to 823,835 on the 512 x 512
    // Q4 cylinder (12-element tiles); the T3 plate (32) is unchanged.
    std::vector<int64_t> tstart;
    {
        // the cuts are in place: the tiles are consecutive ranges of `order`
        // (in bisection order), and halves of more than 2^16 elements are
        // cut on threads of their own
        std::mutex mu;
        std::function<void(int64_t, int64_t)> bisect = [&](int64_t b, int64_t n) {
            if (n <= NE) {
                std::lock_guard<std::mutex> lk(mu);
                tstart.push_back(b);
                return;
            }
            int32_t *p = order.data() + b;
            const int64_t k = (n + NE - 1) / NE, n1 = (k / 2) * NE;
            double lo3[3] = {1e300, 1e300, 1e300}, hi3[3] = {-1e300, -1e300, -1e300};
            for (int64_t i = 0; i < n; ++i)
                for (int d = 0; d < 3; ++d) {
                    lo3[d] = std::min(lo3[d], cen[3 * (int64_t)p[i] + d]);
                    hi3[d] = std::max(hi3[d], cen[3 * (int64_t)p[i] + d]);
                }
            int ax = 0;
            for (int d = 1; d < 3; ++d)
                if (hi3[d] - lo3[d] > hi3[ax] - lo3[ax]) ax = d;
            std::nth_element(p, p + n1, p + n, [&](int32_t u, int32_t v) {
                const double cu = cen[3 * (int64_t)u + ax], cv = cen[3 * (int64_t)v + ax];
                return cu != cv ? cu < cv : u < v;
            });
            if (n > (int64_t(1) << 16)) {
                fs::run_shares(2, [&](int64_t t) { t ? bisect(b + n1, n - n1) : bisect(b, n1); });
            } else {
                bisect(b, n1);
                bisect(b + n1, n - n1);
            }
        };
        for (int64_t b0 = 0; b0 < E;) {
            int64_t b1 = b0;
            while (b1 < E && comp[order[b1]] == comp[order[b0]]) ++b1;
            bisect(b0, b1 - b0);
            b0 = b1;
        }
        std::sort(tstart.begin(), tstart.end());
    }
    const int64_t ntiles = (int64_t)tstart.size();
    tstart.push_back(E);
    if (ntiles >= (int64_t(1) << 31) / 64) return fail(c, FS_ERR_UNSUPPORTED, "fused assembly: too many tiles");
    std::vector<int32_t> telem((size_t)ntiles * NE);
    for (int64_t t = 0; t < ntiles; ++t) {
        std::sort(order.begin() + tstart[t], order.begin() + tstart[t + 1]);
        const int64_t n = tstart[t + 1] - tstart[t];
        for (int le = 0; le < NE; ++le) telem[t * NE + le] = order[tstart[t] + (le < n ? le : 0)];
    }
    // pair entries per tile
    auto slot_of = [&](int64_t I, int64_t J) -> int32_t {
        const int32_t *b0 = m->nbr_list.get() + m->nbr_ptr[I];
        const int32_t *e0 = m->nbr_list.get() + m->nbr_ptr[I + 1];
        return (int32_t)(std::lower_bound(b0, e0, (int32_t)J) - m->nbr_list.get());
    };
    struct Ent {
        int32_t p;
        uint64_t cw;
        int32_t boundary;  // 1: leaves a partial sum
    };
    std::vector<std::vector<Ent>> tent(ntiles);
    std::atomic<int> bad{0};
    fs::parallel_chunks(ntiles, [&](int64_t t0, int64_t t1) {
        std::vector<std::array<int32_t, 4>> tup;  // (pair, element, code, 0)
        for (int64_t t = t0; t < t1; ++t) {
            tup.clear();
            const int64_t n = tstart[t + 1] - tstart[t];
            for (int le = 0; le < n; ++le) {
                const int32_t e = telem[t * NE + le];
                const int32_t *ce = m->conn.data() + (int64_t)e * nen;
                int bl = 0;
                for (int a = 0; a < nen; ++a)
                    for (int b = a; b < nen; ++b, ++bl) {
                        const int32_t na = ce[a], nb = ce[b];
                        const int32_t I = std::min(na, nb), J = std::max(na, nb);
                        const int32_t k = slot_of(I, J);
                        const int32_t pp = B.h_nb_pair[k] >> 1;
                        const int32_t code = le | (bl << 5) | ((na > nb ? 1 : 0) << 9);
                        tup.push_back({pp, e, code, 0});
                    }
            }
            std::sort(tup.begin(), tup.end(), [](const std::array<int32_t, 4> &x, const std::array<int32_t, 4> &y) {
                return x[0] != y[0] ? x[0] < y[0] : x[1] < y[1];
            });
            std::vector<Ent> &out = tent[t];
            for (size_t i = 0; i < tup.size();) {
                size_t j = i;
                while (j < tup.size() && tup[j][0] == tup[i][0]) ++j;
                const int32_t pp = tup[i][0];
                const int cnt = (int)(j - i);
                const int gcnt = B.h_cptr[pp + 1] - B.h_cptr[pp];
                if (cnt > gcnt) bad = 1;
                const bool complete = cnt == gcnt && cnt <= 6;
                for (size_t q = i; q < j; q += 6) {
                    const int nq = (int)std::min<size_t>(6, j - q);
                    uint64_t cw = (uint64_t)nq;
                    for (int r = 0; r < nq; ++r) cw |= (uint64_t)tup[q + r][2] << (3 + 10 * r);
                    out.push_back({pp, cw, complete ? 0 : 1});
                }
                i = j;
            }
            // entries of one kind next to each other, so that the waves of the
            // output phase take one path: completed pairs of two nodes whose
            // dofs are all in the block, completed diagonal pairs, other
            // completed pairs, boundary pairs.  The order within a kind (and
            // of the entries of one pair) stays, so the sums do not change.
            auto kind = [&](const Ent &en) {
                if (en.boundary) return 3;
                const int64_t I = B.h_pnode[2 * (int64_t)en.p], J = B.h_pnode[2 * (int64_t)en.p + 1];
                if (I == J) return 1;
                const bool all = (B.h_node_rec[4 * I + 3] & 0xffffff) == 0x543210 &&
                                 (B.h_node_rec[4 * J + 3] & 0xffffff) == 0x543210;
                return all ? 0 : 2;
            };
            std::stable_sort(out.begin(), out.end(),
                             [&](const Ent &x, const Ent &y) { return kind(x) < kind(y); });
        }
    }, 256);
    if (bad) return fail(c, FS_ERR_STATE, "fused assembly: tile contributions exceed the pair's");
    // flatten; partial slots in tile order; boundary pairs and their slots
    std::vector<int32_t> tp_ptr(ntiles + 1, 0);
    for (int64_t t = 0; t < ntiles; ++t) tp_ptr[t + 1] = tp_ptr[t] + (int32_t)tent[t].size();
    const int64_t nent = tp_ptr[ntiles];
    // the pair of each entry; the placement records are made from them on the device
    HostArray<int32_t> tpair = host_array<int32_t>(nent), tslot = host_array<int32_t>(nent);
    HostArray<uint64_t> tcw = host_array<uint64_t>(nent);
    // partial slots: the slots of one boundary pair are consecutive (its
    // tiles in tile order), so the finalize reads each pair's partials as one
    // stretch
    std::vector<int32_t> pcount(B.npairs + 1, 0);
    for (int64_t t = 0; t < ntiles; ++t)
        for (const Ent &en : tent[t])
            if (en.boundary) pcount[en.p + 1]++;
    std::vector<int32_t> bidx(B.npairs, -1), bpair, bp_ptr(1, 0);
    for (int64_t pp = 0; pp < B.npairs; ++pp)
        if (pcount[pp + 1]) {
            bidx[pp] = (int32_t)(bp_ptr.size() - 1);
            bpair.push_back((int32_t)pp);
            bp_ptr.push_back(bp_ptr.back() + pcount[pp + 1]);
        }
    const int64_t nbnd = (int64_t)bp_ptr.size() - 1;
    const int64_t nslots = bp_ptr.back();
    std::vector<int32_t> bfill(bp_ptr.begin(), bp_ptr.end() - 1);
    for (int64_t t = 0; t < ntiles; ++t)
        for (size_t i = 0; i < tent[t].size(); ++i) {
            const Ent &en = tent[t][i];
            const int64_t q = tp_ptr[t] + (int64_t)i;
            tpair[q] = en.p;
            tcw[q] = en.cw;
            tslot[q] = en.boundary ? bfill[bidx[en.p]]++ : -1;
        }
    int st;
    DevBuf dtpair, dbpair;
    // the tiles' own connectivity (node a of tile element le at (t NE + le) nen + a)
    std::vector<int32_t> tconn(telem.size() * nen);
    for (size_t i = 0; i < telem.size(); ++i)
        for (int a = 0; a < nen; ++a) tconn[i * nen + a] = m->conn[(size_t)telem[i] * nen + a];
    if ((st = upload(c, T.tile_elem, telem.data(), telem.size())) || (st = upload(c, T.tile_conn, tconn.data(), tconn.size())) ||
        (st = upload(c, T.tp_ptr, tp_ptr.data(), tp_ptr.size())) ||
        (st = upload(c, dtpair, tpair.get(), nent)) || (st = upload(c, dbpair, bpair.data(), bpair.size())) ||
        (st = dalloc(c, T.trec, 48 * nent)) || (st = upload(c, T.tcontrib, tcw.get(), nent)) ||
        (st = upload(c, T.tslot, tslot.get(), nent)) || (st = dalloc(c, T.brec, 48 * nbnd)) ||
        (st = upload(c, T.bp_ptr, bp_ptr.data(), bp_ptr.size())) ||
        (st = dalloc(c, T.partial, (size_t)std::max<int64_t>(nslots, 1) * 36 * 8)))
        return st;
    const fs::ScatterPlan sp = plan_of(B);
    for (const bool bnd : {false, true})
        FS_HIP(c, fs::launch_tile_place(bnd ? nbnd : nent, (bnd ? dbpair : dtpair).as<int32_t>(), sp,
                                        B.node_rec.as<int4>(), (bnd ? T.brec : T.trec).as<int4>(), c->stream));
    FS_HIP(c, hipStreamSynchronize(c->stream));
    T.ne = NE;
    T.ntiles = ntiles;
    T.nent = nent;
    T.nbnd = nbnd;
    T.nslots = nslots;
    return FS_OK;
}

// Element-kernel launch on the model's device arrays.
hipError_t launch_elements(fs_model *m, const fs::ElemParams &ep, int variant, hipStream_t st) {
    return fs::launch_element_blocks(ep, m->x.as<double>(), m->y.as<double>(), m->z.as<double>(),
                                     m->dconn.as<int32_t>(), m->nx.as<double>(), m->ny.as<double>(),
                                     m->nz.as<double>(), m->valid.as<uint8_t>(), m->Kb.as<double>(),
                                     m->status.as<int>(), st, variant);
}

// Validate the stiffness parameters, upload the per-group material records,
// size m->Kb, clear the status flag and pick the element-kernel launch shape
// (the autotuner times every shape on the first evaluation of a kind).
int prepare_elements(fs_model *m, const fs_shell_params *p, fs::ElemParams &ep, int *variant_out, bool blocks = true) {
    fs_ctx *c = m->ctx;
    if (!p) return fail(c, FS_ERR_ARG, "stiffness: NULL parameters");
    if (!m->normals_ready) return fail(c, FS_ERR_STATE, "stiffness: normals not computed (associategeometry!)");
    if (p->formulation != FS_SHEAR_AVERAGE_B && p->formulation != FS_SHEAR_AVERAGE_K)
        return fail(c, FS_ERR_ARG, "stiffness: unknown transverse shear formulation %d", p->formulation);
    if (m->nen == FS_Q4 && p->formulation != FS_SHEAR_AVERAGE_B)
        return fail(c, FS_ERR_ARG, "stiffness: the Q4 family has a single (MITC) shear formulation");
    std::memset(&ep, 0, sizeof ep);
    ep.nen = m->nen;
    ep.composite = p->composite ? 1 : 0;
    ep.formulation = p->formulation;
    ep.nelem = (int32_t)m->E;
    ep.ebegin = 0;
    ep.eend = (int32_t)m->E;
    ep.nnodes = m->N;
    ep.thickness = p->thickness;
    ep.stab_c = p->stab_c;
    ep.drill_scale = p->drilling_stiffness_scale;
    int s = 0;
    if (!p->composite) {
        // one material record per group: chol(Dps), chol(5/6 Dt), t, stab_c, drilling scale
        const bool grouped = p->group_homog != nullptr;
        const int ng = grouped ? p->ngroups : 1;
        if (grouped && ng < 1) return fail(c, FS_ERR_ARG, "stiffness: group_homog needs ngroups >= 1");
        std::vector<double> rec(16 * (size_t)ng);
        for (int g = 0; g < ng; ++g) {
            const double *src = grouped ? p->group_homog + 16 * g : nullptr;
            double Dps[9], Dt[4];
            cm2rm(3, grouped ? src : p->Dps, Dps);
            cm2rm(2, grouped ? src + 9 : p->Dt, Dt);
            for (int i = 0; i < 4; ++i) Dt[i] *= 5.0 / 6.0;  // FEMMShellT3FFModule.jl:658-659
            double *r = &rec[16 * g];
            if (!chol_upper(3, Dps, r)) return fail(c, FS_ERR_NUMERIC, "stiffness: Dps of group %d is not positive definite", g);
            if (!chol_upper(2, Dt, r + 9)) return fail(c, FS_ERR_NUMERIC, "stiffness: Dt of group %d is not positive definite", g);
            r[13] = grouped ? src[13] : p->thickness;
            r[14] = grouped ? src[14] : p->stab_c;
            r[15] = grouped ? src[15] : p->drilling_stiffness_scale;
            if (!(r[13] > 0.0)) return fail(c, FS_ERR_ARG, "stiffness: thickness of group %d must be positive", g);
        }
        if ((s = upload(c, m->g_homog, rec.data(), rec.size()))) return s;
        ep.g_homog = m->g_homog.as<double>();
        if (grouped && p->elem_group) {
            for (int64_t e = 0; e < m->E; ++e)
                if (p->elem_group[e] < 0 || p->elem_group[e] >= ng)
                    return fail(c, FS_ERR_ARG, "stiffness: element %lld has group %d", (long long)e, p->elem_group[e]);
            // one group: no group array, so the kernels read one material record
            if (ng > 1) {
                if ((s = upload(c, m->g_group, p->elem_group, (size_t)m->E))) return s;
                ep.elem_group = m->g_group.as<int32_t>();
            }
        }
    } else {
        const int ng = p->ngroups;
        if (ng < 1 || !p->group_ABDH || !p->group_csys || !p->group_thickness)
            return fail(c, FS_ERR_ARG, "stiffness: layered shell needs ngroups >= 1 and group arrays");
        std::vector<double> Labd(36 * ng), Lh(4 * ng), csys(9 * ng), tg(ng);
        for (int g = 0; g < ng; ++g) {
            const double *src = p->group_ABDH + 31 * g;
            double A[9], Bm[9], D[9], H[4], ABD[36];
            cm2rm(3, src, A);
            cm2rm(3, src + 9, Bm);
            cm2rm(3, src + 18, D);
            cm2rm(2, src + 27, H);
            for (int i = 0; i < 3; ++i)
                for (int j = 0; j < 3; ++j) {
                    ABD[i * 6 + j] = A[i * 3 + j];
                    ABD[i * 6 + 3 + j] = Bm[i * 3 + j];
                    ABD[(3 + i) * 6 + j] = Bm[j * 3 + i];
                    ABD[(3 + i) * 6 + 3 + j] = D[i * 3 + j];
                }
            if (!chol_upper(6, ABD, &Labd[36 * g]))
                return fail(c, FS_ERR_NUMERIC, "stiffness: laminate [A B; B D] of group %d is not positive definite", g);
            if (!chol_upper(2, H, &Lh[4 * g]))
                return fail(c, FS_ERR_NUMERIC, "stiffness: laminate H of group %d is not positive definite", g);
            cm2rm(3, p->group_csys + 9 * g, &csys[9 * g]);
            tg[g] = p->group_thickness[g];
        }
        if ((s = upload(c, m->g_Labd, Labd.data(), Labd.size()))) return s;
        if ((s = upload(c, m->g_Lh, Lh.data(), Lh.size()))) return s;
        if ((s = upload(c, m->g_csys, csys.data(), csys.size()))) return s;
        if ((s = upload(c, m->g_t, tg.data(), tg.size()))) return s;
        ep.g_Labd = m->g_Labd.as<double>();
        ep.g_Lh = m->g_Lh.as<double>();
        ep.g_csys = m->g_csys.as<double>();
        ep.g_t = m->g_t.as<double>();
        if (p->elem_group) {
            for (int64_t e = 0; e < m->E; ++e)
                if (p->elem_group[e] < 0 || p->elem_group[e] >= ng)
                    return fail(c, FS_ERR_ARG, "stiffness: element %lld has group %d", (long long)e, p->elem_group[e]);
            if (ng > 1) {
                if ((s = upload(c, m->g_group, p->elem_group, (size_t)m->E))) return s;
                ep.elem_group = m->g_group.as<int32_t>();
            }
        }
    }
    FS_HIP(c, hipMemsetAsync(m->status.p, 0, sizeof(int), c->stream));
    if (!blocks) {
        *variant_out = 0;  // the fused path has one launch shape per family
        return FS_OK;
    }
    const int nblk = m->nen * (m->nen + 1) / 2;
    const size_t kbytes = (size_t)m->E * nblk * 36 * sizeof(double);
    if (m->Kb.bytes < kbytes && (s = dalloc(c, m->Kb, kbytes))) return s;
    int &variant = c->elem_variant[m->nen == 4 ? 1 : 0][ep.formulation == FS_SHEAR_AVERAGE_K ? 1 : 0];
    if (variant < 0 && !c->autotune) variant = 0;
    if (variant < 0) {
        // autotuner: one warm launch and one timed launch per shape on
        // this model; every shape computes bitwise the same blocks
        hipEvent_t e0, e1;
        FS_HIP(c, hipEventCreate(&e0));
        FS_HIP(c, hipEventCreate(&e1));
        float best = 0.f;
        int bestv = 0;
        for (int v = 0; v < fs::element_variants(m->nen); ++v) {
            float t = 0.f;
            for (int rep = 0; rep < 2; ++rep) {
                FS_HIP(c, hipEventRecord(e0, c->stream));
                FS_HIP(c, launch_elements(m, ep, v, c->stream));
                FS_HIP(c, hipEventRecord(e1, c->stream));
                FS_HIP(c, hipEventSynchronize(e1));
                FS_HIP(c, hipEventElapsedTime(&t, e0, e1));
            }
            if (v == 0 || t < best) {
                best = t;
                bestv = v;
            }
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        variant = bestv;
    }
    *variant_out = variant;
    return FS_OK;
}

// After the stream has been synchronised: the singular-metric flag of the
// element kernels, and the bookkeeping of a successful evaluation.
int finish_elements(fs_model *m, const fs::ElemParams &ep, int status) {
    if (status)
        return fail(m->ctx, FS_ERR_NUMERIC, "Singular metric matrix in _gradN_e! (degenerate quadrilateral)");
    m->last_ep = ep;
    ++m->kgen;
    return FS_OK;
}

// Compute element node-pair blocks into m->Kb (device), timed with events.
int element_blocks(fs_model *m, const fs_shell_params *p, float *elem_ms) {
    fs_ctx *c = m->ctx;
    fs::ElemParams ep;
    int variant = 0;
    int s = prepare_elements(m, p, ep, &variant);
    if (s) return s;
    hipEvent_t e0, e1;
    FS_HIP(c, hipEventCreate(&e0));
    FS_HIP(c, hipEventCreate(&e1));
    FS_HIP(c, hipEventRecord(e0, c->stream));
    FS_HIP(c, launch_elements(m, ep, variant, c->stream));
    FS_HIP(c, hipEventRecord(e1, c->stream));
    int st = 0;
    FS_HIP(c, hipMemcpyAsync(&st, m->status.p, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    FS_HIP(c, hipStreamSynchronize(c->stream));
    FS_HIP(c, hipEventElapsedTime(elem_ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return finish_elements(m, ep, st);
}

// Build the mixed-precision operator from the parameters of the last
// stiffness evaluation: split element kernel (membrane + bending blocks,
// shear factor rows, drilling blocks), then the FP32 slices of K_mb and the
// per-node drilling blocks.
int build_mixed(fs_model *m, bool shear_fp32) {
    fs_ctx *c = m->ctx;
    Block &B = m->blk[FS_BLOCK_FF];
    MixedStore &X = m->mixed;
    X.reset();
    const int nen = m->nen;
    const int nblk = nen * (nen + 1) / 2;
    const int K = 6 * nen;
    const int nsr = shear_fp32 ? 0 : nen == 3 ? (m->last_ep.formulation == FS_SHEAR_AVERAGE_K ? 6 : 2) : 8;
    const int64_t N = m->N, E = m->E, nrows = 6 * N;
    if (const int e = host_lists(m)) return e;
    // slices of 10 nodes (60 rows): slot count = largest neighbour count of the slice's nodes
    (void)nrows;
    const int64_t ns = (N + 9) / 10;
    std::vector<int64_t> goff(ns + 1, 0);
    for (int64_t g = 0; g < ns; ++g) {
        const int64_t i0 = 10 * g, i1 = std::min<int64_t>(N - 1, 10 * g + 9);
        int mx = 0;
        for (int64_t i = i0; i <= i1; ++i) mx = std::max(mx, m->nbr_ptr[i + 1] - m->nbr_ptr[i]);
        goff[g + 1] = goff[g] + (int64_t)mx * 3 * 60;
    }
    int s;
    DevBuf kbm, dre;
    if ((s = dalloc(c, kbm, (size_t)E * nblk * 36 * 8)) || (s = dalloc(c, dre, (size_t)E * nen * 9 * 8)) ||
        (nsr > 0 && (s = dalloc(c, X.cs, (size_t)E * nsr * K * 8))) || (s = dalloc(c, X.dr, (size_t)N * 6 * 8)) ||
        (s = upload(c, X.goff, goff.data(), goff.size())) ||
        (s = dalloc(c, X.kmb, (size_t)goff[ns] * sizeof(float2))) ||
        (s = dalloc(c, X.kml, (size_t)goff[ns] * sizeof(short2))))
        return s;
    if (nsr > 0) {
        // incidence records: element and its nodes, in each node's ascending element order
        const int ps = nen == 3 ? 4 : 8;
        std::vector<int32_t> pack((size_t)m->ne_list.size() * ps, 0);
        for (size_t k = 0; k < m->ne_list.size(); ++k) {
            const int32_t e = m->ne_list[k];
            pack[k * ps] = e;
            for (int a = 0; a < nen; ++a) pack[k * ps + 1 + a] = m->conn[(size_t)e * nen + a];
        }
        if ((s = upload(c, X.ne_pack, pack.data(), pack.size()))) return s;
    }
    fs::ElemParams ep = m->last_ep;
    ep.split_cs = nsr > 0 ? X.cs.as<double>() : nullptr;  // nullptr: shear stays in the blocks
    ep.split_dr = dre.as<double>();
    hipEvent_t e0, e1;
    FS_HIP(c, hipEventCreate(&e0));
    FS_HIP(c, hipEventCreate(&e1));
    FS_HIP(c, hipEventRecord(e0, c->stream));
    FS_HIP(c, hipMemsetAsync(X.kmb.p, 0, (size_t)goff[ns] * sizeof(float2), c->stream));
    FS_HIP(c, hipMemsetAsync(X.kml.p, 0, (size_t)goff[ns] * sizeof(short2), c->stream));
    FS_HIP(c, fs::launch_element_blocks(ep, m->x.as<double>(), m->y.as<double>(), m->z.as<double>(),
                                        m->dconn.as<int32_t>(), m->nx.as<double>(), m->ny.as<double>(),
                                        m->nz.as<double>(), m->valid.as<uint8_t>(), kbm.as<double>(),
                                        m->status.as<int>(), c->stream, 0));
    FS_HIP(c, fs::launch_mixed_build(plan_of(B), kbm.as<double>(), X.goff.as<int64_t>(), X.kmb.as<float2>(), X.kml.as<short2>(),
                                     c->stream));
    FS_HIP(c, fs::launch_mixed_drill(nen, N, (int)E, m->dne_ptr.as<int32_t>(), m->dne_list.as<int32_t>(),
                                     m->dconn.as<int32_t>(), dre.as<double>(), X.dr.as<double>(), c->stream));
    FS_HIP(c, hipEventRecord(e1, c->stream));
    FS_HIP(c, hipStreamSynchronize(c->stream));
    FS_HIP(c, hipEventElapsedTime(&X.build_ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    X.nsr = nsr;
    X.shear_fp32 = shear_fp32;
    X.nslices = ns;
    X.kmb_pairs = goff[ns];
    X.kgen = m->kgen;
    X.built = true;
    return FS_OK;
}

fs::MixedOp mixed_op(const fs_model *m) {
    const Block &B = m->blk[FS_BLOCK_FF];
    fs::MixedOp op;
    op.nrows = 6 * m->N;
    op.nnodes = (int32_t)m->N;
    op.nelem = (int32_t)m->E;
    op.goff = m->mixed.goff.as<int64_t>();
    op.kmb = m->mixed.kmb.as<float2>();
    op.kml = m->mixed.kml.as<short2>();
    op.nbr_ptr = B.nbr_ptr;
    op.nbr_node = B.nbr_node;
    op.dr = m->mixed.dr.as<double>();
    op.ne_ptr = m->dne_ptr.as<int32_t>();
    op.ne_pack = m->mixed.ne_pack.as<int32_t>();
    op.cs = m->mixed.cs.as<double>();
    return op;
}

// Places of the one-launch loops on each device: a loop's workgroups wait for
// one another, so all loops in flight have to fit the device together.  A loop
// takes as many places as it has patches and gives them back when it has
// ended; there are two per CU, of the three and more workgroups that a CU holds.
// They are counted within a process, and one process at a time has them: it holds a
// lock on a file of the device's (by its PCI address, in /dev/shm) while loops of
// its own are in flight (two system calls), and the kernel gives the lock back when
// a process ends.  Where no such file is to be had the count stands alone, and loops of
// two processes that do not fit together end by their bounded waits.
class LoopPlaces {
  public:
    ~LoopPlaces() {
        if (n_ == 0) return;
        std::lock_guard<std::mutex> lk(mu());
        Device &d = device(dev_);
        d.used -= n_;
        if (d.used == 0 && d.lock >= 0) (void)flock(d.lock, LOCK_UN);
    }
    bool take(int dev, int64_t n) {
        if (dev < 0 || dev >= 64 || n <= 0) return false;
        std::lock_guard<std::mutex> lk(mu());
        Device &d = device(dev);
        if (d.cus == 0) {
            int v = 0;
            if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return false;
            d.lock = open_lock(dev);
            d.cus = v;
        }
        if (d.used + n > 2 * d.cus) return false;
        if (d.used == 0 && d.lock >= 0 && flock(d.lock, LOCK_EX | LOCK_NB) != 0 && errno == EWOULDBLOCK) return false;
        d.used += n;
        dev_ = dev;
        n_ = n;
        return true;
    }

  private:
    struct Device {
        int64_t cus = 0, used = 0;
        int lock = -1;
    };
    static std::mutex &mu() {
        static std::mutex m;
        return m;
    }
    static Device &device(int dev) {
        static std::array<Device, 64> d;
        return d[dev];
    }
    // read-only, so that it works for a file of another user too
    static int open_lock(int dev) {
        char bus[64] = "";
        if (hipDeviceGetPCIBusId(bus, sizeof bus, dev) != hipSuccess) {
            (void)hipGetLastError();
            return -1;
        }
        const std::string path = std::string("/dev/shm/flexshell-loops-") + bus;
        const int flags = O_RDONLY | O_CLOEXEC | O_NOFOLLOW;
        int fd = open(path.c_str(), flags);
        if (fd < 0) {
            fd = open(path.c_str(), flags | O_CREAT, 0644);
            if (fd >= 0) (void)fchmod(fd, 0644);  // whatever the umask
        }
        return fd;
    }
    int dev_ = 0;
    int64_t n_ = 0;
};

// Polls after which a lane of the one-launch loop gives up: about two seconds.
constexpr uint32_t LOOP_POLLS = 1u << 21;

// Whether the one-launch loop takes a plan at this precision.
int patch_loops(fs_model *m, int precision, bool *yes) {
    fs_ctx *c = m->ctx;
    PatchStore &P = m->blk[FS_BLOCK_FF].patch;
    *yes = false;
    if (!P.loops || c->loop_polls < 0 || c->loop_gave_up) return FS_OK;
    const int f32 = precision == FS_PREC_MIXED_F32;
    if (P.loop_per_cu[f32] == 0) FS_HIP(c, fs::patch_loop_occupancy(patchop_of(P), f32, &P.loop_per_cu[f32]));
    if (P.loop_per_cu[f32] < 3) return FS_OK;  // LoopPlaces counts on it
    if (!c->loop_stop) FS_HIP(c, hipHostMalloc((void **)&c->loop_stop, 64, hipHostMallocDefault));
    *yes = true;
    return FS_OK;
}

// The patch form of a precision's operator (the mixed ones built already): its
// plan, if there is none yet, and its blocks, if they are of another precision
// or other values.  *use becomes false where the form does not take the mesh,
// or there is no memory for it.
int prepare_patches(fs_model *m, int precision, bool *use) {
    fs_ctx *c = m->ctx;
    Block &B = m->blk[FS_BLOCK_FF];
    PatchStore &P = B.patch;
    auto without = [&](int s) {  // no memory: the other forms, for this block
        P.reset();
        if (s != FS_ERR_NOMEM) return s;
        P.planned = true;
        *use = false;
        c->err.clear();
        return FS_OK;
    };
    int s;
    if (!P.planned && (s = build_patches(m))) return without(s);
    *use = P.usable;
    const uint64_t kgen = precision == FS_PREC_FP64 ? 0 : m->mixed.kgen;
    if (!P.usable || (P.kind == precision && P.vgen == B.vgen && P.kgen == kgen)) return FS_OK;
    P.kind = -1;
    const bool f32 = precision == FS_PREC_MIXED_F32;
    if (f32 ? (s = ensure(c, P.kh, (size_t)P.nent * 144)) || (s = ensure(c, P.kl, (size_t)P.nent * 72))
            : (s = ensure(c, P.k2, (size_t)P.nent * 288)))
        return without(s);
    FS_HIP(c, fs::launch_patch_build(patchop_of(P), precision == FS_PREC_FP64 ? 0 : f32 ? 2 : 1, plan_of(B),
                                     B.kval.as<double>(), precision == FS_PREC_FP64 ? fs::MixedOp{} : mixed_op(m),
                                     m->dconn.as<int32_t>(), m->nen, precision == FS_PREC_FP64 ? 0 : m->mixed.nsr,
                                     c->stream));
    P.kind = precision;
    P.vgen = B.vgen;
    P.kgen = kgen;
    return FS_OK;
}

}  // namespace

extern "C" {

const char *fs_version(void) { return "flexshell 0.1.0 (gfx950)"; }

int fs_ctx_create(int device, fs_ctx **out) {
    if (!out) return FS_ERR_ARG;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return FS_ERR_DEVICE;
    if (device < 0 || device >= n) return FS_ERR_ARG;
    fs_ctx *c = new (std::nothrow) fs_ctx;
    if (!c) return FS_ERR_NOMEM;
    c->cache = new (std::nothrow) BufCache;
    if (!c->cache) {
        delete c;
        return FS_ERR_NOMEM;
    }
    c->device = device;
    if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
        delete c->cache;
        delete c;
        return FS_ERR_DEVICE;
    }
    // with `device` current: the device's copy of the allocation-free workspace
    c->scratch_status = fs::noalloc_workspace(device, &c->scratch);
    if (c->scratch_status != hipSuccess) (void)hipGetLastError();
    *out = c;
    return FS_OK;
}

}  // extern "C"

namespace {
// Drops one reference; the last one (the caller's handle or the last live
// model) destroys the streams, events, staging buffers and the context.
void ctx_release(fs_ctx *ctx) {
    if (--ctx->refs > 0) return;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    if (ctx->stream2) {
        (void)hipStreamSynchronize(ctx->stream2);
        (void)hipStreamDestroy(ctx->stream2);
    }
    for (hipEvent_t ev : ctx->ev) (void)hipEventDestroy(ev);
    if (ctx->stage) (void)hipHostFree(ctx->stage);
    for (hipEvent_t ev : ctx->stage_ev)
        if (ev) (void)hipEventDestroy(ev);
    if (ctx->loop_stop) (void)hipHostFree(ctx->loop_stop);
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    delete ctx;
}
}  // namespace

extern "C" {

void fs_ctx_destroy(fs_ctx *ctx) {
    if (!ctx) return;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    if (ctx->stream2) (void)hipStreamSynchronize(ctx->stream2);
    int left;
    {
        std::lock_guard<std::mutex> lk(ctx->cache->mu);
        for (auto &kv : ctx->cache->spare) (void)hipFree(kv.second);
        ctx->cache->spare.clear();
        ctx->cache->spare_bytes = 0;
        ctx->cache->alive = false;  // buffers of models still alive are freed when released
        left = --ctx->cache->refs;
    }
    if (left == 0) delete ctx->cache;
    ctx->cache = nullptr;
    ctx_release(ctx);
}

const char *fs_last_error(const fs_ctx *ctx) { return ctx ? ctx->err.c_str() : "no context"; }

int fs_model_create(fs_ctx *ctx, int nen, int64_t nnodes, const double *xyz, int64_t nelem, const int64_t *conn,
                    int index_base, fs_model **out) {
    if (!ctx || !out) return FS_ERR_ARG;
    *out = nullptr;
    ctx->err.clear();
    if (nen != FS_T3 && nen != FS_Q4) return fail(ctx, FS_ERR_ARG, "nen must be 3 or 4, got %d", nen);
    if (nnodes <= 0 || nelem <= 0 || !xyz || !conn) return fail(ctx, FS_ERR_ARG, "empty mesh or NULL arrays");
    if (nnodes >= (int64_t(1) << 31) || nelem >= (int64_t(1) << 31))
        return fail(ctx, FS_ERR_UNSUPPORTED, "mesh too large for 32-bit node/element indices");
    FS_HIP(ctx, hipSetDevice(ctx->device));
    fs_model *m = new (std::nothrow) fs_model;
    if (!m) return fail(ctx, FS_ERR_NOMEM, "model allocation");
    m->ctx = ctx;
    m->nen = nen;
    m->N = nnodes;
    m->E = nelem;
    m->conn.resize((size_t)nelem * nen);
    for (int64_t i = 0; i < nelem * nen; ++i) {
        const int64_t v = conn[i] - index_base;
        if (v < 0 || v >= nnodes) {
            delete m;
            return fail(ctx, FS_ERR_ARG, "connectivity entry %lld out of range", (long long)i);
        }
        m->conn[i] = (int32_t)v;
    }
    for (int64_t e = 0; e < nelem; ++e)
        for (int a = 0; a < nen; ++a)
            for (int b = a + 1; b < nen; ++b)
                if (m->conn[e * nen + a] == m->conn[e * nen + b]) {
                    delete m;
                    return fail(ctx, FS_ERR_ARG, "element %lld repeats a node", (long long)e);
                }
    // node -> element lists in ascending element order
    m->ne_ptr.assign(nnodes + 1, 0);
    for (int64_t i = 0; i < nelem * nen; ++i) m->ne_ptr[m->conn[i] + 1]++;
    for (int64_t n = 0; n < nnodes; ++n) m->ne_ptr[n + 1] += m->ne_ptr[n];
    m->ne_list.resize(m->ne_ptr[nnodes]);
    {
        std::vector<int32_t> fill(m->ne_ptr.begin(), m->ne_ptr.end() - 1);
        for (int64_t e = 0; e < nelem; ++e)
            for (int a = 0; a < nen; ++a) m->ne_list[fill[m->conn[e * nen + a]]++] = (int32_t)e;
    }
    // device geometry (SoA) and connectivity planes
    int s;
    std::vector<int32_t> planes((size_t)nelem * nen);
    fs::parallel_chunks(nelem, [&](int64_t e0, int64_t e1) {
        for (int64_t e = e0; e < e1; ++e)
            for (int a = 0; a < nen; ++a) planes[(size_t)a * nelem + e] = m->conn[e * nen + a];
    });
    if ((s = upload(ctx, m->x, xyz, nnodes)) || (s = upload(ctx, m->y, xyz + nnodes, nnodes)) ||
        (s = upload(ctx, m->z, xyz + 2 * nnodes, nnodes)) || (s = upload(ctx, m->dconn, planes.data(), planes.size())) ||
        (s = upload(ctx, m->dne_ptr, m->ne_ptr.data(), m->ne_ptr.size())) ||
        (s = upload(ctx, m->dne_list, m->ne_list.data(), m->ne_list.size())) ||
        (s = dalloc(ctx, m->nx, nnodes * 8)) || (s = dalloc(ctx, m->ny, nnodes * 8)) ||
        (s = dalloc(ctx, m->nz, nnodes * 8)) || (s = dalloc(ctx, m->valid, nnodes)) ||
        (s = dalloc(ctx, m->status, sizeof(int))) || (s = make_neighbours(m))) {
        delete m;
        return s;
    }
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) {
        delete m;
        return fail(ctx, FS_ERR_DEVICE, "upload of the mesh failed");
    }
    ++ctx->refs;
    *out = m;
    return FS_OK;
}

void fs_model_destroy(fs_model *m) {
    if (!m) return;
    fs_ctx *c = m->ctx;
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    if (c->stream2) (void)hipStreamSynchronize(c->stream2);
    delete m;  // its buffers go back to the context's spare list, or to hipFree once the context is destroyed
    ctx_release(c);
}

int fs_model_set_dofs(fs_model *m, const int64_t *dofnums, int64_t nalldofs, int64_t nfreedofs, int index_base) {
    if (!m) return FS_ERR_ARG;
    fs_ctx *c = m->ctx;
    c->err.clear();
    if (!dofnums || nalldofs <= 0 || nfreedofs < 0 || nfreedofs > nalldofs)
        return fail(c, FS_ERR_ARG, "set_dofs: bad sizes (nalldofs %lld, nfreedofs %lld)", (long long)nalldofs,
                    (long long)nfreedofs);
    const int64_t N = m->N;
    std::vector<int64_t> dof(N * 6);
    std::vector<uint8_t> seen(nalldofs, 0);
    for (int64_t I = 0; I < N; ++I)
        for (int cc = 0; cc < 6; ++cc) {
            const int64_t d = dofnums[cc * N + I] - index_base;  // column-major N x 6
            if (d < 0 || d >= nalldofs) return fail(c, FS_ERR_ARG, "dof number out of range at node %lld", (long long)I);
            if (seen[d]) return fail(c, FS_ERR_ARG, "dof number %lld used twice", (long long)(d + index_base));
            seen[d] = 1;
            dof[I * 6 + cc] = d;
        }
    if ((int64_t)N * 6 != nalldofs) return fail(c, FS_ERR_ARG, "nalldofs must equal 6 * nnodes");
    FS_HIP(c, hipSetDevice(c->device));
    // the planner's kernels read the device copy: from here on no numbers, until
    // the new ones are there (in the buffer of the old, which have as many)
    int s = ensure(c, m->node_dof, dof.size() * 8);
    if (s) return s;
    m->dofs_ready = false;
    m->blk[0].reset();
    m->blk[1].reset();
    m->mixed.reset();
    FS_HIP(c, hipMemcpyAsync(m->node_dof.p, dof.data(), dof.size() * 8, hipMemcpyHostToDevice, c->stream));
    FS_HIP(c, hipStreamSynchronize(c->stream));
    m->dof.swap(dof);
    m->nall = nalldofs;
    m->nfree = nfreedofs;
    m->dofs_ready = true;
    return FS_OK;
}

int fs_model_number_dofs(fs_model *m, const uint8_t *is_fixed, const int64_t *perm, int64_t *dofnums_out,
                         int64_t *nfree_out) {
    if (!m) return FS_ERR_ARG;
    fs_ctx *c = m->ctx;
    c->err.clear();
    if (!is_fixed) return fail(c, FS_ERR_ARG, "number_dofs: NULL flags");
    const int64_t N = m->N, n = N * 6;
    std::vector<uint8_t> pf;
    if (perm) {
        // flags in numbering order: node perm[k] is the k-th node numbered
        std::vector<uint8_t> seen((size_t)N, 0);
        pf.resize((size_t)n);
        for (int64_t k = 0; k < N; ++k) {
            const int64_t I = perm[k];
            if (I < 0 || I >= N || seen[I]) return fail(c, FS_ERR_ARG, "number_dofs: perm is not a permutation");
            seen[I] = 1;
            for (int cc = 0; cc < 6; ++cc) pf[k * 6 + cc] = is_fixed[I * 6 + cc];
        }
    }
    FS_HIP(c, hipSetDevice(c->device));
    DevBuf dfix, dtile, dtot;
    int s;
    if ((s = upload(c, dfix, perm ? pf.data() : is_fixed, (size_t)n)) ||
        (s = dalloc(c, dtile, fs::number_dofs_tiles(n) * 8 + 8)) || (s = dalloc(c, dtot, 8)) ||
        (s = ensure(c, m->node_dof, (size_t)n * 8)))
        return s;
    // the planner's kernels read the device copy: from here on no numbers, until
    // the new ones are there
    m->dofs_ready = false;
    m->blk[0].reset();
    m->blk[1].reset();
    m->mixed.reset();
    FS_HIP(c, hipMemsetAsync(dtot.p, 0, 8, c->stream));
    FS_HIP(c, fs::launch_number_dofs(n, dfix.as<uint8_t>(), dtile.as<int64_t>(), dtot.as<int64_t>(),
                                     m->node_dof.as<int64_t>(), c->stream));
    std::vector<int64_t> dof((size_t)n);
    int64_t nfree = 0;
    FS_HIP(c, hipMemcpyAsync(&nfree, dtot.p, 8, hipMemcpyDeviceToHost, c->stream));
    FS_HIP(c, hipMemcpyAsync(dof.data(), m->node_dof.p, (size_t)n * 8, hipMemcpyDeviceToHost, c->stream));
    FS_HIP(c, hipStreamSynchronize(c->stream));
    if (perm) {
        // back to node order on the host, and the device copy replaced
        std::vector<int64_t> byn((size_t)n);
        for (int64_t k = 0; k < N; ++k)
            for (int cc = 0; cc < 6; ++cc) byn[perm[k] * 6 + cc] = dof[k * 6 + cc];
        dof.swap(byn);
        FS_HIP(c, hipMemcpyAsync(m->node_dof.p, dof.data(), (size_t)n * 8, hipMemcpyHostToDevice, c->stream));
        FS_HIP(c, hipStreamSynchronize(c->stream));
    }
    // the host copy feeds the pattern planner
    m->dof.swap(dof);
    m->nall = n;
    m->nfree = nfree;
    m->dofs_ready = true;
    if (dofnums_out)
        for (int64_t I = 0; I < m->N; ++I)
            for (int cc = 0; cc < 6; ++cc) dofnums_out[cc * m->N + I] = m->dof[I * 6 + cc];
    if (nfree_out) *nfree_out = nfree;
    return FS_OK;
}

static bool load_rule_ok(int nen, int npts) { return nen == 3 ? (npts == 1 || npts == 3 || npts == 6) : npts == 4; }

int fs_model_surface_load(fs_model *m, int32_t npts, int32_t kind, const double *force, int block, double *F_out) {
    if (!m) return FS_ERR_ARG;
    fs_ctx *c = m->ctx;
    c->err.clear();
    if (!force || !F_out) return fail(c, FS_ERR_ARG, "surface_load: NULL arguments");
    if (kind != FS_LOAD_UNIFORM && kind != FS_LOAD_PER_POINT) return fail(c, FS_ERR_ARG, "surface_load: kind %d", kind);
    if (block != FS_BLOCK_ALL && block != FS_BLOCK_FF) return fail(c, FS_ERR_ARG, "unknown block %d", block);
    if (!m->dofs_ready) return fail(c, FS_ERR_STATE, "surface_load: equation numbers not set");
    if (!load_rule_ok(m->nen, npts)) return fail(c, FS_ERR_ARG, "surface_load: %d-point rule", npts);
    FS_HIP(c, hipSetDevice(c->device));
    const int64_t nrows = block == FS_BLOCK_FF ? m->nfree : m->nall;
    DevBuf dforce, dF;
    int s;
    if ((s = upload(c, dforce, force, kind == FS_LOAD_UNIFORM ? 6 : (size_t)m->E * npts * 6)) ||
        (s = dalloc(c, dF, (size_t)nrows * 8)))
        return s;
    FS_HIP(c, fs::launch_surface_load(m->nen, npts, m->N, (int)m->E, m->x.as<double>(), m->y.as<double>(),
                                      m->z.as<double>(), m->dconn.as<int32_t>(), m->dne_ptr.as<int32_t>(),
                                      m->dne_list.as<int32_t>(), kind == FS_LOAD_PER_POINT ? 1 : 0,
                                      dforce.as<double>(), m->node_dof.as<int64_t>(), nrows, dF.as<double>(),
                                      c->stream));
    return d2h(c, F_out, dF.p, (size_t)nrows * 8);
}

int fs_model_load_points(fs_model *m, int32_t npts, double *xyz_out) {
    if (!m) return FS_ERR_ARG;
    fs_ctx *c = m->ctx;
    c->err.clear();
    if (!xyz_out) return fail(c, FS_ERR_ARG, "load_points: NULL output");
    if (!load_rule_ok(m->nen, npts)) return fail(c, FS_ERR_ARG, "load_points: %d-point rule", npts);
    FS_HIP(c, hipSetDevice(c->device));
    const size_t n = (size_t)m->E * npts * 3;
    DevBuf d;
    int s = dalloc(c, d, n * 8);
    if (s) return s;
    FS_HIP(c, fs::launch_load_points(m->nen, npts, (int)m->E, m->x.as<double>(), m->y.as<double>(), m->z.as<double>(),
                                     m->dconn.as<int32_t>(), d.as<double>(), c->stream));
    return d2h(c, xyz_out, d.p, n * 8);
}

// Normals kernel in either form (gnrm null: isoparametric) and the copies out.
static int normals_common(fs_model *m, double threshold_angle_deg, const double *gnrm, const int32_t *egroup,
                          double *normals_out, uint8_t *valid_out) {
    fs_ctx *c = m->ctx;
    const double s = std::sin(threshold_angle_deg / 180 * M_PI);
    const double ntol = 1 - std::sqrt(1 - s * s);  // FEMMShellT3FFModule.jl:600
    FS_HIP(c, fs::launch_normals(m->nen, m->N, (int)m->E, m->x.as<double>(), m->y.as<double>(), m->z.as<double>(),
                                 m->dconn.as<int32_t>(), m->dne_ptr.as<int32_t>(), m->dne_list.as<int32_t>(), ntol,
                                 gnrm, egroup, m->nx.as<double>(), m->ny.as<double>(), m->nz.as<double>(),
                                 m->valid.as<uint8_t>(), c->stream));
    if (normals_out) {
        FS_HIP(c, hipMemcpyAsync(normals_out, m->nx.p, m->N * 8, hipMemcpyDeviceToHost, c->stream));
        FS_HIP(c, hipMemcpyAsync(normals_out + m->N, m->ny.p, m->N * 8, hipMemcpyDeviceToHost, c->stream));
        FS_HIP(c, hipMemcpyAsync(normals_out + 2 * m->N, m->nz.p, m->N * 8, hipMemcpyDeviceToHost, c->stream));
    }
    if (valid_out) FS_HIP(c, hipMemcpyAsync(valid_out, m->valid.p, m->N, hipMemcpyDeviceToHost, c->stream));
    FS_HIP(c, hipStreamSynchronize(c->stream));
    m->normals_ready = true;
    return FS_OK;
}

int fs_model_normals_isoparametric(fs_model *m, double threshold_angle_deg, double *normals_out, uint8_t *valid_out) {
    if (!m) return FS_ERR_ARG;
    fs_ctx *c = m->ctx;
    c->err.clear();
    FS_HIP(c, hipSetDevice(c->device));
    return normals_common(m, threshold_angle_deg, nullptr, nullptr, normals_out, valid_out);
}

int fs_model_normals_layered(fs_model *m, double threshold_angle_deg, int32_t ngroups, const double *group_normal,
                             const int32_t *elem_group, double *normals_out, uint8_t *valid_out) {
    if (!m) return FS_ERR_ARG;
    fs_ctx *c = m->ctx;
    c->err.clear();
    if (ngroups < 1 || !group_normal) return fail(c, FS_ERR_ARG, "normals: layered form needs ngroups >= 1 normals");
    if (elem_group)
        for (int64_t e = 0; e < m->E; ++e)
            if (elem_group[e] < 0 || elem_group[e] >= ngroups)
                return fail(c, FS_ERR_ARG, "normals: element %lld has group %d", (long long)e, elem_group[e]);
    FS_HIP(c, hipSetDevice(c->device));
    DevBuf dg, de;
    int s;
    if ((s = upload(c, dg, group_normal, (size_t)ngroups * 3))) return s;
    if (elem_group && (s = upload(c, de, elem_group, (size_t)m->E))) return s;
    return normals_common(m, threshold_angle_deg, dg.as<double>(), elem_group ? de.as<int32_t>() : nullptr,
                          normals_out, valid_out);
}

int fs_model_normals_upload(fs_model *m, const double *normals, const uint8_t *valid) {
    if (!m) return FS_ERR_ARG;
    fs_ctx *c = m->ctx;
    c->err.clear();
    if (!normals || !valid) return fail(c, FS_ERR_ARG, "normals_upload: NULL arrays");
    FS_HIP(c, hipSetDevice(c->device));
    FS_HIP(c, hipMemcpyAsync(m->nx.p, normals, m->N * 8, hipMemcpyHostToDevice, c->stream));
    FS_HIP(c, hipMemcpyAsync(m->ny.p, normals + m->N, m->N * 8, hipMemcpyHostToDevice, c->stream));
    FS_HIP(c, hipMemcpyAsync(m->nz.p, normals + 2 * m->N, m->N * 8, hipMemcpyHostToDevice, c->stream));
    FS_HIP(c, hipMemcpyAsync(m->valid.p, valid, m->N, hipMemcpyHostToDevice, c->stream));
    FS_HIP(c, hipStreamSynchronize(c->stream));
    m->normals_ready = true;
    return FS_OK;
}

int fs_model_pattern(fs_model *m, int block, int64_t *nrows, int64_t *nnz) {
    if (!m) return FS_ERR_ARG;
    fs_ctx *c = m->ctx;
    c->err.clear();
    if (block != FS_BLOCK_ALL && block != FS_BLOCK_FF) return fail(c, FS_ERR_ARG, "unknown block %d", block);
    FS_HIP(c, hipSetDevice(c->device));
    int s = build_block(m, block);
    if (s) return s;
    if (nrows) *nrows = m->blk[block].nrows;
    if (nnz) *nnz = m->blk[block].nnz;
    return FS_OK;
}

// Pattern entries that fs_model_pattern_get holds on the device at a time (64 MB).
static constexpr int64_t PATTERN_WINDOW = int64_t(1) << 23;

int fs_model_pattern_get(fs_model *m, int block, int64_t *rowptr, int64_t *colval, int index_base) {
    if (!m) return FS_ERR_ARG;
    int s = fs_model_pattern(m, block, nullptr, nullptr);
    if (s) return s;
    const Block &B = m->blk[block];
    // written on the device as the caller takes them, and copied out in windows, so
    // that the scratch stays within PATTERN_WINDOW entries (less where the device
    // has no room for that)
    fs_ctx *c = m->ctx;
    DevBuf w;
    int64_t win = std::min(std::max(B.nnz, B.nrows + 1), PATTERN_WINDOW);
    while ((s = dalloc(c, w, (size_t)win * 8)) == FS_ERR_NOMEM && win > 65536) win = (win + 1) / 2;
    if (s) return s;
    c->err.clear();
    for (int64_t i0 = 0; rowptr && i0 <= B.nrows; i0 += win) {
        const int64_t n = std::min(B.nrows + 1 - i0, win);
        FS_HIP(c, fs::launch_pattern_rows(n, B.rowptr.as<int32_t>() + i0, index_base, w.as<int64_t>(), c->stream));
        if ((s = d2h(c, rowptr + i0, w.p, (size_t)n * 8))) return s;
    }
    for (int64_t w0 = 0; colval && w0 < B.nnz; w0 += win) {
        const int64_t w1 = std::min(B.nnz, w0 + win);
        FS_HIP(c, fs::launch_pattern_cols(plan_of(B), m->node_dof.as<int64_t>(), index_base, w0, w1, w.as<int64_t>(),
                                          c->stream));
        if ((s = d2h(c, colval + w0, w.p, (size_t)(w1 - w0) * 8))) return s;
    }
    return FS_OK;
}

int fs_model_element_blocks(fs_model *m, const fs_shell_params *p, double *blocks_out) {
    if (!m) return FS_ERR_ARG;
    fs_ctx *c = m->ctx;
    c->err.clear();
    FS_HIP(c, hipSetDevice(c->device));
    float ms = 0.f;
    int s = element_blocks(m, p, &ms);
    if (s) return s;
    m->timing[0] = ms;
    if (blocks_out) {
        const int nblk = m->nen * (m->nen + 1) / 2;
        return d2h(c, blocks_out, m->Kb.p, (size_t)m->E * nblk * 36 * 8);
    }
    return FS_OK;
}

int fs_model_stiffness(fs_model *m, const fs_shell_params *p, int block, double *nzval_out) {
    if (!m) return FS_ERR_ARG;
    fs_ctx *c = m->ctx;
    c->err.clear();
    if (block != FS_BLOCK_ALL && block != FS_BLOCK_FF) return fail(c, FS_ERR_ARG, "unknown block %d", block);
    FS_HIP(c, hipSetDevice(c->device));
    int s = build_block(m, block);
    if (s) return s;
    Block &B = m->blk[block];
    fs::ElemParams ep;
    int variant = 0;
    if (c->assembly == 1) {
        // fused element tiles: one element kernel writes the CSR values of the
        // pairs its tile completes and the partial sums of the others; the
        // finalize kernel adds the partials of the boundary pairs
        const int NE = fs::fused_tile_elems(m->nen);
        if (B.tiles.ne != NE && (s = build_tiles(m, block, NE))) return s;
        if ((s = prepare_elements(m, p, ep, &variant, false))) return s;
        ep.ebegin = 0;
        ep.eend = (int32_t)(B.tiles.ntiles * NE);
        ep.tile_elem = B.tiles.tile_elem.as<int32_t>();
        ep.tile_conn = B.tiles.tile_conn.as<int32_t>();
        const fs::ScatterPlan sp = plan_of(B);
        const fs::TilePlan tp = tileplan_of(B);
        hipEvent_t t0, t1, t2;
        FS_HIP(c, hipEventCreate(&t0));
        FS_HIP(c, hipEventCreate(&t1));
        FS_HIP(c, hipEventCreate(&t2));
        FS_HIP(c, hipEventRecord(t0, c->stream));
        ++B.vgen;
        FS_HIP(c, fs::launch_element_fused(ep, m->x.as<double>(), m->y.as<double>(), m->z.as<double>(),
                                           m->dconn.as<int32_t>(), m->nx.as<double>(), m->ny.as<double>(),
                                           m->nz.as<double>(), m->valid.as<uint8_t>(), m->status.as<int>(), sp, tp,
                                           B.kval.as<double>(), c->stream));
        FS_HIP(c, hipEventRecord(t1, c->stream));
        FS_HIP(c, fs::launch_pair_finalize(sp, tp, B.kval.as<double>(), c->stream));
        FS_HIP(c, hipEventRecord(t2, c->stream));
        int st = 0;
        FS_HIP(c, hipMemcpyAsync(&st, m->status.p, sizeof(int), hipMemcpyDeviceToHost, c->stream));
        FS_HIP(c, hipStreamSynchronize(c->stream));
        float ms_elem = 0.f, ms_all = 0.f;
        FS_HIP(c, hipEventElapsedTime(&ms_elem, t0, t1));
        FS_HIP(c, hipEventElapsedTime(&ms_all, t0, t2));
        (void)hipEventDestroy(t0);
        (void)hipEventDestroy(t1);
        (void)hipEventDestroy(t2);
        ep.tile_elem = nullptr;
        ep.tile_conn = nullptr;
        ep.eend = (int32_t)m->E;
        if ((s = finish_elements(m, ep, st))) return s;
        m->timing[0] = ms_elem;
        m->timing[1] = ms_all - ms_elem;
        m->timing[2] = ms_all;
        B.k_ready = true;
        if (nzval_out) return d2h(c, nzval_out, B.kval.p, (size_t)B.nnz * 8);
        return FS_OK;
    }
    if ((s = prepare_elements(m, p, ep, &variant))) return s;
    // Element ranges of whole workgroups.  After range k the pairs whose
    // contributing elements all lie in ranges 0..k are complete (pair_emax),
    // so their scatter is queued on stream2 behind an event and overlaps the
    // element kernels of the next ranges.  Each pair is still summed by one
    // thread in ascending element order: the values are bitwise those of the
    // unpipelined sequence.
    int ne = 1, wg = 0;
    fs::element_variant_shape(m->nen, variant, &ne, &wg);
    const int64_t E = m->E;
    const int nch = std::max(1, c->asm_chunks);
    int64_t per = (E + nch - 1) / nch;
    per = std::max<int64_t>(ne, (per + ne - 1) / ne * ne);
    const int64_t nranges = E == 0 ? 0 : (E + per - 1) / per;
    while ((int64_t)c->ev.size() < nranges + 1) {
        hipEvent_t ev;
        FS_HIP(c, hipEventCreateWithFlags(&ev, hipEventDisableTiming));
        c->ev.push_back(ev);
    }
    if (!c->stream2) FS_HIP(c, hipStreamCreateWithFlags(&c->stream2, hipStreamNonBlocking));
    const bool piped = nranges > 1;
    if (piped && (s = pair_order(m, B))) return s;
    hipEvent_t t0, t1, t2;
    FS_HIP(c, hipEventCreate(&t0));
    FS_HIP(c, hipEventCreate(&t1));
    FS_HIP(c, hipEventCreate(&t2));
    FS_HIP(c, hipEventRecord(t0, c->stream));
    fs::ScatterPlan sp = plan_of(B);
    ++B.vgen;
    int64_t pdone = 0;
    for (int64_t k = 0; k < nranges; ++k) {
        ep.ebegin = (int32_t)(k * per);
        ep.eend = (int32_t)std::min(E, (k + 1) * per);
        FS_HIP(c, launch_elements(m, ep, variant, c->stream));
        if (!piped) break;
        int64_t pend = B.npairs;
        if (ep.eend < E)
            pend = std::upper_bound(B.pair_emax.begin(), B.pair_emax.end(), ep.eend - 1) - B.pair_emax.begin();
        if (pend > pdone) {
            FS_HIP(c, hipEventRecord(c->ev[k], c->stream));
            FS_HIP(c, hipStreamWaitEvent(c->stream2, c->ev[k], 0));
            sp.pbegin = pdone;
            sp.pend = pend;
            FS_HIP(c, fs::launch_scatter(sp, m->Kb.as<double>(), B.kval.as<double>(), c->stream2));
            pdone = pend;
        }
    }
    FS_HIP(c, hipEventRecord(t1, c->stream));
    if (piped) {
        FS_HIP(c, hipEventRecord(c->ev[nranges], c->stream2));
        FS_HIP(c, hipStreamWaitEvent(c->stream, c->ev[nranges], 0));
    } else {
        FS_HIP(c, fs::launch_scatter(plan_of(B), m->Kb.as<double>(), B.kval.as<double>(), c->stream));
    }
    FS_HIP(c, hipEventRecord(t2, c->stream));
    int st = 0;
    FS_HIP(c, hipMemcpyAsync(&st, m->status.p, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    FS_HIP(c, hipStreamSynchronize(c->stream));
    float ms_elem = 0.f, ms_all = 0.f;
    FS_HIP(c, hipEventElapsedTime(&ms_elem, t0, t1));
    FS_HIP(c, hipEventElapsedTime(&ms_all, t0, t2));
    (void)hipEventDestroy(t0);
    (void)hipEventDestroy(t1);
    (void)hipEventDestroy(t2);
    if ((s = finish_elements(m, ep, st))) return s;
    m->last_ep.ebegin = 0;
    m->last_ep.eend = (int32_t)E;
    m->timing[0] = ms_elem;
    m->timing[1] = ms_all - ms_elem;
    m->timing[2] = ms_all;
    B.k_ready = true;
    if (nzval_out) return d2h(c, nzval_out, B.kval.p, (size_t)B.nnz * 8);
    return FS_OK;
}

int fs_model_mass(fs_model *m, const fs_mass_params *p, int block, double *diag_out) {
    if (!m || !p) return FS_ERR_ARG;
    fs_ctx *c = m->ctx;
    c->err.clear();
    if (block != FS_BLOCK_ALL && block != FS_BLOCK_FF) return fail(c, FS_ERR_ARG, "unknown block %d", block);
    FS_HIP(c, hipSetDevice(c->device));
    int s = build_block(m, block);
    if (s) return s;
    Block &B = m->blk[block];
    const double *ginert = nullptr;
    const int32_t *ggrp = nullptr;
    const double *grt = nullptr;
    if (!p->composite) {
        const bool grouped = p->group_rho_t != nullptr;
        const int ng = grouped ? p->ngroups : 1;
        if (grouped && ng < 1) return fail(c, FS_ERR_ARG, "mass: group_rho_t needs ngroups >= 1");
        std::vector<double> rt(2 * (size_t)ng);
        for (int g = 0; g < ng; ++g) {
            rt[2 * g] = grouped ? p->group_rho_t[2 * g] : p->rho;
            rt[2 * g + 1] = grouped ? p->group_rho_t[2 * g + 1] : p->thickness;
        }
        if ((s = upload(c, m->g_rho_t, rt.data(), rt.size()))) return s;
        grt = m->g_rho_t.as<double>();
        if (grouped && p->elem_group) {
            for (int64_t e = 0; e < m->E; ++e)
                if (p->elem_group[e] < 0 || p->elem_group[e] >= ng)
                    return fail(c, FS_ERR_ARG, "mass: element %lld has group %d", (long long)e, p->elem_group[e]);
            if ((s = upload(c, m->m_group, p->elem_group, (size_t)m->E))) return s;
            ggrp = m->m_group.as<int32_t>();
        }
    } else {
        if (p->ngroups < 1 || !p->group_inertia) return fail(c, FS_ERR_ARG, "mass: layered shell needs group inertia");
        if ((s = upload(c, m->g_inertia, p->group_inertia, (size_t)2 * p->ngroups))) return s;
        ginert = m->g_inertia.as<double>();
        if (p->elem_group) {
            for (int64_t e = 0; e < m->E; ++e)
                if (p->elem_group[e] < 0 || p->elem_group[e] >= p->ngroups)
                    return fail(c, FS_ERR_ARG, "mass: element %lld has group %d", (long long)e, p->elem_group[e]);
            if ((s = upload(c, m->m_group, p->elem_group, (size_t)m->E))) return s;
            ggrp = m->m_group.as<int32_t>();
        }
    }
    FS_HIP(c, fs::launch_mass(m->nen, m->N, (int)m->E, p->composite ? 1 : 0, grt, ginert, ggrp,
                              m->x.as<double>(), m->y.as<double>(), m->z.as<double>(), m->dconn.as<int32_t>(),
                              m->dne_ptr.as<int32_t>(), m->dne_list.as<int32_t>(), m->node_dof.as<int64_t>(),
                              B.nrows, B.mdiag.as<double>(), c->stream));
    if (diag_out)
        FS_HIP(c, hipMemcpyAsync(diag_out, B.mdiag.p, (size_t)B.nrows * 8, hipMemcpyDeviceToHost, c->stream));
    FS_HIP(c, hipStreamSynchronize(c->stream));
    B.m_ready = true;
    return FS_OK;
}

int fs_model_resultants(fs_model *m, const fs_shell_params *p, const double *u, int64_t nlist,
                        const int32_t *felist, int32_t ocs_kind, const double *ocs, int32_t flags, double *out,
                        int32_t *mismatch) {
    if (!m) return FS_ERR_ARG;
    fs_ctx *c = m->ctx;
    c->err.clear();
    if (!p || !u || !out || nlist < 0) return fail(c, FS_ERR_ARG, "resultants: bad arguments");
    if (!m->normals_ready) return fail(c, FS_ERR_STATE, "resultants: normals not computed (associategeometry!)");
    if (ocs_kind < FS_OCSYS_ISOPARAMETRIC || ocs_kind > FS_OCSYS_PER_POINT || (ocs_kind != 0 && !ocs))
        return fail(c, FS_ERR_ARG, "resultants: output csys kind %d", ocs_kind);
    if (flags & ~FS_RES_LAYERED_Q4_SINGLE_T) return fail(c, FS_ERR_ARG, "resultants: unknown flags %d", flags);
    if (nlist > (int64_t)INT32_MAX / 4) return fail(c, FS_ERR_UNSUPPORTED, "resultants: %lld elements", (long long)nlist);
    const int npts = m->nen == 3 ? 1 : 4;
    if (felist)
        for (int64_t l = 0; l < nlist; ++l)
            if (felist[l] < 0 || felist[l] >= m->E)
                return fail(c, FS_ERR_ARG, "resultants: element %d out of range", felist[l]);
    if (!felist && nlist > m->E) return fail(c, FS_ERR_ARG, "resultants: nlist exceeds the element count");
    FS_HIP(c, hipSetDevice(c->device));
    fs::ResParams rp{};
    rp.nlist = (int32_t)nlist;
    rp.nelem = (int32_t)m->E;
    rp.ocs_kind = ocs_kind;
    rp.twice = (p->composite && m->nen == 4 && !(flags & FS_RES_LAYERED_Q4_SINGLE_T)) ? 1 : 0;
    rp.stab_c = p->stab_c;
    int s = 0;
    DevBuf dmat, dgrp, du, dlist, docs, dout, dst;
    std::vector<double> rec;
    int ng = 1;
    const int32_t *egroup = nullptr;
    if (!p->composite) {
        // per group: Dps (row-major), 5/6 Dt, thickness, stab_c
        const bool grouped = p->group_homog != nullptr;
        ng = grouped ? p->ngroups : 1;
        if (ng < 1) return fail(c, FS_ERR_ARG, "resultants: group_homog needs ngroups >= 1");
        rec.assign(16 * (size_t)ng, 0.0);
        for (int g = 0; g < ng; ++g) {
            const double *src = grouped ? p->group_homog + 16 * g : nullptr;
            double *r = &rec[16 * g];
            cm2rm(3, grouped ? src : p->Dps, r);
            cm2rm(2, grouped ? src + 9 : p->Dt, r + 9);
            for (int i = 0; i < 4; ++i) r[9 + i] *= 5.0 / 6.0;  // FEMMShellT3FFModule.jl:875-876, Q4RS :1091-1092
            r[13] = grouped ? src[13] : p->thickness;
            r[14] = grouped ? src[14] : p->stab_c;
            if (!(r[13] > 0.0)) return fail(c, FS_ERR_ARG, "resultants: thickness of group %d must be positive", g);
        }
        if (grouped) egroup = p->elem_group;
    } else {
        ng = p->ngroups;
        if (ng < 1 || !p->group_ABDH || !p->group_csys || !p->group_thickness)
            return fail(c, FS_ERR_ARG, "resultants: layered shell needs ngroups >= 1 and group arrays");
        rec.assign(41 * (size_t)ng, 0.0);
        for (int g = 0; g < ng; ++g) {
            const double *src = p->group_ABDH + 31 * g;
            double *r = &rec[41 * g];
            cm2rm(3, src, r);
            cm2rm(3, src + 9, r + 9);
            cm2rm(3, src + 18, r + 18);
            cm2rm(2, src + 27, r + 27);
            cm2rm(3, p->group_csys + 9 * g, r + 31);
            r[40] = p->group_thickness[g];
        }
        egroup = p->elem_group;
    }
    if (egroup) {
        for (int64_t e = 0; e < m->E; ++e)
            if (egroup[e] < 0 || egroup[e] >= ng)
                return fail(c, FS_ERR_ARG, "resultants: element %lld has group %d", (long long)e, egroup[e]);
        if ((s = upload(c, dgrp, egroup, (size_t)m->E))) return s;
        rp.elem_group = dgrp.as<int32_t>();
    }
    if ((s = upload(c, dmat, rec.data(), rec.size()))) return s;
    rp.g_mat = dmat.as<double>();
    if ((s = upload(c, du, u, (size_t)m->N * 6))) return s;
    rp.u = du.as<double>();
    if (felist) {
        if ((s = upload(c, dlist, felist, (size_t)nlist))) return s;
        rp.felist = dlist.as<int32_t>();
    }
    if (ocs_kind != FS_OCSYS_ISOPARAMETRIC) {
        const size_t nm = ocs_kind == FS_OCSYS_MATRIX ? 1 : (size_t)nlist * npts;
        std::vector<double> rm(9 * nm);
        for (size_t k = 0; k < nm; ++k) cm2rm(3, ocs + 9 * k, &rm[9 * k]);
        if ((s = upload(c, docs, rm.data(), rm.size()))) return s;
        rp.ocs = docs.as<double>();
    }
    if ((s = dalloc(c, dout, (size_t)nlist * npts * 8 * sizeof(double)))) return s;
    if ((s = dalloc(c, dst, 2 * sizeof(int)))) return s;
    rp.out = dout.as<double>();
    rp.status = dst.as<int>();
    FS_HIP(c, hipMemsetAsync(dst.p, 0, 2 * sizeof(int), c->stream));
    hipEvent_t e0, e1;
    FS_HIP(c, hipEventCreate(&e0));
    FS_HIP(c, hipEventCreate(&e1));
    FS_HIP(c, hipEventRecord(e0, c->stream));
    FS_HIP(c, fs::launch_resultants(m->nen, p->composite ? 1 : 0, rp, m->x.as<double>(), m->y.as<double>(),
                                    m->z.as<double>(), m->dconn.as<int32_t>(), m->nx.as<double>(),
                                    m->ny.as<double>(), m->nz.as<double>(), m->valid.as<uint8_t>(), c->stream));
    FS_HIP(c, hipEventRecord(e1, c->stream));
    int st[2] = {0, 0};
    FS_HIP(c, hipMemcpyAsync(st, dst.p, sizeof st, hipMemcpyDeviceToHost, c->stream));
    FS_HIP(c, hipMemcpyAsync(out, dout.p, (size_t)nlist * npts * 8 * sizeof(double), hipMemcpyDeviceToHost,
                             c->stream));
    FS_HIP(c, hipStreamSynchronize(c->stream));
    float ms = 0.f;
    FS_HIP(c, hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    m->timing[5] = ms;
    if (st[0]) return fail(c, FS_ERR_NUMERIC, "resultants: singular metric matrix in _gradN_e!");
    if (mismatch) *mismatch = st[1] ? 1 : 0;
    return FS_OK;
}

int fs_model_explicit(fs_model *m, const fs_cd_params *p, const double *U0, const double *V0, const double *Fmag,
                      const double *g, const int64_t *probe_dofs, int32_t nprobes, double *probe_out, double *U_out,
                      double *V_out) {
    if (!m || !p) return FS_ERR_ARG;
    fs_ctx *c = m->ctx;
    c->err.clear();
    Block &B = m->blk[FS_BLOCK_FF];
    if (!B.k_ready || !B.m_ready)
        return fail(c, FS_ERR_STATE, "explicit: FF-block stiffness and mass must be computed first");
    if (p->precision != FS_PREC_FP64 && p->precision != FS_PREC_MIXED && p->precision != FS_PREC_MIXED_F32)
        return fail(c, FS_ERR_UNSUPPORTED, "explicit: precision %d", p->precision);
    const bool mixed = p->precision != FS_PREC_FP64;
    const bool batch = p->ngroups > 0;
    if (!U0 || !V0 || !Fmag || !g || p->nsteps < 0 || (!batch && !(p->dt > 0.0)))
        return fail(c, FS_ERR_ARG, "explicit: bad arguments");
    if (batch && (!p->row_group || !p->group_dt || !p->group_cdamp))
        return fail(c, FS_ERR_ARG, "explicit: a batch needs row_group, group_dt and group_cdamp");
    const int stride = p->probe_stride > 0 ? p->probe_stride : 1;
    if (nprobes < 0 || (nprobes > 0 && (!probe_dofs || !probe_out))) return fail(c, FS_ERR_ARG, "explicit: probes");
    const int64_t n = B.nrows;
    for (int k = 0; k < nprobes; ++k)
        if (probe_dofs[k] < 0 || probe_dofs[k] >= n) return fail(c, FS_ERR_ARG, "explicit: probe dof out of range");
    const int ng = batch ? p->ngroups : 1;
    if (batch) {
        for (int64_t i = 0; i < n; ++i)
            if (p->row_group[i] < 0 || p->row_group[i] >= ng) return fail(c, FS_ERR_ARG, "explicit: row_group");
        for (int gi = 0; gi < ng; ++gi)
            if (!(p->group_dt[gi] > 0.0)) return fail(c, FS_ERR_ARG, "explicit: group_dt must be positive");
    }
    FS_HIP(c, hipSetDevice(c->device));
    int s;
    double build_ms = 0.0;
    if (mixed) {
        if (m->N > (int64_t)INT32_MAX / 6) return fail(c, FS_ERR_UNSUPPORTED, "explicit: model too large for mixed");
        const bool shear_fp32 = p->precision == FS_PREC_MIXED_F32;
        if (!m->mixed.built || m->mixed.kgen != m->kgen || m->mixed.shear_fp32 != shear_fp32) {
            if ((s = build_mixed(m, shear_fp32))) return s;
            build_ms = m->mixed.build_ms;
        }
    }
    // Loops of PATCH_MIN_STEPS steps or more run on the patch form of K, FP64
    // loops unless the row products were chosen (fs_ctx_set_cd_lanes); a rule
    // on the call's step count alone, so that a model takes the same form
    // alone and in a batch.
    PatchStore &P = B.patch;
    bool patch = (mixed || (c->cd_lanes == 8 && c->cd_pj == 0)) && p->nsteps >= PATCH_MIN_STEPS;
    if (patch && (s = prepare_patches(m, p->precision, &patch))) return s;
    const fs::PatchOp pop = patchop_of(P);
    // in one launch where the mesh is small enough and there is room
    bool loop = false;
    if (patch && p->nsteps < INT32_MAX && (s = patch_loops(m, p->precision, &loop))) return s;
    bool loop_form = loop;
    LoopPlaces places;
    if (loop) loop = places.take(c->device, P.largest_set);
    // State vectors: the free dofs themselves (row products), node-major dof
    // positions 6 i + c (mixed path), or the patches' slot positions; fixed
    // dofs stay zero in the last two.
    bool placed = false;
    int64_t nv = 0;
    const int64_t *map = nullptr;  // dof at each position
    auto lay_out = [&] {
        placed = mixed || patch;
        nv = patch ? P.npatch * fs::PATCH_WG : mixed ? 6 * m->N : n;
        map = patch ? P.map.as<int64_t>() : mixed ? m->node_dof.as<int64_t>() : nullptr;
    };
    lay_out();
    bool damped = false;
    for (int gi = 0; gi < ng; ++gi) damped |= (batch ? p->group_cdamp[gi] : p->cdamp) != 0.0;
    StepCache &sc = m->step;
    DevBuf(&dU)[2] = sc.dU;
    DevBuf &dV = sc.dV, &dA = sc.dA, &dF = sc.dF, &dInv = sc.dInv, &dC = sc.dC, &dSlot = sc.dSlot,
           &dProbe = sc.dProbe, &dRG = sc.dRG, &dGdt = sc.dGdt, &dG = sc.dG;
    const int64_t nrec = p->nsteps / stride + 1;
    // the caller's vectors into the state buffers; placed positions are filled
    // on the device from the free-dof order (through dA, which is free until
    // the loop starts)
    auto set_up = [&]() -> int {
        int e;
        for (DevBuf *b : {&dU[0], &dU[1], &dV, &dA, &dF, &dInv, &dC})
            if ((e = ensure(c, *b, std::max(nv, n) * 8))) return e;
        const struct {
            const double *src;
            double *dst;
        } vec[3] = {{U0, dU[0].as<double>()}, {V0, dV.as<double>()}, {Fmag, dF.as<double>()}};
        for (const auto &v : vec) {
            FS_HIP(c, hipMemcpyAsync(placed ? dA.as<double>() : v.dst, v.src, n * 8, hipMemcpyHostToDevice, c->stream));
            if (placed) FS_HIP(c, fs::launch_cd_place(nv, n, map, dA.as<double>(), v.dst, c->stream));
        }
        if (batch) {
            if ((e = ensure(c, dRG, nv * 4)) || (e = put(c, dGdt, p->group_dt, ng)) ||
                (e = put(c, sc.dGcd, p->group_cdamp, ng)) || (e = put(c, dG, g, (size_t)(p->nsteps + 1) * ng)))
                return e;
            FS_HIP(c, hipMemcpyAsync(placed ? dA.p : dRG.p, p->row_group, n * 4, hipMemcpyHostToDevice, c->stream));
            if (placed)
                FS_HIP(c, fs::launch_cd_place(nv, n, map, dA.as<int32_t>(), dRG.as<int32_t>(), 0, c->stream));
        }
        FS_HIP(c, fs::launch_cd_mass(nv, n, map, B.mdiag.as<double>(), p->dt_mass > 0.0 ? p->dt_mass : p->dt, p->cdamp,
                                     batch ? dRG.as<int32_t>() : nullptr, dGdt.as<double>(), sc.dGcd.as<double>(),
                                     dC.as<double>(), dInv.as<double>(), c->stream));
        if (nprobes > 0) {
            if ((e = ensure(c, dSlot, nv * 4)) || (e = put(c, sc.dPlist, probe_dofs, nprobes)) ||
                (e = ensure(c, dProbe, (size_t)nrec * nprobes * 8)))
                return e;
            int32_t *probe = placed ? dA.as<int32_t>() : dSlot.as<int32_t>();
            FS_HIP(c, fs::launch_cd_probe(n, nprobes, sc.dPlist.as<int64_t>(), probe, c->stream));
            if (placed) FS_HIP(c, fs::launch_cd_place(nv, n, map, probe, dSlot.as<int32_t>(), -1, c->stream));
            for (int k = 0; k < nprobes; ++k) probe_out[k] = U0[probe_dofs[k]];  // peek(0, U0)
        }
        return FS_OK;
    };
    // steps whose load factor is zero for every model skip the Fmag read
    std::vector<uint8_t> forced(p->nsteps + 1, 0);
    for (int64_t step = 0; step <= p->nsteps; ++step)
        for (int gi = 0; gi < ng && !forced[step]; ++gi) forced[step] = g[step * ng + gi] != 0.0;
    s = set_up();
    if (s == FS_ERR_NOMEM && patch) {
        // no memory for the slots of the patches (up to twice the dofs): the other
        // forms, for this block
        sc.drop_graph();
        sc.release();
        P.reset();
        P.planned = true;
        patch = loop = loop_form = false;
        lay_out();
        c->err.clear();
        s = set_up();
    }
    if (s == FS_OK && loop &&
        ((s = ensure(c, sc.dPub, nv * 32)) || (s = put(c, sc.dForced, forced.data(), forced.size())) ||
         (!batch && (s = put(c, dG, g, (size_t)p->nsteps + 1)))) &&
        s == FS_ERR_NOMEM) {
        loop = false;  // step by step
        c->err.clear();
        s = FS_OK;
    }
    if (s) {
        sc.drop_graph();
        return s;
    }
    // rows of the shell stencils hold 7 (T3) to 9 (Q4) neighbour runs: 4 lanes
    // per row, up to three runs per lane loaded together (measured fastest
    // of 2, 4, 8 and 16 lanes per row on both families)
    const int tpr = 4;
    const int cd_pj = node_pj(c, B);
    const int32_t *rg = batch ? dRG.as<int32_t>() : nullptr;
    const double *gdt = batch ? dGdt.as<double>() : nullptr;
    const fs::MixedOp op = mixed ? mixed_op(m) : fs::MixedOp{};
    auto enqueue = [&](hipStream_t st) -> hipError_t {
        hipError_t e = patch ? fs::launch_patch_init(pop, p->dt, batch ? 0.0 : g[0], dInv.as<double>(), dF.as<double>(),
                                                     dU[0].as<double>(), dV.as<double>(), dU[1].as<double>(), rg, gdt,
                                                     batch ? dG.as<double>() : nullptr,
                                                     loop ? sc.dPub.as<unsigned long long>() : nullptr, st)
                             : fs::launch_cd_init(nv, p->dt, batch ? 0.0 : g[0], dInv.as<double>(), dF.as<double>(),
                                          dU[0].as<double>(), dV.as<double>(), dA.as<double>(), dU[1].as<double>(),
                                          rg, gdt, batch ? dG.as<double>() : nullptr, st);
        if (e != hipSuccess) return e;
        if (loop) {
            fs::PatchLoop lp{};
            lp.op = pop;
            lp.U1 = dU[1].as<double>();
            lp.U = dU[p->nsteps % 2].as<double>();
            lp.W = dV.as<double>();
            lp.invMC = dInv.as<double>();
            lp.Cd = dC.as<double>();
            lp.Fmag = dF.as<double>();
            lp.gtab = dG.as<double>();
            lp.forced = sc.dForced.as<uint8_t>();
            lp.row_group = rg;
            lp.group_dt = gdt;
            lp.probe_slot = nprobes > 0 ? dSlot.as<int32_t>() : nullptr;
            lp.probe_dst = dProbe.as<double>();
            lp.pub = sc.dPub.as<unsigned long long>();
            lp.stop = c->loop_stop;
            lp.dt = p->dt;
            lp.nsteps = (int32_t)p->nsteps;
            lp.ng = ng;
            lp.damped = damped ? 1 : 0;
            lp.stride = stride;
            lp.nprobes = nprobes;
            lp.polls = c->loop_polls > 0 ? (uint32_t)std::min<int64_t>(c->loop_polls, LOOP_POLLS) : LOOP_POLLS;
            for (size_t k = 0; k + 1 < P.sets.size() && e == hipSuccess; ++k) {
                lp.first = P.sets[k];
                lp.count = P.sets[k + 1] - P.sets[k];
                e = fs::launch_cd_patch_loop(lp, p->precision == FS_PREC_MIXED_F32, st);
            }
            return e;
        }
        int cur = 1;
        for (int64_t step = 1; step <= p->nsteps; ++step) {
            const bool rec = nprobes > 0 && (step % stride == 0);
            int32_t *slot = rec ? dSlot.as<int32_t>() : nullptr;
            double *pdst = rec ? dProbe.as<double>() + (step / stride) * nprobes : nullptr;
            const double *gt = batch ? dG.as<double>() + step * ng : nullptr;
            if (patch)
                e = fs::launch_cd_patch_step(pop, p->precision == FS_PREC_MIXED_F32, dU[cur].as<double>(),
                                             dU[1 - cur].as<double>(), dV.as<double>(), dInv.as<double>(),
                                             dC.as<double>(), dF.as<double>(), batch ? 0.0 : g[step], p->dt,
                                             damped ? 1 : 0, forced[step] ? 1 : 0, step == p->nsteps ? 1 : 0, slot, pdst,
                                             rg, gdt, gt, st);
            else if (mixed)
                e = fs::launch_cd_mixed_step(m->nen, m->mixed.nsr, op, dU[cur].as<double>(),
                                             dU[1 - cur].as<double>(), dV.as<double>(), dA.as<double>(),
                                             dInv.as<double>(), dC.as<double>(), dF.as<double>(),
                                             batch ? 0.0 : g[step], p->dt, damped ? 1 : 0, forced[step] ? 1 : 0,
                                             slot, pdst, rg, gdt, gt, st);
            else if (c->cd_lanes > 0)
                e = fs::launch_cd_node_step(c->cd_lanes, cd_pj, noderows_of(B), B.slotrec.as<int2>(), B.kval.as<double>(),
                                            dU[cur].as<double>(), dU[1 - cur].as<double>(), dV.as<double>(),
                                            dA.as<double>(), dInv.as<double>(), dC.as<double>(), dF.as<double>(),
                                            batch ? 0.0 : g[step], p->dt, damped ? 1 : 0, slot, pdst, rg, gdt, gt, st);
            else
                e = fs::launch_cd_step(tpr, runrows_of(B), B.kval.as<double>(), dU[cur].as<double>(), dU[1 - cur].as<double>(),
                                       dV.as<double>(), dA.as<double>(), dInv.as<double>(), dC.as<double>(),
                                       dF.as<double>(), batch ? 0.0 : g[step], p->dt, damped ? 1 : 0, slot, pdst, rg,
                                       gdt, gt, st);
            if (e != hipSuccess) return e;
            cur = 1 - cur;
        }
        return hipSuccess;
    };
    hipEvent_t e0, e1;
    FS_HIP(c, hipEventCreate(&e0));
    FS_HIP(c, hipEventCreate(&e1));
    m->timing[6] = 0.0;
    if (loop) __atomic_store_n(c->loop_stop, 0, __ATOMIC_SEQ_CST);
    // a small mesh without room for its loop now runs step by step, beside a
    // graph that it may have of the loop
    if (p->use_graph && loop == loop_form) {
        // everything the captured launches take as arguments
        std::vector<uint64_t> key;
        key.reserve(64 + (size_t)p->nsteps + 1);
        for (const int64_t v : {nv, n, (int64_t)p->nsteps, (int64_t)p->precision, (int64_t)stride, (int64_t)nprobes,
                                (int64_t)ng, (int64_t)batch, (int64_t)damped, (int64_t)c->cd_lanes, (int64_t)cd_pj,
                                (int64_t)tpr, (int64_t)m->nen, (int64_t)m->mixed.nsr, (int64_t)patch, (int64_t)loop, c->loop_polls})
            key_add(key, v);
        key_add(key, p->dt);
        for (const DevBuf *b : {&dU[0], &dU[1], &dV, &dA, &dF, &dInv, &dC, &dSlot, &dProbe, &dRG, &dGdt, &dG})
            key_add(key, b->p);
        key_add(key, B.kval.p);
        key_add(key, B.slotrec.p);
        key_add(key, sc.dPub.p);
        key_add(key, sc.dForced.p);
        if (loop)  // the bounds of its launches
            for (const int32_t b : P.sets) key_add(key, b);
        if (patch) key_add(key, pop);
        else if (mixed) key_add(key, op);
        else if (c->cd_lanes > 0) key_add(key, noderows_of(B));
        else key_add(key, runrows_of(B));
        for (int64_t step = 0; step <= p->nsteps; ++step) {
            key.push_back(forced[step]);
            if (!batch) key_add(key, g[step]);
        }
        if (!sc.exec || key != sc.key) {
            const auto tc0 = std::chrono::steady_clock::now();
            sc.drop_graph();
            FS_HIP(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
            hipError_t ce = enqueue(c->stream);
            hipError_t ee = hipStreamEndCapture(c->stream, &sc.graph);
            if (ce != hipSuccess || ee != hipSuccess) {
                sc.drop_graph();
                return fail(c, FS_ERR_DEVICE, "explicit: graph capture failed: %s",
                            hipGetErrorString(ce != hipSuccess ? ce : ee));
            }
            hipError_t ie = hipGraphInstantiate(&sc.exec, sc.graph, nullptr, nullptr, 0);
            if (ie != hipSuccess) {
                sc.exec = nullptr;
                sc.drop_graph();
                return fail(c, FS_ERR_DEVICE, "explicit: graph instantiation failed: %s", hipGetErrorString(ie));
            }
            sc.key.swap(key);
            m->timing[6] = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - tc0).count();
        } else {
            ++sc.replays;
        }
        FS_HIP(c, hipEventRecord(e0, c->stream));
        FS_HIP(c, hipGraphLaunch(sc.exec, c->stream));
        FS_HIP(c, hipEventRecord(e1, c->stream));
        FS_HIP(c, hipStreamSynchronize(c->stream));
    } else {
        FS_HIP(c, hipEventRecord(e0, c->stream));
        FS_HIP(c, enqueue(c->stream));
        FS_HIP(c, hipEventRecord(e1, c->stream));
        FS_HIP(c, hipStreamSynchronize(c->stream));
    }
    bool restarted = false;
    if (loop && __atomic_load_n(c->loop_stop, __ATOMIC_SEQ_CST) != 0) {
        // a wait ran out: from the start again, step by step, and no such loop
        // on this context any more
        c->loop_gave_up = restarted = true;
        loop = false;
        if ((s = set_up())) {
            sc.drop_graph();
            return s;
        }
        FS_HIP(c, enqueue(c->stream));
        FS_HIP(c, hipEventRecord(e1, c->stream));
        FS_HIP(c, hipStreamSynchronize(c->stream));
    }
    m->cd_form = restarted ? FS_CD_RESTARTED : loop ? FS_CD_ONE_LAUNCH : patch ? FS_CD_PATCHES : FS_CD_ROWS;
    float ms = 0.f;
    FS_HIP(c, hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    m->timing[3] = ms;
    m->timing[4] = build_ms;
    // after the last step the buffer not indexed by the loop's final `cur` holds U_nsteps
    const int fin = (p->nsteps % 2 == 1) ? 1 : 0;
    const double *Ufin = dU[p->nsteps == 0 ? 0 : fin].as<double>();
    const struct {
        const double *src;
        double *out;
    } res[2] = {{Ufin, U_out}, {dV.as<double>(), V_out}};
    for (const auto &r : res) {
        if (!r.out) continue;
        if (placed) FS_HIP(c, fs::launch_cd_collect(nv, n, map, r.src, dA.as<double>(), c->stream));
        if ((s = d2h(c, r.out, placed ? dA.p : r.src, n * 8))) return s;
    }
    if (nprobes > 0 && nrec > 1 &&
        (s = d2h(c, probe_out + nprobes, dProbe.as<double>() + nprobes, (size_t)(nrec - 1) * nprobes * 8)))
        return s;
    return FS_OK;
}

}  // extern "C"

namespace {
// Power iteration of pwr (clamp_cyl_transient_examples.jl:45-60) on the
// resident FF-block K and M, from v (device, overwritten): w (n), sums (n +
// 64: the waves' partial norms), part (512) and ss (4) are device work arrays.
// The vectors are taken in turn as an iteration's start and end; the last one
// keeps its length, which the quotient does not see.
int power_iteration(fs_model *m, double *v, double *w, double *sums, double *part, double *ss, int32_t maxit,
                    double *omega_max) {
    fs_ctx *c = m->ctx;
    Block &B = m->blk[FS_BLOCK_FF];
    const int64_t n = B.nrows;
    const fs::RunRows rows = runrows_of(B);
    const fs::NodeRows nrw = noderows_of(B);
    const double *kv = B.kval.as<double>(), *md = B.mdiag.as<double>();
    const int pj = node_pj(c, B);
    // the step's form of the product (node-grouped unless the row form is set)
    for (int it = 0; it < maxit; ++it) {
        // the length is taken after even iterations, divided out in odd ones
        const double *scale = it % 2 ? ss : nullptr;
        double *norms = it % 2 ? nullptr : sums;
        FS_HIP(c, c->cd_lanes > 0 ? fs::launch_pwr_node(c->cd_lanes, pj, nrw, B.slotrec.as<int2>(), kv, v, w, md, scale,
                                                        norms, ss, c->stream)
                                  : fs::launch_pwr(rows, kv, v, w, md, scale, norms, ss, c->stream));
        std::swap(v, w);
    }
    FS_HIP(c, c->cd_lanes > 0
                  ? fs::launch_spmv_node(c->cd_lanes, pj, nrw, B.slotrec.as<int2>(), kv, v, w, c->stream)
                  : fs::launch_spmv(rows, kv, v, w, c->stream));
    FS_HIP(c, fs::launch_dot(n, w, v, nullptr, part, ss, c->stream));
    FS_HIP(c, fs::launch_dot(n, v, nullptr, md, part, ss + 1, c->stream));
    double h[2];
    FS_HIP(c, hipMemcpyAsync(h, ss, 16, hipMemcpyDeviceToHost, c->stream));
    FS_HIP(c, hipStreamSynchronize(c->stream));
    *omega_max = std::sqrt(h[0] / h[1]);
    return FS_OK;
}
}  // namespace

extern "C" {

int fs_model_omega_max(fs_model *m, const double *v0, int32_t maxit, double *omega_max) {
    if (!m || !v0 || !omega_max || maxit < 0) return FS_ERR_ARG;
    fs_ctx *c = m->ctx;
    c->err.clear();
    Block &B = m->blk[FS_BLOCK_FF];
    if (!B.k_ready || !B.m_ready) return fail(c, FS_ERR_STATE, "omega_max: FF-block K and M must be computed first");
    FS_HIP(c, hipSetDevice(c->device));
    const int64_t n = B.nrows;
    DevBuf dv, dw, dsums, dpart, dss;
    int s;
    if ((s = upload(c, dv, v0, n)) || (s = dalloc(c, dw, n * 8)) || (s = dalloc(c, dsums, (n + 64) * 8)) ||
        (s = dalloc(c, dpart, 512 * 8)) || (s = dalloc(c, dss, 4 * 8)))
        return s;
    return power_iteration(m, dv.as<double>(), dw.as<double>(), dsums.as<double>(), dpart.as<double>(),
                           dss.as<double>(), maxit, omega_max);
}

int fs_model_omega_max_noalloc(fs_model *m, const double *v0, int32_t maxit, double *omega_max) {
    if (!m || !v0 || !omega_max || maxit < 0) return FS_ERR_ARG;
    fs_ctx *c = m->ctx;
    c->err.clear();
    Block &B = m->blk[FS_BLOCK_FF];
    if (!B.k_ready || !B.m_ready) return fail(c, FS_ERR_STATE, "omega_max: FF-block K and M must be computed first");
    const int64_t n = B.nrows;
    if (n > fs::NOALLOC_MAX_ROWS)
        return fail(c, FS_ERR_UNSUPPORTED,
                    "omega_max without allocation: %lld free dofs exceed the workspace's %lld (use fs_model_omega_max)",
                    (long long)n, (long long)fs::NOALLOC_MAX_ROWS);
    if (!c->scratch)
        return fail(c, FS_ERR_DEVICE, "omega_max without allocation: no workspace on device %d (%s)", c->device,
                    hipGetErrorString(c->scratch_status));
    FS_HIP(c, hipSetDevice(c->device));
    double *v = c->scratch, *w = v + fs::NOALLOC_MAX_ROWS, *sums = w + fs::NOALLOC_MAX_ROWS;
    double *part = sums + fs::NOALLOC_MAX_ROWS, *ss = part + 512;
    if (n) FS_HIP(c, hipMemcpyAsync(v, v0, (size_t)n * 8, hipMemcpyHostToDevice, c->stream));
    return power_iteration(m, v, w, sums, part, ss, maxit, omega_max);
}

int fs_ctx_tuning(const fs_ctx *ctx, int nen, int formulation, int32_t *shape) {
    if (!ctx || !shape || (nen != FS_T3 && nen != FS_Q4) ||
        (formulation != FS_SHEAR_AVERAGE_B && formulation != FS_SHEAR_AVERAGE_K))
        return FS_ERR_ARG;
    const int v = ctx->elem_variant[nen == FS_Q4 ? 1 : 0][formulation];
    shape[0] = v;
    int ne = 0, wg = 0;
    if (v >= 0) fs::element_variant_shape(nen, v, &ne, &wg);
    shape[1] = v >= 0 ? ne : 0;
    shape[2] = v >= 0 ? wg : 0;
    return FS_OK;
}

int fs_ctx_set_tuning(fs_ctx *ctx, int nen, int formulation, int32_t variant) {
    if (!ctx || (nen != FS_T3 && nen != FS_Q4) ||
        (formulation != FS_SHEAR_AVERAGE_B && formulation != FS_SHEAR_AVERAGE_K) || variant < -2 ||
        variant >= fs::element_variants(nen))
        return FS_ERR_ARG;
    if (variant == -2) {
        ctx->autotune = false;
        ctx->elem_variant[nen == FS_Q4 ? 1 : 0][formulation] = -1;
        return FS_OK;
    }
    ctx->autotune = true;
    ctx->elem_variant[nen == FS_Q4 ? 1 : 0][formulation] = variant;
    return FS_OK;
}

int fs_ctx_set_pipeline(fs_ctx *ctx, int ranges) {
    if (!ctx || ranges < 1 || ranges > 64) return FS_ERR_ARG;
    ctx->asm_chunks = ranges;
    return FS_OK;
}

int fs_ctx_set_assembly(fs_ctx *ctx, int mode) {
    if (!ctx) return FS_ERR_ARG;
    if (mode != 0 && mode != 1) return fail(ctx, FS_ERR_ARG, "assembly mode %d", mode);
    ctx->assembly = mode;
    return FS_OK;
}

int fs_ctx_set_cd_lanes(fs_ctx *ctx, int lanes_per_node, int positions_per_lane) {
    if (!ctx) return FS_ERR_ARG;
    const int pj = positions_per_lane;
    const bool ok = lanes_per_node == 0 || (lanes_per_node == 8 && (pj == 0 || (pj >= 4 && pj <= 8))) ||
                    (lanes_per_node == 16 && (pj == 0 || (pj >= 2 && pj <= 4)));
    if (!ok) return fail(ctx, FS_ERR_ARG, "cd lanes: %d lanes per node with %d positions per lane", lanes_per_node, pj);
    ctx->cd_lanes = lanes_per_node;
    ctx->cd_pj = lanes_per_node ? pj : 0;
    return FS_OK;
}

int fs_ctx_set_cd_loop(fs_ctx *ctx, int64_t polls) {
    if (!ctx) return FS_ERR_ARG;
    ctx->loop_polls = polls;
    ctx->loop_gave_up = false;
    return FS_OK;
}

int fs_coo_create(fs_ctx *ctx, int64_t nrows, int64_t ncols, int32_t kr, int32_t kc, int64_t nmat,
                  const int64_t *dofnums_row, const int64_t *dofnums_col, int index_base, fs_coo **out) {
    if (!ctx || !out) return FS_ERR_ARG;
    *out = nullptr;
    ctx->err.clear();
    if (nrows < 0 || ncols < 0 || kr < 1 || kc < 1 || kr > 4096 || kc > 4096 || nmat < 0 ||
        (nmat > 0 && (!dofnums_row || !dofnums_col)))
        return fail(ctx, FS_ERR_ARG, "coo: bad sizes (nrows %lld, ncols %lld, k %d x %d, %lld matrices)",
                    (long long)nrows, (long long)ncols, kr, kc, (long long)nmat);
    const int64_t ke = (int64_t)kr * kc;
    for (int64_t i = 0; i < nmat * kr; ++i)
        if (dofnums_row[i] - index_base < 0) return fail(ctx, FS_ERR_ARG, "coo: row dof number below the index base");
    for (int64_t i = 0; i < nmat * kc; ++i)
        if (dofnums_col[i] - index_base < 0) return fail(ctx, FS_ERR_ARG, "coo: column dof number below the index base");
    FS_HIP(ctx, hipSetDevice(ctx->device));
    fs_coo *h = new (std::nothrow) fs_coo;
    if (!h) return fail(ctx, FS_ERR_NOMEM, "coo handle");
    h->ctx = ctx;
    h->nrows = nrows;
    h->ncols = ncols;
    h->nmat = nmat;
    h->kr = kr;
    h->kc = kc;
    // The COO stream of assemble! (element order; within an element
    // column-major: for j in columns, for i in rows) is bucketed by row by
    // threads that each own a row range and scan the stream in order, so a
    // row receives its entries in stream order.
    std::vector<int64_t> cnt(nrows + 1, 0);
    auto rowpass = [&](std::vector<int64_t> *fill, int64_t *bcol, int64_t *bpos) {
        const int64_t nt = std::max<int64_t>(1, std::min<int64_t>(fs::host_threads(), nrows / 4096 + 1));
        fs::run_shares(nt, [&](int64_t t) {
            const int64_t r0 = nrows * t / nt, r1 = nrows * (t + 1) / nt;
            for (int64_t m = 0; m < nmat; ++m) {
                const int64_t *dr = dofnums_row + m * kr, *dc = dofnums_col + m * kc;
                for (int j = 0; j < kc; ++j) {
                    const int64_t c = dc[j] - index_base;
                    if (c >= ncols) continue;
                    for (int i = 0; i < kr; ++i) {
                        const int64_t r = dr[i] - index_base;
                        if (r < r0 || r >= r1) continue;
                        if (!fill) {
                            cnt[r + 1]++;
                        } else {
                            const int64_t q = (*fill)[r]++;
                            bcol[q] = c;
                            bpos[q] = m * ke + (int64_t)j * kr + i;
                        }
                    }
                }
            }
        });
    };
    rowpass(nullptr, nullptr, nullptr);
    for (int64_t r = 0; r < nrows; ++r) cnt[r + 1] += cnt[r];
    const int64_t M = cnt[nrows];
    std::vector<int64_t> bcol(M), bpos(M), fill(cnt.begin(), cnt.end());
    rowpass(&fill, bcol.data(), bpos.data());
    // per row: a stable sort by column keeps stream order among duplicates;
    // each run of equal columns is one stored entry (zeros retained)
    std::vector<int64_t> rlen(nrows, 0), perm(M);
    fs::parallel_chunks(nrows, [&](int64_t r0, int64_t r1) {
        for (int64_t r = r0; r < r1; ++r) {
            const int64_t b = cnt[r], e = cnt[r + 1];
            for (int64_t q = b; q < e; ++q) perm[q] = q;
            std::stable_sort(perm.begin() + b, perm.begin() + e, [&](int64_t x, int64_t y) { return bcol[x] < bcol[y]; });
            int64_t u = 0;
            for (int64_t q = b; q < e; ++q)
                if (q == b || bcol[perm[q]] != bcol[perm[q - 1]]) ++u;
            rlen[r] = u;
        }
    }, 4096);
    h->rowptr.assign(nrows + 1, 0);
    for (int64_t r = 0; r < nrows; ++r) h->rowptr[r + 1] = h->rowptr[r] + rlen[r];
    const int64_t nnz = h->rowptr[nrows];
    h->nnz = nnz;
    h->colval.resize(nnz);
    std::vector<int64_t> cptr(nnz + 1), clist(M);
    fs::parallel_chunks(nrows, [&](int64_t r0, int64_t r1) {
        for (int64_t r = r0; r < r1; ++r) {
            int64_t s = h->rowptr[r] - 1;
            for (int64_t q = cnt[r]; q < cnt[r + 1]; ++q) {
                if (q == cnt[r] || bcol[perm[q]] != bcol[perm[q - 1]]) {
                    ++s;
                    h->colval[s] = bcol[perm[q]];
                    cptr[s] = q;
                }
                clist[q] = bpos[perm[q]];
            }
        }
    }, 4096);
    cptr[nnz] = M;
    int st;
    if ((st = upload(ctx, h->cptr, cptr.data(), cptr.size())) || (st = upload(ctx, h->clist, clist.data(), clist.size())) ||
        (st = dalloc(ctx, h->vals, (size_t)nnz * 8))) {
        delete h;
        return st;
    }
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) {
        delete h;
        return fail(ctx, FS_ERR_DEVICE, "coo: upload of the reduction plan failed");
    }
    ++ctx->refs;
    *out = h;
    return FS_OK;
}

int fs_coo_pattern(const fs_coo *h, int64_t *nnz) {
    if (!h || !nnz) return FS_ERR_ARG;
    *nnz = h->nnz;
    return FS_OK;
}

int fs_coo_pattern_get(const fs_coo *h, int64_t *rowptr, int64_t *colval, int index_base) {
    if (!h || !rowptr || !colval) return FS_ERR_ARG;
    for (int64_t r = 0; r <= h->nrows; ++r) rowptr[r] = h->rowptr[r] + index_base;
    fs::parallel_chunks(h->nnz, [&](int64_t a, int64_t b) {
        for (int64_t q = a; q < b; ++q) colval[q] = h->colval[q] + index_base;
    });
    return FS_OK;
}

int fs_coo_values(fs_coo *h, const double *elmats, double *nzval) {
    if (!h) return FS_ERR_ARG;
    fs_ctx *c = h->ctx;
    c->err.clear();
    const size_t nvals = (size_t)h->nmat * h->kr * h->kc;
    if (nvals > 0 && !elmats) return fail(c, FS_ERR_ARG, "coo: NULL element matrices");
    FS_HIP(c, hipSetDevice(c->device));
    int s;
    if ((s = upload(c, h->mats, elmats, nvals))) return s;
    FS_HIP(c, fs::launch_coo_reduce(h->nnz, h->cptr.as<int64_t>(), h->clist.as<int64_t>(), h->mats.as<double>(),
                                    h->vals.as<double>(), c->stream));
    if (nzval) return d2h(c, nzval, h->vals.p, (size_t)h->nnz * 8);
    FS_HIP(c, hipStreamSynchronize(c->stream));
    return FS_OK;
}

void fs_coo_destroy(fs_coo *h) {
    if (!h) return;
    fs_ctx *c = h->ctx;
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    delete h;
    ctx_release(c);
}

int fs_model_mixed_info(const fs_model *m, int64_t *info) {
    if (!m || !info) return FS_ERR_ARG;
    const MixedStore &X = m->mixed;
    info[0] = X.built ? X.kmb_pairs : 0;
    info[1] = X.built ? X.nsr : 0;
    info[2] = m->nnb;
    info[3] = X.built ? X.nslices : 0;
    return FS_OK;
}

int fs_model_cd_form(const fs_model *m, int32_t *form) {
    if (!m || !form) return FS_ERR_ARG;
    *form = m->cd_form;
    return FS_OK;
}

int fs_model_last_timing(const fs_model *m, int which, double *ms) {
    if (!m || !ms || which < 0 || which > 6) return FS_ERR_ARG;
    *ms = m->timing[which];
    return FS_OK;
}

}  // extern "C"
