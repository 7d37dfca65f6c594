// mplbhip.cpp -- context, HBM layout, launches and the C ABI of
// libmplbhip.so (include/mplbhip.h).
#include "../../include/mplbhip.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <array>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <unordered_map>
#include <vector>

#include "lattice_kernels.hpp"
#include "plan.hpp"

namespace mplbhip {
hipError_t launch_lattice(int dim, int storage, int mode, const KParams& kp,
                          hipStream_t s, int part = 0);
hipError_t launch_materialize_split(int dim, int storage, const KParams& kp, hipStream_t s);
bool pair_shape(int storage, int nt, int* positions);
hipError_t launch_pair(int lat, int storage, const KParams& kp, hipStream_t s);
bool march_shape(int storage, bool obst, int* steps);
hipError_t launch_march(int storage, const KParams& kp, hipStream_t s);
int tile_max_steps(int side);
void tile_wall_classes(int region, uint32_t* in, uint32_t* out, uint32_t* par);
hipError_t launch_tile(int storage, int side, const KParams& kp, hipStream_t s);
hipError_t launch_halo(const HaloParams& hp, hipStream_t s);
hipError_t launch_halo_multi(const HaloParams* links, const int32_t* wg_start, int nlinks,
                             int nwg, int Q, int elem_bytes, hipStream_t s);
hipError_t launch_reduce(const double* partials, const BlockParams* blocks,
                         int nblocks, int ntiles, int nbulk, int nbnd, int split, int fold,
                         double* out, hipStream_t s);
hipError_t launch_fill(void* p, int64_t bytes, hipStream_t s);
hipError_t launch_lift(int dim, const KParams& kp, int64_t nodes, hipStream_t s);
hipError_t launch_rest_macros(const KParams& kp, int b, int64_t nodes, hipStream_t s);
hipError_t launch_copy(const void* src, void* dst, int64_t bytes, hipStream_t s);
hipError_t launch_exchange(void* a, void* b, int64_t bytes, hipStream_t s);
hipError_t scratch_address(double** ptr);
bool swap_masks(const RegionProg* progs, uint32_t* mask);
hipError_t launch_swap_pull(const KParams& kp, int nbnd, bool collide, bool large, hipStream_t s);
hipError_t launch_swap(int part, const KParams& kp, int nbnd, hipStream_t s);
}  // namespace mplbhip

using namespace mplbhip;

namespace {

struct HaloLink {
    HaloParams hp;       // src/dst buffers filled per launch
    int from, to;
    uint8_t* d_flag = nullptr;
    uint32_t* d_sup = nullptr;  // merged launch: populations a later link writes
    bool merged = false;        // copied by the merged launch
};

struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
};

}  // namespace

// the tables of mplbhip_ctx::wg_block (boundary: kWgBnd + fold level)
enum WgTable : int { kWgAll = 0, kWgBulk = 1, kWgBulk3 = 2, kWgH2 = 3, kWgBnd = 4 };

struct mplbhip_ctx {
    int device = -1;
    int dim = 3;
    int lat = 3;  // lattice key of the kernels: 2 D2Q9, 3 D3Q19, 15 D3Q15
    int storage = MPLBHIP_STORE_F64;
    int Q = 19;
    // Collision_BGKThermal4th: per-node relaxation and the 4th-order
    // equilibrium at the Variable_T field temp (host layout, FP64)
    bool thermal = false;
    bool temp_set = false;
    Plan plan;
    double tau = 1.0, dt = 1.0;
    int force_type = 0, force_macros = 0;
    std::vector<std::array<double, 3>> accel;
    bool prepared = false;
    bool initialized = false;
    // Scheme_StreamCollision_Swap: one lattice f (fs[0]) updated in place;
    // swap_formed once f^0 is in it
    bool swap = false;
    bool swap_formed = false;
    // the case runs k_swap_pull, whose steps between a run's first collision
    // and its last stream leave the collided lattice in fs[cur]
    bool swap_pull = false, swap_run = false;
    DevBuf swap_mask;
    bool init_from_f = false;
    bool init_lift = false;  // f^0 = feq + first-order non-equilibrium part
    long long tstep = 0;
    int cur = 0;  // parity of the latest fStage of every active block; also
                  // selects the per-block parity array read by the next step
    std::vector<double> btau, bdt;  // per-block collision overrides (NaN: none)
    std::string err;

    // layout
    std::vector<BlockParams> bp;
    std::vector<int64_t> elem0;  // first element of each block's storage, and the end
    int64_t total_elems = 0;
    int64_t interior_nodes = 0;
    int ntiles = 0;            // whole-lattice tiles
    int nbulk = 0;             // bulk tiles of a step (z planes 1 .. n-2)
    int nbulk3 = 0;            // bulk tiles of a fold-3 step (every z plane)
    int nbnd_v[4] = {0, 0, 0, 0};  // boundary workgroups of a step, [fold]
    bool tuned = false;        // launch configuration chosen (autotune)
    bool fused = false;        // small case: one whole-lattice launch per step
    bool h2 = false;           // FP16: two-node-per-lane bulk kernel (fold level 0)
    bool h2_ok = false, h2_env = false;
    int nbulk2 = 0;            // its workgroups
    double restart_factor = 0.0;     // batched solver: restart a rising instance at rest
    std::vector<int> batch_restarts;  // per block, last iterate_batch
    std::vector<BlockParams> restart_bp;  // block parameters of a restart launch
    bool fused_env = false, fused_full = false;  // MPLBHIP_FUSED given; prepare's choice
    int64_t grid_nodes = 0;    // nodes of the blocks the step launches cover
    bool batch_compact = true;  // iterate_batch shrinks the launches to live blocks
    int fold = 1;              // simple regions the bulk kernel runs inline:
                               // 0 none, 1 x faces, 2 every one of the planes
                               // z = 1 .. n-2, 3 every one (3D: the bulk grid
                               // then spans every z plane)
    bool xcd_remap = false;    // bulk tiles dealt to XCDs in contiguous runs
    int xgroup = 0;            // 1: rows of bulk tiles dealt to one XCD each
    int xgroup_ok = 0;         // 1 when some block allows that grouping
    bool rowwg_ok = false;     // some block allows row workgroups (xgroup 2)
    // split steps: the boundary kernel on a side stream beside the bulk
    // kernel.  On by default for cases with halo links (three-block
    // L-channel: 39.3k -> 40.1k MLUPS) and wherever the boundary launch is
    // small (the eight cavity corners left at fold level 3: its launch then
    // hides behind the bulk kernel).  MPLBHIP_OVERLAP=0/1 overrides.
    bool overlap = false;
    bool overlap_env = false;
    hipStream_t side = nullptr;
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
    bool fold_env = false, xgroup_env = false;  // fixed by the environment
    // two steps per launch (k_pair): allowed by the case (1 forced, -1
    // forbidden by MPLBHIP_PAIR), in use over the blocks the launches cover,
    // each block's tiling, and the block of every workgroup
    bool pair_ok = false, pair = false;
    int pair_env = 0;
    std::vector<PairBlock> pb;
    std::vector<int32_t> wg_pair_host;
    int npair = 0, pair_nt = 0;
    DevBuf dpair, wg_pair;
    // several steps per launch of 2D blocks (k_march), likewise: steps of the
    // form, every wave's share
    bool march_ok = false, march = false;
    int march_steps = 0;
    std::vector<MarchWave> march_host;
    DevBuf dmarch;
    // several steps per launch of small 2D blocks (k_tile): the tiles, their
    // side, and whether the blocks are linked to themselves along x
    bool tile_ok = false, tile = false, wrap_x = false;
    int tile_side = 0, ntile2d = 0, tile_row = 0;
    std::vector<TileWG> tile_host;
    DevBuf dtile;
    bool halo_stale = false;  // the latest fStage's halos are not exchanged
    int singles = 0;  // single steps taken before their launch was tuned
    std::vector<BndSeg> segs;
    std::vector<std::vector<uint8_t>> solid;  // obstacle nodes per block (empty: none)
    std::vector<uint32_t> obst;               // link masks per interior node
    size_t es = 8;

    // device memory
    hipStream_t stream = nullptr;
    DevBuf fs[2], per[2], macro[4], macro_copy[4], progs, blocks, partials,
        red, fhost, parity[2], dsegs, dobst;
    // the block of every workgroup of each grid (KParams::wg_block_*):
    // tables kWgAll, kWgBulk, kWgBulk3, kWgH2, then the boundary grid at
    // fold levels 0-3, concatenated; offsets into wg_block_host
    DevBuf wg_block;
    std::vector<int32_t> wg_block_host;
    size_t wg_block_off[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    // the macros at PreDefinedInitialCondition: f^0 = feq of these, formed
    // at the first step (the collision needs the time step, which the Apps
    // set afterwards); a macro refresh at t = 0 must not change it
    DevBuf macro0[4];
    DevBuf temp;  // Variable_T of the thermal collision
    std::vector<HaloLink> halos;
    // the merged halo launch: its links' parameters for each ping-pong
    // target (into = 0, 1), their workgroup ranges; the other links follow
    // it one launch each, in order
    DevBuf halo_links[2], halo_wgstart;
    int halo_nmerged = 0, halo_nwg = 0;
    bool halo_merge = true;
    std::vector<HaloParams> halo_hps;  // the merged links, buffers not yet filled
    void* halo_fs[2] = {nullptr, nullptr};  // the fStage buffers halo_links point at
    std::vector<double> host_init_f;  // f given by mplbhip_set_f, per block
    std::vector<float> scale, inv_scale;
    hipEvent_t ev[2] = {nullptr, nullptr};
    // device address of this GPU's file-scope scratch array (the
    // allocation-free entry point), taken at create with the device current
    double* scratch = nullptr;
    hipGraph_t graph[2] = {nullptr, nullptr};
    hipGraphExec_t gexec[2] = {nullptr, nullptr};
    int graph_steps = 0;
    double last_ratio[4] = {0, 0, 0, 0};
    double last_bulk_ms = 0.0, last_bnd_ms = 0.0;  // last timed run
    double last_max = -1.0;
};

static int fail(mplbhip_ctx* c, int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (c) c->err = buf;
    return code;
}

#define HIPCHK(c, expr)                                                      \
    do {                                                                     \
        hipError_t e_ = (expr);                                              \
        if (e_ != hipSuccess)                                                \
            return fail((c), MPLBHIP_ERR_HIP, "%s failed: %s", #expr,        \
                        hipGetErrorString(e_));                              \
    } while (0)

static int need_device(mplbhip_ctx* c) {
    if (c->device < 0)
        return fail(c, MPLBHIP_ERR_NODEVICE,
                    "this context was created without a device (plan only)");
    return 0;
}

static int dalloc(mplbhip_ctx* c, DevBuf& b, size_t bytes) {
    if (b.p) {
        (void)hipFree(b.p);
        b.p = nullptr;
    }
    b.bytes = bytes;
    if (bytes == 0) return 0;
    HIPCHK(c, hipMalloc(&b.p, bytes));
    return 0;
}

static void dfree(DevBuf& b) {
    if (b.p) (void)hipFree(b.p);
    b.p = nullptr;
    b.bytes = 0;
}

static double kCSh() { return std::sqrt(3.0); }

// collision constants per block, computed in the reference's order
// (model_kernel.inc:428-429: omega = dt/(tau + 0.5*dt))
static void fill_collision(mplbhip_ctx* c) {
    for (size_t b = 0; b < c->bp.size(); b++) {
        const double tau = std::isnan(c->btau[b]) ? c->tau : c->btau[b];
        const double dt = std::isnan(c->bdt[b]) ? c->dt : c->bdt[b];
        const double omega = dt / (tau + 0.5 * dt);
        BlockParams& B = c->bp[b];
        B.dt = dt;
        B.tau = tau;
        B.omega = omega;
        B.one_minus_omega = 1 - omega;
        B.tau_omega = tau * omega;
        B.fomega = (float)omega;
        B.fone_minus_omega = (float)(1 - omega);
        B.fforce = (float)(tau * omega * kCSh());
        for (int d = 0; d < 3; d++) {
            B.g[d] = c->accel[b][d];
            // half-step shift of the lattice-unit velocity: (dt g/2)/CS
            B.fhalf_dtg[d] = (float)((dt * c->accel[b][d] / 2) / kCSh());
        }
    }
}

static int upload_blocks(mplbhip_ctx* c) {
    fill_collision(c);
    HIPCHK(c, hipMemcpyAsync(c->blocks.p, c->bp.data(),
                             c->bp.size() * sizeof(BlockParams),
                             hipMemcpyHostToDevice, c->stream));
    return 0;
}

static int assign_2d(mplbhip_ctx* c, bool only_active);

static void drop_graphs(mplbhip_ctx* c) {
    for (int i = 0; i < 2; i++) {
        if (c->gexec[i]) (void)hipGraphExecDestroy(c->gexec[i]);
        if (c->graph[i]) (void)hipGraphDestroy(c->graph[i]);
        c->gexec[i] = nullptr;
        c->graph[i] = nullptr;
    }
    c->graph_steps = 0;
}

// fold level of the step in force: the two-node FP16 kernel covers
// interior nodes only (level 0)
static int step_fold(const mplbhip_ctx* c) { return c->h2 ? 0 : c->fold; }
// bulk workgroups of the step in force
static int step_nbulk(const mplbhip_ctx* c) {
    return step_fold(c) == 3 ? c->nbulk3 : c->nbulk;
}

static KParams base_params(mplbhip_ctx* c) {
    KParams kp;
    std::memset(&kp, 0, sizeof kp);
    kp.blocks = static_cast<const BlockParams*>(c->blocks.p);
    kp.nblocks = (int)c->bp.size();
    kp.ntiles = c->ntiles;
    kp.nbulk = step_nbulk(c);
    const int fold = step_fold(c);
    kp.nbnd = c->nbnd_v[fold];
    kp.fold = fold;
    kp.h2 = c->h2 ? 1 : 0;
    kp.nbulk2 = c->nbulk2;
    kp.xcd_remap = c->xcd_remap ? 1 : 0;
    kp.xgroup = c->xgroup;
    kp.fused = c->fused ? 1 : 0;
    kp.segs = static_cast<const BndSeg*>(c->dsegs.p);
    kp.obst = c->obst.empty() ? nullptr : static_cast<const uint32_t*>(c->dobst.p);
    kp.progs = static_cast<const RegionProg*>(c->progs.p);
    for (int v = 0; v < 4; v++) {
        kp.macro[v] = static_cast<double*>(c->macro[v].p);
        kp.macro_copy[v] = static_cast<double*>(c->macro_copy[v].p);
        kp.macro0[v] = static_cast<const double*>(c->macro0[v].p);
    }
    kp.partials = static_cast<double*>(c->partials.p);
    for (int q = 0; q < kMaxQ; q++) {
        kp.scale[q] = q < c->Q ? c->scale[q] : 1.f;
        kp.inv_scale[q] = q < c->Q ? c->inv_scale[q] : 1.f;
    }
    kp.force_type = c->force_type;
    kp.force_macros = c->force_macros;
    kp.thermal = c->thermal ? 1 : 0;
    kp.temp = static_cast<const double*>(c->temp.p);
    for (int i = 0; i < 2; i++) {
        kp.fs_buf[i] = c->fs[i].p;
        kp.per_buf[i] = c->per[i].p;
    }
    kp.cur_in = static_cast<const int32_t*>(c->parity[c->cur].p);
    kp.cur_out = static_cast<int32_t*>(c->parity[1 - c->cur].p);
    const int32_t* wgb = static_cast<const int32_t*>(c->wg_block.p);
    if (wgb) {
        kp.wg_block_all = wgb + c->wg_block_off[kWgAll];
        kp.wg_block_bulk = wgb + c->wg_block_off[kWgBulk];
        kp.wg_block_bulk3 = wgb + c->wg_block_off[kWgBulk3];
        kp.wg_block_h2 = wgb + c->wg_block_off[kWgH2];
        kp.wg_block_bnd = wgb + c->wg_block_off[kWgBnd + fold];
    }
    kp.pair = static_cast<const PairBlock*>(c->dpair.p);
    kp.wg_block_pair = static_cast<const int32_t*>(c->wg_pair.p);
    kp.npair = c->npair;
    kp.pair_nt = c->pair_nt;
    kp.march = static_cast<const MarchWave*>(c->dmarch.p);
    kp.nmarch = (int)c->march_host.size();
    kp.tile = static_cast<const TileWG*>(c->dtile.p);
    kp.ntile2d = c->ntile2d;
    kp.tile_row = c->tile_row;
    kp.wrap_x = c->wrap_x ? 1 : 0;
    kp.swap_mask = static_cast<const uint32_t*>(c->swap_mask.p);
    return kp;
}

// fStage halo exchange into buffer `into` (ops_halo_transfer order); the
// links of frozen instances (iterate_batch) are left alone, so their
// buffers keep the state they converged with.  The swap scheme exchanges
// its one lattice f in place: a halo cell written later in the exchange is
// read as it is (last exchanged, then swapped), as in the reference.
static int exchange(mplbhip_ctx* c, int into) {
    bool all_active = true;
    for (const HaloLink& h : c->halos)
        all_active = all_active && c->bp[h.from].active && c->bp[h.to].active;
    const bool merged = c->halo_merge && c->halo_nmerged >= 2 && all_active &&
                        c->halo_fs[0] == c->fs[0].p && c->halo_fs[1] == c->fs[1].p &&
                        c->halo_links[0].p && c->halo_links[1].p;
    if (merged)
        HIPCHK(c, launch_halo_multi(static_cast<const HaloParams*>(c->halo_links[into].p),
                                    static_cast<const int32_t*>(c->halo_wgstart.p),
                                    c->halo_nmerged, c->halo_nwg, c->Q, (int)c->es, c->stream));
    for (HaloLink& h : c->halos) {
        if (merged && h.merged) continue;
        if (!c->bp[h.from].active || !c->bp[h.to].active) continue;
        HaloParams hp = h.hp;
        hp.src_cur = c->fs[into].p;
        hp.src_other = c->fs[c->swap ? into : 1 - into].p;
        hp.dst = c->fs[into].p;
        hp.other_flag = h.d_flag;
        HIPCHK(c, launch_halo(hp, c->stream));
    }
    return 0;
}

// the boundary kernel of this step runs on the side stream
static bool use_side(const mplbhip_ctx* c, const KParams& kp) {
    if (kp.fused || kp.nbulk <= 0 || kp.nbnd <= 0) return false;
    if (c->overlap_env) return c->overlap;
    return !c->halos.empty() || kp.nbnd <= 256;
}

// The step kernels of one step (no halo exchange).  The bulk and boundary
// kernels touch disjoint nodes and read only the previous fStage: with the
// side stream the boundary kernel runs beside the bulk kernel (a fork and
// join, also in a captured graph).  With ev (four events: bulk start/end on
// the context stream, boundary start/end on the stream it runs on) each
// kernel is bracketed for timing.
static int launch_step_kernels(mplbhip_ctx* c, const KParams& kp, int mode,
                               hipEvent_t* ev = nullptr) {
    if (!use_side(c, kp)) {
        if (!ev) {
            HIPCHK(c, launch_lattice(c->lat, c->storage, mode, kp, c->stream));
            return 0;
        }
        HIPCHK(c, hipEventRecord(ev[0], c->stream));
        HIPCHK(c, launch_lattice(c->lat, c->storage, mode, kp, c->stream, 1));
        HIPCHK(c, hipEventRecord(ev[1], c->stream));
        HIPCHK(c, hipEventRecord(ev[2], c->stream));
        HIPCHK(c, launch_lattice(c->lat, c->storage, mode, kp, c->stream, 2));
        HIPCHK(c, hipEventRecord(ev[3], c->stream));
        return 0;
    }
    HIPCHK(c, hipEventRecord(c->ev_fork, c->stream));
    HIPCHK(c, hipStreamWaitEvent(c->side, c->ev_fork, 0));
    if (ev) HIPCHK(c, hipEventRecord(ev[2], c->side));
    HIPCHK(c, launch_lattice(c->lat, c->storage, mode, kp, c->side, 2));
    if (ev) HIPCHK(c, hipEventRecord(ev[3], c->side));
    if (ev) HIPCHK(c, hipEventRecord(ev[0], c->stream));
    HIPCHK(c, launch_lattice(c->lat, c->storage, mode, kp, c->stream, 1));
    if (ev) HIPCHK(c, hipEventRecord(ev[1], c->stream));
    HIPCHK(c, hipEventRecord(c->ev_join, c->side));
    HIPCHK(c, hipStreamWaitEvent(c->stream, c->ev_join, 0));
    return 0;
}

// A run of the swap scheme's one-pass forms: the collision of f (fs[0]) into
// the buffer from which the run's passes end in fs[0] again, a pass of
// k_swap_pull per step, the last of which streams and applies the walls only.
static int swap_begin(mplbhip_ctx* c, int passes) {
    KParams kp = base_params(c);
    kp.swap_to = c->cur = passes & 1;
    HIPCHK(c, launch_swap(0, kp, 0, c->stream));
    c->swap_run = true;
    return 0;
}
static int swap_pass(mplbhip_ctx* c, bool collide) {
    KParams kp = base_params(c);
    kp.swap_to = 1 - c->cur;
    HIPCHK(c, launch_swap_pull(kp, c->nbnd_v[0], collide, c->fs[0].bytes > ((size_t)1 << 28),
                               c->stream));
    c->cur ^= 1;
    return 0;
}
static int swap_end(mplbhip_ctx* c) {
    c->swap_run = false;
    return swap_pass(c, false);
}

// SwapStreamCollision (evolution.cpp:195-252) on the one lattice f:
// collision and force, halo exchange of f, local swap, swap stream,
// boundaries; with check, the macros (and residual partials) of the result
static int enqueue_swap_step(mplbhip_ctx* c, bool check, bool residual) {
    KParams kp = base_params(c);
    if (c->swap_pull) {
        if (int rc = swap_begin(c, 1)) return rc;
        if (int rc = swap_end(c)) return rc;
        if (check) {
            kp.want_residual = residual ? 1 : 0;
            HIPCHK(c, launch_swap(5, kp, 0, c->stream));
        }
        return 0;
    }
    HIPCHK(c, launch_swap(0, kp, 0, c->stream));
    if (int rc = exchange(c, 0)) return rc;
    HIPCHK(c, launch_swap(1, kp, 0, c->stream));
    HIPCHK(c, launch_swap(2, kp, 0, c->stream));
    HIPCHK(c, launch_swap(3, kp, c->nbnd_v[0], c->stream));
    if (check) {
        kp.want_residual = residual ? 1 : 0;
        HIPCHK(c, launch_swap(5, kp, 0, c->stream));
    }
    return 0;
}

// the per-block sums of the step's partials: split (bulk + boundary slots)
// or one whole-lattice launch's tiles (small cases, the swap scheme)
static int reduce_split(const mplbhip_ctx* c) { return c->fused || c->swap ? 0 : 1; }

// the halo copies that a launch of several steps left out (k_tile wraps by
// itself), ahead of a kernel that reads them
static int fresh_halos(mplbhip_ctx* c) {
    if (c->halo_stale)
        if (int rc = exchange(c, c->cur)) return rc;
    c->halo_stale = false;
    return 0;
}

// one step from parity c->cur (step kernels, then the halo copies, which
// wait for both kernels); leaves c->cur flipped
static int enqueue_step(mplbhip_ctx* c, bool check, bool residual) {
    if (c->swap_run) return swap_pass(c, true);
    if (c->swap) return enqueue_swap_step(c, check, residual);
    if (int rc = fresh_halos(c)) return rc;
    KParams kp = base_params(c);
    kp.want_residual = residual ? 1 : 0;
    const int mode = check ? MODE_STEP_CHECK : MODE_STEP;
    if (int rc = launch_step_kernels(c, kp, mode)) return rc;
    if (int rc = exchange(c, 1 - c->cur)) return rc;
    c->cur ^= 1;
    return 0;
}

// steps per launch in force (1: single steps); a body force turns the forms
// without one off
static int launch_steps(const mplbhip_ctx* c) {
    if (c->swap || c->thermal) return 1;
    if (c->tile) return tile_max_steps(c->tile_side);
    if (c->force_type || c->force_macros) return 1;
    return c->pair ? 2 : c->march ? c->march_steps : 1;
}

// n steps in one launch from parity c->cur (launch_steps(c); k_tile also
// takes fewer); leaves c->cur flipped.  The other fStage buffer then holds
// the state n steps back, so a run whose result is measured by re-streaming
// ends with a single step.
static int enqueue_multi(mplbhip_ctx* c, int n) {
    KParams kp = base_params(c);
    kp.tile_steps = n;
    if (c->tile) HIPCHK(c, launch_tile(c->storage, c->tile_side, kp, c->stream));
    else if (c->pair) HIPCHK(c, launch_pair(c->lat, c->storage, kp, c->stream));
    else HIPCHK(c, launch_march(c->storage, kp, c->stream));
    c->halo_stale = !c->halos.empty();
    c->cur ^= 1;
    return 0;
}

static int build_graphs(mplbhip_ctx* c, int nsteps) {
    drop_graphs(c);
    for (int p = 0; p < 2; p++) {
        HIPCHK(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
        const int saved = c->cur;
        c->cur = p;
        int rc = 0;
        const int ls = launch_steps(c);
        for (int s = 0; s < nsteps && rc == 0; s += ls)
            rc = ls > 1 ? enqueue_multi(c, ls) : enqueue_step(c, false, false);
        c->cur = saved;
        hipGraph_t g = nullptr;
        hipError_t e = hipStreamEndCapture(c->stream, &g);
        if (rc) {
            if (g) (void)hipGraphDestroy(g);
            return rc;
        }
        if (e != hipSuccess)
            return fail(c, MPLBHIP_ERR_HIP, "graph capture failed: %s",
                        hipGetErrorString(e));
        c->graph[p] = g;
        HIPCHK(c, hipGraphInstantiate(&c->gexec[p], g, nullptr, nullptr, 0));
    }
    c->graph_steps = nsteps;
    return 0;
}

static int ensure_init(mplbhip_ctx* c) {
    if (!c->prepared) return fail(c, MPLBHIP_ERR_ARG, "call mplbhip_prepare first");
    if (!c->initialized)
        return fail(c, MPLBHIP_ERR_ARG,
                    "no initial condition: call mplbhip_init_feq or mplbhip_set_f");
    return 0;
}

// materialize the current f: macros always, optionally f in host layout
// (device buffer c->fhost) and the residual against MacroVarsCopy
static int swap_form(mplbhip_ctx* c);

static int materialize(mplbhip_ctx* c, bool want_f, bool residual,
                       std::vector<double>* acc_out) {
    if (int rc = ensure_init(c)) return rc;
    KParams kp = base_params(c);
    const size_t fbytes = (size_t)c->Q * c->interior_nodes * sizeof(double);
    if (c->swap) {
        // the one lattice holds f itself: measure it in place
        if (int rc = swap_form(c)) return rc;
        if (want_f && c->fhost.bytes != fbytes)
            if (int rc = dalloc(c, c->fhost, fbytes)) return rc;
        kp.fhost = want_f ? static_cast<double*>(c->fhost.p) : nullptr;
        kp.want_residual = residual ? 1 : 0;
        HIPCHK(c, launch_swap(5, kp, 0, c->stream));
        if (acc_out) {
            HIPCHK(c, launch_reduce(static_cast<const double*>(c->partials.p),
                                    static_cast<const BlockParams*>(c->blocks.p),
                                    (int)c->bp.size(), c->ntiles, c->nbulk, 0, 0, 0,
                                    static_cast<double*>(c->red.p), c->stream));
            acc_out->resize((c->bp.size() + 1) * kNAcc);
            HIPCHK(c, hipMemcpyAsync(acc_out->data(), c->red.p, acc_out->size() * sizeof(double),
                                     hipMemcpyDeviceToHost, c->stream));
        }
        HIPCHK(c, hipStreamSynchronize(c->stream));
        return 0;
    }
    if ((want_f || c->tstep == 0) && c->fhost.bytes != fbytes) {
        if (int rc = dalloc(c, c->fhost, fbytes)) return rc;
    }
    if (c->tstep == 0) {
        // f^0 is not reachable from a previous fStage: recompute it
        if (c->init_from_f) {
            HIPCHK(c, hipMemcpyAsync(c->fhost.p, c->host_init_f.data(), fbytes,
                                     hipMemcpyHostToDevice, c->stream));
        } else if (c->init_lift) {
            KParams ki = base_params(c);
            ki.fhost = static_cast<double*>(c->fhost.p);
            HIPCHK(c, launch_lift(c->dim, ki, c->interior_nodes, c->stream));
        } else {
            KParams ki = base_params(c);
            ki.fhost = static_cast<double*>(c->fhost.p);
            HIPCHK(c, launch_lattice(c->lat, c->storage, MODE_INIT_FEQ, ki, c->stream));
        }
        kp.fhost = static_cast<double*>(c->fhost.p);
        kp.fhost_in = 1;
    } else {
        kp.fhost = want_f ? static_cast<double*>(c->fhost.p) : nullptr;
    }
    kp.want_residual = residual ? 1 : 0;
    // after the first step, through the step's bulk and boundary kernels
    // (the whole-lattice kernel is the general one, several times slower)
    const bool split = c->tstep > 0 && !c->fused;
    if (split)
        HIPCHK(c, launch_materialize_split(c->lat, c->storage, kp, c->stream));
    else
        HIPCHK(c, launch_lattice(c->lat, c->storage, MODE_MATERIALIZE, kp, c->stream));
    if (acc_out) {
        HIPCHK(c, launch_reduce(static_cast<const double*>(c->partials.p),
                                static_cast<const BlockParams*>(c->blocks.p),
                                (int)c->bp.size(), c->ntiles, kp.nbulk, kp.nbnd, split ? 1 : 0,
                                kp.fold, static_cast<double*>(c->red.p), c->stream));
        acc_out->resize((c->bp.size() + 1) * kNAcc);
        HIPCHK(c, hipMemcpyAsync(acc_out->data(), c->red.p,
                                 acc_out->size() * sizeof(double),
                                 hipMemcpyDeviceToHost, c->stream));
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return 0;
}

// ---------------------------------------------------------------------------
extern "C" {

const char* mplbhip_version(void) {
    return "mplbhip 0.1 gfx950";
}

// the lattice of a context (key 2 D2Q9, 3 D3Q19, 15 D3Q15) and its FP16
// population scales
static void set_lattice(mplbhip_ctx* c, int lat) {
    const LatticeTab L = lattice_tab(lat);
    c->lat = lat;
    c->plan.lat = lat;
    c->Q = L.Q;
    c->scale.assign(c->Q, 1.f);
    c->inv_scale.assign(c->Q, 1.f);
    if (c->storage == MPLBHIP_STORE_F16) {
        // per-population scale s_i = w_i / kF16Scale (the bulk update
        // folds the same constant into its coefficients)
        for (int q = 0; q < c->Q; q++) {
            c->scale[q] = (float)(L.W[q] / kF16Scale);
            c->inv_scale[q] = (float)(kF16Scale / L.W[q]);
        }
    }
}

int mplbhip_create(mplbhip_ctx** out, int device, int space_dim, int storage) {
    if (!out) return MPLBHIP_ERR_ARG;
    *out = nullptr;
    if (space_dim != 2 && space_dim != 3) return MPLBHIP_ERR_ARG;
    if (storage < MPLBHIP_STORE_F64 || storage > MPLBHIP_STORE_F16)
        return MPLBHIP_ERR_ARG;
    mplbhip_ctx* c = new mplbhip_ctx();
    c->device = device;
    c->dim = space_dim;
    c->storage = storage;
    c->plan.dim = space_dim;
    c->es = storage == MPLBHIP_STORE_F64 ? 8 : (storage == MPLBHIP_STORE_F32 ? 4 : 2);
    set_lattice(c, space_dim);
    if (device >= 0) {
        int n = 0;
        if (hipGetDeviceCount(&n) != hipSuccess || device >= n) {
            delete c;
            return MPLBHIP_ERR_NODEVICE;
        }
        if (hipSetDevice(device) != hipSuccess ||
            hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess ||
            hipEventCreate(&c->ev[0]) != hipSuccess ||
            hipEventCreate(&c->ev[1]) != hipSuccess ||
            hipStreamCreateWithFlags(&c->side, hipStreamNonBlocking) != hipSuccess ||
            hipEventCreateWithFlags(&c->ev_fork, hipEventDisableTiming) != hipSuccess ||
            hipEventCreateWithFlags(&c->ev_join, hipEventDisableTiming) != hipSuccess ||
            scratch_address(&c->scratch) != hipSuccess) {
            delete c;
            return MPLBHIP_ERR_HIP;
        }
    }
    *out = c;
    return 0;
}

void mplbhip_destroy(mplbhip_ctx* c) {
    if (!c) return;
    if (c->device >= 0) {
        (void)hipSetDevice(c->device);
        if (c->stream) (void)hipStreamSynchronize(c->stream);
        drop_graphs(c);
        for (int i = 0; i < 2; i++) {
            dfree(c->fs[i]);
            dfree(c->per[i]);
        }
        for (int v = 0; v < 4; v++) {
            dfree(c->macro[v]);
            dfree(c->macro_copy[v]);
            dfree(c->macro0[v]);
        }
        dfree(c->progs);
        dfree(c->blocks);
        dfree(c->partials);
        dfree(c->dsegs);
        for (DevBuf* d : {&c->wg_block, &c->dpair, &c->wg_pair, &c->dmarch, &c->dtile, &c->swap_mask,
                          &c->temp, &c->dobst})
            dfree(*d);
        dfree(c->red);
        dfree(c->fhost);
        dfree(c->parity[0]);
        dfree(c->parity[1]);
        for (HaloLink& h : c->halos) {
            if (h.d_flag) (void)hipFree(h.d_flag);
            if (h.d_sup) (void)hipFree(h.d_sup);
        }
        dfree(c->halo_links[0]);
        dfree(c->halo_links[1]);
        dfree(c->halo_wgstart);
        for (int i = 0; i < 2; i++)
            if (c->ev[i]) (void)hipEventDestroy(c->ev[i]);
        if (c->ev_fork) (void)hipEventDestroy(c->ev_fork);
        if (c->ev_join) (void)hipEventDestroy(c->ev_join);
        if (c->side) (void)hipStreamDestroy(c->side);
        if (c->stream) (void)hipStreamDestroy(c->stream);
    }
    delete c;
}

const char* mplbhip_last_error(const mplbhip_ctx* c) {
    return c ? c->err.c_str() : "null context";
}

int mplbhip_define_block(mplbhip_ctx* c, int id, const int* size) {
    if (!c || !size) return MPLBHIP_ERR_ARG;
    if (c->prepared) return fail(c, MPLBHIP_ERR_ARG, "case already prepared");
    if (id != (int)c->plan.blocks.size())
        return fail(c, MPLBHIP_ERR_ARG, "blocks must be defined in id order");
    if ((int)c->plan.blocks.size() >= kMaxBlocks)
        return fail(c, MPLBHIP_ERR_ARG, "too many blocks");
    BlockDef b;
    for (int a = 0; a < 3; a++) b.n[a] = a < c->dim ? size[a] : 1;
    for (int a = 0; a < c->dim; a++)
        if (b.n[a] < 3)
            return fail(c, MPLBHIP_ERR_ARG, "block %d axis %d has %d < 3 nodes",
                        id, a, b.n[a]);
    c->plan.blocks.push_back(b);
    c->accel.push_back({0.0, 0.0, 0.0});
    c->btau.push_back(std::nan(""));
    c->bdt.push_back(std::nan(""));
    return 0;
}

int mplbhip_define_connection(mplbhip_ctx* c, int from, int fsurf, int to,
                              int tsurf, int vtype) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (c->prepared) return fail(c, MPLBHIP_ERR_ARG, "case already prepared");
    const int nb = (int)c->plan.blocks.size();
    if (from < 0 || from >= nb || to < 0 || to >= nb)
        return fail(c, MPLBHIP_ERR_ARG, "connection names an undefined block");
    for (const LinkDesc& l : c->plan.links)
        if (l.from == from && l.fsurf == fsurf)
            return fail(c, MPLBHIP_ERR_ARG,
                        "a neighbour is already defined for block %d surface %d",
                        from, fsurf);
    c->plan.links.push_back(LinkDesc{from, fsurf, to, tsurf, vtype, 0});
    return 0;
}

int mplbhip_define_rotated_connection(mplbhip_ctx* c, int from, int fsurf, int to,
                                      int tsurf, int vtype) {
    if (!c) return MPLBHIP_ERR_ARG;
    int sf, st;
    const int af = face_axis(fsurf, &sf), at = face_axis(tsurf, &st);
    if (af < 0 || at < 0 || af == at || af >= c->dim || at >= c->dim)
        return fail(c, MPLBHIP_ERR_ARG, "a rotated connection joins two perpendicular faces");
    if (int rc = mplbhip_define_connection(c, from, fsurf, to, tsurf, vtype)) return rc;
    c->plan.links.back().rot = 1;
    return 0;
}

int mplbhip_define_collision(mplbhip_ctx* c, double tau_ref, int force_type,
                             int force_macros) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (force_type != 0 && force_type != 1)
        return fail(c, MPLBHIP_ERR_UNSUPPORTED,
                    "body force type %d: only BodyForce_None and BodyForce_1st",
                    force_type);
    c->tau = tau_ref;
    c->force_type = force_type;
    c->force_macros = force_macros ? 1 : 0;
    if (c->prepared && c->device >= 0) {
        HIPCHK(c, hipSetDevice(c->device));
        drop_graphs(c);
        if (int rc = upload_blocks(c)) return rc;
        // a body force may take 2D steps from rows to tiles, or back
        return assign_2d(c, false);
    }
    return 0;
}

int mplbhip_define_scheme(mplbhip_ctx* c, int scheme) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (c->prepared) return fail(c, MPLBHIP_ERR_ARG, "the scheme is defined before prepare");
    if (scheme != SCHEME_StreamCollision && scheme != SCHEME_Swap)
        return fail(c, MPLBHIP_ERR_UNSUPPORTED, "scheme %d is not implemented", scheme);
    if (scheme == SCHEME_Swap && (c->dim != 3 || c->storage != MPLBHIP_STORE_F64))
        return fail(c, MPLBHIP_ERR_UNSUPPORTED,
                    "the swap scheme runs D3Q19 (the reference's swap kernels are 3D only, "
                    "scheme_kernel.inc:957-1398) with FP64 storage");
    c->plan.scheme = scheme;
    c->swap = scheme == SCHEME_Swap;
    return 0;
}

int mplbhip_define_lattice(mplbhip_ctx* c, int q) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (c->prepared) return fail(c, MPLBHIP_ERR_ARG, "the lattice is defined before prepare");
    int lat = 0;
    if (c->dim == 2 && q == 9) lat = 2;
    if (c->dim == 3 && q == 19) lat = 3;
    if (c->dim == 3 && q == 15) lat = 15;
    if (!lat)
        return fail(c, MPLBHIP_ERR_UNSUPPORTED,
                    "lattice with %d velocities in %dD: d2q9, d3q19 and d3q15 are defined "
                    "(model.cpp:99-150)",
                    q, c->dim);
    set_lattice(c, lat);
    return 0;
}

int mplbhip_define_collision_type(mplbhip_ctx* c, int type) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (c->prepared) return fail(c, MPLBHIP_ERR_ARG, "the collision type is defined before prepare");
    if (type != 0 && type != 1)
        return fail(c, MPLBHIP_ERR_UNSUPPORTED,
                    "collision type %d: Collision_BGKIsothermal2nd (0) and "
                    "Collision_BGKThermal4th (1)",
                    type);
    if (type == 1 && c->storage != MPLBHIP_STORE_F64)
        return fail(c, MPLBHIP_ERR_UNSUPPORTED,
                    "Collision_BGKThermal4th runs with FP64 storage (its equilibrium is "
                    "restated in the reference's FP64 arithmetic)");
    c->thermal = type == 1;
    return 0;
}

int mplbhip_set_temperature(mplbhip_ctx* c, int block, const double* T) {
    if (!c || !T) return MPLBHIP_ERR_ARG;
    if (int rc = need_device(c)) return rc;
    if (!c->prepared) return fail(c, MPLBHIP_ERR_ARG, "call mplbhip_prepare first");
    if (!c->thermal)
        return fail(c, MPLBHIP_ERR_ARG, "the temperature is read by Collision_BGKThermal4th only");
    if (block < 0 || block >= (int)c->bp.size())
        return fail(c, MPLBHIP_ERR_ARG, "undefined block");
    const BlockParams& B = c->bp[block];
    const size_t nn = (size_t)B.n[0] * B.n[1] * B.n[2];
    for (size_t i = 0; i < nn; i++)
        if (!(T[i] > 0.0))
            return fail(c, MPLBHIP_ERR_ARG, "temperature %g at node %zu of block %d", T[i], i,
                        block);
    drop_graphs(c);
    HIPCHK(c, hipMemcpyAsync(static_cast<double*>(c->temp.p) + B.mbase, T, nn * sizeof(double),
                             hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    c->temp_set = true;
    return 0;
}

int mplbhip_define_obstacles(mplbhip_ctx* c, int block, const unsigned char* solid) {
    if (!c || !solid) return MPLBHIP_ERR_ARG;
    if (c->prepared) return fail(c, MPLBHIP_ERR_ARG, "obstacles are defined before prepare");
    if (block < 0 || block >= (int)c->plan.blocks.size())
        return fail(c, MPLBHIP_ERR_ARG, "obstacles on undefined block %d", block);
    const int* n = c->plan.blocks[block].n;
    const size_t cnt = (size_t)n[0] * n[1] * n[2];
    if (c->solid.size() < c->plan.blocks.size()) c->solid.resize(c->plan.blocks.size());
    c->solid[block].assign(solid, solid + cnt);
    for (uint8_t& v : c->solid[block]) v = v ? 1 : 0;
    return 0;
}

int mplbhip_define_boundary(mplbhip_ctx* c, int block, int surface, int scheme,
                            const double* vars, int nvars, int vtype) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (c->prepared) return fail(c, MPLBHIP_ERR_ARG, "case already prepared");
    if (block < 0 || block >= (int)c->plan.blocks.size())
        return fail(c, MPLBHIP_ERR_ARG, "boundary on undefined block %d", block);
    if (nvars < 0 || nvars > 8 || (nvars > 0 && !vars))
        return fail(c, MPLBHIP_ERR_ARG, "bad given variables");
    if (scheme != SCH_EQMDiffuseRefl && scheme != SCH_ExtrapolPressure1ST &&
        scheme != SCH_None && scheme != SCH_MDPeriodic && scheme != SCH_FDPeriodic)
        return fail(c, MPLBHIP_ERR_UNSUPPORTED,
                    "boundary scheme %d is not implemented", scheme);
    if (scheme == SCH_EQMDiffuseRefl && nvars < c->dim)
        return fail(c, MPLBHIP_ERR_ARG, "EQMDiffuseRefl needs the wall velocity");
    if (scheme == SCH_ExtrapolPressure1ST && nvars < 1)
        return fail(c, MPLBHIP_ERR_ARG, "ExtrapolPressure1ST needs the density");
    BCDesc d;
    std::memset(&d, 0, sizeof d);
    d.block = block;
    d.surface = surface;
    d.scheme = scheme;
    d.vtype = vtype;
    d.nvars = nvars;
    for (int i = 0; i < nvars; i++) d.vars[i] = vars[i];
    c->plan.bcs.push_back(d);
    return 0;
}

// The merged halo launch.  A link that reads a halo cell an earlier link
// writes in the same exchange (raw) must see that write: it stays out,
// copied by its own launch after the merged one; so does every later link
// that writes a cell such a link reads or writes (the order of those
// writes matters), to a fixed point.  The merged links never read what
// another merged link writes (an earlier one: they would be raw; a later
// one: they read the previous exchange's buffer, as the single launches
// do), and where two of them write one target element only the later
// writes (sup: per source cell, the target populations later merged links
// write at its target).
struct HaloBox {
    int b, org[3], ext[3];
};
static bool box_overlap(const HaloBox& a, const HaloBox& b) {
    if (a.b != b.b) return false;
    for (int k = 0; k < 3; k++)
        if (a.org[k] + a.ext[k] <= b.org[k] || b.org[k] + b.ext[k] <= a.org[k]) return false;
    return true;
}

static int plan_merged_halos(mplbhip_ctx* c, size_t nl, const std::vector<HaloBox>& src,
                             const std::vector<HaloBox>& dst, const std::vector<LinkMap>& maps,
                             const std::vector<std::vector<uint8_t>>& flags,
                             const std::vector<bool>& raw) {
    c->halo_nmerged = 0;
    c->halo_nwg = 0;
    if (const char* e = std::getenv("MPLBHIP_HALO_MERGE")) c->halo_merge = std::atoi(e) != 0;
    if (nl < 2) return 0;
    auto box = [](const HaloBox& s) { return s; };
    std::vector<bool> deferred(raw);
    for (bool changed = true; changed;) {
        changed = false;
        for (size_t i = 0; i < nl; i++) {
            if (!deferred[i]) continue;
            for (size_t m = i + 1; m < nl; m++)
                if (!deferred[m] && (box_overlap(box(dst[m]), box(src[i])) ||
                                     box_overlap(box(dst[m]), box(dst[i])))) {
                    deferred[m] = true;
                    changed = true;
                }
        }
    }
    std::vector<int> merged;
    for (size_t i = 0; i < nl; i++)
        if (!deferred[i]) merged.push_back((int)i);
    if (merged.size() < 2) return 0;
    const uint32_t all = (1u << c->Q) - 1u;
    // per merged link: target cell -> source cell, and the target
    // populations it writes there
    auto key = [](int x, int y, int z) {
        return ((int64_t)(x + 4) << 42) | ((int64_t)(y + 4) << 21) | (int64_t)(z + 4);
    };
    std::vector<std::unordered_map<int64_t, int>> inv(nl);
    std::vector<uint32_t> inward_t(nl, 0);
    for (int m : merged) {
        const HaloBox& s = src[m];
        const BlockDef& T = c->plan.blocks[dst[m].b];
        const HaloParams& hp = c->halos[m].hp;
        for (int q = 0; q < c->Q; q++)
            if ((hp.inward >> q) & 1u) inward_t[m] |= 1u << hp.qmap[q];
        int idx = 0;
        for (int zz = 0; zz < s.ext[2]; zz++)
            for (int yy = 0; yy < s.ext[1]; yy++)
                for (int xx = 0; xx < s.ext[0]; xx++, idx++) {
                    const int p[3] = {s.org[0] + xx, s.org[1] + yy, s.org[2] + zz};
                    int t[3];
                    link_target(maps[m], T.n, p, t);
                    if (c->dim == 2) t[2] = 0;
                    inv[m][key(t[0], t[1], t[2])] = idx;
                }
    }
    int nwg = 0;
    std::vector<int32_t> wgstart;
    c->halo_hps.clear();
    for (int i : merged) {
        HaloLink& h = c->halos[i];
        const HaloBox& s = src[i];
        const BlockDef& T = c->plan.blocks[dst[i].b];
        const int64_t ncell = (int64_t)s.ext[0] * s.ext[1] * s.ext[2];
        std::vector<uint32_t> sup(ncell, 0);
        bool any = false;
        int idx = 0;
        for (int zz = 0; zz < s.ext[2]; zz++)
            for (int yy = 0; yy < s.ext[1]; yy++)
                for (int xx = 0; xx < s.ext[0]; xx++, idx++) {
                    const int p[3] = {s.org[0] + xx, s.org[1] + yy, s.org[2] + zz};
                    int t[3];
                    link_target(maps[i], T.n, p, t);
                    if (c->dim == 2) t[2] = 0;
                    for (int m : merged) {
                        if (m <= i || dst[m].b != dst[i].b) continue;
                        auto it = inv[m].find(key(t[0], t[1], t[2]));
                        if (it == inv[m].end()) continue;
                        sup[idx] |= (flags[m][it->second] & 2) ? all : inward_t[m];
                    }
                    any = any || sup[idx] != 0;
                }
        if (any && c->device >= 0) {
            HIPCHK(c, hipMalloc(&h.d_sup, ncell * sizeof(uint32_t)));
            HIPCHK(c, hipMemcpy(h.d_sup, sup.data(), ncell * sizeof(uint32_t),
                                hipMemcpyHostToDevice));
        }
        h.merged = true;
        wgstart.push_back(nwg);
        nwg += (int)((ncell + 255) / 256);
        HaloParams hp = h.hp;
        hp.other_flag = h.d_flag;
        hp.sup = h.d_sup;
        c->halo_hps.push_back(hp);
    }
    wgstart.push_back(nwg);
    c->halo_nmerged = (int)merged.size();
    c->halo_nwg = nwg;
    if (c->device >= 0) {
        if (int rc = dalloc(c, c->halo_wgstart, wgstart.size() * sizeof(int32_t))) return rc;
        HIPCHK(c, hipMemcpy(c->halo_wgstart.p, wgstart.data(), wgstart.size() * sizeof(int32_t),
                            hipMemcpyHostToDevice));
    }
    if (std::getenv("MPLBHIP_VERBOSE"))
        std::fprintf(stderr, "mplbhip: halos: %d of %zu links in one launch (%d workgroups)\n",
                     c->halo_nmerged, nl, nwg);
    return 0;
}

// the merged links' parameters with the fStage buffers filled in, one
// array per ping-pong target; once the buffers exist (end of prepare)
static int upload_merged_halos(mplbhip_ctx* c) {
    if (c->halo_nmerged < 2 || c->device < 0) return 0;
    for (int into = 0; into < 2; into++) {
        std::vector<HaloParams> hps = c->halo_hps;
        for (HaloParams& hp : hps) {
            hp.src_cur = c->fs[into].p;
            hp.src_other = c->fs[c->swap ? into : 1 - into].p;
            hp.dst = c->fs[into].p;
        }
        if (int rc = dalloc(c, c->halo_links[into], hps.size() * sizeof(HaloParams))) return rc;
        HIPCHK(c, hipMemcpy(c->halo_links[into].p, hps.data(), hps.size() * sizeof(HaloParams),
                            hipMemcpyHostToDevice));
    }
    c->halo_fs[0] = c->fs[0].p;
    c->halo_fs[1] = c->fs[1].p;
    return 0;
}

static int setup_halos(mplbhip_ctx* c) {
    // ops_halo_transfer order: blocks by id, then surfaces Left, Right, Top,
    // Bottom, Front, Back (std::map<BoundarySurface> order); edge surfaces
    // declare no halo (field.h:395 default).
    const int order[6] = {BS_Left, BS_Right, BS_Top, BS_Bottom, BS_Front, BS_Back};
    std::vector<LinkDesc> seq;
    for (int b = 0; b < (int)c->plan.blocks.size(); b++)
        for (int oi = 0; oi < 6; oi++)
            for (const LinkDesc& l : c->plan.links)
                if (l.from == b && l.fsurf == order[oi]) seq.push_back(l);
    const int hz = c->dim == 3 ? 1 : 0;
    struct Slab { int b; int org[3]; int ext[3]; };
    std::vector<Slab> src(seq.size()), dst(seq.size());
    std::vector<LinkMap> maps(seq.size());
    for (size_t i = 0; i < seq.size(); i++) {
        const LinkDesc& l = seq[i];
        const BlockDef& A = c->plan.blocks[l.from];
        const BlockDef& T = c->plan.blocks[l.to];
        LinkMap& m = maps[i];
        if (!link_map(l, m) || m.af >= c->dim)
            return fail(c, MPLBHIP_ERR_ARG, "connection of block %d names no face of a %dD block",
                        l.from, c->dim);
        for (int d = 0; d < c->dim; d++)
            for (int j = 0; j < c->dim; j++)
                if (d != m.af && m.R[j][d] != 0 && A.n[d] != T.n[j])
                    return fail(c, MPLBHIP_ERR_ARG,
                                "connected blocks %d and %d differ across the face",
                                l.from, l.to);
        // source: the from-face plane with the transverse halo rows
        Slab s{l.from, {-1, -1, -hz}, {A.n[0] + 2, A.n[1] + 2, A.n[2] + 2 * hz}};
        s.org[m.af] = m.sf > 0 ? A.n[m.af] - 1 : 0;
        s.ext[m.af] = 1;
        // target: bounding box of the images of the slab's corners
        Slab d{l.to, {0, 0, 0}, {1, 1, 1}};
        int lo[3] = {1 << 30, 1 << 30, 1 << 30}, hi[3] = {-(1 << 30), -(1 << 30), -(1 << 30)};
        for (int corner = 0; corner < 8; corner++) {
            int p[3], q[3];
            for (int a = 0; a < 3; a++)
                p[a] = s.org[a] + (((corner >> a) & 1) ? s.ext[a] - 1 : 0);
            link_target(m, T.n, p, q);
            if (c->dim == 2) q[2] = 0;
            for (int a = 0; a < 3; a++) {
                lo[a] = std::min(lo[a], q[a]);
                hi[a] = std::max(hi[a], q[a]);
            }
        }
        for (int a = 0; a < 3; a++) {
            d.org[a] = lo[a];
            d.ext[a] = hi[a] - lo[a] + 1;
        }
        src[i] = s;
        dst[i] = d;
    }
    // Source cells outside the source block's interior are halo cells; the
    // reference reads them as last written.  Written earlier in this exchange
    // -> current buffer; written only later -> the previous exchange, which
    // went to the other ping-pong buffer; never written -> zero in both.
    auto covers = [&](const Slab& s, int b, int x, int y, int z) {
        return s.b == b && x >= s.org[0] && x < s.org[0] + s.ext[0] &&
               y >= s.org[1] && y < s.org[1] + s.ext[1] && z >= s.org[2] &&
               z < s.org[2] + s.ext[2];
    };
    c->halos.clear();
    std::vector<std::vector<uint8_t>> flags(seq.size());
    std::vector<bool> raw(seq.size(), false);  // reads a halo cell an earlier link wrote
    for (size_t i = 0; i < seq.size(); i++) {
        const Slab& s = src[i];
        const BlockDef& A = c->plan.blocks[s.b];
        const int64_t ncell = (int64_t)s.ext[0] * s.ext[1] * s.ext[2];
        std::vector<uint8_t>& flag = flags[i];
        flag.assign(ncell, 0);
        bool anyother = false;
        for (int zz = 0; zz < s.ext[2]; zz++)
            for (int yy = 0; yy < s.ext[1]; yy++)
                for (int xx = 0; xx < s.ext[0]; xx++) {
                    const int x = s.org[0] + xx, y = s.org[1] + yy, z = s.org[2] + zz;
                    const bool interior = x >= 0 && x < A.n[0] && y >= 0 &&
                                          y < A.n[1] && z >= 0 && z < A.n[2];
                    if (interior) continue;
                    bool before = false, after = false;
                    for (size_t j = 0; j < seq.size(); j++)
                        if (covers(dst[j], s.b, x, y, z)) {
                            if (j < i) before = true; else after = true;
                        }
                    if (before) raw[i] = true;
                    if (!before && after) {
                        flag[((int64_t)zz * s.ext[1] + yy) * s.ext[0] + xx] = 1;
                        anyother = true;
                    }
                }
        // target cells that another connection reads (as its source, from
        // either buffer) keep every population
        const LinkMap& mi = maps[i];
        const BlockDef& Ti = c->plan.blocks[dst[i].b];
        for (int zz = 0; zz < s.ext[2]; zz++)
            for (int yy = 0; yy < s.ext[1]; yy++)
                for (int xx = 0; xx < s.ext[0]; xx++) {
                    const int p[3] = {s.org[0] + xx, s.org[1] + yy, s.org[2] + zz};
                    int t[3];
                    link_target(mi, Ti.n, p, t);
                    if (c->dim == 2) t[2] = 0;
                    for (size_t j = 0; j < seq.size(); j++)
                        if (j != i && covers(src[j], dst[i].b, t[0], t[1], t[2])) {
                            flag[((int64_t)zz * s.ext[1] + yy) * s.ext[0] + xx] |= 2;
                            anyother = true;
                            break;
                        }
                }
        HaloLink h;
        std::memset(&h.hp, 0, sizeof h.hp);
        h.from = seq[i].from;
        h.to = seq[i].to;
        const BlockParams& SB = c->bp[s.b];
        const BlockParams& DB = c->bp[dst[i].b];
        h.hp.src_base = SB.base;
        h.hp.dst_base = DB.base;
        h.hp.src_sx = SB.sx; h.hp.src_sz = SB.sz; h.hp.src_sq = SB.sq;
        h.hp.dst_sx = DB.sx; h.hp.dst_sz = DB.sz; h.hp.dst_sq = DB.sq;
        const LinkMap& m = maps[i];
        const BlockDef& T = c->plan.blocks[dst[i].b];
        const int64_t stride[3] = {1, DB.sx, DB.sz};
        int q0[3];
        link_target(m, T.n, s.org, q0);
        if (c->dim == 2) q0[2] = 0;
        h.hp.dst_org = 0;
        for (int a = 0; a < 3; a++) {
            h.hp.org_src[a] = s.org[a];
            h.hp.ext[a] = s.ext[a];
            h.hp.dst_org += q0[a] * stride[a];
            h.hp.dstep[a] = 0;
            for (int j = 0; j < 3; j++)
                if (a != m.af && m.R[j][a] != 0) h.hp.dstep[a] = m.R[j][a] * stride[j];
        }
        const int (*cv)[3] = lattice_tab(c->lat).C;
        for (int q = 0; q < c->Q; q++) {
            int v[3] = {0, 0, 0};
            for (int j = 0; j < 3; j++)
                for (int k = 0; k < 3; k++) v[j] += m.R[j][k] * cv[q][k];
            h.hp.qmap[q] = -1;
            for (int r = 0; r < c->Q; r++)
                if (cv[r][0] == v[0] && cv[r][1] == v[1] && cv[r][2] == v[2]) h.hp.qmap[q] = r;
            if (h.hp.qmap[q] < 0)
                return fail(c, MPLBHIP_ERR_ARG, "rotation leaves the velocity set");
        }
        h.hp.Q = c->Q;
        h.hp.elem_bytes = (int)c->es;
        // inward across the target face: against its outward normal st e_at
        h.hp.inward = 0;
        for (int q = 0; q < c->Q; q++)
            if (cv[h.hp.qmap[q]][m.at] * m.st < 0) h.hp.inward |= 1u << q;
        // the swap scheme exchanges the swapped slots and FDPeriodic copies
        // whole halo cells: every population
        if (c->swap) h.hp.inward = (1u << c->Q) - 1u;
        if (anyother && c->device >= 0) {
            HIPCHK(c, hipMalloc(&h.d_flag, ncell));
            HIPCHK(c, hipMemcpy(h.d_flag, flag.data(), ncell, hipMemcpyHostToDevice));
        }
        c->halos.push_back(h);
    }
    std::vector<HaloBox> sbox(seq.size()), dbox(seq.size());
    for (size_t i = 0; i < seq.size(); i++) {
        sbox[i].b = src[i].b;
        dbox[i].b = dst[i].b;
        for (int k = 0; k < 3; k++) {
            sbox[i].org[k] = src[i].org[k];
            sbox[i].ext[k] = src[i].ext[k];
            dbox[i].org[k] = dst[i].org[k];
            dbox[i].ext[k] = dst[i].ext[k];
        }
    }
    return plan_merged_halos(c, seq.size(), sbox, dbox, maps, flags, raw);
}

static bool full_pull_type(int vt) {
    return vt == VT_Fluid || vt == VT_MDPeriodic || vt == VT_VirtualBoundary;
}

// Obstacle link masks (bit q: the pull source x - c_q is an obstacle node;
// kObstSolid: x is one).  Sources in a halo are resolved through the block
// connections, as the halo exchange would copy them.  A node pulling from
// an obstacle must pull every population; obstacles sit on Fluid or
// MDPeriodic nodes only.
static int build_obstacles(mplbhip_ctx* c) {
    c->obst.clear();
    const int nb = (int)c->plan.blocks.size();
    bool any = false;
    for (int b = 0; b < (int)c->solid.size(); b++) any = any || !c->solid[b].empty();
    if (!any) return 0;
    c->solid.resize(nb);
    const int hz = c->dim == 3 ? 1 : 0;
    // halo-extended obstacle flags per block
    std::vector<std::vector<uint8_t>> ext(nb);
    auto eidx = [&](int b, int i, int j, int k) {
        const int* n = c->plan.blocks[b].n;
        return ((size_t)(k + hz) * (n[1] + 2) + (j + 1)) * (n[0] + 2) + (i + 1);
    };
    for (int b = 0; b < nb; b++) {
        const int* n = c->plan.blocks[b].n;
        ext[b].assign((size_t)(n[0] + 2) * (n[1] + 2) * (n[2] + 2 * hz), 0);
        if (c->solid[b].empty()) continue;
        size_t p = 0;
        for (int k = 0; k < n[2]; k++)
            for (int j = 0; j < n[1]; j++)
                for (int i = 0; i < n[0]; i++, p++) ext[b][eidx(b, i, j, k)] = c->solid[b][p];
    }
    for (const LinkDesc& l : c->plan.links) {
        if (c->solid[l.from].empty()) continue;
        LinkMap m;
        if (!link_map(l, m)) continue;
        const int* na = c->plan.blocks[l.from].n;
        const int* nt = c->plan.blocks[l.to].n;
        int lo[3] = {0, 0, 0}, hi[3] = {na[0], na[1], na[2]};
        lo[m.af] = m.sf > 0 ? na[m.af] - 1 : 0;
        hi[m.af] = lo[m.af] + 1;
        for (int k = lo[2]; k < hi[2]; k++)
            for (int j = lo[1]; j < hi[1]; j++)
                for (int i = lo[0]; i < hi[0]; i++) {
                    const int p[3] = {i, j, k};
                    int d[3];
                    link_target(m, nt, p, d);
                    if (c->dim == 2) d[2] = 0;
                    ext[l.to][eidx(l.to, d[0], d[1], d[2])] =
                        c->solid[l.from][((size_t)k * na[1] + j) * na[0] + i];
                }
    }
    c->obst.assign((size_t)c->interior_nodes, 0u);
    const int (*cv)[3] = lattice_tab(c->lat).C;
    for (int b = 0; b < nb; b++) {
        const int* n = c->plan.blocks[b].n;
        bool has = false;
        size_t p = 0;
        for (int k = 0; k < n[2]; k++)
            for (int j = 0; j < n[1]; j++)
                for (int i = 0; i < n[0]; i++, p++) {
                    // the node type is constant over a region (Plan::build)
                    const int vt = c->plan.region_vt[(size_t)b * c->plan.nregions +
                                                     c->plan.region_of(b, i, j, k)];
                    uint32_t mask = 0;
                    if (ext[b][eidx(b, i, j, k)]) {
                        if (vt != VT_Fluid && vt != VT_MDPeriodic)
                            return fail(c, MPLBHIP_ERR_ARG,
                                        "obstacle on a node that is not Fluid or MDPeriodic "
                                        "(block %d node %d,%d,%d)", b, i, j, k);
                        mask = kObstSolid;
                    } else {
                        for (int q = 0; q < c->Q; q++)
                            if (ext[b][eidx(b, i - cv[q][0], j - cv[q][1], k - cv[q][2])])
                                mask |= 1u << q;
                        if (mask && !full_pull_type(vt))
                            return fail(c, MPLBHIP_ERR_ARG,
                                        "obstacle next to a boundary node (block %d node "
                                        "%d,%d,%d)", b, i, j, k);
                    }
                    has = has || mask != 0;
                    c->obst[(size_t)c->bp[b].mbase + p] = mask;
                }
        c->bp[b].has_obst = has ? 1 : 0;
    }
    return 0;
}

// Workgroup ranges of the blocks in the step launches (whole tiles, the
// two-node FP16 tiles, the bulk tiles and the three boundary segment
// lists) and the per-block XCD row grouping.  With only_active, frozen
// blocks get empty ranges that start where the next block's range does,
// so the launches' block search (the last block whose start <= the
// workgroup) never lands on them.  Returns the number of row-grouped blocks.
static int assign_tiles(mplbhip_ctx* c, bool only_active) {
    int tiles = 0, bulk = 0, bulk3 = 0, bulk2 = 0, bnd_v[4] = {0, 0, 0, 0};
    int64_t nodes = 0;
    for (BlockParams& B : c->bp) {
        const bool on = !only_active || B.active;
        const int zb = c->dim == 3 ? B.n[2] - 2 : 1;
        const int zb3 = c->dim == 3 ? B.n[2] : 1;
        B.tile_start = tiles;
        B.bulk_tile_start = bulk;
        B.bulk_tile_start3 = bulk3;
        B.h2_tile_start = bulk2;
        if (on) {
            tiles += B.tiles_x * B.tiles_y * B.n[2];
            bulk += B.tiles_x * B.tiles_y * zb;
            bulk3 += B.tiles_x * B.tiles_y * zb3;
            bulk2 += B.tiles_x2 * B.tiles_y * zb;
            nodes += (int64_t)B.n[0] * B.n[1] * B.n[2];
        }
        for (int v = 0; v < 4; v++) {
            B.bnd_wg_start[v] = bnd_v[v];
            if (!on) continue;
            int count = 0;
            for (int k = B.seg_start[v]; k < B.seg_start[v] + B.seg_count[v]; k++)
                count += (c->segs[(size_t)k].count + kBndWG - 1) / kBndWG;
            bnd_v[v] += count;
        }
    }
    c->ntiles = tiles;
    c->nbulk = bulk;
    c->nbulk3 = bulk3;
    c->nbulk2 = bulk2;
    for (int v = 0; v < 4; v++) c->nbnd_v[v] = bnd_v[v];
    c->grid_nodes = nodes;
    // the x tiles of a row share their edge cache lines: deal each row's
    // tiles to one XCD (hardware hands workgroups to the 8 XCDs round
    // robin) where the block's tiles start on a multiple of 8 and fill
    // whole groups of 8 rows
    const int nb = (int)c->bp.size();
    int grouped = 0;
    for (int b = 0; b < nb; b++) {
        BlockParams& B = c->bp[b];
        const int next = b + 1 < nb ? c->bp[b + 1].bulk_tile_start : bulk;
        const int cnt = next - B.bulk_tile_start;
        const bool ok = cnt > 0 && B.bulk_tile_start % 8 == 0 && cnt % (8 * B.tiles_x) == 0 &&
                        !c->xcd_remap;
        B.xgroup = ok ? B.tiles_x : 0;
        grouped += ok ? 1 : 0;
        const int next3 = b + 1 < nb ? c->bp[b + 1].bulk_tile_start3 : bulk3;
        const int cnt3 = next3 - B.bulk_tile_start3;
        B.xgroup3 = cnt3 > 0 && B.bulk_tile_start3 % 8 == 0 && cnt3 % (8 * B.tiles_x) == 0 &&
                            !c->xcd_remap
                        ? B.tiles_x
                        : 0;
        B.rowwg = B.tiles_x % kTY == 0 && B.n[1] % kTY == 0 ? 1 : 0;
    }
    // each grid's workgroup -> block table: block b owns workgroups
    // [its first, the next block's first) of that grid
    c->wg_block_host.clear();
    auto table = [&](int k, int total, auto first) {
        c->wg_block_off[k] = c->wg_block_host.size();
        for (int b = 0; b < nb; b++) {
            const int lo = first(c->bp[b]);
            const int hi = b + 1 < nb ? first(c->bp[b + 1]) : total;
            for (int w = lo; w < hi; w++) c->wg_block_host.push_back(b);
        }
    };
    table(kWgAll, tiles, [](const BlockParams& B) { return B.tile_start; });
    table(kWgBulk, bulk, [](const BlockParams& B) { return B.bulk_tile_start; });
    table(kWgBulk3, bulk3, [](const BlockParams& B) { return B.bulk_tile_start3; });
    table(kWgH2, bulk2, [](const BlockParams& B) { return B.h2_tile_start; });
    for (int v = 0; v < 4; v++)
        table(kWgBnd + v, bnd_v[v], [v](const BlockParams& B) { return B.bnd_wg_start[v]; });
    return grouped;
}

// Whether the case can take two steps per launch: 3D blocks without
// connections or obstacles, BGK without a body force, every envelope region a
// wall (masked pulls and at most one EQM application), populations persisted
// at single corner nodes only, and rows long enough to tile.
static bool pair_allowed(const mplbhip_ctx* c) {
    if (c->dim != 3 || c->swap || c->thermal) return false;
    if (!c->plan.links.empty() || !c->obst.empty()) return false;
    for (size_t b = 0; b < c->plan.blocks.size(); b++) {
        if (c->bp[b].n[0] < 16 || c->bp[b].n[1] < 4) return false;
        for (int r = 1; r < c->plan.nregions; r++) {
            const RegionProg& P = c->plan.progs[b * c->plan.nregions + r];
            const bool corner = r % 3 && (r / 3) % 3 && r / 9;
            if (P.kind != RK_MASKED || P.nops > 1) return false;
            if (P.nops == 1 && P.op[0].type != OP_EQM) return false;
            if (P.persist >= 0 && !corner) return false;
        }
    }
    return true;
}

// Whether every tile of a w x h tiling of a block fits a k_pair workgroup of
// nt threads and np positions: the grown tile's positions, and for either
// step the threads of its nodes (the first wave for the x-face nodes).
static bool pair_fits(const int* n, int w, int h, int nt, int np) {
    if ((w + 2) * (h + 2) > np) return false;
    for (int xa = 0; xa < n[0]; xa += w) {
        const bool lo1 = xa <= 1, hi1 = xa + w + 1 >= n[0];
        const bool lo = xa == 0, hi = xa + w >= n[0];
        const int rw1 = (hi1 ? n[0] - 1 : xa + w + 1) - (lo1 ? 1 : xa - 1);
        const int rows1 = std::min(h + 2, n[1]), rows = std::min(h, n[1]);
        if ((lo1 || hi1 ? 64 : 0) + rw1 * rows1 > nt) return false;
        if ((lo || hi ? 64 : 0) + w * rows > nt) return false;
        if (rows1 * ((lo1 ? 1 : 0) + (hi1 ? 1 : 0)) > 64) return false;
    }
    return true;
}

static int upload_pairs(mplbhip_ctx* c) {
    if (int rc = dalloc(c, c->dpair, c->pb.size() * sizeof(PairBlock))) return rc;
    if (int rc = dalloc(c, c->wg_pair, std::max<size_t>(1, c->wg_pair_host.size()) * sizeof(int32_t)))
        return rc;
    HIPCHK(c, hipMemcpyAsync(c->dpair.p, c->pb.data(), c->dpair.bytes, hipMemcpyHostToDevice,
                             c->stream));
    HIPCHK(c, hipMemcpyAsync(c->wg_pair.p, c->wg_pair_host.data(),
                             c->wg_pair_host.size() * sizeof(int32_t), hipMemcpyHostToDevice,
                             c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return 0;
}

// The two-step tiling of one of nblk blocks, by a model of the launch: its
// workgroups run in rounds of one per CU, each for lz + 3 planes (the planes
// below and above its range, and the start); a plane costs a fixed latency,
// worth that of 16 waves, and the work of the tile's waves, and the two ends
// of its rows add a quarter of a 128-byte line.  Fitted to some 700 tilings
// of 48^3 to 256^3 in the three storage forms, where its pick is within 8% of
// the fastest.  Tile widths are multiples of 64 bytes (or the whole row):
// rows that share such a piece with the next tile's cost twice the time
// (D3Q19 FP32 256^3: 0.70 ms per step in tiles of 43 x 19, 0.28 in 64 x 13;
// FP64 160^3: 0.27 in 20 x 18, 0.16 in 32 x 11).
static void pair_tiling(const int* n, int es, long long nblk, int nt, int np, PairBlock* P) {
    double best = 1e300;
    const int unit = 64 / es;
    for (int w = unit; w < n[0] + unit; w += unit) {
        const int wt = w < n[0] ? w : n[0];
        // (each height and range once: 160^3 in 0.04 ms instead of 0.23)
        for (int ty = 1, last = 0; ty <= n[1]; ty++) {
            const int h = (n[1] + ty - 1) / ty;
            if (h == last) continue;
            last = h;
            if (!pair_fits(n, wt, h, nt, np)) continue;
            const int waves = ((wt + 2) * (h + 2) + 63) / 64;
            const long long columns = nblk * ((n[0] + wt - 1) / wt) * ((n[1] + h - 1) / h);
            for (int tz = 1, lz0 = 0; tz <= n[2]; tz++) {
                const int lz = (n[2] + tz - 1) / tz;
                if (lz == lz0) continue;
                lz0 = lz;
                const long long wgs = columns * ((n[2] + lz - 1) / lz);
                const double cost = (double)((wgs + 255) / 256) * (lz + 3) * (16.0 + waves) *
                                    (1.0 + 32.0 / (wt * es));
                if (cost < best) {
                    best = cost;
                    P->w = wt;
                    P->h = h;
                    P->lz = lz;
                }
            }
            if (h < 4) break;
        }
    }
}

// Whether a region is a wall as known_wall and lane_wall have it: masked
// pulls and one EQM application with the classes of its place.
static bool plain_wall2(const RegionProg& P, int r) {
    if (P.kind != RK_MASKED || P.nops != 1 || P.op[0].type != OP_EQM || P.persist >= 0)
        return false;
    uint32_t in, out, par;
    tile_wall_classes(r, &in, &out, &par);
    const BCOp& op = P.op[0];
    return op.m_in == in && op.m_out == out && op.m_par == par;
}

// Whether the case can take several steps per launch of k_march: 2D blocks
// without connections, BGK without a body force, every envelope region a
// wall.
static bool march_allowed(const mplbhip_ctx* c) {
    if (c->dim != 2 || c->swap || c->thermal || !c->plan.links.empty()) return false;
    // (a block is one buffer resource, of 32-bit byte offsets)
    for (const BlockParams& B : c->bp)
        if ((int64_t)B.sz * (int64_t)c->es >= (int64_t)1 << 31) return false;
    for (size_t b = 0; b < c->plan.blocks.size(); b++)
        for (int r = 1; r < c->plan.nregions; r++)
            if (!plain_wall2(c->plan.progs[b * c->plan.nregions + r], r)) return false;
    return true;
}

// Whether the case can run in tiles (k_tile): such blocks, with or without a
// body force, or blocks without obstacles that are linked to themselves along
// x (their x faces pull every population) and long enough to wrap once.
static bool tile_allowed(mplbhip_ctx* c) {
    if (c->dim != 2 || c->swap || c->thermal) return false;
    std::vector<int> sides(c->plan.blocks.size(), 0);
    for (const LinkDesc& l : c->plan.links) {
        if (l.rot || l.from != l.to) return false;
        if (l.fsurf == BS_Left && l.tsurf == BS_Right) sides[l.from] |= 1;
        else if (l.fsurf == BS_Right && l.tsurf == BS_Left) sides[l.from] |= 2;
        else return false;
    }
    c->wrap_x = !c->plan.links.empty();
    if (c->wrap_x && !c->obst.empty()) return false;
    for (size_t b = 0; b < c->plan.blocks.size(); b++) {
        if (sides[b] != (c->wrap_x ? 3 : 0)) return false;
        if (c->wrap_x && c->bp[b].n[0] < 32) return false;
        for (int r = 1; r < c->plan.nregions; r++) {
            const RegionProg& P = c->plan.progs[b * c->plan.nregions + r];
            if (c->wrap_x && r < 3) {
                if (P.kind != RK_FULL || P.nops != 0 || P.persist >= 0) return false;
            } else if (!plain_wall2(P, r)) {
                return false;
            }
        }
    }
    return true;
}

static int upload_table(mplbhip_ctx* c, DevBuf& d, const void* v, size_t bytes) {
    if (d.bytes < bytes)
        if (int rc = dalloc(c, d, bytes)) return rc;
    HIPCHK(c, hipMemcpyAsync(d.p, v, bytes, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return 0;
}

// the tiles of k_tile; a single block's follow from the workgroup's number
static int assign_tiles2d(mplbhip_ctx* c, bool only_active) {
    auto count = [&](int w) {
        c->tile_side = w;
        c->tile_row = (c->bp[0].n[0] + w - 1) / w;
        c->ntile2d = 0;
        for (const BlockParams& B : c->bp)
            if (!only_active || B.active)
                c->ntile2d += ((B.n[0] + w - 1) / w) * ((B.n[1] + w - 1) / w);
        return c->ntile2d;
    };
    if (count(8) > 256 && count(16) > 768) count(24);
    if (c->bp.size() == 1) return 0;
    const int w = c->tile_side;
    c->tile_host.clear();
    for (size_t b = 0; b < c->bp.size(); b++) {
        const BlockParams& B = c->bp[b];
        if (only_active && !B.active) continue;
        for (int y = 0; y < B.n[1]; y += w)
            for (int x = 0; x < B.n[0]; x += w)
                c->tile_host.push_back(TileWG{(int32_t)b, x, y, x == 0 && y == 0});
    }
    return upload_table(c, c->dtile, c->tile_host.data(), c->tile_host.size() * sizeof(TileWG));
}

// The waves of k_march.  Rows per chunk: 16 read and compute 2K of K + 16
// rows again, 8 twice that share, for twice the waves.
// (us per step with 8, 12, 16 rows: FP32 1024^2 10.1, 10.4, 11.2; 1448^2 16.5,
// 16.3, 15.9; 2048^2 27.7, 26.4, 25.0; FP64 1024^2 18.1, 17.7, 18.7)
static int assign_march(mplbhip_ctx* c, bool only_active) {
    march_shape(c->storage, !c->obst.empty(), &c->march_steps);
    const int K = c->march_steps, own = 64 - 2 * K;
    auto group = [&](int nx) { return nx <= 16 ? 16 : nx <= 32 ? 32 : 64; };
    // strips: the first and the last one need no margin on the wall's side
    auto strips = [&](int nx) { return nx <= 64 ? 1 : (nx - 64 + own - 1) / own + 1; };
    auto list = [&](int rows) {
        c->march_host.clear();
        for (size_t b = 0; b < c->bp.size(); b++) {
            const BlockParams& B = c->bp[b];
            if (only_active && !B.active) continue;
            const int G = group(B.n[0]), T = strips(B.n[0]), chunks = (B.n[1] + rows - 1) / rows;
            for (int t = 0; t < T; t++)
                for (int k = 0; k < chunks; k += 64 / G) {
                    MarchWave M;
                    M.block = (int32_t)b;
                    M.x0 = t * own;
                    M.xs = t ? M.x0 + K : 0;
                    M.xe = t + 1 < T ? M.x0 + 64 - K : B.n[0];
                    M.group = G;
                    M.chunk0 = k;
                    M.rows = rows;
                    M.first = t == 0 && k == 0;
                    c->march_host.push_back(M);
                }
        }
        return (int)c->march_host.size();
    };
    if (list(16) < 2048) list(8);
    return upload_table(c, c->dmarch, c->march_host.data(), c->march_host.size() * sizeof(MarchWave));
}

// The several-step form of 2D cases over the (active) blocks, by measured
// steps (us, cavities of n^2 nodes; single steps, tiles, march):
//   FP64  512: 16.1, 6.3, 8.6   1024: 26.2, 16.0, 17.7   1448: -, 29.0, 28.7
//   FP32  512: 14.0, 3.9, 6.0    860: -, 8.3, 8.5        1024: 17.3, 10.6, 10.1
// so tiles up to 2^20 nodes in FP64 and below that in reduced storage, where
// k_march reads less per node, and above it where k_march cannot run
// (periodic or with a body force; 4096 x 2048 channel, single against tiles:
// FP64 232 and 165, FP32 112 and 62, FP16 66 and 56).  The tile's side by the
// number of workgroups: small ones while the chip has a CU for each (128^2
// FP64: 1.7 with side 8, 2.2 with 16; 192^2: 3.1 and 2.5), the large,
// four-step ones when there are several rounds of them (400^2 FP32: 3.1
// either way; 512^2 FP64: 6.7 with 16, 6.3 with 24).
static int assign_2d(mplbhip_ctx* c, bool only_active) {
    const int64_t most = c->storage == MPLBHIP_STORE_F64 ? 1 << 20 : (1 << 20) - 1;
    c->tile = c->tile_ok && c->pair_env >= 0 && c->pair_env != 2 &&
              (c->grid_nodes <= most || !c->march_ok || c->force_type || c->force_macros);
    c->march = c->march_ok && c->pair_env >= 0 && !c->tile;
    return c->tile ? assign_tiles2d(c, only_active) : c->march ? assign_march(c, only_active) : 0;
}

// the swap scheme in one pass per step (k_swap_pull) where no block is
// connected and every region allows it
static int assign_swap(mplbhip_ctx* c) {
    c->swap_pull = c->swap && c->plan.links.empty();
    const size_t nb = c->plan.blocks.size();
    std::vector<uint32_t> mask(c->swap_pull ? nb * 54 : 0);
    for (size_t b = 0; b < nb && c->swap_pull; b++)
        c->swap_pull = swap_masks(&c->plan.progs[b * c->plan.nregions], &mask[b * 54]);
    return c->swap_pull ? upload_table(c, c->swap_mask, mask.data(), mask.size() * 4) : 0;
}

// Two-step launches over the (active) blocks: from 2^16 nodes on.  Below, a
// step is bound by the launch and its latency either way (32^3 FP64: 11.1 us
// per step against 9.8 in one whole-lattice launch; 48^3: 14.0 against 21.8).
static int assign_pairs(mplbhip_ctx* c, bool only_active) {
    c->pair = c->pair_ok && c->pair_env >= 0 && (c->pair_env > 0 || c->grid_nodes >= (1 << 16));
    if (!c->pair) return 0;
    int np = 0;
    c->pair_nt = c->storage == MPLBHIP_STORE_F64 ? 512 : 1024;
    if (!pair_shape(c->storage, c->pair_nt, &np))
        return fail(c, MPLBHIP_ERR_HIP, "no two-step kernel for this storage");
    long long nblk = 0;
    for (const BlockParams& B : c->bp) nblk += !only_active || B.active ? 1 : 0;
    c->pb.assign(c->bp.size(), PairBlock{});
    c->wg_pair_host.clear();
    for (size_t b = 0; b < c->bp.size(); b++) {
        const BlockParams& B = c->bp[b];
        PairBlock& P = c->pb[b];
        P.start = (int32_t)c->wg_pair_host.size();
        if (only_active && !B.active) continue;
        if (b > 0 && std::equal(B.n, B.n + 3, c->bp[b - 1].n) && c->pb[b - 1].w > 0) {
            P.w = c->pb[b - 1].w;
            P.h = c->pb[b - 1].h;
            P.lz = c->pb[b - 1].lz;
        } else {
            pair_tiling(B.n, (int)c->es, nblk, c->pair_nt, np, &P);
        }
        if (P.w <= 0) {  // no tile fits
            c->pair = false;
            return 0;
        }
        P.tx = (B.n[0] + P.w - 1) / P.w;
        P.ty = (B.n[1] + P.h - 1) / P.h;
        P.tz = (B.n[2] + P.lz - 1) / P.lz;
        fast_div_params(P.tx, &P.div_m[0], &P.div_sh[0]);
        fast_div_params(P.ty, &P.div_m[1], &P.div_sh[1]);
        c->wg_pair_host.insert(c->wg_pair_host.end(), (size_t)P.tx * P.ty * P.tz, (int32_t)b);
    }
    c->npair = (int)c->wg_pair_host.size();
    return upload_pairs(c);
}

// the workgroup -> block tables to the device (after assign_tiles; the
// buffer holds the tables over every block, compaction only shrinks them)
static int upload_wg_blocks(mplbhip_ctx* c) {
    const size_t bytes = c->wg_block_host.size() * sizeof(int32_t);
    if (bytes > c->wg_block.bytes)
        return fail(c, MPLBHIP_ERR_HIP, "workgroup tables outgrew their buffer");
    if (bytes)
        HIPCHK(c, hipMemcpyAsync(c->wg_block.p, c->wg_block_host.data(), bytes,
                                 hipMemcpyHostToDevice, c->stream));
    // the host tables change at the next compaction: the copy must be done
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return 0;
}

int mplbhip_prepare(mplbhip_ctx* c) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (c->prepared) return fail(c, MPLBHIP_ERR_ARG, "case already prepared");
    if (c->plan.blocks.empty()) return fail(c, MPLBHIP_ERR_ARG, "no blocks defined");
    if (c->swap && (c->lat != 3 || c->thermal))
        return fail(c, MPLBHIP_ERR_UNSUPPORTED,
                    "the swap scheme has D3Q19 Collision_BGKIsothermal2nd_Swap kernels only "
                    "(scheme_kernel.inc:957-1398)");
    if (!c->plan.build()) return fail(c, MPLBHIP_ERR_UNSUPPORTED, "%s", c->plan.error.c_str());
    // HBM layout: one halo node per axis, x = 0 and every row aligned to a
    // 128-byte cache line, so a wave's 64-node row segment spans whole lines
    const int nb = (int)c->plan.blocks.size();
    const int hz = c->dim == 3 ? 1 : 0;
    const int align = (int)(128 / c->es);
    c->bp.assign(nb, BlockParams{});
    c->elem0.assign(1, 0);
    int64_t off = 0, moff = 0;
    c->segs.clear();
    // measured at 256^3: folding the x faces pays for 4- and 8-byte
    // populations; with 2-byte ones the extra lanes cost more than the
    // strided boundary loads.  The first step's autotuning decides for
    // large cases.
    c->fold = c->storage != MPLBHIP_STORE_F16 ? 1 : 0;
    if (const char* e = std::getenv("MPLBHIP_XFACE_FOLD")) {
        c->fold = std::min(c->dim == 3 ? 3 : 2, std::max(0, std::atoi(e)));
        c->fold_env = true;
    }
    if (const char* e = std::getenv("MPLBHIP_XCD_REMAP")) c->xcd_remap = std::atoi(e) != 0;
    for (int b = 0; b < nb; b++) {
        const int* n = c->plan.blocks[b].n;
        BlockParams& B = c->bp[b];
        std::memset(&B, 0, sizeof B);
        for (int a = 0; a < 3; a++) B.n[a] = n[a];
        // z-slab interleaved populations: element (q, x, y, z) at
        // base + z*sz + q*sq + y*sx + x with sq = one padded xy plane and
        // sz = Q planes, so the Q streams of a z plane share one
        // contiguous slab (fewer DRAM pages and TLB entries per wave than
        // Q whole-lattice arrays)
        const int ox = align;
        int64_t row = (int64_t)ox + n[0] + 1;
        // FP16: the two-node bulk kernel's lanes load x0 - 1 .. x0 + 2 over
        // whole 128-node tiles; keep all of that inside the row
        if (c->storage == MPLBHIP_STORE_F16)
            row = std::max<int64_t>(row, (int64_t)ox + 2 * kTX * ((n[0] + 2 * kTX - 1) / (2 * kTX)) + 2);
        const int64_t sx = (row + align - 1) / align * align;
        const int64_t sq = sx * (n[1] + 2);
        const int64_t sz = sq * c->Q;
        const int64_t elems = sz * (n[2] + 2 * hz);
        if (elems >= (1LL << 31) || elems * (int64_t)c->es >= (1LL << 32))
            return fail(c, MPLBHIP_ERR_UNSUPPORTED,
                        "block %d too large for 32-bit node offsets", b);
        B.sx = (int32_t)sx;
        B.sz = (int32_t)sz;
        B.sq = (int32_t)sq;
        B.base = off + hz * sz + sx + ox;
        off += (elems + 255) / 256 * 256;
        c->elem0.push_back(off);
        {
            const int (*cv)[3] = lattice_tab(c->lat).C;
            const int64_t shift = (c->dim == 3 ? sz : 0) + sx + 1;
            B.pull_shift = (int32_t)shift;
            for (int q = 0; q < c->Q; q++) {
                const int64_t delta = cv[q][0] + cv[q][1] * sx + cv[q][2] * sz;
                const int64_t pull = (q * sq - delta + shift) * (int64_t)c->es;
                const int64_t put = q * sq * (int64_t)c->es;
                // the lane offset (below elems * es) plus the scalar one stays
                // below 4 GiB, so no 32-bit offset sum can wrap
                if (pull < 0 || pull + elems * (int64_t)c->es >= (1LL << 32) ||
                    put + elems * (int64_t)c->es >= (1LL << 32))
                    return fail(c, MPLBHIP_ERR_UNSUPPORTED,
                                "block %d too large for 32-bit population offsets", b);
                B.pull_off[q] = (uint32_t)pull;
                B.put_off[q] = (uint32_t)put;
            }
        }
        B.tiles_x = (n[0] + kTX - 1) / kTX;
        B.tiles_y = (n[1] + kTY - 1) / kTY;
        B.tiles_x2 = (n[0] + 2 * kTX - 1) / (2 * kTX);
        const int32_t divisors[4] = {B.tiles_x, B.tiles_y, (int32_t)n[1], B.tiles_x / kTY};
        for (int k = 0; k < 4; k++) fast_div_params(divisors[k], &B.div_m[k], &B.div_sh[k]);
        // the step's split: bulk tiles over z = 1 .. n-2 (3D; every z plane
        // at fold level 3), and the boundary regions as segments, 256 nodes
        // per workgroup, in four lists: [0] every boundary region, [1]
        // without the simple x-face interiors, [2] without every simple
        // region of the planes z = 1 .. n-2, [3] without every simple region
        // (the bulk kernel runs those inline at that fold level)
        for (int v = 0; v < 4; v++) {
            B.seg_start[v] = (int)c->segs.size();
            int count = 0;
            for (int r = 1; r < c->plan.nregions; r++) {
                const int code[3] = {r % 3, (r / 3) % 3, r / 9};
                const bool simple = c->plan.progs[(size_t)b * c->plan.nregions + r].simple;
                if (v == 1 && r < 3 && simple) continue;
                // every region in 2D; rz = 0, i.e. r < 9, in 3D
                if (v == 2 && (c->dim == 2 || r < 9) && simple) continue;
                if (v == 3 && simple) continue;
                BndSeg S;
                for (int a = 0; a < 3; a++) {
                    if (a == 2 && c->dim == 2) {
                        S.org[a] = 0;
                        S.ext[a] = 1;
                    } else {
                        S.org[a] = code[a] == 0 ? 1 : code[a] == 1 ? 0 : n[a] - 1;
                        S.ext[a] = code[a] == 0 ? n[a] - 2 : 1;
                    }
                }
                // every segment starts on a workgroup boundary, so a
                // workgroup's lanes share one region program
                S.start = count;
                S.count = S.ext[0] * S.ext[1] * S.ext[2];
                if (S.count <= 0) continue;
                count += (S.count + kBndWG - 1) / kBndWG * kBndWG;
                c->segs.push_back(S);
            }
            B.seg_count[v] = (int)c->segs.size() - B.seg_start[v];
        }
        B.prog_base = b * c->plan.nregions;
        B.mbase = moff;
        B.fbase = moff * c->Q;
        moff += (int64_t)n[0] * n[1] * n[2];
        B.active = 1;
    }
    c->total_elems = off;
    c->interior_nodes = moff;
    // workgroup ranges of every launch form
    const int grouped = assign_tiles(c, false);
    c->xgroup = grouped > 0 ? 1 : 0;
    c->xgroup_ok = c->xgroup;
    c->rowwg_ok = false;
    for (const BlockParams& B : c->bp) c->rowwg_ok = c->rowwg_ok || B.rowwg;
    // below a quarter million nodes a step is launch-bound: one launch
    c->fused = c->interior_nodes < (1 << 18);
    if (const char* e = std::getenv("MPLBHIP_FUSED")) {
        c->fused = std::atoi(e) != 0;
        c->fused_env = true;
    }
    c->fused_full = c->fused;
    if (const char* e = std::getenv("MPLBHIP_BATCH_COMPACT")) c->batch_compact = std::atoi(e) != 0;
    if (const char* e = std::getenv("MPLBHIP_XGROUP")) {
        const int v = std::atoi(e);
        if (v == 0) c->xgroup = 0;
        if (v == 2 && c->rowwg_ok) c->xgroup = 2;
        c->xgroup_env = true;
    }
    if (int rc = setup_halos(c)) return rc;
    if (const char* e = std::getenv("MPLBHIP_OVERLAP")) {
        c->overlap = std::atoi(e) != 0;
        c->overlap_env = true;
    }
    if (int rc = build_obstacles(c)) return rc;
    if (c->swap && !c->obst.empty())
        return fail(c, MPLBHIP_ERR_UNSUPPORTED, "obstacles are not supported by the swap scheme");
    // the two-node FP16 kernel has no obstacle path
    c->h2_ok = c->storage == MPLBHIP_STORE_F16 && c->obst.empty() && c->lat != 15;
    c->h2 = c->h2_ok;
    if (const char* e = std::getenv("MPLBHIP_H2")) {
        c->h2 = c->h2_ok && std::atoi(e) != 0;
        c->h2_env = true;
    }
    c->prepared = true;
    if (c->device < 0) return 0;
    HIPCHK(c, hipSetDevice(c->device));
    const size_t tbytes = (size_t)c->total_elems * c->es;
    const size_t tsz = c->storage == MPLBHIP_STORE_F64 ? 8 : 4;
    for (int i = 0; i < 2; i++) {
        if (int rc = dalloc(c, c->fs[i], tbytes)) return rc;
        if (int rc = dalloc(c, c->per[i],
                            std::max<size_t>(64, c->plan.persist_total * c->Q * tsz)))
            return rc;
        HIPCHK(c, launch_fill(c->fs[i].p, (int64_t)tbytes, c->stream));
        HIPCHK(c, launch_fill(c->per[i].p, (int64_t)c->per[i].bytes, c->stream));
    }
    for (int v = 0; v < 4; v++) {
        const size_t mb = (size_t)c->interior_nodes * sizeof(double);
        if (int rc = dalloc(c, c->macro[v], mb)) return rc;
        if (int rc = dalloc(c, c->macro_copy[v], mb)) return rc;
        HIPCHK(c, launch_fill(c->macro[v].p, (int64_t)mb, c->stream));
        HIPCHK(c, launch_fill(c->macro_copy[v].p, (int64_t)mb, c->stream));
    }
    if (c->thermal)
        if (int rc = dalloc(c, c->temp, (size_t)c->interior_nodes * sizeof(double))) return rc;
    if (int rc = dalloc(c, c->progs, c->plan.progs.size() * sizeof(RegionProg))) return rc;
    HIPCHK(c, hipMemcpyAsync(c->progs.p, c->plan.progs.data(), c->progs.bytes,
                             hipMemcpyHostToDevice, c->stream));
    if (int rc = dalloc(c, c->blocks, nb * sizeof(BlockParams))) return rc;
    if (!c->obst.empty()) {
        if (int rc = dalloc(c, c->dobst, c->obst.size() * sizeof(uint32_t))) return rc;
        HIPCHK(c, hipMemcpyAsync(c->dobst.p, c->obst.data(), c->dobst.bytes,
                                 hipMemcpyHostToDevice, c->stream));
    }
    // partial slots of the launches over every block (compaction only shrinks them)
    const size_t nslots = (size_t)std::max(
        c->ntiles, std::max(c->nbulk + std::max(c->nbnd_v[0], std::max(c->nbnd_v[1], c->nbnd_v[2])),
                            c->nbulk3 + c->nbnd_v[3]));
    if (int rc = dalloc(c, c->partials, nslots * kNAcc * sizeof(double))) return rc;
    if (int rc = dalloc(c, c->dsegs, std::max<size_t>(1, c->segs.size()) * sizeof(BndSeg)))
        return rc;
    if (int rc = dalloc(c, c->wg_block,
                        std::max<size_t>(1, c->wg_block_host.size()) * sizeof(int32_t)))
        return rc;
    if (int rc = upload_wg_blocks(c)) return rc;
    if (!c->segs.empty())
        HIPCHK(c, hipMemcpyAsync(c->dsegs.p, c->segs.data(), c->segs.size() * sizeof(BndSeg),
                                 hipMemcpyHostToDevice, c->stream));
    if (int rc = dalloc(c, c->red, (size_t)(nb + 1) * kNAcc * sizeof(double))) return rc;
    for (int i = 0; i < 2; i++) {
        if (int rc = dalloc(c, c->parity[i], (size_t)std::max(nb, 16) * sizeof(int32_t)))
            return rc;
        HIPCHK(c, launch_fill(c->parity[i].p, (int64_t)c->parity[i].bytes, c->stream));
    }
    if (int rc = upload_blocks(c)) return rc;
    if (int rc = upload_merged_halos(c)) return rc;
    // a single-step form chosen by the environment is the one that runs
    if (int rc = assign_swap(c)) return rc;
    c->pair_ok = pair_allowed(c);
    c->pair_env = c->fused_env || c->fold_env || c->xgroup_env || c->h2_env || c->xcd_remap ? -1 : 0;
    if (const char* e = std::getenv("MPLBHIP_PAIR")) c->pair_env = std::atoi(e) > 0 ? std::atoi(e) : -1;
    if (int rc = assign_pairs(c, false)) return rc;
    c->march_ok = march_allowed(c);
    c->tile_ok = tile_allowed(c);
    if (int rc = assign_2d(c, false)) return rc;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return 0;
}

int mplbhip_node_info(mplbhip_ctx* c, int block, int which, int* out) {
    if (!c || !out) return MPLBHIP_ERR_ARG;
    if (!c->prepared) return fail(c, MPLBHIP_ERR_ARG, "call mplbhip_prepare first");
    if (block < 0 || block >= (int)c->plan.blocks.size())
        return fail(c, MPLBHIP_ERR_ARG, "undefined block");
    if (which < 0 || which > 3) return fail(c, MPLBHIP_ERR_ARG, "which must be 0 .. 3");
    const int* n = c->plan.blocks[block].n;
    const int R = c->plan.nregions;
    size_t p = 0;
    for (int k = 0; k < n[2]; k++)
        for (int j = 0; j < n[1]; j++)
            for (int i = 0; i < n[0]; i++) {
                const int r = c->plan.region_of(block, i, j, k);
                const bool obst = !c->obst.empty() &&
                                  (c->obst[(size_t)c->bp[block].mbase + p] & kObstSolid);
                const RegionProg& P = c->plan.progs[(size_t)block * R + r];
                if (which == 0)
                    out[p] = obst ? (int)VT_ImmersedSolid : c->plan.region_vt[(size_t)block * R + r];
                else if (which == 1)
                    out[p] = c->plan.region_vg[(size_t)block * R + r];
                else if (which == 2)
                    out[p] = P.simple;
                else
                    out[p] = (int)P.adj;
                p++;
            }
    return 0;
}

int mplbhip_set_macros(mplbhip_ctx* c, int block, const double* rho,
                       const double* u, const double* v, const double* w) {
    if (!c || !rho || !u || !v || (c->dim == 3 && !w)) return MPLBHIP_ERR_ARG;
    if (int rc = need_device(c)) return rc;
    if (!c->prepared) return fail(c, MPLBHIP_ERR_ARG, "call mplbhip_prepare first");
    if (block < 0 || block >= (int)c->bp.size())
        return fail(c, MPLBHIP_ERR_ARG, "undefined block");
    const BlockParams& B = c->bp[block];
    const size_t nn = (size_t)B.n[0] * B.n[1] * B.n[2];
    const double* src[4] = {rho, u, v, w};
    for (int var = 0; var < 1 + c->dim; var++) {
        double* dst = static_cast<double*>(c->macro[var].p) + B.mbase;
        HIPCHK(c, hipMemcpyAsync(dst, src[var], nn * sizeof(double),
                                 hipMemcpyHostToDevice, c->stream));
        double* dc = static_cast<double*>(c->macro_copy[var].p) + B.mbase;
        HIPCHK(c, hipMemcpyAsync(dc, src[var], nn * sizeof(double),
                                 hipMemcpyHostToDevice, c->stream));
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return 0;
}

int mplbhip_init_feq(mplbhip_ctx* c) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (int rc = need_device(c)) return rc;
    if (!c->prepared) return fail(c, MPLBHIP_ERR_ARG, "call mplbhip_prepare first");
    drop_graphs(c);
    c->cur = 0;
    c->tstep = 0;
    c->init_from_f = false;
    c->init_lift = false;
    c->initialized = true;
    c->swap_formed = false;
    // fStage^0 = collide(feq) is formed lazily at the first step, once the
    // time step is known (the Apps call SetTimeStep after this), from the
    // macros as they are now (PreDefinedInitialCondition reads them here,
    // model_wrapper.cpp:347-391)
    const size_t mb = (size_t)c->interior_nodes * sizeof(double);
    for (int v = 0; v < 4; v++) {
        if (c->macro0[v].bytes != mb)
            if (int rc = dalloc(c, c->macro0[v], mb)) return rc;
        HIPCHK(c, hipMemcpyAsync(c->macro0[v].p, c->macro[v].p, mb, hipMemcpyDeviceToDevice,
                                 c->stream));
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return 0;
}

int mplbhip_init_lift(mplbhip_ctx* c) {
    if (c && c->swap)
        return fail(c, MPLBHIP_ERR_UNSUPPORTED, "the swap scheme starts from feq or a given f");
    if (c && (c->lat == 15 || c->thermal))
        return fail(c, MPLBHIP_ERR_UNSUPPORTED,
                    "the lifted start is built for D2Q9/D3Q19 with the isothermal collision");
    if (int rc = mplbhip_init_feq(c)) return rc;
    c->init_lift = true;
    return 0;
}

int mplbhip_set_f(mplbhip_ctx* c, int block, const double* f) {
    if (!c || !f) return MPLBHIP_ERR_ARG;
    if (int rc = need_device(c)) return rc;
    if (!c->prepared) return fail(c, MPLBHIP_ERR_ARG, "call mplbhip_prepare first");
    if (block < 0 || block >= (int)c->bp.size())
        return fail(c, MPLBHIP_ERR_ARG, "undefined block");
    const BlockParams& B = c->bp[block];
    const size_t nn = (size_t)B.n[0] * B.n[1] * B.n[2];
    if (c->host_init_f.size() != (size_t)c->Q * c->interior_nodes)
        c->host_init_f.assign((size_t)c->Q * c->interior_nodes, 0.0);
    std::memcpy(c->host_init_f.data() + B.fbase, f, nn * c->Q * sizeof(double));
    drop_graphs(c);
    c->cur = 0;
    c->tstep = 0;
    c->init_from_f = true;
    c->init_lift = false;
    c->initialized = true;
    c->swap_formed = false;
    return 0;
}

int mplbhip_set_timestep(mplbhip_ctx* c, double dt) {
    if (!c) return MPLBHIP_ERR_ARG;
    c->dt = dt;
    if (c->prepared && c->device >= 0) {
        drop_graphs(c);
        return upload_blocks(c);
    }
    return 0;
}

int mplbhip_set_accel(mplbhip_ctx* c, int block, const double* g) {
    if (!c || !g) return MPLBHIP_ERR_ARG;
    if (block < 0 || block >= (int)c->accel.size())
        return fail(c, MPLBHIP_ERR_ARG, "undefined block");
    for (int d = 0; d < 3; d++) c->accel[block][d] = d < c->dim ? g[d] : 0.0;
    if (c->prepared && c->device >= 0) {
        drop_graphs(c);
        return upload_blocks(c);
    }
    return 0;
}

// Launch-configuration autotuning, once per context: which simple boundary
// regions the bulk kernel runs inline (none, the x faces, all of its grid's),
// and keeping a row's tiles on one XCD or not.  Each candidate runs the step
// kernels a few times from the current state into the other buffer, which
// holds the step before the latest, that macros and f are re-streamed from: a
// real single step has to follow, whose writes replace those.  Cases under
// 2^20 nodes keep the defaults (their steps are launch-bound).
static int autotune(mplbhip_ctx* c) {
    if (c->tuned) return 0;
    c->tuned = true;
    if (c->interior_nodes < (1 << 20)) return 0;
    std::vector<std::array<int, 3>> cand;  // fold, xgroup, h2
    std::vector<int> folds;
    if (c->fold_env) {
        folds = {c->fold};
    } else {
        folds = {0};
        if (c->nbnd_v[1] != c->nbnd_v[0]) folds.push_back(1);
        if (c->nbnd_v[2] != c->nbnd_v[1]) folds.push_back(2);
        if (c->dim == 3 && c->nbnd_v[3] != c->nbnd_v[2]) folds.push_back(3);
    }
    std::vector<int> groups;
    if (c->xgroup_env) {
        groups = {c->xgroup};
    } else {
        if (c->xgroup_ok) groups.push_back(1);
        groups.push_back(0);
        if (c->rowwg_ok) groups.push_back(2);
    }
    if (!(c->h2_env && c->h2))
        for (int f : folds)
            for (int g : groups) cand.push_back({f, g, 0});
    if (c->h2_ok && !(c->h2_env && !c->h2)) cand.push_back({0, 0, 1});
    if (cand.size() < 2) return 0;
    // three interleaved rounds of 5 dry steps per candidate; each keeps its
    // fastest round (clock and neighbour noise only ever add time)
    constexpr int kRounds = 3, kSteps = 5;
    std::vector<float> tmin(cand.size(), 1e30f);
    for (int r = 0; r < kRounds; r++)
        for (size_t i = 0; i < cand.size(); i++) {
            c->fold = cand[i][0];
            c->xgroup = cand[i][1];
            c->h2 = cand[i][2] != 0;
            KParams kp = base_params(c);
            if (int rc = launch_step_kernels(c, kp, MODE_STEP)) return rc;
            HIPCHK(c, hipEventRecord(c->ev[0], c->stream));
            for (int k = 0; k < kSteps; k++)
                if (int rc = launch_step_kernels(c, kp, MODE_STEP)) return rc;
            HIPCHK(c, hipEventRecord(c->ev[1], c->stream));
            HIPCHK(c, hipEventSynchronize(c->ev[1]));
            float ms = 0.f;
            HIPCHK(c, hipEventElapsedTime(&ms, c->ev[0], c->ev[1]));
            tmin[i] = std::min(tmin[i], ms / kSteps);
        }
    // the first candidate within 1% of the fastest: near-ties go to the
    // earlier (simpler) form, so repeated runs pick the same one
    const float fastest = *std::min_element(tmin.begin(), tmin.end());
    size_t ipick = 0;
    while (tmin[ipick] > 1.01f * fastest) ipick++;
    const std::array<int, 3> pick = cand[ipick];
    const float best = tmin[ipick];
    if (std::getenv("MPLBHIP_VERBOSE"))
        for (size_t i = 0; i < cand.size(); i++)
            std::fprintf(stderr, "mplbhip: autotune fold=%d xgroup=%d h2=%d: %.4f ms/step\n",
                         cand[i][0], cand[i][1], cand[i][2], tmin[i]);
    c->fold = pick[0];
    c->xgroup = pick[1];
    c->h2 = pick[2] != 0;
    drop_graphs(c);
    if (std::getenv("MPLBHIP_VERBOSE"))
        std::fprintf(stderr, "mplbhip: autotune picked fold=%d xgroup=%d h2=%d (%.4f ms/step)\n",
                     c->fold, c->xgroup, (int)c->h2, best);
    return 0;
}

// The tuning, ahead of a single step of the stream-collision scheme over every
// block: at once where single steps are what runs; beside launches of several
// steps, where single ones only end a run, from the 65th on.  period: a check
// step's, which counts if no launch of several steps fits before it (else one
// step in hundreds is single: at 256^3 tuning takes 0.1 s, for at most 0.02 ms
// of each).
static int tune_single(mplbhip_ctx* c, int period = 0) {
    if (c->tuned || c->swap || c->grid_nodes != c->interior_nodes) return 0;
    const int ls = launch_steps(c);
    if (ls > 1 && (period > ls || ++c->singles <= 64)) return 0;
    return autotune(c);
}

// the swap scheme's f^0 in its one lattice: feq of the initial macros, or
// the f given by mplbhip_set_f; the halos start at zero like a new dat
static int swap_form(mplbhip_ctx* c) {
    if (c->swap_formed) return 0;
    HIPCHK(c, hipSetDevice(c->device));
    HIPCHK(c, launch_fill(c->fs[0].p, (int64_t)c->fs[0].bytes, c->stream));
    KParams kp = base_params(c);
    if (c->init_from_f) {
        const size_t fbytes = (size_t)c->Q * c->interior_nodes * sizeof(double);
        if (c->fhost.bytes != fbytes)
            if (int rc = dalloc(c, c->fhost, fbytes)) return rc;
        HIPCHK(c, hipMemcpyAsync(c->fhost.p, c->host_init_f.data(), fbytes,
                                 hipMemcpyHostToDevice, c->stream));
        kp.fhost = static_cast<double*>(c->fhost.p);
        kp.fhost_in = 1;
    }
    HIPCHK(c, launch_swap(4, kp, 0, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    c->swap_formed = true;
    return 0;
}

// the collision of f^0 happens here, with the time step then in force
static int first_collision(mplbhip_ctx* c) {
    if (c->swap) return swap_form(c);
    if (c->thermal && !c->temp_set)
        return fail(c, MPLBHIP_ERR_ARG,
                    "Collision_BGKThermal4th reads Variable_T: call mplbhip_set_temperature");
    // every block starts from buffer 0
    for (int i = 0; i < 2; i++)
        HIPCHK(c, launch_fill(c->parity[i].p, (int64_t)c->parity[i].bytes, c->stream));
    c->cur = 0;
    c->halo_stale = false;
    KParams kp = base_params(c);
    int mode = MODE_INIT_FEQ;
    if (c->init_from_f) {
        const size_t fbytes = (size_t)c->Q * c->interior_nodes * sizeof(double);
        if (c->fhost.bytes != fbytes)
            if (int rc = dalloc(c, c->fhost, fbytes)) return rc;
        HIPCHK(c, hipMemcpyAsync(c->fhost.p, c->host_init_f.data(), fbytes,
                                 hipMemcpyHostToDevice, c->stream));
        kp.fhost = static_cast<double*>(c->fhost.p);
        mode = MODE_INIT_F;
    } else if (c->init_lift) {
        const size_t fbytes = (size_t)c->Q * c->interior_nodes * sizeof(double);
        if (c->fhost.bytes != fbytes)
            if (int rc = dalloc(c, c->fhost, fbytes)) return rc;
        kp.fhost = static_cast<double*>(c->fhost.p);
        HIPCHK(c, launch_lift(c->dim, kp, c->interior_nodes, c->stream));
        mode = MODE_INIT_F;
    }
    HIPCHK(c, launch_lattice(c->lat, c->storage, mode, kp, c->stream));
    if (int rc = exchange(c, 0)) return rc;
    // beside launches of several steps the single ones only end a run: not
    // tuned yet
    return launch_steps(c) > 1 ? 0 : autotune(c);
}

// the steps of a launch of several for which `left` of a run's steps are left,
// 1: a single step is next
static int next_launch(const mplbhip_ctx* c, int left) {
    const int ls = launch_steps(c);
    return left >= (c->tile ? 2 : ls) ? std::min(ls, left) : 1;
}

// The launches of mplbhip_step (without captured graphs, which cannot carry
// events), each step kernel between two events on the stream it runs on: a
// bulk and a boundary kernel each, any other launch as the bulk share.
static int timed_steps(mplbhip_ctx* c, int nsteps, double* ms_total, double* ms_kernel) {
    if (launch_steps(c) == 1 && nsteps > 0)
        if (int rc = tune_single(c)) return rc;
    std::vector<hipEvent_t> evs(4 * ((size_t)nsteps + 1));
    for (auto& e : evs) HIPCHK(c, hipEventCreate(&e));
    std::vector<char> split;  // per launch: a bulk and a boundary kernel
    auto bracket = [&](auto&& enqueue) -> int {
        hipEvent_t* ev = &evs[4 * split.size()];
        split.push_back(0);
        HIPCHK(c, hipEventRecord(ev[0], c->stream));
        if (int rc = enqueue()) return rc;
        HIPCHK(c, hipEventRecord(ev[1], c->stream));
        return 0;
    };
    HIPCHK(c, hipEventRecord(c->ev[0], c->stream));
    int left = nsteps;
    if (c->swap_pull && nsteps > 0) {
        if (int rc = bracket([&] { return swap_begin(c, nsteps); })) return rc;
        for (; left > 1; left--, c->tstep++)
            if (int rc = bracket([&] { return swap_pass(c, true); })) return rc;
        if (int rc = bracket([&] { return swap_end(c); })) return rc;
        left = 0;
        c->tstep++;
    }
    while (left > 0) {
        const int n = next_launch(c, left - 1);  // the last step is a single one
        if (n > 1) {
            if (int rc = bracket([&] { return enqueue_multi(c, n); })) return rc;
        } else if (c->swap) {
            if (int rc = bracket([&] { return enqueue_swap_step(c, false, false); })) return rc;
        } else {
            if (int rc = fresh_halos(c)) return rc;
            const KParams kp = base_params(c);
            if (kp.fused) {
                if (int rc = bracket([&]() -> int {
                        HIPCHK(c, launch_lattice(c->lat, c->storage, MODE_STEP, kp, c->stream));
                        return 0;
                    }))
                    return rc;
            } else {
                split.push_back(1);
                if (int rc = launch_step_kernels(c, kp, MODE_STEP, &evs[4 * (split.size() - 1)]))
                    return rc;
            }
            if (int rc = exchange(c, 1 - c->cur)) return rc;
            c->cur ^= 1;
        }
        c->tstep += n;
        left -= n;
    }
    HIPCHK(c, hipEventRecord(c->ev[1], c->stream));
    HIPCHK(c, hipEventSynchronize(c->ev[1]));
    float ms = 0.f;
    HIPCHK(c, hipEventElapsedTime(&ms, c->ev[0], c->ev[1]));
    if (ms_total) *ms_total = ms;
    c->last_bulk_ms = c->last_bnd_ms = 0.0;
    for (size_t l = 0; l < split.size(); l++) {
        HIPCHK(c, hipEventElapsedTime(&ms, evs[4 * l], evs[4 * l + 1]));
        c->last_bulk_ms += ms;
        if (!split[l]) continue;
        HIPCHK(c, hipEventElapsedTime(&ms, evs[4 * l + 2], evs[4 * l + 3]));
        c->last_bnd_ms += ms;
    }
    for (auto& e : evs) (void)hipEventDestroy(e);
    if (ms_kernel) *ms_kernel = c->last_bulk_ms + c->last_bnd_ms;
    return 0;
}

// tail: a check step follows, so the last step need not be a single one
static int run_steps(mplbhip_ctx* c, int nsteps, bool timed, double* ms_total,
                     double* ms_kernel, bool tail = false) {
    if (int rc = need_device(c)) return rc;
    if (int rc = ensure_init(c)) return rc;
    if (nsteps < 0) return fail(c, MPLBHIP_ERR_ARG, "negative step count");
    HIPCHK(c, hipSetDevice(c->device));
    c->swap_run = false;
    if (c->tstep == 0)
        if (int rc = first_collision(c)) return rc;
    if (timed) return timed_steps(c, nsteps, ms_total, ms_kernel);
    // untimed: replay captured graphs of G steps (even, so the parity after
    // a graph of single steps is unchanged; MPLBHIP_GRAPH_STEPS overrides),
    // the remainder launch by launch.  32 steps, or 16 launches of several:
    // replaying a graph costs some 10 us more than its launches one by one,
    // which a run of fewer than 16 takes as fast (2D cavity 128^2, FP64, 100
    // steps between checks: 1,000 steps in 2.18 ms with graphs of 4 launches,
    // 2.09 of 8, 2.11 of 16, that is none).
    const int ls = launch_steps(c);
    if (ls == 1 && nsteps > 0)
        if (int rc = tune_single(c)) return rc;
    int G = std::max(32, 16 * ls);
    if (const char* e = std::getenv("MPLBHIP_GRAPH_STEPS")) {
        const int g = std::atoi(e);
        if (g >= 2 && g <= 1024 && g % 2 == 0) G = g;
    }
    int left = nsteps;
    const bool pull = c->swap_pull && left > 0;
    if (pull) {
        if (int rc = swap_begin(c, left)) return rc;
        left--;
    }
    // launches of several steps leave the last step to a single one
    const int keep = ls > 1 && !tail ? 1 : 0;
    G -= G % ls;  // whole launches
    if (G > 0 && left - keep >= G) {
        if (c->graph_steps != G)
            if (int rc = build_graphs(c, G)) return rc;
        while (left - keep >= G) {
            HIPCHK(c, hipGraphLaunch(c->gexec[c->cur], c->stream));
            // every launch flips the parity
            if ((G / ls) % 2) c->cur ^= 1;
            c->halo_stale = ls > 1 && !c->halos.empty();
            c->tstep += G;
            left -= G;
        }
    }
    while (ls > 1) {
        const int n = next_launch(c, left - keep);
        if (n == 1) break;
        if (int rc = enqueue_multi(c, n)) return rc;
        c->tstep += n;
        left -= n;
    }
    while (left > 0) {
        if (int rc = tune_single(c)) return rc;
        if (int rc = enqueue_step(c, false, false)) return rc;
        c->tstep++;
        left--;
    }
    if (pull) {
        if (int rc = swap_end(c)) return rc;
        c->tstep++;
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return 0;
}

int mplbhip_iterate(mplbhip_ctx* c, double criteria, int check_period,
                    long long max_steps, long long* steps_done, double* residual) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (int rc = need_device(c)) return rc;
    if (int rc = ensure_init(c)) return rc;
    if (check_period <= 0 || max_steps < 0)
        return fail(c, MPLBHIP_ERR_ARG, "bad check period or step limit");
    const bool converge = criteria >= 0;
    long long done = 0;
    double res = -1.0;
    while (done < max_steps) {
        // steps until the next check step (iteration counts from tstep)
        long long to_check = check_period - (c->tstep % check_period) - 1;
        long long plain = std::min<long long>(to_check, max_steps - done);
        while (plain > 0) {
            const int chunk = (int)std::min<long long>(plain, 1 << 20);
            if (int rc = run_steps(c, chunk, false, nullptr, nullptr,
                                   plain == chunk && done + chunk < max_steps))
                return rc;
            plain -= chunk;
            done += chunk;
        }
        if (done >= max_steps) break;
        if (c->tstep == 0)
            if (int rc = first_collision(c)) return rc;
        if (int rc = tune_single(c, check_period)) return rc;
        if (int rc = enqueue_step(c, true, converge)) return rc;
        c->tstep++;
        done++;
        if (converge) {
            double acc[kNAcc];
            HIPCHK(c, launch_reduce(static_cast<const double*>(c->partials.p),
                                    static_cast<const BlockParams*>(c->blocks.p),
                                    (int)c->bp.size(), c->ntiles, step_nbulk(c),
                                    c->nbnd_v[step_fold(c)], reduce_split(c),
                                    step_fold(c), static_cast<double*>(c->red.p), c->stream));
            HIPCHK(c, hipMemcpyAsync(acc, static_cast<double*>(c->red.p) +
                                              c->bp.size() * kNAcc,
                                     sizeof acc, hipMemcpyDeviceToHost, c->stream));
            HIPCHK(c, hipStreamSynchronize(c->stream));
            // CalcResidualError ratios, GetMaximumResidual (flowfield.cpp:148-158)
            double mx = 0.0;
            for (int v = 0; v < 1 + c->dim; v++) {
                c->last_ratio[v] = acc[v] / acc[4 + v];
                const double rel = c->last_ratio[v] / (check_period * c->dt);
                if (mx <= rel) mx = rel;
            }
            res = mx;
            c->last_max = mx;
            if (!(res >= criteria)) break;
        }
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (steps_done) *steps_done = done;
    if (residual) *residual = res;
    return 0;
}

int mplbhip_define_block_collision(mplbhip_ctx* c, int block, double tau_ref, double dt) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (block < 0 || block >= (int)c->btau.size())
        return fail(c, MPLBHIP_ERR_ARG, "undefined block %d", block);
    if (!(dt > 0) || !(tau_ref > 0))
        return fail(c, MPLBHIP_ERR_ARG, "tau and dt must be positive");
    c->btau[block] = tau_ref;
    c->bdt[block] = dt;
    if (c->prepared && c->device >= 0) {
        drop_graphs(c);
        return upload_blocks(c);
    }
    return 0;
}

// Shrink the step launches to the active blocks (on) or restore them to
// every block (off).  Blocks outside the launches carry no parity forward,
// so both parity arrays first take the current parities; the launches'
// grids change, so captured graphs go.  The caller uploads c->bp.
static int compact_grid(mplbhip_ctx* c, bool on) {
    const size_t nb = c->bp.size();
    if (on)
        HIPCHK(c, hipMemcpyAsync(c->parity[1 - c->cur].p, c->parity[c->cur].p,
                                 nb * sizeof(int32_t), hipMemcpyDeviceToDevice, c->stream));
    assign_tiles(c, on);
    if (int rc = upload_wg_blocks(c)) return rc;
    // a small remainder runs as one launch per step, as small cases do
    c->fused = c->fused_env ? c->fused_full
                            : (on ? c->grid_nodes < (1 << 18) : c->fused_full);
    drop_graphs(c);
    if (int rc = assign_pairs(c, on)) return rc;
    return assign_2d(c, on);
}

// Restart the listed blocks at rest, as a rest start forms its first
// fStage: macros (and residual copies) rho = 1, u = 0, then an INIT_FEQ
// launch in which only these blocks are active.  INIT_FEQ rewrites each
// node's latest fStage in place from its own macros, so the parities stay.
// The caller re-uploads the block parameters afterwards.
static int restart_at_rest(mplbhip_ctx* c, const std::vector<int>& blocks) {
    KParams kp = base_params(c);
    // the restarted blocks start from the rest macros just written
    for (int v = 0; v < 4; v++) kp.macro0[v] = nullptr;
    for (int b : blocks) {
        const BlockParams& B = c->bp[b];
        HIPCHK(c, launch_rest_macros(kp, b, (int64_t)B.n[0] * B.n[1] * B.n[2], c->stream));
    }
    c->restart_bp = c->bp;
    for (auto& B : c->restart_bp) B.active = 0;
    for (int b : blocks) c->restart_bp[b].active = 1;
    HIPCHK(c, hipMemcpyAsync(c->blocks.p, c->restart_bp.data(),
                             c->restart_bp.size() * sizeof(BlockParams), hipMemcpyHostToDevice,
                             c->stream));
    HIPCHK(c, launch_lattice(c->lat, c->storage, MODE_INIT_FEQ, kp, c->stream));
    // the host copy must outlive the upload
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return 0;
}

// Bring every block to the buffer c->cur.  A frozen instance keeps its parity
// while the launches go on, and the halo copies take one buffer for every
// block (exchange), so an instance that stopped an odd number of launches
// before the others has its two buffers exchanged, whole: halos, the step
// before the latest, kept boundary populations.
static int align_parity(mplbhip_ctx* c) {
    const size_t nb = c->bp.size();
    std::vector<int32_t> par(nb);
    HIPCHK(c, hipMemcpyAsync(par.data(), c->parity[c->cur].p, nb * sizeof(int32_t),
                             hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    const size_t slot = c->Q * (c->storage == MPLBHIP_STORE_F64 ? 8 : 4);
    auto exchange = [&](DevBuf* pair, size_t at, size_t bytes) {
        return launch_exchange(static_cast<char*>(pair[0].p) + at,
                               static_cast<char*>(pair[1].p) + at, (int64_t)bytes, c->stream);
    };
    for (size_t b = 0; b < nb; b++) {
        if (par[b] == c->cur) continue;
        HIPCHK(c, exchange(c->fs, c->elem0[b] * c->es, (c->elem0[b + 1] - c->elem0[b]) * c->es));
        for (int r = 1; r < c->plan.nregions; r++) {
            const size_t i = b * c->plan.nregions + r;
            if (c->plan.progs[i].persist >= 0)
                HIPCHK(c, exchange(c->per, c->plan.progs[i].persist * slot,
                                   c->plan.persist_nodes[i] * slot));
        }
        par[b] = c->cur;
    }
    HIPCHK(c, hipMemcpyAsync(c->parity[c->cur].p, par.data(), nb * sizeof(int32_t),
                             hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return 0;
}

int mplbhip_iterate_batch(mplbhip_ctx* c, double criteria, int check_period,
                          long long max_steps, long long* steps_b, double* res_b,
                          long long* steps_done) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (int rc = need_device(c)) return rc;
    if (int rc = ensure_init(c)) return rc;
    if (check_period <= 0 || max_steps < 0 || criteria < 0)
        return fail(c, MPLBHIP_ERR_ARG, "bad criteria, check period or step limit");
    if (c->restart_factor > 0 && c->plan.persist_total > 0)
        return fail(c, MPLBHIP_ERR_UNSUPPORTED,
                    "instances with persisted boundary state cannot restart at rest");
    if (c->restart_factor > 0 && !c->plan.links.empty())
        return fail(c, MPLBHIP_ERR_UNSUPPORTED,
                    "instances with block connections cannot restart at rest");
    if (c->swap)
        return fail(c, MPLBHIP_ERR_UNSUPPORTED, "batched instances run the stream-collision scheme");
    const int nb = (int)c->bp.size();
    // instances: the blocks joined by connections (a periodic channel's
    // self-linked block, or several linked blocks) converge and freeze
    // together; each instance's blocks share one time step
    std::vector<int> root(nb);
    for (int b = 0; b < nb; b++) root[b] = b;
    auto find = [&](int b) {
        while (root[b] != b) b = root[b] = root[root[b]];
        return b;
    };
    for (const LinkDesc& l : c->plan.links) root[find(l.from)] = find(l.to);
    std::vector<std::vector<int>> inst_blocks(nb);
    for (int b = 0; b < nb; b++) inst_blocks[find(b)].push_back(b);
    for (int r = 0; r < nb; r++)
        for (int b : inst_blocks[r])
            if (c->bp[b].dt != c->bp[inst_blocks[r][0]].dt)
                return fail(c, MPLBHIP_ERR_ARG,
                            "linked blocks %d and %d have different time steps", b,
                            inst_blocks[r][0]);
    std::vector<long long> conv(nb, -1);
    std::vector<double> res(nb, -1.0);
    std::vector<double> minres(nb, INFINITY);
    c->batch_restarts.assign(nb, 0);
    for (int b = 0; b < nb; b++) c->bp[b].active = 1;
    if (int rc = upload_blocks(c)) return rc;
    long long done = 0;
    int remaining = nb;
    std::vector<double> acc((size_t)(nb + 1) * kNAcc);
    // MPLBHIP_VERBOSE=2: one line per check (time step, live instances and
    // nodes, wall milliseconds since the previous check)
    const char* verbose = std::getenv("MPLBHIP_VERBOSE");
    const bool trace = verbose && std::atoi(verbose) >= 2;
    auto t_last = std::chrono::steady_clock::now();
    while (done < max_steps && remaining > 0) {
        long long to_check = check_period - (c->tstep % check_period) - 1;
        long long plain = std::min<long long>(to_check, max_steps - done);
        while (plain > 0) {
            const int chunk = (int)std::min<long long>(plain, 1 << 20);
            if (int rc = run_steps(c, chunk, false, nullptr, nullptr,
                                   plain == chunk && done + chunk < max_steps))
                return rc;
            plain -= chunk;
            done += chunk;
        }
        if (done >= max_steps) break;
        if (c->tstep == 0)
            if (int rc = first_collision(c)) return rc;
        if (int rc = tune_single(c, check_period)) return rc;
        if (int rc = enqueue_step(c, true, true)) return rc;
        c->tstep++;
        done++;
        HIPCHK(c, launch_reduce(static_cast<const double*>(c->partials.p),
                                static_cast<const BlockParams*>(c->blocks.p), nb,
                                c->ntiles, step_nbulk(c), c->nbnd_v[step_fold(c)],
                                c->fused ? 0 : 1, step_fold(c),
                                static_cast<double*>(c->red.p), c->stream));
        HIPCHK(c, hipMemcpyAsync(acc.data(), c->red.p, acc.size() * sizeof(double),
                                 hipMemcpyDeviceToHost, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
        bool changed = false, linked_frozen = false;
        std::vector<int> restart;
        for (int b = 0; b < nb; b++) {
            if (!c->bp[b].active || find(b) != b) continue;
            // the instance's sums over its blocks (CalcResidualError sums
            // over every block of a case, flowfield_wrapper.cpp:31-89)
            double a[kNAcc] = {0};
            for (int m : inst_blocks[b])
                for (int k = 0; k < kNAcc; k++) a[k] += acc[(size_t)m * kNAcc + k];
            double mx = 0.0;
            for (int v = 1; v < 1 + c->dim; v++) {
                const double rel = (a[v] / a[4 + v]) / (check_period * c->bp[b].dt);
                if (mx <= rel) mx = rel;
            }
            for (int m : inst_blocks[b]) res[m] = mx;
            // fallback: an instance whose residual climbs well above the
            // lowest it reached (or is no longer a number) restarts once at rest
            if (c->restart_factor > 0 && c->batch_restarts[b] == 0 &&
                !(mx <= c->restart_factor * minres[b])) {
                restart.push_back(b);
                c->batch_restarts[b]++;
                minres[b] = INFINITY;
                continue;
            }
            if (mx < minres[b]) minres[b] = mx;
            if (mx < criteria) {
                for (int m : inst_blocks[b]) {
                    c->bp[m].active = 0;
                    conv[m] = c->tstep;
                    remaining--;
                }
                changed = true;
                linked_frozen = linked_frozen || inst_blocks[b].size() > 1 || !c->halos.empty();
            }
        }
        // captured graphs hold the halo copies of the instances live when
        // they were captured: a frozen instance's links must drop out
        if (linked_frozen) drop_graphs(c);
        if (!restart.empty())
            if (int rc = restart_at_rest(c, restart)) return rc;
        if (changed && remaining > 0) {
            // compaction: once the launches cover a quarter more nodes than
            // the unconverged instances hold, they shrink to those
            int64_t live = 0;
            for (int b = 0; b < nb; b++)
                if (c->bp[b].active)
                    live += (int64_t)c->bp[b].n[0] * c->bp[b].n[1] * c->bp[b].n[2];
            if (c->batch_compact && c->grid_nodes > live + live / 4)
                if (int rc = compact_grid(c, true)) return rc;
        }
        if (changed || !restart.empty())
            HIPCHK(c, hipMemcpyAsync(c->blocks.p, c->bp.data(), nb * sizeof(BlockParams),
                                     hipMemcpyHostToDevice, c->stream));
        if (trace) {
            const auto now = std::chrono::steady_clock::now();
            std::fprintf(stderr, "mplbhip: check t=%lld live=%d grid_nodes=%lld fused=%d %.3f ms\n",
                         (long long)c->tstep, remaining, (long long)c->grid_nodes, (int)c->fused,
                         std::chrono::duration<double, std::milli>(now - t_last).count());
            t_last = now;
        }
    }
    // freezing lasts for this call only: later steps, macros and f reads
    // see every instance again
    bool frozen = false;
    for (int b = 0; b < nb; b++) {
        frozen = frozen || !c->bp[b].active;
        c->bp[b].active = 1;
    }
    if (c->grid_nodes != c->interior_nodes)
        if (int rc = compact_grid(c, false)) return rc;
    if (frozen)
        HIPCHK(c, hipMemcpyAsync(c->blocks.p, c->bp.data(), nb * sizeof(BlockParams),
                                 hipMemcpyHostToDevice, c->stream));
    if (frozen && !c->halos.empty())
        if (int rc = align_parity(c)) return rc;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (steps_b)
        for (int b = 0; b < nb; b++) steps_b[b] = conv[b];
    if (res_b)
        for (int b = 0; b < nb; b++) res_b[b] = res[b];
    if (steps_done) *steps_done = done;
    return 0;
}

int mplbhip_set_batch_restart(mplbhip_ctx* c, double factor) {
    if (!c || factor < 0) return MPLBHIP_ERR_ARG;
    if (factor > 0 && c->prepared && c->plan.persist_total > 0)
        return fail(c, MPLBHIP_ERR_UNSUPPORTED,
                    "instances with persisted boundary state cannot restart at rest");
    c->restart_factor = factor;
    return 0;
}

int mplbhip_batch_restarts(mplbhip_ctx* c, int* restarts) {
    if (!c || !restarts) return MPLBHIP_ERR_ARG;
    for (size_t b = 0; b < c->bp.size(); b++)
        restarts[b] = b < c->batch_restarts.size() ? c->batch_restarts[b] : 0;
    return 0;
}

int mplbhip_step(mplbhip_ctx* c, int nsteps) {
    if (!c) return MPLBHIP_ERR_ARG;
    return run_steps(c, nsteps, false, nullptr, nullptr);
}

int mplbhip_step_timed(mplbhip_ctx* c, int nsteps, double* ms_total, double* ms_kernel) {
    if (!c) return MPLBHIP_ERR_ARG;
    return run_steps(c, nsteps, true, ms_total, ms_kernel);
}

int mplbhip_kernel_times(mplbhip_ctx* c, double* ms_bulk, double* ms_boundary) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (ms_bulk) *ms_bulk = c->last_bulk_ms;
    if (ms_boundary) *ms_boundary = c->last_bnd_ms;
    return 0;
}

int mplbhip_launch_shape(mplbhip_ctx* c, int* fold, int* xgroup, int* h2,
                         long long* bulk_nodes) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (!c->prepared) return fail(c, MPLBHIP_ERR_ARG, "call mplbhip_prepare first");
    const int fl = step_fold(c);
    if (fold) *fold = fl;
    if (xgroup) *xgroup = c->xgroup;
    if (h2) *h2 = c->h2 ? 1 : 0;
    if (bulk_nodes) {
        // the bulk kernel's lanes: interior nodes of its planes, plus (fold
        // 1) the simple x-face regions or (fold 2) every simple region of
        // the planes z = 1 .. n-2 or (fold 3, 3D) every simple region, as in
        // its lane selection
        long long total = 0;
        for (size_t b = 0; b < c->bp.size(); b++) {
            const int* n = c->plan.blocks[b].n;
            const int rzmax = (c->dim == 3 && fl == 3) ? 3 : 1;
            for (int rz = 0; rz < rzmax; rz++)
                for (int ry = 0; ry < 3; ry++)
                    for (int rx = 0; rx < 3; rx++) {
                        const int r = rx + 3 * ry + 9 * rz;
                        const long long planes = c->dim == 3 ? (rz == 0 ? n[2] - 2 : 1) : 1;
                        const long long cnt = (long long)(rx == 0 ? n[0] - 2 : 1) *
                                              (ry == 0 ? n[1] - 2 : 1) * planes;
                        bool lane = r == 0;
                        if (!lane && fl > 0 && (fl >= 2 || (ry == 0 && rz == 0)))
                            lane = c->plan.progs[b * c->plan.nregions + r].simple != 0;
                        if (lane) total += cnt;
                    }
        }
        *bulk_nodes = total;
    }
    return 0;
}

int mplbhip_step_form(mplbhip_ctx* c, int* form, int* steps) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (int rc = need_device(c)) return rc;
    if (!c->prepared) return fail(c, MPLBHIP_ERR_ARG, "call mplbhip_prepare first");
    const int ls = launch_steps(c);
    if (form)
        *form = c->swap_pull ? MPLBHIP_FORM_SWAP
                : ls == 1    ? MPLBHIP_FORM_SINGLE
                : c->tile    ? MPLBHIP_FORM_TILE
                : c->pair    ? MPLBHIP_FORM_PAIR
                             : MPLBHIP_FORM_MARCH;
    if (steps) *steps = ls;
    return 0;
}

int mplbhip_update_macros(mplbhip_ctx* c) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (int rc = need_device(c)) return rc;
    return materialize(c, false, false, nullptr);
}

int mplbhip_get_f(mplbhip_ctx* c, int block, double* out) {
    if (!c || !out) return MPLBHIP_ERR_ARG;
    if (int rc = need_device(c)) return rc;
    if (block < 0 || block >= (int)c->bp.size())
        return fail(c, MPLBHIP_ERR_ARG, "undefined block");
    if (int rc = materialize(c, true, false, nullptr)) return rc;
    const BlockParams& B = c->bp[block];
    const size_t nn = (size_t)B.n[0] * B.n[1] * B.n[2];
    HIPCHK(c, hipMemcpy(out, static_cast<double*>(c->fhost.p) + B.fbase,
                        nn * c->Q * sizeof(double), hipMemcpyDeviceToHost));
    return 0;
}

int mplbhip_get_macro(mplbhip_ctx* c, int block, int var, double* out) {
    if (!c || !out) return MPLBHIP_ERR_ARG;
    if (int rc = need_device(c)) return rc;
    if (block < 0 || block >= (int)c->bp.size() || var < 0 || var > c->dim)
        return fail(c, MPLBHIP_ERR_ARG, "bad block or variable");
    const BlockParams& B = c->bp[block];
    const size_t nn = (size_t)B.n[0] * B.n[1] * B.n[2];
    HIPCHK(c, hipStreamSynchronize(c->stream));
    HIPCHK(c, hipMemcpy(out, static_cast<double*>(c->macro[var].p) + B.mbase,
                        nn * sizeof(double), hipMemcpyDeviceToHost));
    return 0;
}

int mplbhip_residual(mplbhip_ctx* c, int check_period, double* per_var, double* max) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (int rc = need_device(c)) return rc;
    if (check_period <= 0) return fail(c, MPLBHIP_ERR_ARG, "check period must be > 0");
    std::vector<double> acc;
    if (int rc = materialize(c, false, true, &acc)) return rc;
    const double* tot = acc.data() + c->bp.size() * kNAcc;
    double mx = 0.0;
    for (int v = 0; v < 1 + c->dim; v++) {
        c->last_ratio[v] = tot[v] / tot[4 + v];
        const double rel = c->last_ratio[v] / (check_period * c->dt);
        if (per_var) per_var[v] = c->last_ratio[v];
        if (mx <= rel) mx = rel;
    }
    c->last_max = mx;
    if (max) *max = mx;
    return 0;
}

int mplbhip_last_residual(mplbhip_ctx* c, double* per_var, double* max) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (per_var)
        for (int v = 0; v < 1 + c->dim; v++) per_var[v] = c->last_ratio[v];
    if (max) *max = c->last_max;
    return 0;
}

int mplbhip_mass(mplbhip_ctx* c, double* mass) {
    if (!c || !mass) return MPLBHIP_ERR_ARG;
    if (int rc = need_device(c)) return rc;
    std::vector<double> acc;
    if (int rc = materialize(c, false, false, &acc)) return rc;
    *mass = acc[c->bp.size() * kNAcc + 8];
    return 0;
}

int mplbhip_mass_noalloc(mplbhip_ctx* c, double* mass) {
    if (!c || !mass) return MPLBHIP_ERR_ARG;
    if (!c->prepared) return fail(c, MPLBHIP_ERR_ARG, "call mplbhip_prepare first");
    // the same launches and partial-sum slots as mplbhip_mass after the
    // first step: the bulk and boundary kernels, or the whole-lattice one
    const bool split = !c->swap && !c->fused;
    KParams kp = base_params(c);
    const long long slots = split ? (long long)kp.nbulk + kp.nbnd : (long long)c->ntiles;
    const long long need = (slots + (long long)c->bp.size() + 1) * kNAcc;
    if (need > kScratchDoubles)
        return fail(c, MPLBHIP_ERR_UNSUPPORTED,
                    "mplbhip_mass_noalloc: the case needs %lld doubles of scratch, the limit is "
                    "%lld (%lld workgroups of 256 nodes); use mplbhip_mass",
                    need, (long long)kScratchDoubles, slots);
    if (int rc = need_device(c)) return rc;
    if (int rc = ensure_init(c)) return rc;
    if (c->tstep == 0)
        return fail(c, MPLBHIP_ERR_ARG,
                    "mplbhip_mass_noalloc: no step taken yet (f^0 is formed on the device only "
                    "by the first step); use mplbhip_mass at t = 0");
    if (!c->scratch) return fail(c, MPLBHIP_ERR_HIP, "no scratch address for this device");
    HIPCHK(c, hipSetDevice(c->device));
    // every workgroup of the launches writes its partial slot and the block
    // sums overwrite theirs, so nothing needs clearing
    kp.partials = c->scratch;
    kp.fhost = nullptr;
    kp.want_residual = 0;
    if (c->swap) HIPCHK(c, launch_swap(5, kp, 0, c->stream));
    else if (split) HIPCHK(c, launch_materialize_split(c->lat, c->storage, kp, c->stream));
    else HIPCHK(c, launch_lattice(c->lat, c->storage, MODE_MATERIALIZE, kp, c->stream));
    double* out = c->scratch + (size_t)slots * kNAcc;
    HIPCHK(c, launch_reduce(c->scratch, static_cast<const BlockParams*>(c->blocks.p),
                            (int)c->bp.size(), c->ntiles, kp.nbulk, kp.nbnd, split ? 1 : 0,
                            kp.fold, out, c->stream));
    HIPCHK(c, hipMemcpyAsync(mass, out + c->bp.size() * kNAcc + 8, sizeof(double),
                             hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return 0;
}

int mplbhip_time_step(mplbhip_ctx* c, long long* step) {
    if (!c || !step) return MPLBHIP_ERR_ARG;
    *step = c->tstep;
    return 0;
}

int mplbhip_sync(mplbhip_ctx* c) {
    if (!c) return MPLBHIP_ERR_ARG;
    if (c->device < 0) return 0;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return 0;
}

int mplbhip_copy_probe(int device, long long nbytes, int iters,
                       double* ms_per_iter) {
    if (nbytes < 16 || iters < 1 || !ms_per_iter) return MPLBHIP_ERR_ARG;
    nbytes = nbytes / 16 * 16;
    if (hipSetDevice(device) != hipSuccess) return MPLBHIP_ERR_NODEVICE;
    void *a = nullptr, *b = nullptr;
    hipStream_t s = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = 0;
    if (hipMalloc(&a, nbytes) != hipSuccess || hipMalloc(&b, nbytes) != hipSuccess ||
        hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        rc = MPLBHIP_ERR_HIP;
    } else {
        (void)launch_fill(a, nbytes, s);
        (void)launch_copy(a, b, nbytes, s);  // warm up
        (void)hipEventRecord(e0, s);
        for (int i = 0; i < iters; i++) (void)launch_copy(a, b, nbytes, s);
        (void)hipEventRecord(e1, s);
        if (hipEventSynchronize(e1) != hipSuccess) {
            rc = MPLBHIP_ERR_HIP;
        } else {
            float ms = 0.f;
            (void)hipEventElapsedTime(&ms, e0, e1);
            *ms_per_iter = ms / iters;
        }
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (s) (void)hipStreamDestroy(s);
    if (a) (void)hipFree(a);
    if (b) (void)hipFree(b);
    return rc;
}

}  // extern "C"
