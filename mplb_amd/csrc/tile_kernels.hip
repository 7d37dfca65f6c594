// tile_kernels.hip -- several time steps per launch of 2D blocks: a workgroup
// holds a tile of the lattice, grown by a node per step on every side, in LDS
// and steps it there.
#include "lattice_device.hpp"

namespace mplbhip {


// the wall-velocity terms of the block's regions
template <typename T> struct TileWalls {
    T c[9][9];  // BCOp::cq (or eq_c)
    T den[9];   // BCOp::den (or eq_k)
    T win[9];   // BCOp::eq_win
    uint32_t in[9];  // wall_in, 0: the region applies none
    int32_t force[9];
};

// a population as the next step reads it (rounded to storage)
template <int ST> struct TileSink {
    using T = typename Store<ST>::T;
    T* h;
    const float* scale;
    __device__ __forceinline__ void operator()(int q, T v) const {
        if constexpr (ST == MPLBHIP_STORE_F16) h[q] = h2f_scaled(__float2half_rn(v), scale[q]);
        else h[q] = v;
    }
};

constexpr uint32_t kWallIn[9] = {0u,           wall_in<2>(1), wall_in<2>(2),
                                 wall_in<2>(3), wall_in<2>(4), wall_in<2>(5),
                                 wall_in<2>(6), wall_in<2>(7), wall_in<2>(8)};

// Bound: launch and latency up to some 256 tiles, vector issue above.  A
// single step of a small block costs its launch (4.8 us of 5.9 at 128^2 FP64);
// S steps per launch of a SIDE^2 tile compute the (SIDE + 2m)^2 nodes of every
// margin m < S.  128^2 FP64 takes 1.7 us per step with SIDE = 8, S = 8 (of
// 14 us per launch 4.8 are the launch, 2 the loads and stores and 0.9 each
// step: reads and barrier 0.4, walls 0.25, the node update 0.25), 1.9 with
// S = 6.  One copy of the populations in LDS, read by all before any writes:
// two copies saved a barrier (3% at 128^2) and halved the workgroups of a CU
// (512^2 FP64 8.1 against 6.4 us).  us per step, single and tiles: FP64 64^2
// 5.9 and 1.65, 256^2 6.0 and 2.6, 512^2 16.1 and 6.3, 301 x 127 channel 8.1
// and 2.8; FP32 128^2 6.2 and 1.4, 512^2 14.2 and 3.9.
template <int ST, int SIDE, int S, bool OBST, bool FORCE>
__global__ __launch_bounds__((SIDE + 2 * S) * (SIDE + 2 * S)) void k_tile(KParams kp) {
    using T = typename Store<ST>::T;
    using E = typename Store<ST>::E;
    constexpr int Q = 9, EW = SIDE + 2 * S, NT = EW * EW;
    __shared__ T s_f[Q][NT];
    __shared__ TileWalls<T> s_w;
    __shared__ uint32_t s_om[OBST ? NT : 1];
    // one block: neither its tiles nor its parameters wait for a table
    TileWG G{0, 0, 0, blockIdx.x == 0};
    if (kp.nblocks == 1) {
        const int ty = (int)blockIdx.x / kp.tile_row;
        G.x0 = ((int)blockIdx.x - ty * kp.tile_row) * SIDE;
        G.y0 = ty * SIDE;
    } else {
        __builtin_memcpy(&G, (const TileWG*)&const_view(kp.tile)[blockIdx.x], sizeof G);
    }
    const int b = G.block;
    const BlockParams B = load_block(kp, b);
    const int cur = load_parity(kp, b);
    const int tid = (int)threadIdx.x;
    if (G.first && tid == 0) kp.cur_out[b] = B.active ? 1 - cur : cur;
    if (!B.active) return;
    const int nx = B.n[0], ny = B.n[1], K = kp.tile_steps;
    const E* prev = static_cast<const E*>(kp.fs_buf[cur]) + B.base;
    E* next = static_cast<E*>(kp.fs_buf[1 - cur]) + B.base;
    const int xend = G.x0 + SIDE < nx ? G.x0 + SIDE : nx;
    const int yend = G.y0 + SIDE < ny ? G.y0 + SIDE : ny;
    // the nodes of step s are the tile grown by K - s; they are dealt out anew
    // for every step, so no wave is partly outside of them but the last
    struct Spot {
        int x, y, at;
        bool on;
    };
    auto spot = [&](int s) {
        const int m = K - s;
        const int xlo = G.x0 - m > 0 || kp.wrap_x ? G.x0 - m : 0;
        const int xhi = xend + m < nx || kp.wrap_x ? xend + m : nx;
        const int ylo = G.y0 - m > 0 ? G.y0 - m : 0, yhi = yend + m < ny ? yend + m : ny;
        const int w = xhi - xlo;
        const int iy = (int)(((float)tid + 0.5f) * __builtin_amdgcn_rcpf((float)w));
        const int x = xlo + tid - iy * w, y = ylo + iy;
        return Spot{kp.wrap_x ? x < 0 ? x + nx : x >= nx ? x - nx : x : x, y,
                    (y - G.y0 + S) * EW + x - G.x0 + S, y < yhi};
    };
    {
        // the state's loads are under way before those of the tables
        const Spot P = spot(0);
        E v[Q];
        uint32_t om = 0;
        if (P.on) {
#pragma unroll
            for (int q = 0; q < Q; q++)
                v[q] = *at_u(prev, (int64_t)q * B.sq, (uint32_t)(P.y * B.sx + P.x));
            if constexpr (OBST) om = obst_mask(kp, B, B.mbase + (int64_t)P.y * nx + P.x);
        }
        const RegionProg* progs = kp.progs + B.prog_base;
        for (int i = tid; i < 9 * 16; i += NT) {
            const int r = i >> 4, w = i & 15;
            const BCOp& op = progs[r].op[0];
            if constexpr (ST == MPLBHIP_STORE_F64) {
                if (w < Q) s_w.c[r][w] = op.cq[w];
                if (w == 9) s_w.den[r] = op.den;
            } else {
                if (w < Q) s_w.c[r][w] = op.eq_c[w];
                if (w == 9) s_w.den[r] = op.eq_k;
            }
            if (w == 10) s_w.win[r] = T(op.eq_win);
            if (w == 11) s_w.in[r] = r && progs[r].nops > 0 ? kWallIn[r] : 0u;
            if (w == 12) s_w.force[r] = progs[r].force;
        }
        if (P.on) {
            if constexpr (OBST) s_om[P.at] = om;
#pragma unroll
            for (int q = 0; q < Q; q++) {
                if constexpr (ST == MPLBHIP_STORE_F16) s_f[q][P.at] = h2f_scaled(v[q], kp.scale[q]);
                else s_f[q][P.at] = v[q];
            }
        }
    }
    double acc[1];
    for (int s = 1; s <= K; s++) {
        const auto [x, y, at, on] = spot(s);
        const int32_t node = y * B.sx + x;
        const int64_t mnode = B.mbase + (int64_t)y * nx + x;
        __syncthreads();
        T f[Q];
        uint32_t om = 0;
        int r = 0;
        if (on) {
#pragma unroll
            for (int q = 0; q < Q; q++) f[q] = s_f[q][at - (cvel(2, q, 1) * EW + cvel(2, q, 0))];
            if constexpr (OBST) {
                // an obstacle source bounces the node's own opposite value
                om = s_om[at];
                if (om) {
#pragma unroll
                    for (int q = 1; q < Q; q++)
                        if (om >> q & 1u) f[q] = s_f[opp(2, q)][at];
                }
            }
            r = region_code(x, nx) + 3 * region_code(y, ny);
        }
        // (every wave has read before any writes the next step's values)
        if (s < K) __syncthreads();
        if (!on || (om & kObstSolid)) continue;
        const uint32_t in = s_w.in[r];
        if (__builtin_amdgcn_ballot_w64(in != 0) != 0)
            lane_wall<2, ST>(f, in, s_w.win[r], s_w.den[r], s_w.c[r]);
        const bool force_node = !FORCE || r == 0 || s_w.force[r] != 0;
        if (s < K) {
            T h[Q];
            finish_node<2, ST, MODE_STEP, FORCE ? 1 : 0>(kp, B, f, false, force_node, mnode,
                                                         TileSink<ST>{h, kp.scale}, x, y, 0, acc);
#pragma unroll
            for (int q = 0; q < Q; q++) s_f[q][at] = h[q];
        } else {
            finish_node<2, ST, MODE_STEP, FORCE ? 1 : 0>(kp, B, f, false, force_node, mnode,
                                                         NodeStore<ST, false>{B, next, node}, x, y,
                                                         0, acc);
        }
    }
}

// the forms: side of the tile, steps per launch
#define MPLB_TILE_FORMS(X) X(8, 8) X(16, 8) X(24, 4)

int tile_max_steps(int side) {
#define X(SIDE, S) \
    if (side == SIDE) return S;
    MPLB_TILE_FORMS(X)
#undef X
    return 0;
}

// the classes of the populations (wall_class) that k_tile takes a region's
// wall to have
void tile_wall_classes(int region, uint32_t* in, uint32_t* out, uint32_t* par) {
    *in = *out = *par = 0;
    for (int q = 0; q < 9; q++) {
        const int t = wall_class(2, region, q);
        *(t == 1 ? in : t == 2 ? out : par) |= 1u << q;
    }
}

template <int ST, int SIDE, int S>
static void launch_form(bool obst, bool force, const KParams& kp, hipStream_t s) {
    const dim3 grid(kp.ntile2d), wg((SIDE + 2 * S) * (SIDE + 2 * S));
    if (obst && force) hipLaunchKernelGGL((k_tile<ST, SIDE, S, true, true>), grid, wg, 0, s, kp);
    else if (obst) hipLaunchKernelGGL((k_tile<ST, SIDE, S, true, false>), grid, wg, 0, s, kp);
    else if (force) hipLaunchKernelGGL((k_tile<ST, SIDE, S, false, true>), grid, wg, 0, s, kp);
    else hipLaunchKernelGGL((k_tile<ST, SIDE, S, false, false>), grid, wg, 0, s, kp);
}

hipError_t launch_tile(int storage, int side, const KParams& kp, hipStream_t s) {
    if (kp.ntile2d <= 0) return hipSuccess;
    if (kp.tile_steps < 1 || kp.tile_steps > tile_max_steps(side)) return hipErrorInvalidValue;
    const bool obst = kp.obst != nullptr, force = kp.force_type || kp.force_macros;
#define X(SIDE, S)                                                                        \
    if (side == SIDE) {                                                                   \
        if (storage == MPLBHIP_STORE_F64)                                                 \
            launch_form<MPLBHIP_STORE_F64, SIDE, S>(obst, force, kp, s);                  \
        else if (storage == MPLBHIP_STORE_F32)                                            \
            launch_form<MPLBHIP_STORE_F32, SIDE, S>(obst, force, kp, s);                  \
        else                                                                              \
            launch_form<MPLBHIP_STORE_F16, SIDE, S>(obst, force, kp, s);                  \
    }
    MPLB_TILE_FORMS(X)
#undef X
    return hipGetLastError();
}

}  // namespace mplbhip
