// march_kernels.hip -- several time steps per launch for 2D blocks without
// halo links: a wave marches through the rows of a strip of columns and keeps
// the rows that the steps in flight still need in registers, so HBM sees one
// read and one write of the lattice per K steps and no wave waits for another.
#include "lattice_device.hpp"

namespace mplbhip {

// the populations by c_y: kRow[s][i] is the i-th with c_y = s - 1
constexpr int kRow[3][3] = {{3, 4, 5}, {0, 2, 6}, {1, 7, 8}};

// value of the lane before (DIR 1) or after (DIR -1) this one; 0 past the wave
template <int DIR>
__device__ __forceinline__ float lane_shift(float v) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(
        0, (int)__float_as_uint(v), DIR > 0 ? 0x138 : 0x130, 0xf, 0xf, true));
}
template <int DIR>
__device__ __forceinline__ double lane_shift(double v) {
    const uint2 u = __builtin_bit_cast(uint2, v);
    const uint2 r{(uint32_t)__builtin_amdgcn_update_dpp(0, (int)u.x, DIR > 0 ? 0x138 : 0x130, 0xf,
                                                        0xf, true),
                  (uint32_t)__builtin_amdgcn_update_dpp(0, (int)u.y, DIR > 0 ? 0x138 : 0x130, 0xf,
                                                        0xf, true)};
    return __builtin_bit_cast(double, r);
}

// a node's new populations as the next step reads them (rounded to storage)
template <int ST> struct StateSink {
    using T = typename Store<ST>::T;
    T* h;
    const float* scale;
    __device__ __forceinline__ void operator()(int q, T v) const {
        if constexpr (ST == MPLBHIP_STORE_F16) h[q] = h2f_scaled(__float2half_rn(v), scale[q]);
        else h[q] = v;
    }
};
template <int ST> struct ElemSink {
    using T = typename Store<ST>::T;
    using E = typename Store<ST>::E;
    E* h;
    __device__ __forceinline__ void operator()(int q, T v) const {
        if constexpr (ST == MPLBHIP_STORE_F16) h[q] = __float2half_rn(v);
        else h[q] = v;
    }
};

// the wall of region R (block-uniform constants, scalar loads)
template <int ST, int R>
__device__ __forceinline__ void march_wall(const MPLB_CONST RegionProg* progs,
                                           typename Store<ST>::T* f) {
    using T = typename Store<ST>::T;
    const MPLB_CONST BCOp& op = progs[R].op[0];
    if constexpr (ST == MPLBHIP_STORE_F64)
        known_wall<2, ST, R, false>(f, T(0), op.den, [&](int q) { return op.cq[q]; });
    else
        known_wall<2, ST, R, true>(f, op.eq_win, op.eq_k, [&](int q) { return op.eq_c[q]; });
}

// Bound: vector issue, then HBM.  A step of its own is HBM-bound (2048^2 FP32
// 56 us at 5.4 TB/s); a march of K steps moves (64 / (64 - 2K)) (1 + 2K / rows)
// reads and one write of the lattice per K steps.  One wave per workgroup and
// no LDS, so no wave waits for another; K as many rows as the registers of W
// waves per SIMD hold and the ends of a strip leave worth it (2048^2, us per
// step: FP32 K = 5 at W = 5 24.6, 6 at 4 26.4, 7 at 4 24.8, 8 at 4 27.8, 256
// blocks of 104^2 20.3, 21.2, 19.4, 21.9; FP64 4 at 3 50.9, 5 at 3 46.7, 6 at 2
// 50.3, 8 at 2 55.5; FP16 4 at 5 22.8, 5 at 4 23.3; with obstacles, 96 blocks
// of 128^2, FP32 3 at 5 16.6, 4 at 4 15.7, 5 at 4 15.8, FP64 3 at 3 29.2, 4 at
// 2 31.4).  Loads of the next row are issued before this row's
// arithmetic; the wall constants come by scalar loads, and the rows that make
// no result store out of range, since a vector load or a store under a branch
// would make the wait for the row wait for those too.  us per step, single
// steps and march (rows 16): FP32 2048^2 56 and 24.8 (K = 7), 256 blocks of 64
// to 256 rows 94 and 37 (K = 7); FP64 2048^2 112 and 46 (K = 5); FP16 2048^2 34 and 22.8
// (K = 4); FP32 with obstacles, 96 blocks of 128^2, 25.3 and 16.0 (K = 4).
template <int ST, int K, bool OBST, int W>
__global__ __launch_bounds__(64, W) void k_march(KParams kp) {
    using T = typename Store<ST>::T;
    using E = typename Store<ST>::E;
    constexpr int Q = 9;
    constexpr uint32_t kE = sizeof(E);
    const int wv = (int)blockIdx.x;
    MarchWave M;
    __builtin_memcpy(&M, (const MarchWave*)&const_view(kp.march)[wv], sizeof M);
    const int b = M.block;
    const BlockParams B = load_block(kp, b);
    const int cur = load_parity(kp, b);
    const int lane = (int)threadIdx.x;
    if (M.first && lane == 0) kp.cur_out[b] = B.active ? 1 - cur : cur;
    if (!B.active) return;
    const int nx = B.n[0], ny = B.n[1];
    const int g = lane / M.group;
    const int x = M.x0 + (lane - g * M.group);
    const int ys = (M.chunk0 + g) * M.rows;
    const int ye = ys + M.rows < ny ? ys + M.rows : ny;
    const E* prev = static_cast<const E*>(kp.fs_buf[cur]) + B.base;
    E* next = static_cast<E*>(kp.fs_buf[1 - cur]) + B.base;
    // the block's memory from node (0, 0) on; an offset of `bytes` is outside
    const uint32_t bytes = (uint32_t)(B.sz - B.sx - 128 / (int)kE) * kE;
    const __amdgpu_buffer_rsrc_t rget =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<E*>(prev), 0, (int)bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rput =
        __builtin_amdgcn_make_buffer_rsrc(next, 0, (int)bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t robst = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(kp.obst) + (OBST ? B.mbase : 0), 0,
        OBST && B.has_obst ? nx * ny * 4 : 0, 0x00020000);
    const MPLB_CONST RegionProg* progs = const_view(kp.progs) + B.prog_base;

    // rows of the steps in flight: stage s holds the results of step s (0:
    // as loaded); z the row before the newest one (c_y = 0), p0 that row
    // and p1 the one before it (c_y > 0), m that row (c_y < 0, which bounces)
    T z[K][3], p0[K][3], p1[K][3], m[OBST ? K : 1][3];
    uint32_t om[OBST ? K : 1];
#pragma unroll
    for (int s = 0; s < K; s++)
#pragma unroll
        for (int k = 0; k < 3; k++) {
            z[s][k] = p0[s][k] = p1[s][k] = T(0);
            if constexpr (OBST) m[s][k] = T(0), om[s] = 0;
        }
    E in[Q];
    uint32_t oin = 0;
    auto load = [&](int y) {
        const bool on = x < nx && y >= 0 && y < ny;
        const uint32_t off = on ? (uint32_t)(y * B.sx + x) * kE : bytes;
#pragma unroll
        for (int q = 0; q < Q; q++) in[q] = buf_ld<E>(rget, off, B.put_off[q]);
        if constexpr (OBST)
            oin = __builtin_amdgcn_raw_buffer_load_b32(
                robst, on ? (uint32_t)(y * nx + x) * 4u : 0xFFFFFFF0u, 0, 0);
    };
    double acc[1];
    load(ys - K);
    const int total = M.rows + 2 * K;
    for (int i = 0; i < total; i++) {
        const int row0 = ys - K + i;  // the newest row of stage 0
        T n[Q];                       // newest row of the stage at hand
        uint32_t mask = oin;
#pragma unroll
        for (int q = 0; q < Q; q++) {
            if constexpr (ST == MPLBHIP_STORE_F16) n[q] = h2f_scaled(in[q], kp.scale[q]);
            else n[q] = in[q];
        }
        load(row0 + 1);
#pragma unroll
        for (int s = 0; s < K; s++) {
            const int y = row0 - 1 - s;  // the row step s + 1 makes now
            auto move_on = [&]() {
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    p1[s][k] = p0[s][k];
                    p0[s][k] = n[kRow[2][k]];
                    z[s][k] = n[kRow[1][k]];
                    if constexpr (OBST) m[s][k] = n[kRow[0][k]];
                }
            };
            if (i < 2 * (s + 1)) {
                // before the first row that any later one needs: the later
                // stages have none either
                move_on();
                if constexpr (OBST) om[s] = mask;
#pragma unroll
                for (int q = 0; q < Q; q++) buf_st<E, 2>(E{}, rput, bytes, B.put_off[q]);
                break;
            }
            // c_x = 1 of the lane before, -1 of the one after
            T f[Q];
            f[0] = z[s][0];
            f[4] = n[4];
            f[8] = p1[s][2];
            f[5] = lane_shift<1>(n[5]);
            f[6] = lane_shift<1>(z[s][2]);
            f[7] = lane_shift<1>(p1[s][1]);
            f[3] = lane_shift<-1>(n[3]);
            f[2] = lane_shift<-1>(z[s][1]);
            f[1] = lane_shift<-1>(p1[s][0]);
            uint32_t w = 0;
            if constexpr (OBST) {
                w = om[s];
                om[s] = mask;
                mask = w;
                // an obstacle source bounces the node's own opposite value
                if (__builtin_amdgcn_ballot_w64(w != 0) != 0) {
                    const T own[Q] = {T(0),     m[s][2], z[s][2], p0[s][1], p0[s][2],
                                      p0[s][0], z[s][1], m[s][0], m[s][1]};
#pragma unroll
                    for (int q = 1; q < Q; q++) f[q] = (w >> q & 1u) ? own[q] : f[q];
                }
            }
            move_on();
            if (__builtin_amdgcn_ballot_w64(y <= 0 || y >= ny - 1) == 0) {
                if (x == 0) march_wall<ST, 1>(progs, f);
                if (x == nx - 1) march_wall<ST, 2>(progs, f);
            } else {
                const int r = region_code(x, nx) + 3 * region_code(y, ny);
                if (r == 1) march_wall<ST, 1>(progs, f);
                if (r == 2) march_wall<ST, 2>(progs, f);
                if (r == 3) march_wall<ST, 3>(progs, f);
                if (r == 6) march_wall<ST, 6>(progs, f);
                if (r == 4) march_wall<ST, 4>(progs, f);
                if (r == 5) march_wall<ST, 5>(progs, f);
                if (r == 7) march_wall<ST, 7>(progs, f);
                if (r == 8) march_wall<ST, 8>(progs, f);
            }
            if (s < K - 1) {
                finish_node<2, ST, MODE_STEP, 0>(kp, B, f, false, true, 0, StateSink<ST>{n, kp.scale},
                                                 x, y, 0, acc);
            } else {
                // the last step's row to HBM
                E e[Q];
                finish_node<2, ST, MODE_STEP, 0>(kp, B, f, false, true, 0, ElemSink<ST>{e}, x, y, 0,
                                                 acc);
                const bool on = y >= ys && y < ye && x >= M.xs && x < M.xe && !(w & kObstSolid);
                const uint32_t at = on ? (uint32_t)(y * B.sx + x) * kE : bytes;
#pragma unroll
                for (int q = 0; q < Q; q++) buf_st<E, 2>(e[q], rput, at, B.put_off[q]);
            }
        }
    }
}

// the forms: storage, obstacles, steps per launch, waves per SIMD
#define MPLB_MARCH_FORMS(X)           \
    X(MPLBHIP_STORE_F64, false, 5, 3) \
    X(MPLBHIP_STORE_F32, false, 7, 4) \
    X(MPLBHIP_STORE_F16, false, 4, 5) \
    X(MPLBHIP_STORE_F64, true, 3, 3)  \
    X(MPLBHIP_STORE_F32, true, 4, 4)  \
    X(MPLBHIP_STORE_F16, true, 4, 4)

// steps per launch of the form
bool march_shape(int storage, bool obst, int* steps) {
#define X(ST, OB, K, W)                \
    if (storage == ST && obst == OB) { \
        *steps = K;                    \
        return true;                   \
    }
    MPLB_MARCH_FORMS(X)
#undef X
    return false;
}

hipError_t launch_march(int storage, const KParams& kp, hipStream_t s) {
    if (kp.nmarch <= 0) return hipSuccess;
    const bool obst = kp.obst != nullptr;
#define X(ST, OB, K, W)                                                                    \
    if (storage == ST && obst == OB) {                                                     \
        hipLaunchKernelGGL((k_march<ST, K, OB, W>), dim3(kp.nmarch), dim3(64), 0, s, kp);  \
        return hipGetLastError();                                                          \
    }
    MPLB_MARCH_FORMS(X)
#undef X
    return hipErrorInvalidValue;
}

}  // namespace mplbhip
