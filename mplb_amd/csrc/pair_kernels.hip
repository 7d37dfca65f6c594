// pair_kernels.hip -- two time steps per launch for 3D cases without halo
// links: a workgroup marches through the z planes of a tile of columns, takes
// the first step of plane z and the second of plane z - 1, and passes the
// intermediate populations through LDS, so HBM sees one read and one write
// of the lattice per two steps.
#include "lattice_device.hpp"

namespace mplbhip {

// ---- boundary programs from LDS ------------------------------------------------
// Every workgroup waits for its wall lanes twice per plane, so what they do
// must not wait on memory: a program read from global memory costs a chain of
// loads per application, and any vector load in the loop makes the compiler
// wait for the next plane's populations too (the load counter is shared; D3Q19
// FP32 256^3: 0.36 ms per step with the programs read from memory against
// 0.30 without any).  The workgroup copies the wall applications of the
// block's regions into LDS once; a lane then runs its own region's by LDS
// reads and bit masks, without branches on populations.
// (Plan::build leaves one application per region.)
template <int D, typename T> struct PairWalls {
    T c[27][lq(D)];            // BCOp::cq (or eq_c) of the region's application
    T den[27];                 // BCOp::den (or eq_k)
    T win[27];                 // BCOp::eq_win
    uint32_t mask[27][3];      // populations: incoming, outgoing, parallel
    uint32_t pull[27];
    int32_t nops[27];
    int32_t persist[27];       // slot of a corner's kept populations, -1: none
    T kept[8][lq(D)];          // the corners' f before the first step ...
    T mid[8][lq(D)];           // ... and between the two
};

// corner number of a region, axis by axis (low 0, high 1)
__device__ __forceinline__ int pair_corner(int r) {
    return (r % 3 == 2) + 2 * (r / 3 % 3 == 2) + 4 * (r / 9 == 2);
}

template <int D, int ST>
__device__ void load_walls(PairWalls<D, typename Store<ST>::T>& W, const RegionProg* progs,
                           const typename Store<ST>::T* per_prev, int tid, int nt) {
    using T = typename Store<ST>::T;
    constexpr int Q = lq(D);
    for (int i = tid; i < 27 * 32; i += nt) {
        const int word = i & 31, r = i >> 5;
        const RegionProg& P = progs[r];
        if (word == 31) {
            W.pull[r] = P.pull;
            W.nops[r] = P.nops;
            W.persist[r] = P.persist;
        }
        const bool dev = ST == MPLBHIP_STORE_F16 && P.persist < 0;
        const BCOp& op = P.op[0];
        if (word < Q) {
            if constexpr (ST == MPLBHIP_STORE_F64) W.c[r][word] = op.cq[word];
            else W.c[r][word] = dev ? op.eq_c[word] : op.fcq[word];
        }
        if (word == 20) {
            if constexpr (ST == MPLBHIP_STORE_F64) W.den[r] = op.den;
            else W.den[r] = dev ? op.eq_k : op.fden;
        }
        if (word == 21) W.win[r] = T(op.eq_win);
        if (word == 22) W.mask[r][0] = op.m_in;
        if (word == 23) W.mask[r][1] = op.m_out;
        if (word == 24) W.mask[r][2] = op.m_par;
    }
    for (int i = tid; i < 8 * Q; i += nt) {
        const int k = i / Q;
        const RegionProg& P = progs[(k & 1 ? 2 : 1) + 3 * (k & 2 ? 2 : 1) + 9 * (k & 4 ? 2 : 1)];
        W.kept[k][i - k * Q] = P.persist >= 0 ? per_prev[(int64_t)P.persist * Q + i - k * Q] : T(0);
    }
}

// pair_boundary of a face or edge whose populations' classes are known at
// compile time: the faces, and the edges that every plane has.  The general
// form issues about 350 instructions; one wave per tile runs it while the
// others wait at the barrier, 0.09 of 0.27 ms per step for the four z edges
// of D3Q19 FP32 256^3 alone.
template <int D, int ST, int R>
__device__ __forceinline__ void pair_wall(PairWalls<D, typename Store<ST>::T>& W,
                                          typename Store<ST>::T* f) {
    known_wall<D, ST, R, ST == MPLBHIP_STORE_F16>(
        f, W.win[R], W.den[R], [&](int q) { return W.c[R][q]; });
}

// The boundary program of region r (not the interior) on a lane's gathered
// populations (raw: FP64 f, reduced storage g = f - w), with the arithmetic
// of the bulk kernel for simple regions and of the boundary kernel for the
// corners whose unpulled populations persist: the first step reads those from
// W.kept and leaves its own in W.mid (own: the lane's tile owns the node),
// the second reads W.mid and stores to per_next.
template <int D, int ST, bool SECOND>
__device__ __forceinline__ void pair_boundary(PairWalls<D, typename Store<ST>::T>& W, int r,
                                              typename Store<ST>::T* f, bool own,
                                              typename Store<ST>::T* per_next) {
#pragma clang fp contract(off)
    using T = typename Store<ST>::T;
    constexpr int Q = lq(D);
    const bool wall = W.nops[r] != 0;
    if (wall) {
        if (r == 1) return pair_wall<D, ST, 1>(W, f);
        if (r == 2) return pair_wall<D, ST, 2>(W, f);
        if (r == 3) return pair_wall<D, ST, 3>(W, f);
        if (r == 6) return pair_wall<D, ST, 6>(W, f);
        if (r == 9) return pair_wall<D, ST, 9>(W, f);
        if (r == 18) return pair_wall<D, ST, 18>(W, f);
        if (r == 4) return pair_wall<D, ST, 4>(W, f);
        if (r == 5) return pair_wall<D, ST, 5>(W, f);
        if (r == 7) return pair_wall<D, ST, 7>(W, f);
        if (r == 8) return pair_wall<D, ST, 8>(W, f);
    }
    const uint32_t pull = W.pull[r];
    const int persist = W.persist[r];
    if (ST == MPLBHIP_STORE_F16 && persist < 0) {
        // apply_eqm_dev
#pragma unroll
        for (int q = 0; q < Q; q++) f[q] = bit_and(f[q], pull, q);
        if (wall) {
            const int s = r;
            const uint32_t m_in = W.mask[s][0], m_out = W.mask[s][1], m_par = W.mask[s][2];
            const uint32_t m_set = m_out | m_par;
            T rin = W.win[s];
#pragma unroll
            for (int q = 0; q < Q; q++) rin += bit_and(f[q], m_in, q);
            const T rw = rin * W.den[s];
#pragma unroll
            for (int q = 0; q < Q; q++) {
                const int p = opp(D, q);
                if (p < q) continue;
                const T bq = bit_or(bit_and(f[p], m_out, q), bit_and(-T(wgt(D, q)), m_par, q));
                const T bp = bit_or(bit_and(f[q], m_out, p), bit_and(-T(wgt(D, p)), m_par, p));
                const T vq = fma_t(rw, W.c[s][q], bq), vp = fma_t(rw, W.c[s][p], bp);
                f[q] = bit_sel(m_set, q, vq, f[q]);
                if (p != q) f[p] = bit_sel(m_set, p, vp, f[p]);
            }
        }
        return;
    }
#pragma unroll
    for (int q = 0; q < Q; q++) {
        if constexpr (ST != MPLBHIP_STORE_F64) f[q] += T(wgt(D, q));
        f[q] = bit_and(f[q], pull, q);
    }
    const int corner = pair_corner(r);
    if (persist >= 0) {
        const T* kept = SECOND ? W.mid[corner] : W.kept[corner];
#pragma unroll
        for (int q = 0; q < Q; q++) f[q] = bit_or(f[q], bit_and(kept[q], ~pull, q));
    }
    // apply_eqm
    if (wall) {
        const int s = r;
        const uint32_t m_in = W.mask[s][0], m_out = W.mask[s][1];
        const uint32_t m_set = m_out | W.mask[s][2];
        T rin = T(0);
#pragma unroll
        for (int q = 0; q < Q; q++) rin += bit_and(f[q], m_in, q);
        const T rw = T(2) * rin / W.den[s];
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const int p = opp(D, q);
            if (p < q) continue;
            const T wr = T(wgt(D, q)) * rw;
            const T vq = wr * W.c[s][q] + bit_and(f[p], m_out, q);
            const T vp = wr * W.c[s][p] + bit_and(f[q], m_out, p);
            f[q] = bit_sel(m_set, q, vq, f[q]);
            if (p != q) f[p] = bit_sel(m_set, p, vp, f[p]);
        }
    }
    if (persist >= 0 && own) {
#pragma unroll
        for (int q = 0; q < Q; q++) {
            if constexpr (SECOND) per_next[(int64_t)persist * Q + q] = f[q];
            else W.mid[corner][q] = f[q];
        }
    }
    if constexpr (ST != MPLBHIP_STORE_F64) {
#pragma unroll
        for (int q = 0; q < Q; q++) f[q] -= T(wgt(D, q));
    }
}

// populations with c_z of the given sign, and a population's place among
// those of its sign
__host__ __device__ constexpr int pair_count(int D, int sign) {
    int n = 0;
    for (int q = 0; q < lq(D); q++) n += cvel(D, q, 2) == sign ? 1 : 0;
    return n;
}
__host__ __device__ constexpr int pair_slot(int D, int q) {
    int n = 0;
    for (int p = 0; p < q; p++) n += cvel(D, p, 2) == cvel(D, q, 2) ? 1 : 0;
    return n;
}

// keeps a node's new populations in registers, as they are stored
template <int ST> struct RegSink {
    using T = typename Store<ST>::T;
    using E = typename Store<ST>::E;
    E* h;
    __device__ __forceinline__ void operator()(int q, T v) const {
        if constexpr (ST == MPLBHIP_STORE_F16) h[q] = __float2half_rn(v);
        else h[q] = v;
    }
};

// A thread's node of a tile: columns [xa, xb) x [ya, yb) cut to the block.
// Nodes of the block's x faces go to the first wave alone, so that one wave
// runs their boundary programs instead of a few lanes of every wave; the
// others follow row by row, in rows of rw threads from column xr on.
struct TileNode {
    int x, y;
    bool valid;
};
__device__ __forceinline__ TileNode tile_node(int tid, bool lo, bool hi, int xr, int rw, int ya,
                                              int rows, int nx) {
    const int faces = (lo || hi) ? 64 : 0;
    TileNode n{0, 0, false};
    if (tid < faces) {
        const int c = tid / rows;
        n.y = ya + tid - c * rows;
        n.x = c == 0 && lo ? 0 : nx - 1;
        n.valid = c < (lo ? 1 : 0) + (hi ? 1 : 0);
    } else if (tid - faces < rw * rows) {
        const int r = (tid - faces) / rw;
        n.x = xr + tid - faces - r * rw;
        n.y = ya + r;
        n.valid = n.x > 0 && n.x < nx - 1;
    }
    return n;
}

// Two steps of one tile.  A single-step launch is bound by HBM (D3Q19 FP32
// 256^3: 5.8 of the 6.3 TB/s a plain copy reaches), so the lattice is read and
// written once per two steps: each workgroup computes the first step on its
// tile grown by one node and marches along z, where nothing is computed twice
// but one plane at either end of its range.  Tile height and width are what
// the positions in LDS allow: all populations of one to three planes (38
// values per position in D3Q19), one workgroup per CU.
// 256^3 FP32: HBM reads 1.46 GB and writes 1.28 GB per two steps, 4.9 TB/s;
// 0.445 -> 0.281 ms per step (FP64 0.957 -> 0.595, FP16 0.237 -> 0.214, where
// the arithmetic of 16 waves per CU bounds it).  160^3 FP64 0.238 -> 0.159,
// 81 x 67 x 53 FP64 30.6 -> 24.2 us.  What remains above HBM's time is the
// barriers': the four phases of a plane do not overlap within a workgroup.
// Two workgroups of 512 threads per CU were slower (0.337: more is computed
// twice), and so were loads two planes ahead (0.285).
// NT threads, NP positions of a grown tile
template <int D, int ST, int NT, int NP>
__global__ __launch_bounds__(NT, ST == MPLBHIP_STORE_F64 ? 2 : 4) void k_pair(KParams kp) {
    using T = typename Store<ST>::T;
    using E = typename Store<ST>::E;
    constexpr int Q = lq(D);
    // Populations of the first step by position in the grown tile.  Plane z
    // needs those with c_z < 0 of plane z + 1, c_z = 0 of plane z and c_z > 0
    // of plane z - 1: one, two and three planes are kept.
    constexpr int QM = pair_count(D, -1), Q0 = pair_count(D, 0), QP = pair_count(D, 1);
    __shared__ E s_m[QM][NP], s_0[2][Q0][NP], s_p[3][QP][NP];
    __shared__ PairWalls<D, T> s_w;
    // neighbouring tiles on one XCD: their grown rows share cache lines (HBM
    // reads 1.15 times the lattice per launch, against 1.85 dealt in order)
    const int wg = logical_wg(blockIdx.x, gridDim.x);
    const int b = wg_block(kp, kp.wg_block_pair, wg);
    const BlockParams B = load_block(kp, b);
    PairBlock PB;
    __builtin_memcpy(&PB, (const PairBlock*)&const_view(kp.pair)[b], sizeof PB);
    const int cur = load_parity(kp, b);
    const int t = wg - PB.start;
    const int tid = (int)threadIdx.x;
    if (t == 0 && tid == 0) kp.cur_out[b] = B.active ? 1 - cur : cur;
    if (!B.active) return;
    const int tr = fast_div(t, PB.div_m[0], PB.div_sh[0]);
    const int tx = t - tr * PB.tx;
    const int tz = fast_div(tr, PB.div_m[1], PB.div_sh[1]);
    const int ty = tr - tz * PB.ty;
    const int exw = PB.w + 2;
    const int nz = B.n[2];
    const int zs = tz * PB.lz;
    const int ze = zs + PB.lz < nz ? zs + PB.lz : nz;
    const int xa = tx * PB.w, ya = ty * PB.h;  // the tile's first column
    // first step: the tile grown by one node on every side; second: the tile
    const bool lo1 = xa <= 1, hi1 = xa + PB.w + 1 >= B.n[0];
    const int xr1 = lo1 ? 1 : xa - 1, ya1 = ya > 0 ? ya - 1 : 0;
    const TileNode n1 = tile_node(tid, lo1, hi1, xr1,
                                  (hi1 ? B.n[0] - 1 : xa + PB.w + 1) - xr1, ya1,
                                  (ya + PB.h + 1 < B.n[1] ? ya + PB.h + 1 : B.n[1]) - ya1, B.n[0]);
    // (whole rows of w, so that a row's stores stay whole cache lines)
    const bool xlo = xa == 0, xhi = xa + PB.w >= B.n[0];
    const TileNode n2 = tile_node(tid, xlo, xhi, xa, PB.w, ya,
                                  ya + PB.h < B.n[1] ? PB.h : B.n[1] - ya, B.n[0]);
    const bool xface = xlo || xhi;
    const bool own1 = n1.x >= xa && n1.x < xa + PB.w && n1.y >= ya && n1.y < ya + PB.h;
    const int rc1 = region_code(n1.x, B.n[0]) + 3 * region_code(n1.y, B.n[1]);
    const int rc2 = region_code(n2.x, B.n[0]) + 3 * region_code(n2.y, B.n[1]);
    const int at1 = n1.valid ? (n1.y - ya + 1) * exw + n1.x - xa + 1 : 0;
    const int at2 = n2.valid ? (n2.y - ya + 1) * exw + n2.x - xa + 1 : exw + 1;
    const E* prev = static_cast<const E*>(kp.fs_buf[cur]) + B.base;
    E* next = static_cast<E*>(kp.fs_buf[1 - cur]) + B.base;
    const T* per_prev = static_cast<const T*>(kp.per_buf[cur]);
    T* per_next = static_cast<T*>(kp.per_buf[1 - cur]);
    // Every wave issues the same loads and stores in every iteration, lanes
    // without a node at an offset outside the buffer (loads give 0, stores
    // are dropped): a store under a branch would make the compiler wait for
    // it together with the loads issued before it.
    const uint32_t bytes = (uint32_t)B.sz * (uint32_t)(nz + 2) * (uint32_t)sizeof(E);
    const __amdgpu_buffer_rsrc_t rpull = __builtin_amdgcn_make_buffer_rsrc(
        reinterpret_cast<char*>(const_cast<E*>(prev)) - (int64_t)B.pull_shift * sizeof(E), 0,
        (int)bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rput =
        __builtin_amdgcn_make_buffer_rsrc(next, 0, (int)bytes, 0x00020000);
    const uint32_t node1 = (uint32_t)(n1.y * B.sx + n1.x), node2 = (uint32_t)(n2.y * B.sx + n2.x);

    const bool any2 = __builtin_amdgcn_ballot_w64(n2.valid) != 0;

    // pulled populations of a plane of the first step
    auto load = [&](E* pre, int z, bool on) {
        const uint32_t off = on ? (node1 + (uint32_t)(z * B.sz)) * (uint32_t)sizeof(E) : bytes;
#pragma unroll
        for (int q = 0; q < Q; q++) pre[q] = buf_ld<E>(rpull, off, B.pull_off[q]);
    };
    load_walls<D, ST>(s_w, kp.progs + B.prog_base, per_prev, tid, NT);
    __syncthreads();
    const int k0 = zs > 0 ? zs - 1 : 0;
    const int k1 = ze < nz ? ze : nz - 1;  // last plane of the first step
    // Two register sets in turn: with one, the loads of the next plane would
    // go to registers that are copied at the end of the iteration, and the
    // copy waits for them there.
    E pa[Q], pb[Q];
    load(pa, k0, n1.valid);
    // (dropped) as many stores after these loads as every iteration leaves:
    // the wait for the loads at the top of the loop then counts them on both
    // ways in, and does not wait for the stores themselves
#pragma unroll
    for (int q = 0; q < Q; q++) buf_st<E, 2>(E(0), rput, bytes, B.put_off[q]);
    double acc[1];
    int i2 = 0, i3 = 0;  // ring positions of plane k
    auto plane = [&](int k, const E* pre, E* ahead) {
        E h[Q];
        {
            T f[Q];
#pragma unroll
            for (int q = 0; q < Q; q++) {
                if constexpr (ST == MPLBHIP_STORE_F16) f[q] = h2f_scaled(pre[q], kp.scale[q]);
                else f[q] = pre[q];
            }
            const int r = rc1 + 9 * region_code(k, nz);
            if (r && n1.valid)
                pair_boundary<D, ST, false>(s_w, r, f, own1 && k >= zs && k < ze, per_next);
            finish_node<D, ST, MODE_STEP, 0>(kp, B, f, false, true, 0, RegSink<ST>{h}, n1.x,
                                                 n1.y, k, acc);
        }
        // the second step of the plane before has read what is replaced
        __syncthreads();
        if (n1.valid && k <= k1) {
#pragma unroll
            for (int q = 0; q < Q; q++) {
                const int cz = cvel(D, q, 2), s = pair_slot(D, q);
                if (cz < 0) s_m[s][at1] = h[q];
                if (cz == 0) s_0[i2][s][at1] = h[q];
                if (cz > 0) s_p[i3][s][at1] = h[q];
            }
        }
        // the next plane's loads, ahead of this iteration's stores, which
        // they would otherwise queue behind (0.281 against 0.305 ms per step
        // of D3Q19 FP32 256^3 with the loads at the top of the iteration)
        load(ahead, k + 1, n1.valid && k < k1);
        __syncthreads();
        if (!any2) {
#pragma unroll
            for (int q = 0; q < Q; q++) buf_st<E, 0>(E(0), rput, bytes, B.put_off[q]);
        } else {
            const int z = k - 1;
            const bool on = n2.valid && z >= zs && z < ze;
            const int j2 = 1 - i2;                // plane z
            const int j3 = i3 == 2 ? 0 : i3 + 1;  // plane z - 1
            T f[Q];
#pragma unroll
            for (int q = 0; q < Q; q++) {
                const int cz = cvel(D, q, 2), s = pair_slot(D, q);
                const int at = at2 - cvel(D, q, 1) * exw - cvel(D, q, 0);
                const E v = cz < 0 ? s_m[s][at] : cz == 0 ? s_0[j2][s][at] : s_p[j3][s][at];
                if constexpr (ST == MPLBHIP_STORE_F16) f[q] = h2f_scaled(v, kp.scale[q]);
                else f[q] = v;
            }
            const int r = rc2 + 9 * region_code(z, nz);
            if (r && on) pair_boundary<D, ST, true>(s_w, r, f, true, per_next);
            E o[Q];
            finish_node<D, ST, MODE_STEP, 0>(kp, B, f, false, true, 0, RegSink<ST>{o}, n2.x,
                                                 n2.y, z, acc);
            // nontemporal rows, except in tiles whose x-face nodes another
            // wave stores: those lines meet in L2
            const uint32_t off = on ? (node2 + (uint32_t)(z * B.sz)) * (uint32_t)sizeof(E) : bytes;
            if (xface) {
#pragma unroll
                for (int q = 0; q < Q; q++) buf_st<E, 0>(o[q], rput, off, B.put_off[q]);
            } else {
#pragma unroll
                for (int q = 0; q < Q; q++) buf_st<E, 2>(o[q], rput, off, B.put_off[q]);
            }
        }
        i2 = 1 - i2;
        i3 = i3 == 2 ? 0 : i3 + 1;
    };
    for (int k = k0; k <= ze; k += 2) {
        plane(k, pa, pb);
        plane(k + 1, pb, pa);
    }
}

// a workgroup's threads and the positions its LDS holds
bool pair_shape(int storage, int nt, int* positions) {
    *positions = 0;
    if (storage == MPLBHIP_STORE_F64 && nt == 512) *positions = 448;
    if (storage == MPLBHIP_STORE_F32 && nt == 1024) *positions = 992;
    if (storage == MPLBHIP_STORE_F16 && nt == 1024) *positions = 1024;
    return *positions > 0;
}

hipError_t launch_pair(int lat, int storage, const KParams& kp, hipStream_t s) {
    if (kp.npair <= 0) return hipSuccess;
    const dim3 g(kp.npair), blk(kp.pair_nt);
#define MPLB_PAIR(D, ST, NT, NP)                                         \
    if (lat == D && storage == ST && kp.pair_nt == NT) {                 \
        hipLaunchKernelGGL((k_pair<D, ST, NT, NP>), g, blk, 0, s, kp);   \
        return hipGetLastError();                                        \
    }
    MPLB_PAIR(3, MPLBHIP_STORE_F64, 512, 448)
    MPLB_PAIR(3, MPLBHIP_STORE_F32, 1024, 992)
    MPLB_PAIR(3, MPLBHIP_STORE_F16, 1024, 1024)
    MPLB_PAIR(15, MPLBHIP_STORE_F64, 512, 448)
    MPLB_PAIR(15, MPLBHIP_STORE_F32, 1024, 992)
    MPLB_PAIR(15, MPLBHIP_STORE_F16, 1024, 1024)
#undef MPLB_PAIR
    return hipErrorInvalidValue;
}

}  // namespace mplbhip
