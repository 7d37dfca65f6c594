// lattice_device.hpp -- device functions of the lattice update: velocity
// tables, storage traits, the reference arithmetic, boundary programs, node
// addressing and the macros + collision of one node.
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/mplbhip.h"
#include "lattice_kernels.hpp"

namespace mplbhip {

// sqrt(3) rounded to double: equals the host's sqrt(3.0) (model.cpp:67-68)
constexpr double kCS = 1.7320508075688772935274463415059;

// The lattice key D of every template below: 2 = D2Q9, 3 = D3Q19,
// 15 = D3Q15 (Src/model.cpp:133-150); ldim(D) is its space dimension and
// lq(D) its number of velocities.
__host__ __device__ constexpr int ldim(int D) { return D == 2 ? 2 : 3; }
__host__ __device__ constexpr int lq(int D) { return D == 2 ? 9 : (D == 15 ? 15 : 19); }

__host__ __device__ constexpr int cvel(int D, int q, int a) {
    constexpr int t2[9][2] = {{0, 0},  {-1, 1}, {-1, 0}, {-1, -1}, {0, -1},
                              {1, -1}, {1, 0},  {1, 1},  {0, 1}};
    constexpr int t3[19][3] = {
        {0, 0, 0},  {-1, 0, 0},  {0, -1, 0}, {0, 0, -1}, {-1, -1, 0},
        {-1, 1, 0}, {-1, 0, -1}, {-1, 0, 1}, {0, -1, -1}, {0, -1, 1},
        {1, 0, 0},  {0, 1, 0},   {0, 0, 1},  {1, 1, 0},  {1, -1, 0},
        {1, 0, 1},  {1, 0, -1},  {0, 1, 1},  {0, 1, -1}};
    constexpr int t15[15][3] = {
        {0, 0, 0},    {-1, 0, 0},  {0, -1, 0},  {0, 0, -1}, {-1, -1, -1},
        {-1, -1, 1},  {-1, 1, -1}, {-1, 1, 1},  {1, 0, 0},  {0, 1, 0},
        {0, 0, 1},    {1, 1, 1},   {1, 1, -1},  {1, -1, 1}, {1, -1, -1}};
    return D == 2 ? (a < 2 ? t2[q][a] : 0) : (D == 15 ? t15[q][a] : t3[q][a]);
}
__host__ __device__ constexpr double wgt(int D, int q) {
    constexpr double w2[9] = {4.0 / 9.0,  1.0 / 36.0, 1.0 / 9.0,
                              1.0 / 36.0, 1.0 / 9.0,  1.0 / 36.0,
                              1.0 / 9.0,  1.0 / 36.0, 1.0 / 9.0};
    constexpr double w3[19] = {
        1.0 / 3.0,  1.0 / 18.0, 1.0 / 18.0, 1.0 / 18.0, 1.0 / 36.0,
        1.0 / 36.0, 1.0 / 36.0, 1.0 / 36.0, 1.0 / 36.0, 1.0 / 36.0,
        1.0 / 18.0, 1.0 / 18.0, 1.0 / 18.0, 1.0 / 36.0, 1.0 / 36.0,
        1.0 / 36.0, 1.0 / 36.0, 1.0 / 36.0, 1.0 / 36.0};
    // 2/9, 1/9, 1/72 as the reference writes them: 2 / ((Real)9) ...
    constexpr double w15[15] = {
        2.0 / 9.0,  1.0 / 9.0,  1.0 / 9.0,  1.0 / 9.0,  1.0 / 72.0,
        1.0 / 72.0, 1.0 / 72.0, 1.0 / 72.0, 1.0 / 9.0,  1.0 / 9.0,
        1.0 / 9.0,  1.0 / 72.0, 1.0 / 72.0, 1.0 / 72.0, 1.0 / 72.0};
    return D == 2 ? w2[q] : (D == 15 ? w15[q] : w3[q]);
}
__host__ __device__ constexpr int opp(int D, int q) {
    constexpr int o2[9] = {0, 5, 6, 7, 8, 1, 2, 3, 4};
    constexpr int o3[19] = {0, 10, 11, 12, 13, 14, 15, 16, 17, 18,
                            1, 2,  3,  4,  5,  6,  7,  8,  9};
    constexpr int o15[15] = {0, 8, 9, 10, 11, 12, 13, 14, 1, 2, 3, 4, 5, 6, 7};
    return D == 2 ? o2[q] : (D == 15 ? o15[q] : o3[q]);
}

// ---- storage traits -------------------------------------------------------
template <int ST> struct Store;
template <> struct Store<MPLBHIP_STORE_F64> { using E = double; using T = double; };
template <> struct Store<MPLBHIP_STORE_F32> { using E = float; using T = float; };
template <> struct Store<MPLBHIP_STORE_F16> { using E = __half; using T = float; };

// a stored FP16 value times its population scale: one mixed-precision
// multiply-add (v_fma_mix) instead of a conversion and a multiply
__device__ __forceinline__ float h2f_scaled(__half h, float sc) {
    return __builtin_fmaf(__half2float(h), sc, 0.0f);
}

template <int ST>
__device__ __forceinline__ typename Store<ST>::T ld(const typename Store<ST>::E* p,
                                                    int64_t i, float sc) {
    if constexpr (ST == MPLBHIP_STORE_F16) return h2f_scaled(p[i], sc);
    else return p[i];
}
template <int ST>
__device__ __forceinline__ void st(typename Store<ST>::E* p, int64_t i,
                                   typename Store<ST>::T v, float isc) {
    if constexpr (ST == MPLBHIP_STORE_F16) p[i] = __float2half_rn(v * isc);
    else p[i] = v;
}
// non-temporal store for the streamed post-collision state
template <int ST>
__device__ __forceinline__ void st_nt(typename Store<ST>::E* p, int64_t i,
                                      typename Store<ST>::T v, float isc) {
    if constexpr (ST == MPLBHIP_STORE_F16) {
        p[i] = __float2half_rn(v * isc);
    } else {
        __builtin_nontemporal_store(v, p + i);
    }
}

// ---- reference arithmetic (any T; exact for double) -------------------------
// CalcBGKFeq, T = 1, polyOrder = 2 (model_host_device.h:34-83).  The
// (T-1)(c2-D) term is an exact zero and is left out.
template <int D, typename T>
__device__ __forceinline__ T feq_ref(int q, T rho, T u, T v, T w) {
#pragma clang fp contract(off)
    const T cs = T(kCS);
    T cu;
    T u2;
    if constexpr (D == 2) {
        cu = cs * T(cvel(D, q, 0)) * u + cs * T(cvel(D, q, 1)) * v;
        u2 = u * u + v * v;
    } else {
        cu = cs * T(cvel(D, q, 0)) * u + cs * T(cvel(D, q, 1)) * v +
             cs * T(cvel(D, q, 2)) * w;
        u2 = u * u + v * v + w * w;
    }
    const T cu2 = cu * cu;
    const T res = T(1.0) + cu + T(0.5) * (cu2 - u2);
    return T(wgt(D, q)) * rho * res;
}

// CalcBGKFeq at temperature Tm with polyOrder 4 (model_host_device.h:34-83),
// every term in the reference's order; LATTDIM enters as an int
template <int D>
__device__ __forceinline__ double feq4_ref(int q, double rho, double u, double v, double w,
                                           double Tm) {
#pragma clang fp contract(off)
    constexpr int LD = ldim(D);
    const double cs = kCS;
    double cu, c2, u2;
    if constexpr (LD == 2) {
        cu = (cs * double(cvel(D, q, 0)) * u + cs * double(cvel(D, q, 1)) * v);
        c2 = (cs * double(cvel(D, q, 0)) * cs * double(cvel(D, q, 0)) +
              cs * double(cvel(D, q, 1)) * cs * double(cvel(D, q, 1)));
        u2 = u * u + v * v;
    } else {
        cu = (cs * double(cvel(D, q, 0)) * u + cs * double(cvel(D, q, 1)) * v +
              cs * double(cvel(D, q, 2)) * w);
        c2 = (cs * double(cvel(D, q, 0)) * cs * double(cvel(D, q, 0)) +
              cs * double(cvel(D, q, 1)) * cs * double(cvel(D, q, 1)) +
              cs * double(cvel(D, q, 2)) * cs * double(cvel(D, q, 2)));
        u2 = u * u + v * v + w * w;
    }
    const double cu2 = cu * cu;
    double res = 1.0 + cu + 0.5 * (cu2 - u2 + (Tm - 1.0) * (c2 - LD));
    res = res + cu * (cu2 - 3.0 * u2 + 3.0 * (Tm - 1.0) * (c2 - LD - 2.0)) / 6.0;
    res = res + (cu2 * cu2 - 6.0 * cu2 * u2 + 3.0 * u2 * u2) / 24.0 +
          (Tm - 1.0) * ((c2 - (LD + 2)) * (cu2 - u2) - 2.0 * cu2) / 4.0 +
          (Tm - 1.0) * (Tm - 1.0) * (c2 * c2 - 2.0 * (LD + 2) * c2 + LD * (LD + 2)) / 8.0;
    return wgt(D, q) * rho * res;
}

__device__ __forceinline__ double fma_t(double a, double b, double c) {
    return __builtin_fma(a, b, c);
}
__device__ __forceinline__ float fma_t(float a, float b, float c) {
    return __builtin_fmaf(a, b, c);
}
template <typename OP> __device__ __forceinline__ double eq_den(const OP& op, double) { return op.den; }
template <typename OP> __device__ __forceinline__ float eq_den(const OP& op, float) { return op.fden; }
template <typename OP> __device__ __forceinline__ double eq_coef(const OP& op, int q, double) {
    return op.cq[q];
}
template <typename OP> __device__ __forceinline__ float eq_coef(const OP& op, int q, float) {
    return op.fcq[q];
}

// v where bit q of m is set, else +0; a where it is set, else b: exact
// whatever they hold
__device__ __forceinline__ float bit_and(float v, uint32_t m, int q) {
    return __uint_as_float(__float_as_uint(v) & (uint32_t)((int32_t)(m << (31 - q)) >> 31));
}
__device__ __forceinline__ double bit_and(double v, uint32_t m, int q) {
    const int64_t k = (int32_t)(m << (31 - q)) >> 31;
    return __builtin_bit_cast(double, __builtin_bit_cast(int64_t, v) & k);
}
__device__ __forceinline__ float bit_or(float a, float b) {
    return __uint_as_float(__float_as_uint(a) | __float_as_uint(b));
}
__device__ __forceinline__ double bit_or(double a, double b) {
    return __builtin_bit_cast(double,
                              __builtin_bit_cast(int64_t, a) | __builtin_bit_cast(int64_t, b));
}
__device__ __forceinline__ float bit_sel(uint32_t m, int q, float a, float b) {
    const uint32_t k = (uint32_t)((int32_t)(m << (31 - q)) >> 31);
    return __uint_as_float((__float_as_uint(a) & k) | (__float_as_uint(b) & ~k));
}
__device__ __forceinline__ double bit_sel(uint32_t m, int q, double a, double b) {
    const int64_t k = (int32_t)(m << (31 - q)) >> 31;
    return __builtin_bit_cast(double, (__builtin_bit_cast(int64_t, a) & k) |
                                          (__builtin_bit_cast(int64_t, b) & ~k));
}

// KerCutCellEQMDiffuseRefl[3D] (boundary_kernel.inc:534-613, 1184-1276).
// With the wall-velocity terms from the host (BCOp::den, cq): rho_w = 2
// sum_in f / den, a parallel population (w rho_w) res, an outgoing one f_opp
// + (w rho_w) (2 cu).  Every rounding is the reference's: a factor two and an
// added zero are exact.  The classes are chosen by bit masks, so the code has
// no branch, and only incoming populations are read (the opposite of an
// outgoing one is incoming, that of a parallel one parallel), so that no other
// one, finite or not, has a part in the result.  With a scalar branch per
// population and class an application took some 60 branches and as many
// dependent scalar loads, which set the pace of every workgroup that waits
// for its wall lanes.
template <int D, typename T, typename OP>
__device__ __forceinline__ void apply_eqm(T* f, const OP& op) {
#pragma clang fp contract(off)
    constexpr int Q = lq(D);
    const uint32_t m_in = op.m_in, m_set = op.m_out | op.m_par;
    T rin = T(0), in[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        in[q] = bit_and(f[q], m_in, q);
        rin += in[q];
    }
    const T rw = T(2) * rin / eq_den(op, T(0));
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int p = opp(D, q);
        if (p < q) continue;
        const T wr = T(wgt(D, q)) * rw;
        const T vq = wr * eq_coef(op, q, T(0)) + in[p];
        const T vp = wr * eq_coef(op, p, T(0)) + in[q];
        f[q] = bit_sel(m_set, q, vq, f[q]);
        if (p != q) f[p] = bit_sel(m_set, p, vp, f[p]);
    }
}

// apply_eqm on deviations g = f - w (reduced storage, FP32 arithmetic),
// with the terms that depend on the wall velocity only computed by the
// host (BCOp::eq_*): rho_in = sum_in w + sum_in g, rho_w = 2 rho_in /
// (1 - dRho - rhoPar), parallel g = rho_w w res - w, outgoing g = g_opp +
// 2 rho_w w c.u (the w of a population and its opposite are equal)
template <int D, typename OP>
__device__ __forceinline__ void apply_eqm_dev(float* g, const OP& op) {
    constexpr int Q = lq(D);
    const uint32_t m_in = op.m_in, m_par = op.m_par, m_set = op.m_out | m_par;
    float rin = op.eq_win, in[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        in[q] = bit_and(g[q], m_in, q);
        rin += in[q];
    }
    const float rw = rin * op.eq_k;
    auto value = [&](int q, int p) {
        const float b = bit_or(in[p], bit_and(-float(wgt(D, q)), m_par, q));
        return __builtin_fmaf(rw, op.eq_c[q], b);
    };
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int p = opp(D, q);
        if (p < q) continue;
        const float vq = value(q, p), vp = value(p, q);
        g[q] = bit_sel(m_set, q, vq, g[q]);
        if (p != q) g[p] = bit_sel(m_set, p, vp, g[p]);
    }
}

// FindBdyDvType[3D] (boundary_host_device.h:47-183, 191-706) of a face or an
// edge region (2D: a corner): 1 streams into the wall, 2 comes out of it, 3 along it
__host__ __device__ constexpr int wall_class(int D, int r, int q) {
    const int code[3] = {r % 3, r / 3 % 3, r / 9};
    int n = 0, cn[3] = {0, 0, 0};
    for (int a = 0; a < 3; a++)
        if (code[a]) cn[n++] = (code[a] == 1 ? 1 : -1) * cvel(D, q, a);
    if (n == 1) return cn[0] < 0 ? 1 : cn[0] > 0 ? 2 : 3;
    if ((cn[0] <= 0 && cn[1] < 0) || (cn[0] < 0 && cn[1] == 0)) return 1;
    if ((cn[0] >= 0 && cn[1] > 0) || (cn[0] > 0 && cn[1] == 0)) return 2;
    return 3;
}

// apply_eqm (DEV: apply_eqm_dev, on deviations) of region R with its
// populations' classes known at compile time: every incoming population is
// pulled, and every other one is written.  Reduced storage takes and leaves
// deviations either way.
template <int D, int ST, int R, bool DEV, typename T, typename COEF>
__device__ __forceinline__ void known_wall(T* f, T win, T den, const COEF& coef) {
#pragma clang fp contract(off)
    constexpr int Q = lq(D);
    if constexpr (DEV) {
        T rin = win;
#pragma unroll
        for (int q = 0; q < Q; q++)
            if (wall_class(D, R, q) == 1) rin += f[q];
        const T rw = rin * den;
#pragma unroll
        for (int q = 0; q < Q; q++) {
            if (wall_class(D, R, q) == 3) f[q] = fma_t(rw, coef(q), -T(wgt(D, q)));
            if (wall_class(D, R, q) == 2) f[q] = fma_t(rw, coef(q), f[opp(D, q)]);
        }
    } else {
        T rin = T(0);
#pragma unroll
        for (int q = 0; q < Q; q++)
            if (wall_class(D, R, q) == 1) {
                if constexpr (ST != MPLBHIP_STORE_F64) f[q] += T(wgt(D, q));
                rin += f[q];
            }
        const T rw = T(2) * rin / den;
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const T wr = T(wgt(D, q)) * rw;
            if (wall_class(D, R, q) == 3) f[q] = wr * coef(q);
            if (wall_class(D, R, q) == 2) f[q] = wr * coef(q) + f[opp(D, q)];
        }
        if constexpr (ST != MPLBHIP_STORE_F64) {
#pragma unroll
            for (int q = 0; q < Q; q++) f[q] -= T(wgt(D, q));
        }
    }
}

// The bits of wall_class 1 of a region; class 2 are the opposite ones, as
// every wall region has them.
template <int D> __host__ __device__ constexpr uint32_t wall_in(int r) {
    uint32_t m = 0;
    for (int q = 0; q < lq(D); q++)
        if (wall_class(D, r, q) == 1) m |= 1u << q;
    return m;
}

// known_wall for lanes of different regions at once, by the lane's wall_in
// mask (0: no wall, f stays) and values: the lanes of a corner tile take one
// pass and one division instead of one each per face and corner.
template <int D, int ST, typename T>
__device__ __forceinline__ void lane_wall(T* f, uint32_t in, T win, T den, const T* c) {
#pragma clang fp contract(off)
    constexpr int Q = lq(D);
    T rin = ST == MPLBHIP_STORE_F64 ? T(0) : win;
#pragma unroll
    for (int q = 1; q < Q; q++) rin += (in >> q & 1u) ? f[q] : T(0);
    const T rw = ST == MPLBHIP_STORE_F64 ? T(2) * rin / den : rin * den;
    const bool wall = in != 0;
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int p = opp(D, q);
        if (p < q) continue;
        const bool qi = in >> q & 1u, pi = in >> p & 1u;
        if constexpr (ST == MPLBHIP_STORE_F64) {
            const T wr = T(wgt(D, q)) * rw;
            const T vq = wr * c[q] + (pi ? f[p] : T(0)), vp = wr * c[p] + (qi ? f[q] : T(0));
            f[q] = wall && !qi ? vq : f[q];
            if (p != q) f[p] = wall && !pi ? vp : f[p];
        } else {
            const T w = -T(wgt(D, q));
            const T vq = fma_t(rw, c[q], pi ? f[p] : w), vp = fma_t(rw, c[p], qi ? f[q] : w);
            f[q] = wall && !qi ? vq : f[q];
            if (p != q) f[p] = wall && !pi ? vp : f[p];
        }
    }
}

// rescale part of KerCutCellExtrapolPressure1ST[3D]
// (boundary_kernel.inc:404-488, 894-1182); f already holds the copied
// populations.  The loop stops before the last population (:484, :1178).
template <int D, typename T>
__device__ void extrapol_rescale(T* f, double rho_given) {
#pragma clang fp contract(off)
    constexpr int Q = lq(D);
    T rho = T(0);
#pragma unroll
    for (int q = 0; q < Q; q++) rho += f[q];
    const T ratio = T(rho_given) / rho;
#pragma unroll
    for (int q = 0; q < Q - 1; q++) f[q] *= ratio;
}

// ---- node addressing --------------------------------------------------------
template <int D>
__device__ __forceinline__ int32_t pull_delta(const BlockParams& B, int q) {
    return cvel(D, q, 0) + cvel(D, q, 1) * B.sx + cvel(D, q, 2) * B.sz;
}

// element q*sq + node - delta of a block array: the uniform part forms a
// scalar base, the per-thread part a 32-bit byte offset (saddr addressing)
template <typename E>
__device__ __forceinline__ const E* at_u(const E* base, int64_t uniform, uint32_t node) {
    return reinterpret_cast<const E*>(reinterpret_cast<const char*>(base + uniform) +
                                      node * (uint32_t)sizeof(E));
}
template <typename E>
__device__ __forceinline__ E* at_u(E* base, int64_t uniform, uint32_t node) {
    return reinterpret_cast<E*>(reinterpret_cast<char*>(base + uniform) +
                                node * (uint32_t)sizeof(E));
}

// Raw buffer accesses (address = resource base + lane offset + scalar
// offset): the per-population part of an address is a scalar operand of
// the instruction, so a population costs no vector address arithmetic.
// Word 3 0x00020000 is the raw (untyped) buffer format; the record count
// 0xFFFFFFFF leaves every offset below 4 GiB in range.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(uint64_t base) {
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(base), 0, -1, 0x00020000);
}
template <typename E>
__device__ __forceinline__ E buf_ld(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    if constexpr (sizeof(E) == 2)
        return __ushort_as_half(__builtin_amdgcn_raw_buffer_load_b16(r, voff, soff, 0));
    else if constexpr (sizeof(E) == 4)
        return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
    else
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
// AUX: cache policy, 0 plain, 2 nontemporal (nt)
template <typename E, int AUX>
__device__ __forceinline__ void buf_st(E v, __amdgpu_buffer_rsrc_t r, uint32_t voff,
                                       uint32_t soff) {
    if constexpr (sizeof(E) == 2)
        __builtin_amdgcn_raw_buffer_store_b16(__half_as_ushort(v), r, voff, soff, AUX);
    else if constexpr (sizeof(E) == 4)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, voff, soff, AUX);
    else
        __builtin_amdgcn_raw_buffer_store_b64(
            __builtin_bit_cast(decltype(__builtin_amdgcn_raw_buffer_load_b64(r, 0, 0, 0)), v), r,
            voff, soff, AUX);
}

__device__ __forceinline__ int region_code(int x, int n) {
    return x == 0 ? 1 : (x == n - 1 ? 2 : 0);
}

template <int D, typename PR = RegionProg>
__device__ __forceinline__ int64_t persist_slot(const PR& P, int x, int y, int z) {
    const int l0 = P.ext[0] > 1 ? x - 1 : 0;
    const int l1 = P.ext[1] > 1 ? y - 1 : 0;
    const int l2 = (D != 2 && P.ext[2] > 1) ? z - 1 : 0;
    return (int64_t)P.persist + l0 + (int64_t)P.ext[0] * (l1 + (int64_t)P.ext[1] * l2);
}

// obstacle link mask of interior node mnode (0 when the block has none)
__device__ __forceinline__ uint32_t obst_mask(const KParams& kp, const BlockParams& B,
                                              int64_t mnode) {
    return (kp.obst && B.has_obst) ? kp.obst[mnode] : 0u;
}

// residual terms of a node whose macros do not change (ImmersedSolid):
// (m - m_copy)^2 and m^2, with the copy refreshed, as the whole-range sums
// of CalcResidualError include them (flowfield_wrapper.cpp:31-89)
template <int D, int MODE>
__device__ __forceinline__ void solid_residual(const KParams& kp, int64_t mnode, double* acc) {
    if constexpr (MODE == MODE_STEP_CHECK || MODE == MODE_MATERIALIZE) {
        if (kp.want_residual) {
#pragma unroll
            for (int v = 0; v < ldim(D) + 1; v++) {
                const double m = kp.macro[v][mnode];
                const double old = kp.macro_copy[v][mnode];
                acc[v] = (m - old) * (m - old);
                acc[4 + v] = m * m;
                kp.macro_copy[v][mnode] = m;
            }
        }
    }
}

// full-value state of a node at the start of the boundary stage: streamed
// populations from the neighbours, unstreamed ones from the persist buffer
// PR: RegionProg, or the constant-address-space RegionProg of a
// wave-uniform program (scalar loads)
template <int D, int ST, typename PR = RegionProg>
__device__ void gather_masked(const KParams& kp, const BlockParams& B,
                              const PR& P, int x, int y, int z,
                              typename Store<ST>::T* f, const void* fs_prev,
                              const void* per_prev, uint32_t om) {
    using T = typename Store<ST>::T;
    using E = typename Store<ST>::E;
    constexpr int Q = lq(D);
    const E* prev = static_cast<const E*>(fs_prev) + B.base;
    const int32_t node = z * B.sz + y * B.sx + x;
    const T* per = static_cast<const T*>(per_prev);
    int64_t slot = P.persist >= 0 ? persist_slot<D, PR>(P, x, y, z) : 0;
#pragma unroll
    for (int q = 0; q < Q; q++) {
        T v;
        if (P.pull >> q & 1u) {
            // an obstacle source bounces back the node's own opposite value
            if (om >> q & 1u)
                v = ld<ST>(prev, (int64_t)opp(D, q) * B.sq + node, kp.scale[opp(D, q)]);
            else
                v = ld<ST>(prev, (int64_t)q * B.sq + node - pull_delta<D>(B, q),
                           kp.scale[q]);
            if constexpr (ST != MPLBHIP_STORE_F64) v += T(wgt(D, q));
        } else if (P.persist >= 0) {
            v = per[slot * Q + q];
        } else {
            v = T(0);
        }
        f[q] = v;
    }
}

// one population of a neighbour, as the extrapolation reads it: after the
// neighbour's boundary applications that precede it in definition order
template <int D, int ST>
__device__ void neighbour_values(const KParams& kp, const BlockParams& B,
                                 const BCOp& op, int x, int y, int z,
                                 typename Store<ST>::T* f, const void* fs_prev,
                                 const void* per_prev) {
    using T = typename Store<ST>::T;
    constexpr int Q = lq(D);
    const RegionProg& N = kp.progs[B.prog_base + op.nb_region];
    const int nx = x + op.off[0], ny = y + op.off[1], nz = z + op.off[2];
    const int64_t nm = B.mbase + ((int64_t)nz * B.n[1] + ny) * B.n[0] + nx;
    T g[Q];
    gather_masked<D, ST>(kp, B, N, nx, ny, nz, g, fs_prev, per_prev, obst_mask(kp, B, nm));
    for (int o = 0; o < op.nb_nops; o++) {
        if (N.op[o].type == OP_EQM) apply_eqm<D, T>(g, N.op[o]);
    }
#pragma unroll
    for (int q = 0; q < Q; q++)
        if (op.m_ext >> q & 1u) f[q] = g[q];
}

template <int D, int ST, typename PR = RegionProg>
__device__ void boundary_program(const KParams& kp, const BlockParams& B,
                                 const PR& P, int x, int y, int z,
                                 typename Store<ST>::T* f, const void* fs_prev,
                                 const void* per_prev) {
    using T = typename Store<ST>::T;
    for (int o = 0; o < P.nops; o++) {
        BCOp op;
        __builtin_memcpy(&op, (const BCOp*)&P.op[o], sizeof op);
        if (op.type == OP_EQM) {
            apply_eqm<D, T>(f, op);
        } else if (op.type == OP_EXTRAPOL) {
            if (op.m_ext) neighbour_values<D, ST>(kp, B, op, x, y, z, f, fs_prev, per_prev);
            extrapol_rescale<D, T>(f, op.vars[0]);
        }
    }
}

// ---- workgroup reduction of the residual accumulators ------------------------
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__device__ void reduce_store(double* acc, double* out) {
    __shared__ double red[kTY][kNAcc];
    const int lane = threadIdx.x, wv = threadIdx.y;
#pragma unroll
    for (int a = 0; a < kNAcc; a++) {
        const double s = wave_sum(acc[a]);
        if (lane == 0) red[wv][a] = s;
    }
    __syncthreads();
    if (lane == 0 && wv == 0) {
        for (int a = 0; a < kNAcc; a++) {
            double s = 0.0;
            for (int k = 0; k < kTY; k++) s += red[k][a];
            out[a] = s;
        }
    }
}

// logical workgroup -> XCD-contiguous chunk: hardware deals workgroups to
// the 8 XCDs round robin; this hands each XCD a contiguous run of tiles so
// that neighbouring tiles (and their halo re-reads) share an L2.
__device__ __forceinline__ int logical_wg(int wg, int n) {
    if ((n & 7) != 0) return wg;
    return (wg & 7) * (n >> 3) + (wg >> 3);
}

// workgroup -> tile such that the tx tiles of one row go to the same XCD
// (workgroups b, b+8, b+16, ... share an XCD) while consecutive rows are
// spread over the 8 XCDs; a bijection when the grid is a multiple of 8*tx
__device__ __forceinline__ int fast_div(int n, uint32_t m, int sh) {
    return (int)(((uint64_t)(uint32_t)n * m) >> sh);
}

// (the division by tx as the block's multiply-high-and-shift pair m, sh)
__device__ __forceinline__ int row_group_wg(int b, int tx, uint32_t m, int sh) {
    const int j = b >> 3;
    const int jq = fast_div(j, m, sh);
    return (jq * 8 + (b & 7)) * tx + (j - jq * tx);
}

// Block parameters and parities are never written while a step kernel
// runs.  Read through the constant address space, a wave-uniform index
// turns their loads into scalar loads: one batched round trip per wave
// instead of a chain of dependent vector loads ahead of the population
// loads.
#define MPLB_CONST __attribute__((address_space(4)))
template <typename T>
__device__ __forceinline__ const MPLB_CONST T* const_view(const T* p) {
    return (const MPLB_CONST T*)(p);
}

__device__ __forceinline__ BlockParams load_block(const KParams& kp, int b) {
    BlockParams B;
    __builtin_memcpy(&B, (const BlockParams*)&const_view(kp.blocks)[b], sizeof B);
    return B;
}

// the pointer held by the first active lane, as a wave-uniform value
template <typename T>
__device__ __forceinline__ const T* first_lane_ptr(const T* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<const T*>(((uint64_t)hi << 32) | lo);
}

__device__ __forceinline__ int load_parity(const KParams& kp, int b) {
    return const_view(kp.cur_in)[b];
}

// block of logical workgroup wg of a grid, from that grid's table (wg is
// wave-uniform: a scalar load); a one-block case reads nothing
__device__ __forceinline__ int wg_block(const KParams& kp, const int32_t* table, int wg) {
    return kp.nblocks == 1 ? 0 : const_view(table)[wg];
}

// where a node's new populations go: HBM, nontemporal.  BUF: raw buffer
// stores (next is wave-uniform), else global ones.
template <int ST, bool BUF>
struct NodeStore {
    using T = typename Store<ST>::T;
    using E = typename Store<ST>::E;
    const BlockParams& B;
    E* next;
    int32_t node;
    // v: the new value in storage units (h = g / s_q for FP16)
    __device__ __forceinline__ void operator()(int q, T v) const {
        if constexpr (BUF) {
            const __amdgpu_buffer_rsrc_t rput = buf_rsrc(reinterpret_cast<uint64_t>(next));
            const uint32_t voff = (uint32_t)node * (uint32_t)sizeof(E);
            if constexpr (ST == MPLBHIP_STORE_F16)
                buf_st<E, 2>(__float2half_rn(v), rput, voff, B.put_off[q]);
            else buf_st<E, 2>(v, rput, voff, B.put_off[q]);
            return;
        }
        E* p = at_u(next, (int64_t)q * B.sq, (uint32_t)node);
        if constexpr (ST == MPLBHIP_STORE_F64) *p = v;
        else if constexpr (ST == MPLBHIP_STORE_F16)
            __builtin_nontemporal_store(__half_as_ushort(__float2half_rn(v)),
                                        reinterpret_cast<unsigned short*>(p));
        else __builtin_nontemporal_store(v, p);
    }
};

// macros (+ residual partials), then the MATERIALIZE output or the BGK
// collision, whose new populations go to `store` (population, value in
// storage units).  f holds full values when `full` (boundary path), else
// (reduced storage) deviations g = f - w.
// EXTRA: what the case may have besides plain BGK: 0 nothing, 1 a body force,
// 2 that and Collision_BGKThermal4th (FP64).
template <int D, int ST, int MODE, int EXTRA = 2, typename SINK = NodeStore<ST, false>>
__device__ __forceinline__ void finish_node(const KParams& kp, const BlockParams& B,
                                            typename Store<ST>::T* f, bool full,
                                            bool force_node, int64_t mnode, const SINK& store,
                                            int x, int y, int z, double* acc) {
    using T = typename Store<ST>::T;
    constexpr int Q = lq(D);
    constexpr bool EXACT = ST == MPLBHIP_STORE_F64;
    (void)full;
    if constexpr (EXACT) {
#pragma clang fp contract(off)
        // UpdateMacroVars: density then each velocity component
        double rho = 0;
#pragma unroll
        for (int q = 0; q < Q; q++) rho += f[q];
        double uvw[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int d = 0; d < ldim(D); d++) {
            // u = sum_q (CS c_qd) f_q: the terms with c_qd = 0 add a zero and
            // are left out, and (-CS) f is -(CS f) exactly
            double u = 0;
#pragma unroll
            for (int q = 0; q < Q; q++) {
                if (cvel(D, q, d) > 0) u += kCS * f[q];
                if (cvel(D, q, d) < 0) u -= kCS * f[q];
            }
            u /= rho;
            if (EXTRA > 0 && kp.force_macros && force_node) u += (B.dt * B.g[d] / 2);
            uvw[d] = u;
        }
        if constexpr (MODE == MODE_MATERIALIZE || MODE == MODE_STEP_CHECK) {
            const double m[4] = {rho, uvw[0], uvw[1], uvw[2]};
#pragma unroll
            for (int v = 0; v < ldim(D) + 1; v++) {
                if (kp.want_residual) {
                    const double old = kp.macro_copy[v][mnode];
                    acc[v] = (m[v] - old) * (m[v] - old);
                    acc[4 + v] = m[v] * m[v];
                    kp.macro_copy[v][mnode] = m[v];
                }
                kp.macro[v][mnode] = m[v];
            }
            double mass = 0;
#pragma unroll
            for (int q = 0; q < Q; q++) mass += f[q];
            acc[8] = mass;
        }
        if constexpr (MODE == MODE_MATERIALIZE) {
            if (kp.fhost && !kp.fhost_in) {
                const int64_t nn = (int64_t)B.n[0] * B.n[1] * B.n[2];
                const int64_t h = B.fbase + ((int64_t)z * B.n[1] + y) * B.n[0] + x;
#pragma unroll
                for (int q = 0; q < Q; q++) kp.fhost[h + q * nn] = f[q];
            }
        } else if (EXTRA == 2 && kp.thermal) {
            // KerCollideBGKThermal[3D] (model_kernel.inc:267-310, 457-502):
            // tau = tauRef / (rho sqrt(T)) per node, the 4th-order
            // equilibrium at T, and f - w (f - feq) (+ tau w F)
            const double Tm = kp.temp[mnode];
            const double tau = B.tau / (rho * sqrt(Tm));
            const double om = B.dt / (tau + 0.5 * B.dt);
            const bool addf = force_node && kp.force_type == 1;
#pragma unroll
            for (int q = 0; q < Q; q++) {
                const double fe = feq4_ref<D>(q, rho, uvw[0], uvw[1], uvw[2], Tm);
                double fsq = f[q] - om * (f[q] - fe);
                if (addf) {
                    double cf = 0;
#pragma unroll
                    for (int d = 0; d < ldim(D); d++)
                        cf += kCS * double(cvel(D, q, d)) * B.g[d];
                    const double F = wgt(D, q) * rho * cf;
                    fsq = fsq + tau * om * F;
                }
                store(q, fsq);
            }
        } else {
            // BGK collision with the optional first-order force source
            const double tw = B.tau_omega, om1 = B.one_minus_omega;
            const bool addf = EXTRA > 0 && force_node && kp.force_type == 1;
            // CalcBGKFeq (feq_ref) with the same operations on the same
            // values in the same order: terms with c = 0 add a zero and are
            // left out, and an opposite velocity's cu is the exact negative,
            // so the pair shares cu^2 and 0.5 (cu^2 - u^2).  Per node of
            // D3Q19 this issues 60% of the plain form's instructions.
            double u2 = uvw[0] * uvw[0] + uvw[1] * uvw[1];
            if constexpr (ldim(D) == 3) u2 = u2 + uvw[2] * uvw[2];
            auto put = [&](int q, double fe) {
                double fsq = fe + om1 * (f[q] - fe);
                if (addf) {
                    double cf = 0;
#pragma unroll
                    for (int d = 0; d < ldim(D); d++)
                        cf += kCS * double(cvel(D, q, d)) * B.g[d];
                    const double F = wgt(D, q) * rho * cf;
                    fsq = fsq + tw * F;
                }
                store(q, fsq);
            };
            put(0, wgt(D, 0) * rho * (1.0 + 0.5 * (0.0 - u2)));
#pragma unroll
            for (int q = 1; q < Q; q++) {
                const int p = opp(D, q);
                if (p < q) continue;
                double cu = 0;
                bool any = false;
#pragma unroll
                for (int d = 0; d < ldim(D); d++) {
                    if (cvel(D, q, d) == 0) continue;
                    const double t = kCS * uvw[d];
                    if (cvel(D, q, d) > 0) cu = any ? cu + t : t;
                    else cu = any ? cu - t : -t;
                    any = true;
                }
                const double e = 0.5 * (cu * cu - u2);
                const double wr = wgt(D, q) * rho;
                put(q, wr * (1.0 + cu + e));
                put(p, wr * (1.0 - cu + e));
            }
        }
    } else {
#pragma clang fp contract(off)
        // deviation form g = f - w, FP32 arithmetic; the multiply-adds are
        // written out, so that every kernel built on this function rounds
        // alike
        if (full) {
#pragma unroll
            for (int q = 0; q < Q; q++) f[q] -= T(wgt(D, q));
        }
        float drho = 0.f, j[3] = {0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < Q; q++) {
            drho += f[q];
#pragma unroll
            for (int d = 0; d < ldim(D); d++) {
                if (cvel(D, q, d) > 0) j[d] += f[q];
                if (cvel(D, q, d) < 0) j[d] -= f[q];
            }
        }
        const float rho = 1.f + drho;
        const float inv = __builtin_amdgcn_rcpf(rho);  // v_rcp_f32, 1 ulp
        float ul[3] = {0.f, 0.f, 0.f};
#pragma unroll
        for (int d = 0; d < ldim(D); d++) {
            ul[d] = j[d] * inv;
            if (EXTRA > 0 && kp.force_macros && force_node) ul[d] = __builtin_fmaf(j[d], inv, B.fhalf_dtg[d]);
        }
        float usq = __builtin_fmaf(ul[0], ul[0], ul[1] * ul[1]);
        if constexpr (ldim(D) == 3) usq = __builtin_fmaf(ul[2], ul[2], usq);
        if constexpr (MODE == MODE_MATERIALIZE || MODE == MODE_STEP_CHECK) {
            double dr = 0.0;
#pragma unroll
            for (int q = 0; q < Q; q++) dr += double(f[q]);
            const double m[4] = {1.0 + dr, kCS * double(ul[0]), kCS * double(ul[1]),
                                 kCS * double(ul[2])};
#pragma unroll
            for (int v = 0; v < ldim(D) + 1; v++) {
                if (kp.want_residual) {
                    const double old = kp.macro_copy[v][mnode];
                    acc[v] = (m[v] - old) * (m[v] - old);
                    acc[4 + v] = m[v] * m[v];
                    kp.macro_copy[v][mnode] = m[v];
                }
                kp.macro[v][mnode] = m[v];
            }
            acc[8] = 1.0 + dr;
        }
        if constexpr (MODE == MODE_MATERIALIZE) {
            if (kp.fhost && !kp.fhost_in) {
                const int64_t nn = (int64_t)B.n[0] * B.n[1] * B.n[2];
                const int64_t h = B.fbase + ((int64_t)z * B.n[1] + y) * B.n[0] + x;
#pragma unroll
                for (int q = 0; q < Q; q++)
                    kp.fhost[h + q * nn] = double(f[q]) + wgt(D, q);
            }
        } else {
            const float om = B.fomega, om1 = B.fone_minus_omega;
            const bool addf = EXTRA > 0 && force_node && kp.force_type == 1;
            const float c0 = __builtin_fmaf(rho, -1.5f * usq, drho);
            if constexpr (ST == MPLBHIP_STORE_F16) {
                // g' = (1 - om) g + om geq in storage units h = g / s_q
                // (s_q = w_q / kF16Scale).  Opposite velocities share the
                // even part of the equilibrium: geq(q), geq(opp q) = w_q (A
                // +- B) with A = drho + rho (4.5 cu^2 - 1.5 u^2), B = 3 rho
                // cu, so h' = m_q g + k (A +- B), m_q = (1 - om) / s_q, k =
                // om kF16Scale (w_q cancels); the force term changes sign too
                const float k = om * float(kF16Scale);
                auto m_of = [&](int q) { return om1 * float(kF16Scale / wgt(D, q)); };
                store(0, __builtin_fmaf(m_of(0), f[0], k * c0));
                const float ka = (k * 4.5f) * rho, kb = (k * 3.f) * rho, kc = k * c0;
#pragma unroll
                for (int q = 1; q < Q; q++) {
                    const int p = opp(D, q);
                    if (p < q) continue;
                    // c.u without a leading 0 + (which would not fold away)
                    float cu = 0.f;
                    bool any = false;
#pragma unroll
                    for (int d = 0; d < ldim(D); d++) {
                        if (cvel(D, q, d) > 0) { cu = any ? cu + ul[d] : ul[d]; any = true; }
                        if (cvel(D, q, d) < 0) { cu = any ? cu - ul[d] : -ul[d]; any = true; }
                    }
                    const float a = __builtin_fmaf(ka, cu * cu, kc);
                    float hq = __builtin_fmaf(kb, cu, a), hp = __builtin_fmaf(-kb, cu, a);
                    if (addf) {
                        float cg = 0.f;
#pragma unroll
                        for (int d = 0; d < ldim(D); d++)
                            cg += float(cvel(D, q, d)) * float(B.g[d]);
                        const float fq = B.fforce * float(kF16Scale) * cg;
                        hq = __builtin_fmaf(fq, rho, hq);
                        hp = __builtin_fmaf(-fq, rho, hp);
                    }
                    const float m = m_of(q);
                    store(q, __builtin_fmaf(m, f[q], hq));
                    store(p, __builtin_fmaf(m, f[p], hp));
                }
            } else {
                // opposite velocities share the even part of the
                // equilibrium: geq(q), geq(opp q) = A +- Bq with A = w (drho
                // + rho (4.5 cu^2 - 1.5 u^2)), Bq = 3 w rho cu, and the force
                // term changes sign
                store(0, __builtin_fmaf(om1, f[0], om * (float(wgt(D, 0)) * c0)));
#pragma unroll
                for (int q = 1; q < Q; q++) {
                    const int p = opp(D, q);
                    if (p < q) continue;
                    float cu = 0.f;
#pragma unroll
                    for (int d = 0; d < ldim(D); d++) {
                        if (cvel(D, q, d) > 0) cu += ul[d];
                        if (cvel(D, q, d) < 0) cu -= ul[d];
                    }
                    const float wq = float(wgt(D, q));
                    const float a = __builtin_fmaf(rho, (4.5f * cu) * cu, c0);
                    const float bq = (wq * rho) * (3.f * cu);
                    float gq = __builtin_fmaf(om1, f[q], om * __builtin_fmaf(a, wq, bq));
                    float gp = __builtin_fmaf(om1, f[p], om * __builtin_fmaf(a, wq, -bq));
                    if (addf) {
                        float cg = 0.f;
#pragma unroll
                        for (int d = 0; d < ldim(D); d++)
                            cg += float(cvel(D, q, d)) * float(B.g[d]);
                        const float fq = (B.fforce * wq) * rho;
                        gq = __builtin_fmaf(fq, cg, gq);
                        gp = __builtin_fmaf(-fq, cg, gp);
                    }
                    store(q, gq);
                    store(p, gp);
                }
            }
        }
    }
}

}  // namespace mplbhip
