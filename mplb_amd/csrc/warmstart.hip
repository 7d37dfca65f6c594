// warmstart.hip -- kernels of the learned warm start (a small U-Net that
// predicts the steady cavity flow from the obstacle mask and Re): 3x3
// convolutions as implicit GEMMs on the gfx950 matrix cores
// (v_mfma_f32_32x32x16_bf16: BF16 operands, FP32 accumulation), their data
// and weight gradients, and the element-wise layers, loss and optimiser.
// C ABI in include/mplbws.h.  No reference counterpart: the reference
// starts every run from its initial macros.
//
// Tensors are FP32 in HBM, channels last: x[n][y][x][c].  Operands are
// rounded to BF16 (nearest even) as they are loaded into the MFMA
// fragments.  Convolution weights are laid out [tap = 3*ky + kx][cin][cout].
#include "../../include/mplbws.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

namespace {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWaves = 4;  // waves per workgroup

// Forward 3x3 convolution as an implicit GEMM, out[m][co] = sum_{tap, ci}
// in[shift_tap(m)][ci] * w[tap][ci][co], zero padding at the image edges.
//
// A workgroup (4 waves) owns a tile of TP = 128 WM output pixels -- R rows of
// W0 <= 32 columns, nearly square so that its halo is small -- and CG = 32 WN
// output channels.  Input channels go in chunks of kCC: the chunk's input tile
// with its one-pixel halo is converted to BF16 once into LDS (zeros outside
// the image), and so are the chunk's weights, in the MFMA operand layout; the
// waves then run the 9 taps from LDS only.  Wave v takes pixels
// [32 WM v, 32 WM (v + 1)) of the tile and all CG channels: WM x WN
// accumulators of 32x32.  The weights are the A operand, so a lane's
// accumulators hold four consecutive channels of one pixel, one 16-byte store.
//
// Bound: the staging, whose latency two to three workgroups per CU hide in
// part: 32 images of 128 x 128, 72 to 24 channels read and write 201 MB, 32 us
// of HBM, and take 62 us (135 with tiles of one row of 128 pixels, products of
// 8 channels, integer rounding to BF16 and 64-bit addresses).  64 x 64, 48 to
// 48 channels 51 -> 20 us, 128 to 64 channels at 128 x 128 266 -> 140 us.
//
// MFMA 32x32x16 (BF16 in, FP32 accumulate) lane layout: lane l holds
// A[l%32][8(l/32) .. +7] and B[8(l/32) .. +7][l%32]; the accumulator
// element 4i+j of lane l is C[8i + 4(l/32) + j][l%32].
constexpr int kCC = 32;              // input channels per LDS chunk
constexpr int kPixStride = kCC + 8;  // BF16 elements per staged pixel (the
                                     // 16-byte pad spreads a wave's reads
                                     // over all LDS banks)

struct ConvTile {
    int W0, R, tiles_x, tiles_y;
};

// pixels staged for a tile of tp pixels: the largest (R + 2)(W0 + 2)
__host__ __device__ constexpr int conv_max_staged(int tp) { return tp == 256 ? 340 : 204; }

// equal columns of at most 32, or (wide) of as many more as an image of few
// rows leaves pixels for, and as many rows as the tile's pixels and the staged
// ones allow
inline ConvTile conv_tile(int h, int wd, int tp, bool wide) {
    ConvTile t;
    int most = 32;
    if (wide && h < 8) {
        const int row = tp / h, fit = conv_max_staged(tp) / (h + 2) - 2;
        const int w = row < fit ? row : fit;
        if (w > most) most = w;
    }
    t.tiles_x = (wd + most - 1) / most;
    t.W0 = (wd + t.tiles_x - 1) / t.tiles_x;
    t.R = tp / t.W0;
    const int fit = conv_max_staged(tp) / (t.W0 + 2) - 2;
    if (t.R > fit) t.R = fit;
    if (t.R > h) t.R = h;
    t.tiles_y = (h + t.R - 1) / t.R;
    return t;
}

// q = e / d, r = e - q d for 0 <= e < 2^22 and 1 <= d <= 2^10 through a
// float reciprocal (error below one unit before the correction)
struct FastDiv {
    float inv;
    int d;
};
__device__ __forceinline__ FastDiv fast_div(int d) { return FastDiv{1.0f / (float)d, d}; }
__device__ __forceinline__ int fdiv(int e, const FastDiv& f, int* r) {
    int q = (int)((float)e * f.inv);
    int rr = e - q * f.d;
    if (rr < 0) { q--; rr += f.d; }
    if (rr >= f.d) { q++; rr -= f.d; }
    *r = rr;
    return q;
}

// eight floats as BF16 (nearest even), one v_cvt_pk_bf16_f32 per pair
__device__ __forceinline__ bf16x8 to_bf16x8(const float4& a, const float4& b) {
    const f32x8 f = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    return __builtin_convertvector(f, bf16x8);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf(const float* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float4 buf_ld4(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
__device__ __forceinline__ float buf_ld1(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}

// 8 floats from p + off on, `left` of them real; zeros past them
__device__ __forceinline__ void load8_wide(float4* f, const float* p, int64_t off, int left) {
    float v[8];
#pragma unroll
    for (int c = 0; c < 8; c++) v[c] = left > c ? p[off + c] : 0.f;
    f[0] = float4{v[0], v[1], v[2], v[3]};
    f[1] = float4{v[4], v[5], v[6], v[7]};
}

// workgroups are dealt to the 8 XCDs in turn: consecutive tiles, which share
// their halos, on one of them
__device__ __forceinline__ int tile_order(int i, int count) {
    const int per = count / 8, whole = per * 8;
    return i < whole ? (i % 8) * per + i / 8 : i;
}

// How a convolution addresses its operands: by buffer offsets of 32 bits, in
// 16-byte accesses where channel counts and alignment allow them (kFormVec) or
// not; by 64 bits (kFormWide) where a tile's rows, a chunk's or the weights are
// 4 GiB and more.
enum { kFormAny = 0, kFormVec = 1, kFormWide = 2 };
template <int FORM> using Offset = std::conditional_t<FORM == kFormWide, int64_t, uint32_t>;

// kFormVec: cout is a multiple of four, and w and out are aligned for 16-byte
// accesses
template <int WM, int WN, int FORM>
__global__ __launch_bounds__(64 * kWaves, WN == 1 ? 3 : 2) void k_conv_fwd(const float* __restrict__ in,
                                                          const float* __restrict__ w,
                                                          const float* __restrict__ bias,
                                                          float* __restrict__ out, int n,
                                                          int h, int wd, int cin, int cout,
                                                          int relu, ConvTile T) {
    constexpr int TP = 128 * WM, CG = 32 * WN, NT = 64 * kWaves;
    constexpr bool WIDE = FORM == kFormWide, VEC = FORM == kFormVec;
    using Off = Offset<FORM>;
    constexpr Off unit = WIDE ? 1 : 4;  // offsets in floats, or in bytes
    __shared__ __attribute__((aligned(16))) short s_in[conv_max_staged(TP) * kPixStride];
    // A fragments: [tap][8 input channels][co 0 .. CG-1][8]
    __shared__ __attribute__((aligned(16))) short s_w[9 * (kCC / 8) * CG * 8];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int row = lane & 31, g = lane >> 5;
    const int tiles = T.tiles_x * T.tiles_y;
    const int bid = tile_order((int)blockIdx.x, (int)gridDim.x);
    const int pn = bid / tiles;
    const int t = bid % tiles;
    const int y0 = (t / T.tiles_x) * T.R, x0 = (t % T.tiles_x) * T.W0;
    const int co0 = (int)blockIdx.y * CG;
    const int SW = T.W0 + 2, SP = (T.R + 2) * SW;
    const FastDiv dW0 = fast_div(T.W0), dsw = fast_div(SW);
    // this lane's pixel in its WM pixel tiles, and the first of the 3 x 3
    // staged ones it reads; a lane past the tile reads those of pixel (0, 0)
    // instead (its results are never stored)
    int pbase[WM], px[WM], py[WM];
#pragma unroll
    for (int mt = 0; mt < WM; mt++) {
        int tx;
        int ty = fdiv(wave * 32 * WM + mt * 32 + row, dW0, &tx);
        px[mt] = x0 + tx;
        py[mt] = ty < T.R ? y0 + ty : h;
        if (ty >= T.R) ty = tx = 0;
        pbase[mt] = (ty * SW + tx) * kPixStride + 8 * g;
    }
    // Loads by buffer offsets that hold for every chunk, with the chunk and
    // the weight row as scalar offsets and zeros (an offset past the end)
    // outside the image and the weights: with 64-bit addresses and selects
    // the staging issued three quarters of the kernel's instructions.
    // Input item k: 8 channels of a staged pixel.
    constexpr int kIn = (conv_max_staged(TP) * (kCC / 8) + NT - 1) / NT;
    const int ya = y0 > 0 ? y0 - 1 : 0, yb = y0 + T.R + 1 < h ? y0 + T.R + 1 : h;
    const uint32_t ibytes = (uint32_t)(yb - ya) * (uint32_t)wd * (uint32_t)cin * 4u;
    const float* rows_in = in + ((int64_t)pn * h + ya) * wd * cin;
    const __amdgpu_buffer_rsrc_t rin = buf(rows_in, ibytes);
    const Off inone = WIDE ? Off(-1) : Off(ibytes);
    const int c8 = (int)threadIdx.x & 3;
    Off ioff[kIn];
#pragma unroll
    for (int k = 0; k < kIn; k++) {
        const int sp = ((int)threadIdx.x + k * NT) >> 2;
        int sx;
        const int sy = fdiv(sp, dsw, &sx);
        const int yy = y0 + sy - 1, xx = x0 + sx - 1;
        ioff[k] = sp < SP && yy >= 0 && yy < h && xx >= 0 && xx < wd
                      ? (((Off)(yy - ya) * (Off)wd + (Off)xx) * (Off)cin + 8 * c8) * unit
                      : inone;
    }
    // Weight item k: 8 input channels of one tap by 4 output channels.
    constexpr int kTot = 9 * (kCC / 8) * (CG / 4), kW = (kTot + NT - 1) / NT;
    const uint32_t wbytes = 9u * (uint32_t)cin * (uint32_t)cout * 4u;
    const __amdgpu_buffer_rsrc_t rw = buf(w, wbytes);
    const Off wnone = WIDE ? Off(-1) : Off(wbytes);
    Off woff[kW];
#pragma unroll
    for (int k = 0; k < kW; k++) {
        const int e = (int)threadIdx.x + k * NT;
        const int oc = co0 + (e % (CG / 4)) * 4, j = e / (CG / 4);
        woff[k] = e < kTot && oc < cout
                      ? (((Off)(j >> 2) * cin + 8 * (j & 3)) * (Off)cout + oc) * unit
                      : wnone;
    }
    f32x16 acc[WM][WN] = {};
    for (int c0 = 0; c0 < cin; c0 += kCC) {
        const int cc = cin - c0 < kCC ? cin - c0 : kCC;  // a multiple of 8
        const int g8 = (cc + 15) / 16 * 2;  // groups of 8 staged, zeros past cc
        float4 f[kIn][2];
#pragma unroll
        for (int k = 0; k < kIn; k++) {
            const Off off = 8 * c8 < cc ? ioff[k] : inone;
            if constexpr (WIDE) {
                load8_wide(f[k], rows_in, off + c0, off < 0 ? 0 : 8);
            } else {
                f[k][0] = buf_ld4(rin, off, c0 * 4u);
                f[k][1] = buf_ld4(rin, off, c0 * 4u + 16u);
            }
        }
        float4 u[8];
        auto load_w = [&](int k) {
            const int j = ((int)threadIdx.x + k * NT) / (CG / 4);
            const Off off = 8 * (j & 3) < cc ? woff[k] : wnone;
#pragma unroll
            for (int r = 0; r < 8; r++) {
                const Off so = (Off)(c0 + r) * (Off)cout * unit;
                if constexpr (WIDE) {
                    const int left = off < 0 ? 0 : cout - (int)(off % cout);
                    const float* p = w + off + so;
                    u[r].x = left > 0 ? p[0] : 0.f;
                    u[r].y = left > 1 ? p[1] : 0.f;
                    u[r].z = left > 2 ? p[2] : 0.f;
                    u[r].w = left > 3 ? p[3] : 0.f;
                } else if constexpr (VEC) {
                    u[r] = buf_ld4(rw, off, so);
                } else {
                    const int left = off < wbytes ? cout - (int)((off / 4u) % (uint32_t)cout) : 0;
                    u[r].x = buf_ld1(rw, off, so);
                    u[r].y = buf_ld1(rw, left > 1 ? off + 4u : wbytes, so);
                    u[r].z = buf_ld1(rw, left > 2 ? off + 8u : wbytes, so);
                    u[r].w = buf_ld1(rw, left > 3 ? off + 12u : wbytes, so);
                }
            }
        };
        load_w(0);
        if (c0) __syncthreads();  // the previous chunk's reads are done
#pragma unroll
        for (int k = 0; k < kIn; k++) {
            const int sp = ((int)threadIdx.x + k * NT) >> 2;
            if (sp < SP && c8 < g8)
                *reinterpret_cast<bf16x8*>(&s_in[sp * kPixStride + 8 * c8]) =
                    to_bf16x8(f[k][0], f[k][1]);
        }
#pragma unroll
        for (int k = 0; k < kW; k++) {
            if (k) load_w(k);
            const int e = (int)threadIdx.x + k * NT;
            const int co4 = (e % (CG / 4)) * 4, j = e / (CG / 4);
            if (e >= kTot || (j & 3) >= g8) continue;
            short* dst = &s_w[(j * CG + co4) * 8];
            auto put = [&](int c, float4 a, float4 b) {
                *reinterpret_cast<bf16x8*>(dst + 8 * c) = to_bf16x8(a, b);
            };
            put(0, float4{u[0].x, u[1].x, u[2].x, u[3].x}, float4{u[4].x, u[5].x, u[6].x, u[7].x});
            put(1, float4{u[0].y, u[1].y, u[2].y, u[3].y}, float4{u[4].y, u[5].y, u[6].y, u[7].y});
            put(2, float4{u[0].z, u[1].z, u[2].z, u[3].z}, float4{u[4].z, u[5].z, u[6].z, u[7].z});
            put(3, float4{u[0].w, u[1].w, u[2].w, u[3].w}, float4{u[4].w, u[5].w, u[6].w, u[7].w});
        }
        __syncthreads();
        // the taps' offsets are immediate ones but for the row's
        auto products = [&](auto steps) {
#pragma unroll
            for (int dy = 0; dy < 3; dy++) {
                const short* rows[WM];
#pragma unroll
                for (int mt = 0; mt < WM; mt++)
                    rows[mt] = &s_in[pbase[mt] + dy * SW * kPixStride];
                const short* wl = &s_w[(g * CG + row) * 8];
#pragma unroll
                for (int dx = 0; dx < 3; dx++)
#pragma unroll
                    for (int ks = 0; ks < decltype(steps)::value; ks++) {
                        bf16x8 a[WN], b[WM];
#pragma unroll
                        for (int mt = 0; mt < WM; mt++)
                            b[mt] = *reinterpret_cast<const bf16x8*>(rows[mt] + dx * kPixStride +
                                                                     ks * 16);
#pragma unroll
                        for (int nt = 0; nt < WN; nt++)
                            a[nt] = *reinterpret_cast<const bf16x8*>(
                                wl + (((3 * dy + dx) * (kCC / 8) + 2 * ks) * CG + nt * 32) * 8);
#pragma unroll
                        for (int mt = 0; mt < WM; mt++)
#pragma unroll
                            for (int nt = 0; nt < WN; nt++)
                                acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                                    a[nt], b[mt], acc[mt][nt], 0, 0, 0);
                    }
            }
        };
        if (g8 == 4) products(std::integral_constant<int, 2>{});
        else products(std::integral_constant<int, 1>{});
    }
    // epilogue: bias, relu, FP32 store
#pragma unroll
    for (int nt = 0; nt < WN; nt++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int co = co0 + nt * 32 + 8 * i + 4 * g;
            float bv[4];
#pragma unroll
            for (int j = 0; j < 4; j++) bv[j] = bias && co + j < cout ? bias[co + j] : 0.f;
#pragma unroll
            for (int mt = 0; mt < WM; mt++) {
                if (py[mt] >= h || px[mt] >= wd || co >= cout) continue;
                float v[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    v[j] = acc[mt][nt][4 * i + j] + bv[j];
                    if (relu) v[j] = v[j] > 0.f ? v[j] : 0.f;
                }
                float* dst = out + (((int64_t)pn * h + py[mt]) * wd + px[mt]) * cout + co;
                if constexpr (VEC) {
                    *reinterpret_cast<float4*>(dst) = float4{v[0], v[1], v[2], v[3]};
                } else {
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        if (co + j < cout) dst[j] = v[j];
                }
            }
        }
}

// weights of the data gradient: wt[tap][co][ci] = w[8 - tap][ci][co]
__global__ void k_flip_weights(const float* __restrict__ w, float* __restrict__ wt, int cin,
                               int cout) {
    const int64_t total = 9LL * cin * cout;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int ci = (int)(i % cin);
        const int co = (int)((i / cin) % cout);
        const int tap = (int)(i / ((int64_t)cin * cout));
        wt[i] = w[((int64_t)(8 - tap) * cin + ci) * cout + co];
    }
}

// Pixel chunks of the weight gradient: whole rows of one image, about
// MPLBWS_WGRAD_CHUNK pixels each, so that a chunk's pixel coordinates need
// no division.
__host__ __device__ inline int wgrad_rows(int h, int wd) {
    int r = MPLBWS_WGRAD_CHUNK / wd;
    if (r < 1) r = 1;
    if (r > h) r = h;
    return r;
}

// Weight gradient partials of one chunk of whole rows: partial[chunk][tap][ci]
// [co] = sum over its pixels m of in[shift_tap(m)][ci] dout[m][co], products
// of 16 pixels.  A workgroup takes 32 input and 32 output channels, one wave
// per tap; sub-tiles of at most kGPix pixels (RT lines of SEG positions, a
// multiple of 16) of dout, and of the input with a pixel around them, are
// converted to BF16 once into LDS as they lie in HBM, a pixel's 32 channels in
// a row, and read transposed (ds_read_b64_tr_b16): the product's reduction
// runs over pixels, and a tap is a shift by whole pixels, which needs no
// alignment.  Lines are the chunk's rows, or (TURN) its columns.  The
// workgroups of the first input channels also sum the dout values they load
// (FP32, fixed order) into bpart[chunk][co] when it is given.
//
// Bound: the loads of one sub-tile per workgroup in flight, and too few
// workgroups for the chip when the chunks are few (one image of 64 x 64: 2 us
// per sub-tile either way).  With both sums, us: 32 images of 64 x 64, 48 to 48
// channels 123 -> 47, 128 x 128, 72 to 24 356 -> 100 and 128 to 64 731 -> 204,
// 8 x 8, 128 to 64 18.7 -> 13.3 (before: every operand by 4-byte loads from
// HBM, again for each of the 9 cin / 32 tiles, one wave's rows at a time).  A
// workgroup per row of taps with the pixels dealt to 4 or 8 waves and their
// tiles summed in LDS took 52 to 103, its staging three times as much.
constexpr int kGWaves = 9;
constexpr int kGPix = 256;   // pixels of dout staged
constexpr int kGIn = 396;    // and of the input: (RT + 2)(SEG + 2), 4 lines of 64 the most

// positions and lines of a sub-tile, by those of a whole chunk
struct GradTile {
    int seg, segs, rt;
};
inline GradTile grad_tile(int lines, int positions) {
    GradTile t;
    const int most = lines == 1 ? 128 : lines == 2 ? 96 : 64;
    t.segs = (positions + most - 1) / most;
    t.seg = ((positions + t.segs - 1) / t.segs + 15) / 16 * 16;
    t.rt = kGPix / t.seg < lines ? kGPix / t.seg : lines;
    return t;
}
// sub-tiles of a chunk
inline int64_t grad_tiles(int lines, int positions) {
    const GradTile t = grad_tile(lines, positions);
    return (int64_t)((lines + t.rt - 1) / t.rt) * t.segs;
}

// four pixels of one channel: the 16 lanes of a row each point at 4 channels
// of one of them
__device__ __forceinline__ s16x4 lds_tr(const short* p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
}

// 8 channels at a byte offset, `left` of them (kFormVec: a multiple of 4) real;
// zeros past them and for off = bytes.  kFormAny's loads are as wide, at any
// multiple of four bytes, and what is not this pixel's is dropped (8
// images of 64 x 64, 35 to 33 channels: 105 us by single floats, 48).
template <int FORM>
__device__ __forceinline__ void load8(float4* f, __amdgpu_buffer_rsrc_t r, uint32_t off, int left,
                                      uint32_t bytes) {
    f[0] = buf_ld4(r, left > 0 ? off : bytes, 0);
    f[1] = buf_ld4(r, left > 4 ? off + 16u : bytes, 0);
    if constexpr (FORM == kFormAny) {
        f[0].y = left > 1 ? f[0].y : 0.f;
        f[0].z = left > 2 ? f[0].z : 0.f;
        f[0].w = left > 3 ? f[0].w : 0.f;
        f[1].y = left > 5 ? f[1].y : 0.f;
        f[1].z = left > 6 ? f[1].z : 0.f;
        f[1].w = left > 7 ? f[1].w : 0.f;
    }
}

// kFormVec: cin and cout are multiples of four, in and dout aligned for 16-byte
// accesses.
// TURN: where the chunk is in fewer sub-tiles by columns than by rows (1 x 4096
// pixels by rows would be 256 sub-tiles of 16 columns each, one of them real:
// 64 to 64 channels 1270 us, 55; 8 columns 166, 40).
template <int FORM, bool TURN>
__global__ __launch_bounds__(64 * kGWaves) void k_conv_wgrad(const float* __restrict__ in,
                                                                const float* __restrict__ dout,
                                                                float* __restrict__ partial,
                                                                float* __restrict__ bpart, int h,
                                                                int wd, int cin, int cout,
                                                                int rows, GradTile T) {
    constexpr int NT = 64 * kGWaves, NP = NT / 4;
    constexpr bool WIDE = FORM == kFormWide;
    using Off = Offset<FORM>;
    constexpr Off unit = WIDE ? 1 : 4;  // offsets in floats, or in bytes
    // [pixel][32 channels]
    __shared__ __attribute__((aligned(16))) short s_x[kGIn * 32];
    __shared__ __attribute__((aligned(16))) short s_d[kGPix * 32];
    const int lane = threadIdx.x & 63, tap = threadIdx.x >> 6;
    const int ci0 = (int)blockIdx.x * 32, co0 = (int)blockIdx.y * 32;
    const int per_image = (h + rows - 1) / rows;
    const int pn = (int)blockIdx.z / per_image;
    const int r0 = ((int)blockIdx.z % per_image) * rows;
    const int r1 = r0 + rows < h ? r0 + rows : h;
    // the chunk's lines and their positions, the pixels from one to the next
    const int nl = TURN ? wd : r1 - r0, np = TURN ? r1 - r0 : wd;
    const int ls = TURN ? 1 : wd, ps = TURN ? wd : 1;
    // the chunk's rows of dout, and of the input with one around
    const int ya = r0 > 0 ? r0 - 1 : 0, yb = r1 < h ? r1 + 1 : h;
    const uint32_t xbytes = (uint32_t)(yb - ya) * (uint32_t)wd * (uint32_t)cin * 4u;
    const uint32_t dbytes = (uint32_t)(r1 - r0) * (uint32_t)wd * (uint32_t)cout * 4u;
    const float* px0 = in + ((int64_t)pn * h + ya) * wd * cin;
    const float* pd0 = dout + ((int64_t)pn * h + r0) * wd * cout;
    const __amdgpu_buffer_rsrc_t rx = buf(px0, xbytes), rd = buf(pd0, dbytes);
    // the input's lines and positions, from the chunk's first
    const int la = TURN ? 0 : ya - r0, lb = TURN ? wd : yb - r0;
    const int pa = TURN ? ya - r0 : 0, pb = TURN ? yb - r0 : wd;
    const int xw = T.seg + 2;
    const FastDiv dseg = fast_div(T.seg), dxw = fast_div(xw);
    // staging items: 8 channels of a pixel; a thread keeps its channels
    constexpr int kX = (kGIn + NP - 1) / NP, kD = (kGPix + NP - 1) / NP;
    const int c8 = (int)threadIdx.x % 4 * 8, p0 = (int)threadIdx.x / 4;
    const int xleft = cin - ci0 - c8, dleft = cout - co0 - c8;
    // the items' pixels in a sub-tile (lines past it: none), and their byte
    // offsets from its first one
    int xty[kX], xtx[kX], dty[kD], dtx[kD];
    Off xrel[kX], drel[kD];
#pragma unroll
    for (int k = 0; k < kX; k++) {
        xty[k] = fdiv(p0 + k * NP, dxw, &xtx[k]) - 1;
        xtx[k]--;
        xrel[k] = (((Off)xty[k] * (Off)ls + (Off)xtx[k] * (Off)ps + (Off)(r0 - ya) * (Off)wd) *
                       (Off)cin + ci0 + c8) * unit;
        if (xty[k] > T.rt) xty[k] = 1 << 30;
    }
#pragma unroll
    for (int k = 0; k < kD; k++) {
        dty[k] = fdiv(p0 + k * NP, dseg, &dtx[k]);
        drel[k] = (((Off)dty[k] * (Off)ls + (Off)dtx[k] * (Off)ps) * (Off)cout + co0 + c8) * unit;
        if (dty[k] >= T.rt) dty[k] = 1 << 30;
    }
    float4 fx[kX][2], fd[kD][2];
    // sub-tile: lines from l, positions from p
    auto load = [&](int l, int p) {
        const Off at = (Off)l * (Off)ls + (Off)p * (Off)ps;
        const Off xb = at * (Off)cin * unit, db = at * (Off)cout * unit;
#pragma unroll
        for (int k = 0; k < kX; k++) {
            const bool on = (uint32_t)(xty[k] + l - la) < (uint32_t)(lb - la) &&
                            (uint32_t)(xtx[k] + p - pa) < (uint32_t)(pb - pa);
            if constexpr (WIDE) load8_wide(fx[k], px0, xrel[k] + xb, on ? xleft : 0);
            else load8<FORM>(fx[k], rx, xrel[k] + xb, on ? xleft : 0, xbytes);
        }
#pragma unroll
        for (int k = 0; k < kD; k++) {
            const bool on = dty[k] + l < nl && dtx[k] + p < np;
            if constexpr (WIDE) load8_wide(fd[k], pd0, drel[k] + db, on ? dleft : 0);
            else load8<FORM>(fd[k], rd, drel[k] + db, on ? dleft : 0, dbytes);
        }
    };
    // this lane's part of a transposed read: group l / 16 reads channels
    // 16 (l / 16 % 2) .. and pixels 8 (l / 32) .. of a product's 16
    const int tr = (8 * (lane >> 5) + (lane & 15) / 4) * 32 + 16 * (lane >> 4 & 1) + 4 * (lane & 3);
    const int shift = (TURN ? tap % 3 * xw + tap / 3 : tap / 3 * xw + tap % 3) * 32;
    f32x16 acc = {};
    float bsum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    load(0, 0);
    for (int ry = 0, cx = 0; ry < nl;) {
        const int nx = cx + T.seg < np ? cx + T.seg : 0, ny = nx ? ry : ry + T.rt;
        if (ry || cx) __syncthreads();  // the products before have read
#pragma unroll
        for (int k = 0; k < kX; k++)
            if (p0 + k * NP < kGIn)
                *reinterpret_cast<bf16x8*>(&s_x[(p0 + k * NP) * 32 + c8]) =
                    to_bf16x8(fx[k][0], fx[k][1]);
#pragma unroll
        for (int k = 0; k < kD; k++) {
            if (p0 + k * NP < kGPix)
                *reinterpret_cast<bf16x8*>(&s_d[(p0 + k * NP) * 32 + c8]) =
                    to_bf16x8(fd[k][0], fd[k][1]);
            const float v[8] = {fd[k][0].x, fd[k][0].y, fd[k][0].z, fd[k][0].w,
                                fd[k][1].x, fd[k][1].y, fd[k][1].z, fd[k][1].w};
#pragma unroll
            for (int c = 0; c < 8; c++) bsum[c] += v[c];
        }
        __syncthreads();
        if (ny < nl) load(ny, nx);
        const int nrows = nl - ry < T.rt ? nl - ry : T.rt;
        // N products of a line, their reads ahead of them
        auto products = [&](auto steps, const short* d, const short* x, int px) {
            constexpr int N = decltype(steps)::value;
            s16x8 a[N], b[N];
#pragma unroll
            for (int i = 0; i < N; i++) {
                b[i] = __builtin_shufflevector(lds_tr(d + (px + 16 * i) * 32),
                                               lds_tr(d + (px + 16 * i + 4) * 32), 0, 1, 2, 3, 4, 5,
                                               6, 7);
                a[i] = __builtin_shufflevector(lds_tr(x + (px + 16 * i) * 32),
                                               lds_tr(x + (px + 16 * i + 4) * 32), 0, 1, 2, 3, 4, 5,
                                               6, 7);
            }
            // pixels past the line's end: their dout is zero, and so has to be
            // the input beside it, whatever it holds
            if (np - cx - px < 16 * N) {
#pragma unroll
                for (int i = 0; i < N; i++)
#pragma unroll
                    for (int t = 0; t < 8; t++)
                        a[i][t] =
                            px + 16 * i + 8 * (lane >> 5) + t < np - cx ? a[i][t] : (short)0;
            }
#pragma unroll
            for (int i = 0; i < N; i++)
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[i]),
                                                              __builtin_bit_cast(bf16x8, b[i]), acc,
                                                              0, 0, 0);
        };
        for (int ty = 0; ty < nrows; ty++) {
            const short* d = &s_d[ty * T.seg * 32 + tr];
            const short* x = &s_x[ty * xw * 32 + tr + shift];
            int px = 0;
            for (; px + 64 <= T.seg; px += 64) products(std::integral_constant<int, 4>{}, d, x, px);
            for (; px < T.seg; px += 16) products(std::integral_constant<int, 1>{}, d, x, px);
        }
        ry = ny;
        cx = nx;
    }
    const int row = lane & 31, g = lane >> 5;
    if (co0 + row < cout) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int ci = ci0 + 8 * i + 4 * g + j;
                if (ci < cin)
                    partial[(((int64_t)blockIdx.z * 9 + tap) * cin + ci) * cout + co0 + row] =
                        acc[4 * i + j];
            }
    }
    if (bpart && blockIdx.x == 0) {
        __syncthreads();
        float* red = reinterpret_cast<float*>(s_x);  // [thread / 4][channel]
        static_assert(sizeof(float) * NT * 8 <= sizeof(s_x), "bias sums");
#pragma unroll
        for (int c = 0; c < 8; c++) red[threadIdx.x * 8 + c] = bsum[c];
        __syncthreads();
        // 16 threads per channel, then one
        const int c = (int)threadIdx.x & 31, v0 = (int)threadIdx.x >> 5;
        float s = 0.f;
        if (v0 < 16)
            for (int v = v0; v < NP; v += 16) s += red[v * 32 + c];
        __syncthreads();
        if (v0 < 16) red[v0 * 32 + c] = s;
        __syncthreads();
        if (threadIdx.x < 32 && co0 + c < cout) {
            s = 0.f;
            for (int v = 0; v < 16; v++) s += red[v * 32 + c];
            bpart[(int64_t)blockIdx.z * cout + co0 + c] = s;
        }
    }
}

// dst[i] = sum over the chunks of partial[c][i], and the same of the bias
// partials in the workgroups after those of dst (bdst: none if 0): a workgroup
// takes 64 consecutive i, its four waves the chunks c = w, w + 4, ... (so each
// wave has a quarter of the dependent adds, eight loads in flight), and the
// waves' sums are added in wave order through LDS: a fixed order, reproducible
// sums.
constexpr int kSumWaves = 4;
__global__ __launch_bounds__(64 * kSumWaves) void k_sum_partials(const float* __restrict__ partial,
                                                                 float* __restrict__ dst,
                                                                 int64_t count,
                                                                 const float* __restrict__ bpart,
                                                                 float* __restrict__ bdst,
                                                                 int64_t bcount, int nchunks) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int64_t i = (int64_t)blockIdx.x * 64 + lane;
    const int64_t whole = (count + 63) / 64;
    if (blockIdx.x >= whole) {
        i -= whole * 64;
        partial = bpart;
        dst = bdst;
        count = bcount;
    }
    float s = 0.f;
    if (i < count) {
#pragma unroll 8
        for (int c = w; c < nchunks; c += kSumWaves) s += partial[(int64_t)c * count + i];
    }
    __shared__ float red[kSumWaves][64];
    red[w][lane] = s;
    __syncthreads();
    if (w == 0 && i < count) {
        float t = red[0][lane];
        for (int v = 1; v < kSumWaves; v++) t += red[v][lane];
        dst[i] = t;
    }
}

// V consecutive floats: 4 where the channel counts are multiples of four and
// the arrays are aligned for it, else 1
template <int V> struct Vec;
template <> struct Vec<1> {
    float v[1];
    __device__ static Vec ld(const float* p) { return Vec{{*p}}; }
    __device__ void st(float* p) const { *p = v[0]; }
};
template <> struct Vec<4> {
    float v[4];
    __device__ static Vec ld(const float* p) {
        const float4 f = *reinterpret_cast<const float4*>(p);
        return Vec{{f.x, f.y, f.z, f.w}};
    }
    __device__ void st(float* p) const {
        *reinterpret_cast<float4*>(p) = float4{v[0], v[1], v[2], v[3]};
    }
};

__global__ void k_relu_bwd(const float* __restrict__ dout, const float* __restrict__ out,
                           float* __restrict__ din, int64_t count) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < count;
         i += (int64_t)gridDim.x * blockDim.x)
        din[i] = out[i] > 0.f ? dout[i] : 0.f;
}

// 2x2 average pooling and its adjoint (h, wd: the fine size)
__global__ void k_pool_fwd(const float* __restrict__ in, float* __restrict__ out, int n, int h,
                           int wd, int c) {
    const int ho = h / 2, wo = wd / 2;
    const int64_t total = (int64_t)n * ho * wo * c;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int ch = (int)(i % c);
        const int64_t p = i / c;
        const int x = (int)(p % wo), y = (int)((p / wo) % ho);
        const int64_t b = p / ((int64_t)wo * ho);
        const float* s = in + ((b * h + 2 * y) * wd + 2 * x) * c + ch;
        out[i] = 0.25f * ((s[0] + s[c]) + (s[(int64_t)wd * c] + s[(int64_t)wd * c + c]));
    }
}

__global__ void k_pool_bwd(const float* __restrict__ dout, float* __restrict__ din, int n,
                           int h, int wd, int c) {
    const int64_t total = (int64_t)n * h * wd * c;
    const int ho = h / 2, wo = wd / 2;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int ch = (int)(i % c);
        const int64_t p = i / c;
        const int x = (int)(p % wd), y = (int)((p / wd) % h);
        const int64_t b = p / ((int64_t)wd * h);
        din[i] = 0.25f * dout[((b * ho + y / 2) * wo + x / 2) * c + ch];
    }
}

// These three take their items (V channels of a pixel) by one 32-bit index over
// all of them, with 32-bit divisions (some 20 instructions each; of 64-bit
// ones, 100); the host cuts larger calls into slabs (slabs).  HBM bounds them.
constexpr int64_t kSlab = (int64_t)1 << 30;

// nearest 2x upsampling (wd: the coarse width) of items / (cols cv) rows of
// cols columns into channels of a tensor with ctot channels, and its adjoint.
// (fine row 2 y of image b is row 2 (b h + y) of all)
// 32 images of 64 x 64 x 48 and 128 x 128 x 72, forward 18.5 us (one channel
// and an index of 64 bits: 73), backward 23.5 (four channels: 25.1).
template <int V>
__global__ void k_up_fwd(const float* __restrict__ in, float* __restrict__ out, uint32_t items,
                         uint32_t cols, uint32_t cv, int wd, int ctot) {
    const int64_t W = 2 * (int64_t)wd, c = (int64_t)cv * V;
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < items; i += gridDim.x * 256u) {
        const uint32_t q = i / cv, k = (i - q * cv) * V, r = q / cols, x = q - r * cols;
        const Vec<V> v = Vec<V>::ld(in + ((int64_t)r * wd + x) * c + k);
        float* f = out + (2 * (int64_t)r * W + 2 * (int64_t)x) * ctot + k;
        v.st(f);
        v.st(f + ctot);
        v.st(f + W * ctot);
        v.st(f + W * ctot + ctot);
    }
}

__global__ void k_up_bwd(const float* __restrict__ dout, float* __restrict__ din, uint32_t items,
                         uint32_t cols, uint32_t c, int wd, int ctot) {
    const int64_t W = 2 * (int64_t)wd;
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < items; i += gridDim.x * 256u) {
        const uint32_t q = i / c, k = i - q * c, r = q / cols, x = q - r * cols;
        const float* f = dout + (2 * (int64_t)r * W + 2 * (int64_t)x) * ctot + k;
        din[((int64_t)r * wd + x) * c + k] =
            (f[0] + f[ctot]) + (f[W * ctot] + f[W * ctot + ctot]);
    }
}

// copy channels [0, c) of src (c channels) into channels [c0, c0 + c) of
// dst (ctot channels) (dir = 0), or back (dir = 1), or add them back (dir =
// 2); the tensor of ctot channels from channel c0 on.  32 images of 128 x 128
// x 24 into 72: 15.6 us (one channel and an index of 64 bits: 18.6).
template <int V>
__global__ void k_channels(const float* __restrict__ a, float* __restrict__ b, uint32_t items,
                           uint32_t cv, int ctot, int dir) {
    const int64_t c = (int64_t)cv * V;
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < items; i += gridDim.x * 256u) {
        const uint32_t p = i / cv, k = (i - p * cv) * V;
        const int64_t thin = p * c + k, wide = (int64_t)p * ctot + k;
        if (dir == 0) {
            Vec<V>::ld(a + thin).st(b + wide);
        } else {
            Vec<V> v = Vec<V>::ld(a + wide);
            if (dir != 1) {
                const Vec<V> o = Vec<V>::ld(b + thin);
#pragma unroll
                for (int j = 0; j < V; j++) v.v[j] = o.v[j] + v.v[j];
            }
            v.st(b + thin);
        }
    }
}

// dst[p][ch] = src[p][ch] on pixels with mask[p] == 0 and ch < cu, else 0
__global__ void k_mask_channels(const float* src, const float* __restrict__ mask, float* dst,
                                int64_t pixels, int c, int cu) {
    const int64_t total = pixels * c;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int ch = (int)(i % c);
        const int64_t p = i / c;
        dst[i] = (ch < cu && mask[p] == 0.f) ? src[i] : 0.f;
    }
}

// dst[i][:] = src[idx[i]][:] for rows of `elems` floats (a mini-batch
// from a device-resident training set)
__global__ void k_gather(const float* __restrict__ src, float* __restrict__ dst,
                         const int32_t* __restrict__ idx, int count, int64_t elems) {
    const int64_t total = (int64_t)count * elems;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int r = (int)(i / elems);
        dst[i] = src[(int64_t)idx[r] * elems + (i - (int64_t)r * elems)];
    }
}

// masked mean squared error over channels [0, cu) of pred (ctot channels):
// per-block partial sums of the loss; grad = 2 (pred - target) / count on
// fluid pixels (mask == 0), zero elsewhere and in channels >= cu
__global__ void k_mse(const float* __restrict__ pred, const float* __restrict__ target,
                      const float* __restrict__ mask, float* __restrict__ grad,
                      float* __restrict__ partial, int64_t pixels, int cu, int ctot,
                      float inv_count) {
    __shared__ float red[256];
    float s = 0.f;
    const int64_t total = pixels * ctot;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int ch = (int)(i % ctot);
        const int64_t p = i / ctot;
        float gv = 0.f;
        if (ch < cu && mask[p] == 0.f) {
            const float d = pred[i] - target[p * cu + ch];
            s += d * d;
            gv = 2.f * d * inv_count;
        }
        grad[i] = gv;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// Adam (Kingma & Ba 2015) with bias correction folded into the step size
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, int64_t count, float lr, float b1, float b2,
                       float eps, float c1, float c2) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < count;
         i += (int64_t)gridDim.x * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.f - b1) * gi;
        const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        p[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
    }
}

__global__ void k_zero(float* __restrict__ p, int64_t count) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < count;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0.f;
}

int grid_for(int64_t total) {
    int64_t g = (total + 255) / 256;
    if (g > 8192) g = 8192;
    if (g < 1) g = 1;
    return (int)g;
}

// whether four-float accesses of arrays with these channel counts and the
// first of them c0 are aligned
bool vec4(const void* p, const void* q, int64_t c, int64_t ctot, int64_t c0) {
    return ((reinterpret_cast<uintptr_t>(p) | reinterpret_cast<uintptr_t>(q)) & 15) == 0 &&
           ((c | ctot | c0) & 3) == 0;
}

// launch(first row, first column, items, columns, cv, grid) over rows of wd
// columns of cv items, in slabs of at most kSlab items (or of one column)
// (8192 workgroups that loop against one per 256 items: 32.5 and 42 us for
// 32 images of 128 x 128 x 47 channels into 72, one at a time)
template <typename F> void slabs(int64_t rows, int64_t wd, int64_t cv, const F& launch) {
    const int64_t cols = std::max<int64_t>(1, std::min(wd, kSlab / cv));
    const int64_t some = std::max<int64_t>(1, std::min(rows, kSlab / (cols * cv)));
    for (int64_t r = 0; r < rows; r += some)
        for (int64_t x = 0; x < wd; x += cols) {
            const int64_t nc = std::min(cols, wd - x), items = std::min(some, rows - r) * nc * cv;
            launch(r, x, (uint32_t)items, (uint32_t)nc, (uint32_t)cv, dim3(grid_for(items)));
        }
}

int status() { return hipGetLastError() == hipSuccess ? 0 : MPLBWS_ERR_HIP; }

}  // namespace

extern "C" {

int mplbws_conv3x3_fwd(const float* in, const float* w, const float* bias, float* out, int n,
                       int h, int wd, int cin, int cout, int relu) {
    if (!in || !w || !out || n <= 0 || h <= 0 || wd <= 0 || cin <= 0 || cout <= 0 ||
        cin % 8 != 0)
        return MPLBWS_ERR_ARG;
    // WN = 1 for at most 32 output channels; WM = 2 (256-pixel tiles) while
    // that gives every CU two workgroups (64 x 64 x 48, 32 images: 512 of
    // them and 22.6 us, 28.8 with WM = 1; 128 or fewer: the same within 0.3 us)
    const int wn = cout > 32 ? 2 : 1;
    const int64_t groups = (cout + 32 * wn - 1) / (32 * wn);
    auto tiles = [&](int tp, bool longer) {
        const ConvTile t = conv_tile(h, wd, tp, longer);
        return (int64_t)n * t.tiles_x * t.tiles_y;
    };
    // longer tiles for few rows once there are two short ones for every CU (1 x
    // 100000, 16 to 16 channels: 22.4 us in columns of 32, 11.8; 1 x 4096, 64 to
    // 64: 10.1, 10.7)
    const bool longer = tiles(128, false) * groups >= 512;
    const int wm = tiles(256, longer) * groups >= 512 ? 2 : 1;
    const ConvTile T = conv_tile(h, wd, 128 * wm, longer);
    const int64_t wgs = (int64_t)n * T.tiles_x * T.tiles_y;
    if (wgs >= ((int64_t)1 << 31)) return MPLBWS_ERR_ARG;
    const dim3 grd((unsigned)wgs, (unsigned)groups), blk(64 * kWaves);
    const bool wide = (int64_t)(T.R + 2) * wd >= (((int64_t)1 << 30) + cin - 1) / cin ||
                      9LL * cin * cout >= (int64_t)1 << 30;
    const int form = wide ? kFormWide : vec4(w, out, cout, 0, 0) ? kFormVec : kFormAny;
#define X(WM, WN, FORM)                                                                        \
    if (wm == WM && wn == WN && form == FORM)                                                  \
        hipLaunchKernelGGL((k_conv_fwd<WM, WN, FORM>), grd, blk, 0, 0, in, w, bias, out, n, h, \
                           wd, cin, cout, relu, T);
    X(2, 2, kFormAny) X(2, 1, kFormAny) X(1, 2, kFormAny) X(1, 1, kFormAny)
    X(2, 2, kFormVec) X(2, 1, kFormVec) X(1, 2, kFormVec) X(1, 1, kFormVec)
    X(2, 2, kFormWide) X(2, 1, kFormWide) X(1, 2, kFormWide) X(1, 1, kFormWide)
#undef X
    return status();
}

int mplbws_flip_weights(const float* w, float* wt, int cin, int cout) {
    if (!w || !wt || cin <= 0 || cout <= 0) return MPLBWS_ERR_ARG;
    hipLaunchKernelGGL(k_flip_weights, dim3(grid_for(9LL * cin * cout)), dim3(256), 0, 0, w, wt,
                       cin, cout);
    return status();
}

int64_t mplbws_wgrad_workspace(int n, int h, int wd, int cin, int cout) {
    if (n <= 0 || h <= 0 || wd <= 0) return 0;
    const int rows = wgrad_rows(h, wd);
    const int64_t chunks = (int64_t)n * ((h + rows - 1) / rows);
    return chunks * 9LL * cin * cout + chunks * cout;
}

int mplbws_conv3x3_wgrad(const float* in, const float* dout, float* dw, float* dbias,
                         float* workspace, int n, int h, int wd, int cin, int cout) {
    if (!in || !dout || !dw || !workspace || n <= 0 || h <= 0 || wd <= 0 || cin <= 0 ||
        cout <= 0)
        return MPLBWS_ERR_ARG;
    const int rows = wgrad_rows(h, wd);
    const int64_t chunks = (int64_t)n * ((h + rows - 1) / rows);
    if (chunks > 65535) return MPLBWS_ERR_ARG;
    const int K = 9 * cin;
    const int64_t cnt = (int64_t)K * cout;
    float* bp = dbias ? workspace + chunks * cnt : nullptr;
    const dim3 grd((unsigned)((cin + 31) / 32), (unsigned)((cout + 31) / 32), (unsigned)chunks);
    const bool turn = grad_tiles(wd, rows) < grad_tiles(rows, wd);
    const GradTile T = turn ? grad_tile(wd, rows) : grad_tile(rows, wd);
    const int64_t most = std::max(cin, cout);
    const bool wide = (int64_t)(rows + 2) * wd >= (((int64_t)1 << 30) + most - 1) / most;
    const int form = wide ? kFormWide : vec4(in, dout, cin, cout, 0) ? kFormVec : kFormAny;
#define X(FORM, TURN)                                                                           \
    if (form == FORM && turn == TURN)                                                           \
        hipLaunchKernelGGL((k_conv_wgrad<FORM, TURN>), grd, dim3(64 * kGWaves), 0, 0, in, dout, \
                           workspace, bp, h, wd, cin, cout, rows, T);
    X(kFormAny, false) X(kFormVec, false) X(kFormWide, false)
    X(kFormAny, true) X(kFormVec, true) X(kFormWide, true)
#undef X
    const int64_t sums = (cnt + 63) / 64 + (dbias ? (cout + 63) / 64 : 0);
    hipLaunchKernelGGL(k_sum_partials, dim3((unsigned)sums), dim3(64 * kSumWaves), 0, 0, workspace,
                       dw, cnt, bp, dbias, (int64_t)cout, (int)chunks);
    return status();
}

int mplbws_relu_bwd(const float* dout, const float* out, float* din, int64_t count) {
    if (!dout || !out || !din || count < 0) return MPLBWS_ERR_ARG;
    hipLaunchKernelGGL(k_relu_bwd, dim3(grid_for(count)), dim3(256), 0, 0, dout, out, din, count);
    return status();
}

int mplbws_pool2_fwd(const float* in, float* out, int n, int h, int wd, int c) {
    if (!in || !out || h % 2 || wd % 2) return MPLBWS_ERR_ARG;
    hipLaunchKernelGGL(k_pool_fwd, dim3(grid_for((int64_t)n * h * wd * c / 4)), dim3(256), 0, 0,
                       in, out, n, h, wd, c);
    return status();
}

int mplbws_pool2_bwd(const float* dout, float* din, int n, int h, int wd, int c) {
    if (!dout || !din || h % 2 || wd % 2) return MPLBWS_ERR_ARG;
    hipLaunchKernelGGL(k_pool_bwd, dim3(grid_for((int64_t)n * h * wd * c)), dim3(256), 0, 0, dout,
                       din, n, h, wd, c);
    return status();
}

int mplbws_up2_fwd(const float* in, float* out, int n, int h, int wd, int c, int ctot, int c0) {
    if (!in || !out || c0 < 0 || c0 + c > ctot) return MPLBWS_ERR_ARG;
    if (n <= 0 || h <= 0 || wd <= 0 || c <= 0) return status();
    const bool v4 = vec4(in, out, c, ctot, c0);
    slabs((int64_t)n * h, wd, v4 ? c / 4 : c, [&](int64_t r, int64_t x, uint32_t items,
                                                  uint32_t cols, uint32_t cv, dim3 grd) {
        const float* i = in + (r * wd + x) * c;
        float* o = out + (4 * r * wd + 2 * x) * ctot + c0;
        if (v4) hipLaunchKernelGGL(k_up_fwd<4>, grd, dim3(256), 0, 0, i, o, items, cols, cv, wd, ctot);
        else hipLaunchKernelGGL(k_up_fwd<1>, grd, dim3(256), 0, 0, i, o, items, cols, cv, wd, ctot);
    });
    return status();
}

int mplbws_up2_bwd(const float* dout, float* din, int n, int h, int wd, int c, int ctot, int c0) {
    if (!dout || !din || c0 < 0 || c0 + c > ctot) return MPLBWS_ERR_ARG;
    if (n <= 0 || h <= 0 || wd <= 0 || c <= 0) return status();
    slabs((int64_t)n * h, wd, c, [&](int64_t r, int64_t x, uint32_t items, uint32_t cols, uint32_t,
                                     dim3 grd) {
        hipLaunchKernelGGL(k_up_bwd, grd, dim3(256), 0, 0, dout + (4 * r * wd + 2 * x) * ctot + c0,
                           din + (r * wd + x) * c, items, cols, (uint32_t)c, wd, ctot);
    });
    return status();
}

int mplbws_channels(const float* src, float* dst, int64_t pixels, int c, int ctot, int c0,
                    int direction) {
    if (!src || !dst || c0 < 0 || c0 + c > ctot) return MPLBWS_ERR_ARG;
    if (pixels <= 0 || c <= 0) return status();
    const bool v4 = vec4(src, dst, c, ctot, c0);
    slabs(pixels, 1, v4 ? c / 4 : c, [&](int64_t p, int64_t, uint32_t items, uint32_t, uint32_t cv,
                                         dim3 grd) {
        const int64_t thin = p * c, wide = p * ctot + c0;
        const float* a = src + (direction == 0 ? thin : wide);
        float* b = dst + (direction == 0 ? wide : thin);
        if (v4) hipLaunchKernelGGL(k_channels<4>, grd, dim3(256), 0, 0, a, b, items, cv, ctot, direction);
        else hipLaunchKernelGGL(k_channels<1>, grd, dim3(256), 0, 0, a, b, items, cv, ctot, direction);
    });
    return status();
}

int mplbws_mask_channels(const float* src, const float* mask, float* dst, int64_t pixels, int c,
                         int cu) {
    if (!src || !mask || !dst || pixels < 0 || c <= 0 || cu < 0) return MPLBWS_ERR_ARG;
    hipLaunchKernelGGL(k_mask_channels, dim3(grid_for(pixels * c)), dim3(256), 0, 0, src, mask,
                       dst, pixels, c, cu);
    return status();
}

int mplbws_gather(const float* src, float* dst, const int32_t* idx, int count,
                  int64_t elems) {
    if (!src || !dst || !idx || count < 0 || elems < 0) return MPLBWS_ERR_ARG;
    hipLaunchKernelGGL(k_gather, dim3(grid_for((int64_t)count * elems)), dim3(256), 0, 0, src,
                       dst, idx, count, elems);
    return status();
}

int mplbws_mse(const float* pred, const float* target, const float* mask, float* grad,
               float* partial, int npartial, int64_t pixels, int cu, int ctot, float inv_count) {
    if (!pred || !target || !mask || !grad || !partial || npartial <= 0 || cu > ctot)
        return MPLBWS_ERR_ARG;
    hipLaunchKernelGGL(k_mse, dim3(npartial), dim3(256), 0, 0, pred, target, mask, grad, partial,
                       pixels, cu, ctot, inv_count);
    return status();
}

int mplbws_adam(float* p, const float* g, float* m, float* v, int64_t count, float lr, float b1,
                float b2, float eps, int step) {
    if (!p || !g || !m || !v || count < 0 || step < 1) return MPLBWS_ERR_ARG;
    const float c1 = 1.f / (1.f - powf(b1, (float)step));
    const float c2 = 1.f / (1.f - powf(b2, (float)step));
    hipLaunchKernelGGL(k_adam, dim3(grid_for(count)), dim3(256), 0, 0, p, g, m, v, count, lr, b1,
                       b2, eps, c1, c2);
    return status();
}

int mplbws_sync(void) { return hipDeviceSynchronize() == hipSuccess ? 0 : MPLBWS_ERR_HIP; }

int mplbws_alloc(void** p, int64_t bytes) {
    if (!p || bytes < 0) return MPLBWS_ERR_ARG;
    *p = nullptr;
    if (bytes == 0) return 0;
    return hipMalloc(p, (size_t)bytes) == hipSuccess ? 0 : MPLBWS_ERR_HIP;
}

int mplbws_free(void* p) {
    if (!p) return 0;
    return hipFree(p) == hipSuccess ? 0 : MPLBWS_ERR_HIP;
}

int mplbws_upload(void* dst, const void* src, int64_t bytes) {
    if (!dst || !src || bytes < 0) return MPLBWS_ERR_ARG;
    return hipMemcpy(dst, src, (size_t)bytes, hipMemcpyHostToDevice) == hipSuccess
               ? 0
               : MPLBWS_ERR_HIP;
}

int mplbws_download(void* dst, const void* src, int64_t bytes) {
    if (!dst || !src || bytes < 0) return MPLBWS_ERR_ARG;
    return hipMemcpy(dst, src, (size_t)bytes, hipMemcpyDeviceToHost) == hipSuccess
               ? 0
               : MPLBWS_ERR_HIP;
}

int mplbws_zero(void* p, int64_t bytes) {
    if (!p || bytes < 0 || bytes % 4) return MPLBWS_ERR_ARG;
    hipLaunchKernelGGL(k_zero, dim3(grid_for(bytes / 4)), dim3(256), 0, 0,
                       static_cast<float*>(p), bytes / 4);
    return status();
}

}  // extern "C"
