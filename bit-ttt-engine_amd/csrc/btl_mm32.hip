// btl_mm32.hip -- gfx950 kernels that run fixed-order f32 sums on the f32 matrix
// instructions.
//
// v_mfma_f32_16x16x4_f32 adds its four products to the accumulator one after
// the other, in k order, each as one fused multiply-add rounded to nearest even
// with subnormals kept: D = fma(a3, b3, fma(a2, b2, fma(a1, b1, fma(a0, b0, C)))).
// v_mfma_f32_16x16x1_f32 is one such step for four independent 16 x 16 blocks.
// So a sum that this library defines as a sequential chain of fused
// multiply-adds gives the same bits through them (measured on MI355X against
// fmaf over normal, wide-exponent, subnormal, infinite and NaN operands; the
// tests compare every kernel here with the oracle bit for bit), at 138 and 128
// TFLOP/s against 79 for v_fma_f32, with the vector ALU left to the unpacking
// and one operand register per 1024 products instead of an LDS read per few.
//
// Kernels:
//   k_ref_mm    BTL_ACT_F32_REF of many token rows (BitLinearCpu::forward,
//               src/kernels/cpu.rs:86-123: eight chains per output)
//   k_dense_mm  btl_dense_linear of several token rows (candle_nn::Linear,
//               src/model/llama.rs:129-141; src/layers/adaptive_linear.rs:131-160)
#include <hip/hip_runtime.h>

#include <algorithm>

#include "btl_device.hpp"
#include "btl_internal.hpp"

namespace btl {

typedef float v4f __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// k_ref_mm
// ---------------------------------------------------------------------------
// Chain b of an output takes the inputs k = 8 j + b in increasing j.  One
// v_mfma_f32_16x16x4_f32 advances chain b of 16 tokens x 16 weight rows by four
// steps: lane 16 q + r holds x[token r][32 i + 8 q + b] and the coefficient of
// the same element of weight row r, i counting blocks of 32 inputs.  A lane's
// operands of all eight chains are therefore eight consecutive inputs (32
// bytes of x) and 16 consecutive bits of the packed row, so both come straight
// from global memory in vector loads with no exchange between lanes.
//
// A wave computes 16 TB tokens x 16 NB rows for CH of the eight chains (4 TB NB
// CH accumulator registers); a workgroup is 8 / CH waves per output tile and WN
// tiles along the rows.  With CH < 8 the chains meet in LDS at the end.  The
// loads of a 32-input block are issued D blocks ahead of its matrix
// instructions, each pinned in its place: left to the scheduler they all moved
// to the end of the loop body, right before their first use (q|k|v at m = 512:
// 236 -> 224 us).
//
// What bounds it: the f32 matrix rate.  Llama-3-8B shapes, f32 in and out, us
// (k_ref_f32_st before -> now): q|k|v (k = 4096) at m = 512 754-800 -> 224
// (115 TFLOP/s), gate|up 3227 -> 993 (121), down (k = 14336) 2929 -> 511
// (118); at m = 64 103 -> 51, 436 -> 145, 392 -> 122.  Up to 13 % more is lost
// where the tiles of a launch do not divide over the SIMDs.
struct RefMm {
    const void* x;
    RefGroup g;  // wg_begin in tiles of 16 NB WN rows
    int m, k;
};

__device__ __forceinline__ uint4 bload_s(__amdgpu_buffer_rsrc_t r, int voff, int soff)
{
    return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// CH consecutive inputs of a row, as stored
template <int XK, int CH>
struct RefX {
    static constexpr int kBytes = CH * (XK == XK_BF16 ? 2 : 4);
    uint32_t u[kBytes / 4];
};

template <int XK, int CH>
__device__ __forceinline__ RefX<XK, CH> ref_load_x(__amdgpu_buffer_rsrc_t r, int voff, int soff)
{
    RefX<XK, CH> o;
    if constexpr (RefX<XK, CH>::kBytes >= 16) {
#pragma unroll
        for (int i = 0; i < RefX<XK, CH>::kBytes / 16; ++i) {
            const uint4 v = bload_s(r, voff + 16 * i, soff);
            o.u[4 * i] = v.x; o.u[4 * i + 1] = v.y; o.u[4 * i + 2] = v.z; o.u[4 * i + 3] = v.w;
        }
    } else {
        typedef uint32_t u2 __attribute__((ext_vector_type(2)));
        const u2 v = __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
        o.u[0] = v.x; o.u[1] = v.y;
    }
    return o;
}

template <int XK, int CH>
__device__ __forceinline__ float ref_x(const RefX<XK, CH>& v, int b)
{
    if constexpr (XK == XK_BF16) {
        const uint32_t u = v.u[b >> 1];
        return __uint_as_float((b & 1) ? (u & 0xFFFF0000u) : (u << 16));
    }
    return __uint_as_float(v.u[b]);
}

template <int XK, int YK, int TB, int NB, int CH, int WN, int D>
__global__ __launch_bounds__(64 * WN * (8 / CH), TB * NB * CH >= 32 ? 2 : 4) void k_ref_mm(RefMm a)
{
    static_assert((CH == 8 || CH == 4) && D % 2 == 0, "eight or four chains a wave, pairs of blocks");
    constexpr int WC = 8 / CH;  // waves that share an output tile, CH chains each
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, r = lane & 15;
    const int wc = wave % WC, wn = wave / WC, c0 = wc * CH;
    int li = 0;
#pragma unroll
    for (int i = 1; i < kMaxGroup; ++i)
        if (i < a.g.count && (int)blockIdx.x >= a.g.wg_begin[i]) li = i;
    const int K = a.k, rb = K >> 2;
    const int64_t n = a.g.n[li];
    const int64_t col0 = ((int64_t)((int)blockIdx.x - a.g.wg_begin[li]) * WN + wn) * 16 * NB;
    const int64_t row0 = (int64_t)blockIdx.y * 16 * TB;
    const int nrow = (int)min((int64_t)16 * TB, a.m - row0);                   // token rows of the tile
    const int ncol = (int)max((int64_t)0, min((int64_t)16 * NB, n - col0));    // weight rows (0: past the layer)
    constexpr int XB = XK == XK_BF16 ? 2 : 4;
    // rows past the end read as zero (outside the descriptor) and are not stored
    const char* xbase = (const char*)a.x + row0 * K * XB;
    const uint8_t* wbase = a.g.w[li] + (ncol ? col0 * rb : 0);
    const uint32_t xbytes = (uint32_t)(nrow * K * XB), wbytes = (uint32_t)(ncol * rb);
    int xo[TB], wo[NB];
#pragma unroll
    for (int t = 0; t < TB; ++t) xo[t] = ((16 * t + r) * K + 8 * q + c0) * XB;
#pragma unroll
    for (int u = 0; u < NB; ++u) wo[u] = (16 * u + r) * rb;
    // the 16 bits of quarter q: half word q of each 8 bytes
    const uint32_t sel = (q & 1) ? 0x07060302u : 0x05040100u;
    const bool hi = q >= 2;

    v4f acc[TB][NB][CH];
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
        for (int u = 0; u < NB; ++u)
#pragma unroll
            for (int b = 0; b < CH; ++b) acc[t][u][b] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    // D blocks of 32 inputs in flight (and the weights of D / 2 pairs of blocks);
    // a block past the row reads zeros (an empty descriptor), which leave every
    // chain as it is: fma(0, 0, acc) = acc for an acc that is never -0
    const int blocks = K >> 5;
    RefX<XK, CH> xa[D][TB];
    uint4 wv[D / 2][NB];
    const auto load_x = [&](int i, int d) {
        const __amdgpu_buffer_rsrc_t xr = make_rsrc(xbase, i + d < blocks ? xbytes : 0u);
#pragma unroll
        for (int t = 0; t < TB; ++t) xa[d][t] = ref_load_x<XK, CH>(xr, xo[t], (i + d) * 32 * XB);
    };
    const auto load_w = [&](int i, int p) {
        const __amdgpu_buffer_rsrc_t wr = make_rsrc(wbase, i + 2 * p < blocks ? wbytes : 0u);
#pragma unroll
        for (int u = 0; u < NB; ++u) wv[p][u] = bload_s(wr, wo[u], (i + 2 * p) * 8);
    };
#pragma unroll
    for (int d = 0; d < D; ++d) {
        if (!(d & 1)) load_w(0, d >> 1);
        load_x(0, d);
    }
    for (int i = 0; i < blocks; i += D) {
#pragma unroll
        for (int p = 0; p < D / 2; ++p) {
            v4i co[NB];  // coefficients, byte 2 s + b / 4 of word b % 4: chain b of block s
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                const uint32_t lo = hi ? wv[p][u].y : wv[p][u].x, up = hi ? wv[p][u].w : wv[p][u].z;
                co[u] = unpack16(__builtin_amdgcn_perm(up, lo, sel));
            }
            load_w(i + D, p);
            __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the matrix instructions
#pragma unroll
            for (int s = 0; s < 2; ++s) {
#pragma unroll
                for (int b = 0; b < CH; ++b) {
                    float wf[NB];
#pragma unroll
                    for (int u = 0; u < NB; ++u) {
                        if constexpr (CH == 8) {
                            wf[u] = (float)(int8_t)((uint32_t)co[u][b & 3] >> (16 * s + 8 * (b >> 2)));
                        } else {
                            wf[u] = (float)(int8_t)((uint32_t)co[u][b] >> (16 * s + 8 * wc));
                        }
                    }
#pragma unroll
                    for (int t = 0; t < TB; ++t)
#pragma unroll
                        for (int u = 0; u < NB; ++u)
                            acc[t][u][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(ref_x<XK, CH>(xa[2 * p + s][t], b), wf[u],
                                                                                acc[t][u][b], 0, 0, 0);
                }
                load_x(i + D, 2 * p + s);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }

    // y = (the lanes 0..7 added in order, cpu.rs:236-238) * scale
    const float scale = a.g.scale[li];
    void* y = a.g.y[li];
    if constexpr (CH == 8) {
#pragma unroll
        for (int t = 0; t < TB; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = 16 * t + 4 * q + v;
#pragma unroll
                for (int u = 0; u < NB; ++u) {
                    float z = -0.0f;
#pragma unroll
                    for (int b = 0; b < 8; ++b) z = __fadd_rn(z, acc[t][u][b][v]);
                    if (row < nrow && 16 * u + r < ncol)
                        store_y<YK>(y, (row0 + row) * n + col0 + 16 * u + r, __fmul_rn(__fadd_rn(0.0f, z), scale));
                }
            }
    } else {
        constexpr int TILE = TB * NB * 256;
        __shared__ float s_acc[WN][8][TILE];
#pragma unroll
        for (int t = 0; t < TB; ++t)
#pragma unroll
            for (int u = 0; u < NB; ++u)
#pragma unroll
                for (int b = 0; b < CH; ++b)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        s_acc[wn][c0 + b][(16 * t + 4 * q + v) * 16 * NB + 16 * u + r] = acc[t][u][b][v];
        __syncthreads();
        for (int e = wc * 64 + lane; e < TILE; e += WC * 64) {
            const int row = e / (16 * NB), col = e % (16 * NB);
            float z = -0.0f;
#pragma unroll
            for (int b = 0; b < 8; ++b) z = __fadd_rn(z, s_acc[wn][b][e]);
            if (row < nrow && col < ncol)
                store_y<YK>(y, (row0 + row) * n + col0 + col, __fmul_rn(__fadd_rn(0.0f, z), scale));
        }
    }
}

template <int XK, int YK, int TB, int NB, int CH, int WN, int D>
static void launch_ref_mm_t(RefMm a, hipStream_t st)
{
    const int rows = 16 * NB * WN;
    int b = 0;
    for (int i = 0; i < a.g.count; ++i) {
        a.g.wg_begin[i] = b;
        b += (int)((a.g.n[i] + rows - 1) / rows);
    }
    a.g.wg_begin[a.g.count] = b;
    const dim3 grid((unsigned)b, (unsigned)((a.m + 16 * TB - 1) / (16 * TB)));
    hipLaunchKernelGGL((k_ref_mm<XK, YK, TB, NB, CH, WN, D>), grid, dim3(64 * WN * (8 / CH)), 0, st, a);
}

hipError_t launch_ref_mm(const void* x, int xkind, int64_t m, int64_t k, const RefGroup& g, int ykind, hipStream_t st)
{
    RefMm a{};
    a.x = x;
    a.g = g;
    a.m = (int)m;
    a.k = (int)k;
    // The form of least cost: rounds of the launch's waves over the 1024 SIMDs
    // times what one round of the form takes (us at k = 4096, measured with at
    // most one wave per SIMD).  Few tokens or rows: smaller tiles and the chains
    // split over waves, so that the launch still covers the chip (q|k|v at m =
    // 32: 33 us with 1 x 2 blocks and 4 chains a wave, 76 with 2 x 2 and 8).
    const auto cost = [&](int tb, int nb, int ch, int wn, float us) {
        int64_t waves = 0;
        for (int i = 0; i < g.count; ++i) waves += (g.n[i] + 16 * nb * wn - 1) / (16 * nb * wn) * wn;
        waves *= (m + 16 * tb - 1) / (16 * tb) * (8 / ch);
        return (float)((waves + 1023) / 1024) * us;
    };
    const float c[4] = {cost(2, 2, 8, 4, 74.0f), cost(2, 2, 4, 2, 47.0f), cost(1, 2, 4, 2, 31.0f),
                        cost(1, 1, 4, 2, 19.5f)};
    const int form = (int)(std::min_element(c, c + 4) - c);
#define BTL_REF_MM(XKV, YKV)                                                 \
    if (xkind == XKV && ykind == YKV) {                                      \
        if (form == 0) launch_ref_mm_t<XKV, YKV, 2, 2, 8, 4, 2>(a, st);      \
        else if (form == 1) launch_ref_mm_t<XKV, YKV, 2, 2, 4, 2, 4>(a, st); \
        else if (form == 2) launch_ref_mm_t<XKV, YKV, 1, 2, 4, 2, 4>(a, st); \
        else launch_ref_mm_t<XKV, YKV, 1, 1, 4, 2, 8>(a, st);                \
        return hipGetLastError();                                            \
    }
    BTL_REF_MM(XK_F32, YK_F32)
    BTL_REF_MM(XK_F32, YK_BF16)
    BTL_REF_MM(XK_BF16, YK_F32)
    BTL_REF_MM(XK_BF16, YK_BF16)
#undef BTL_REF_MM
    return hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------
// k_dense_mm
// ---------------------------------------------------------------------------
// btl_dense_linear of several token rows: lane l of 64 (a chain) folds the
// 4-element chunks l, l + 64, ... of a row in element order, then the chains
// are added in the butterfly's order (xor 32, 16, 8, 4, 2, 1).  One
// v_mfma_f32_16x16x1_f32 advances four chains of 16 tokens x 16 weight rows by
// one element: lane 16 c + r holds the element of chain c's chunk for token
// (weight row) r, so the 16 bytes of a chunk feed four of them and nothing is
// exchanged between lanes.  Wave s of eight holds the chains 4 s .. 4 s + 3 and
// 32 + 4 s .. 35 + 4 s of a tile of 16 TB tokens x 16 NB rows (32 TB NB
// accumulator registers); the first level of the butterfly is then in its
// registers, the rest in LDS after the main loop.
//
// The operands go through LDS: with direct loads the lanes of a quarter wave
// read 16 different rows, which the address unit takes one line per lane (128
// tokens x 5632 rows, k = 2048: 63 us, 45 with the copies, whose consecutive
// lanes read consecutive bytes).  A wave copies and reads only its own chains,
// so the main loop has no barrier, two stages of 256 elements.
//
// What bounds it: the f32 matrix rate from about 64 token rows, below that the
// weights.  us, k_dense_gemv (which reads the weights again for every token
// row) -> now: n = 5632, k = 2048, f32: m = 2 15 -> 12, 16 80 -> 14, 128 711 ->
// 45, 256 1483 -> 79; n = 16384, k = 4096, bf16: m = 2 40 -> 26, 16 279 -> 35,
// 256 5102 -> 368 (93 TFLOP/s).
typedef float v16f __attribute__((ext_vector_type(16)));

struct DenseMm {
    const void* w;  // [n, k]
    const float* x;  // [m, k]
    float* y;        // [m, n]
    int64_t n;
    int m, k;
    int mt;          // token tiles
};

template <int WK>
struct DenseW {
    uint4 v;
};
template <>
struct DenseW<XK_BF16> {
    uint2 v;
};

template <int WK>
__device__ __forceinline__ void dense_load_w(DenseW<WK>& o, __amdgpu_buffer_rsrc_t r, int voff, int soff)
{
    if constexpr (WK == XK_BF16) {
        typedef uint32_t u2 __attribute__((ext_vector_type(2)));
        const u2 t = __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
        o.v = make_uint2(t.x, t.y);
    } else {
        o.v = bload_s(r, voff, soff);
    }
}

template <int WK>
__device__ __forceinline__ float dense_w(const DenseW<WK>& o, int e)
{
    if constexpr (WK == XK_BF16) {
        const uint32_t u = e < 2 ? o.v.x : o.v.y;
        return __uint_as_float((e & 1) ? (u & 0xFFFF0000u) : (u << 16));
    } else {
        return __uint_as_float(e == 0 ? o.v.x : (e == 1 ? o.v.y : (e == 2 ? o.v.z : o.v.w)));
    }
}

template <int WK, int TB, int NB>
__global__ __launch_bounds__(512, 2) void k_dense_mm(DenseMm a)
{
    constexpr int WB = WK == XK_BF16 ? 2 : 4;
    constexpr int XS = 128, WS = 32 * WB;                 // bytes of a row per wave and block
    constexpr int XW = 16 * TB * XS, WW = 16 * NB * WS;   // one stage of a wave
    constexpr int XC = XW / 1024, WC = WW / 1024;         // its copies
    constexpr int kSums = 32 * 256 * 4;                   // a tile's chains, after the main loop
    constexpr int kStage = 8 * (XW + WW) > kSums ? 8 * (XW + WW) : kSums;
    constexpr int D = 2;
    // an array per stage: the compiler then knows which copies a read depends on
    __shared__ __align__(1024) uint8_t lds0[kStage];
    __shared__ __align__(1024) uint8_t lds1[kStage];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane >> 4, r = lane & 15;
    // consecutive workgroups (on the 8 XCDs in turn) take different weight
    // tiles; an XCD walks the token tiles of its weight tile
    const int b8 = (int)blockIdx.x >> 3;
    const int64_t col0 = (int64_t)((b8 / a.mt) * 8 + (blockIdx.x & 7)) * 16 * NB;
    const int row0 = (b8 % a.mt) * 16 * TB;
    if (col0 >= a.n) return;  // uniform
    const int K = a.k;
    const int nrow = min(16 * TB, a.m - row0), ncol = (int)min((int64_t)16 * NB, a.n - col0);
    const float* xbase = a.x + (int64_t)row0 * K;
    const char* wbase = (const char*)a.w + col0 * K * WB;
    // rows past the end read as zero and are not stored
    const uint32_t xbytes = (uint32_t)nrow * K * 4, wbytes = (uint32_t)ncol * K * WB;

    // copies: lane -> (row, 16-byte unit); units 0 .. half - 1 are the chains
    // 4 wave .. 4 wave + 3, the others the chains 32 above them.  Unit u of a
    // row sits at u ^ swizzle(row), so a quarter wave's operand reads (16 rows)
    // cover the banks once.
    int xo[XC], wo[WC];
#pragma unroll
    for (int i = 0; i < XC; ++i) {
        const int row = 8 * i + (lane >> 3), u = (lane & 7) ^ ((row >> 1) & 7);
        xo[i] = row * K * 4 + 64 * wave + 512 * (u >> 2) + 16 * (u & 3);
    }
#pragma unroll
    for (int i = 0; i < WC; ++i) {
        if constexpr (WK == XK_BF16) {
            const int row = 16 * i + (lane >> 2), u = (lane & 3) ^ ((row >> 2) & 3);
            wo[i] = row * K * 2 + 32 * wave + 256 * (u >> 1) + 16 * (u & 1);
        } else {
            const int row = 8 * i + (lane >> 3), u = (lane & 7) ^ ((row >> 1) & 7);
            wo[i] = row * K * 4 + 64 * wave + 512 * (u >> 2) + 16 * (u & 3);
        }
    }
    const int xrd = r * XS + ((c ^ ((r >> 1) & 7)) << 4);  // chains 4 wave + c; the others at xrd ^ 64
    const int wrd = WK == XK_BF16 ? r * WS + (((c >> 1) ^ ((r >> 2) & 3)) << 4) + 8 * (c & 1) : xrd;

    v16f acc[TB][NB][2];
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
        for (int u = 0; u < NB; ++u)
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[t][u][g][v] = 0.0f;

    const int full = K >> 8;  // blocks of 256 elements
    const auto issue = [&](int j, int d) {
        const __amdgpu_buffer_rsrc_t xr = make_rsrc(xbase, j < full ? xbytes : 0u);
        const __amdgpu_buffer_rsrc_t wr = make_rsrc(wbase, j < full ? wbytes : 0u);
        uint8_t* st = (d ? lds1 : lds0) + wave * (XW + WW);
#pragma unroll
        for (int i = 0; i < WC; ++i) copy_to_lds(wr, st + XW + 1024 * i, wo[i] + j * 256 * WB);
#pragma unroll
        for (int i = 0; i < XC; ++i) copy_to_lds(xr, st + 1024 * i, xo[i] + j * 1024);
    };
    const auto mfma4 = [&](const uint4 (&xv)[TB], const DenseW<WK> (&wv)[NB], int g) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int t = 0; t < TB; ++t) {
                const uint4 q = xv[t];
                const float xe = __uint_as_float(e == 0 ? q.x : (e == 1 ? q.y : (e == 2 ? q.z : q.w)));
#pragma unroll
                for (int u = 0; u < NB; ++u)
                    acc[t][u][g] =
                        __builtin_amdgcn_mfma_f32_16x16x1f32(xe, dense_w<WK>(wv[u], e), acc[t][u][g], 0, 0, 0);
            }
    };
    const auto step = [&](int d) {
        const uint8_t* st = (d ? lds1 : lds0) + wave * (XW + WW);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            uint4 xv[TB];
            DenseW<WK> wv[NB];
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                const uint8_t* p = st + XW + 16 * u * WS + (WK == XK_BF16 ? wrd ^ (32 * g) : wrd ^ (64 * g));
                if constexpr (WK == XK_BF16) wv[u].v = *(const uint2*)p;
                else wv[u].v = *(const uint4*)p;
            }
#pragma unroll
            for (int t = 0; t < TB; ++t) xv[t] = *(const uint4*)(st + 16 * t * XS + (xrd ^ (64 * g)));
            mfma4(xv, wv, g);
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d) issue(d, d);
    int j = 0;
    for (; j + D <= full; j += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            // this wave's copies of block j + d have landed (it reads no other wave's)
            __builtin_amdgcn_s_waitcnt(vmcnt_imm((D - 1) * (XC + WC)));
            __asm__ volatile("" ::: "memory");
            step(d);
            __asm__ volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);  // every read of stage d is done (its products are issued)
            issue(j + D + d, d);
        }
    }
    wait_loads();
    __asm__ volatile("" ::: "memory");
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (j + d < full) step(d);
    if (K & 255) {
        // the row's last chunks: a chain past the end takes fma(0, -0, acc) = acc
        const __amdgpu_buffer_rsrc_t xr = make_rsrc(xbase, xbytes), wr = make_rsrc(wbase, wbytes);
        const int rem = (K & 255) >> 2;
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const int ch = 32 * g + 4 * wave + c;
            const bool in = ch < rem;
            uint4 xv[TB];
            DenseW<WK> wv[NB];
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                dense_load_w<WK>(wv[u], wr, in ? (16 * u + r) * K * WB + 4 * WB * (64 * full + ch) : kOOB, 0);
                if (!in) {
                    if constexpr (WK == XK_BF16) wv[u].v = make_uint2(0x80008000u, 0x80008000u);
                    else wv[u].v = make_uint4(0x80000000u, 0x80000000u, 0x80000000u, 0x80000000u);
                }
            }
#pragma unroll
            for (int t = 0; t < TB; ++t) xv[t] = bload_s(xr, in ? (16 * t + r) * K * 4 + 16 * (64 * full + ch) : kOOB, 0);
            mfma4(xv, wv, g);
        }
    }

    // two tiles at a time, one in each array: [chain][16 x 16 outputs]
#pragma unroll
    for (int p = 0; p < TB * NB; p += 2) {
        __syncthreads();  // the arrays are no longer read
#pragma unroll
        for (int i = p; i < p + 2 && i < TB * NB; ++i) {
            float* s_c = (float*)(i & 1 ? lds1 : lds0);
#pragma unroll
            for (int v = 0; v < 16; ++v)
                s_c[(4 * wave + (v >> 2)) * 256 + (4 * c + (v & 3)) * 16 + r] =
                    __fadd_rn(acc[i / NB][i % NB][0][v], acc[i / NB][i % NB][1][v]);
        }
        __syncthreads();
        const int i = p + (tid >> 8), e = tid & 255;
        if (i < TB * NB) {
            const int row = i / NB * 16 + (e >> 4), col = i % NB * 16 + (e & 15);
            const float* s_c = (const float*)(tid >> 8 ? lds1 : lds0) + e;
            float z[16];
#pragma unroll
            for (int l = 0; l < 16; ++l) z[l] = __fadd_rn(s_c[l * 256], s_c[(l + 16) * 256]);
#pragma unroll
            for (int h = 8; h >= 1; h >>= 1)
#pragma unroll
                for (int l = 0; l < h; ++l) z[l] = __fadd_rn(z[l], z[l + h]);
            if (row < nrow && col < ncol) a.y[(int64_t)(row0 + row) * a.n + col0 + col] = z[0];
        }
    }
}

template <int WK, int TB, int NB>
static void launch_dense_mm_t(DenseMm a, hipStream_t st)
{
    a.mt = (a.m + 16 * TB - 1) / (16 * TB);
    const int64_t nt = (a.n + 16 * NB - 1) / (16 * NB);
    hipLaunchKernelGGL((k_dense_mm<WK, TB, NB>), dim3((unsigned)((nt + 7) / 8 * 8 * a.mt)), dim3(512), 0, st, a);
}

hipError_t launch_dense_mm(const void* w, int wkind, int64_t n, int64_t k, const float* x, int64_t m, float* y,
                           hipStream_t st)
{
    DenseMm a{w, x, y, n, (int)m, (int)k, 0};
    // 32 x 32 tiles (one workgroup per CU) when more than 16 tokens make enough
    // of them, else 16 x 16 (two per CU); us with 16 x 16 / 32 x 32 tiles: k =
    // 4096, n = 1024: m = 64 11 / 21, 128 20 / 23, 256 38 / 26; n = 5632: m = 16
    // 25 / 25, 32 30 / 28, 128 91 / 70
    const bool big = m > 16 && ((m + 31) / 32) * ((n + 31) / 32) >= 160;
#define BTL_DENSE_MM(WKV)                                    \
    if (wkind == WKV) {                                      \
        if (big) launch_dense_mm_t<WKV, 2, 2>(a, st);        \
        else launch_dense_mm_t<WKV, 1, 1>(a, st);            \
        return hipGetLastError();                            \
    }
    BTL_DENSE_MM(XK_F32)
    BTL_DENSE_MM(XK_BF16)
#undef BTL_DENSE_MM
    return hipErrorInvalidValue;
}

}  // namespace btl
