// zq_gemm_skinny.hip -- fp32-activation GEMM for few tokens, and without a
// workspace.
//
// Y[t][n] = sum_k X[t][k] * W[n][k], fp32 activations, every format.  At a few
// tokens the weights are the traffic and the launches the time, so this kernel
// needs no activation pass, no workspace and no K planes: a workgroup takes 32
// (or 64) tokens x 32 weight rows, its waves share the tile's K (a group
// of 32 elements each in turn) and add their sums through LDS at the end.  The
// weights go from memory straight to the matrix core's operand registers, the
// activations through a part of LDS that belongs to the wave, in whole lines;
// there is no barrier in the loop.
//
// Products: an fp32 activation is the exact sum of three bf16 values (8 + 8 +
// 8 significant bits), a weight code is a whole number of at most 8 bits, so
// v_mfma_f32_32x32x16_bf16 gives exact products in fp32 sums, three
// instructions for each 16 k.  A group's sum is scaled by its fp32 scale into
// the accumulator; the offset of Q4_K / Q5_K multiplies the group's sum of x on
// the fp32 MFMA.  Sums that are not finite are formed again in fp32 with the
// dequantised weights (see the kernel).
//
// Bound: at a few tokens the launch and the chain of a wave's K groups (loads,
// decoding, products; 16 and 8 waves sharing K measured the same), at many the
// VALU work of decoding each weight again for every 64 tokens.  Where the split
// kernels are faster depends on rows, K and workspace as well as tokens: the
// estimates of plan_gemm_skinny_f32 and plan_gemm_split.  Q4_K, 19 tokens, 4096 +
// 1024 + 1024 rows x 4096: 94 us in nine launches -> 16.9 in one.
#include "zq_device.hpp"
#include "zq_internal.hpp"

#include <algorithm>

namespace zq {
namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u4a2_t __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u4a4_t __attribute__((ext_vector_type(4), aligned(4)));
typedef __bf16 b8_t __attribute__((ext_vector_type(8)));

// Waves of a workgroup: 16 for one token tile; for two (their registers) 8, or 4
// or 2 where K is short and the grid large, so that a CU has 2 or 4 workgroups
// and their starts and ends overlap (see plan_gemm_skinny_f32).

// The weight matrices of one launch: task i's 32-row tiles start at tile[i].
struct SkinnyTasks {
    const uint8_t* w[kMaxTasks];
    float* y[kMaxTasks];
    uint32_t rows[kMaxTasks];
    uint32_t tile[kMaxTasks + 1];
    int count;
    float* partial;       // planes 1.. of the one task of a K split
    uint32_t groups;      // groups of 32 per split
};

__device__ __forceinline__ uint32_t fbits(float f) { return __builtin_bit_cast(uint32_t, f); }
__device__ __forceinline__ float bitsf(uint32_t u) { return __builtin_bit_cast(float, u); }
// the upper halves of two fp32 words as a bf16 pair
__device__ __forceinline__ uint32_t hi_pair(float a, float b) {
    return __builtin_amdgcn_perm(fbits(b), fbits(a), 0x07060302u);
}

// x (8 elements) as bf16 planes: p0 + p1 + p2 == x exactly, down to 2^-110 (below,
// to 2^-133 absolutely).  An infinity or a NaN gives a NaN in p1.
__device__ __forceinline__ void split3(const float (&x)[8], b8_t& p0, b8_t& p1, b8_t& p2) {
    float r1[8], r2[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) r1[i] = x[i] - bitsf(fbits(x[i]) & 0xffff0000u);
#pragma unroll
    for (int i = 0; i < 8; ++i) r2[i] = r1[i] - bitsf(fbits(r1[i]) & 0xffff0000u);
    u4_t a, b, c;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        a[i] = hi_pair(x[2 * i], x[2 * i + 1]);
        b[i] = hi_pair(r1[2 * i], r1[2 * i + 1]);
        c[i] = hi_pair(r2[2 * i], r2[2 * i + 1]);
    }
    p0 = __builtin_bit_cast(b8_t, a);
    p1 = __builtin_bit_cast(b8_t, b);
    p2 = __builtin_bit_cast(b8_t, c);
}

// Eight signed code bytes as bf16 (|value| <= 128: exact), the bits `flip` of
// each pair changed.
__device__ __forceinline__ b8_t codes8(uint32_t a, uint32_t b, uint32_t flip) {
    u4_t o;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        o[i] = hi_pair(sbyte(a, 2 * i), sbyte(a, 2 * i + 1));
        o[2 + i] = hi_pair(sbyte(b, 2 * i), sbyte(b, 2 * i + 1));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] ^= flip;
    return __builtin_bit_cast(b8_t, o);
}

// One group of 32 elements of a weight row, as one lane (half h of the wave)
// holds it: 16 elements.  The codes are carried centred and shifted to the top
// of a signed byte: 1, 16, 16, 8, 4 times the code (Q8_0, Q4_0, Q4_K, Q5_K,
// Q6_K).
template <int FMT>
constexpr bool kOffset = FMT == kQ4_K || FMT == kQ5_K;
template <int FMT>
struct Group {
    u4_t q;
    u4_t h[FMT == kQ5_K || FMT == kQ6_K ? 1 : 0];  // fifth bits / the codes' upper two bits
    u4_t head[kOffset<FMT> ? 1 : 0];               // d, dmin, the 12 scale bytes
    uint32_t d;
    uint32_t sc;  // Q6_K: the two int8 scales
};
// First of the 8 elements of MFMA step s (0, 1) for lane half h, from the
// group's first.  Q6_K's steps are its 16-element scale groups.
template <int FMT>
__device__ __forceinline__ uint32_t step_k(uint32_t s, uint32_t h) {
    return FMT == kQ6_K ? 16 * s + 8 * h : 16 * h + 8 * s;
}
template <int FMT>
__device__ __forceinline__ void load_group(const uint8_t* row, uint32_t b, uint32_t h, Group<FMT>& r) {
    const uint32_t g = b & 7u;
    if constexpr (FMT == kQ8_0 || FMT == kQ4_0) {
        const uint8_t* p = row + size_t(b) * (FMT == kQ8_0 ? 34 : 18);
        r.q = *reinterpret_cast<const u4a2_t*>(p + 2 + (FMT == kQ8_0 ? 16 * h : 0));
        r.d = *reinterpret_cast<const uint16_t*>(p);
    } else if constexpr (kOffset<FMT>) {
        const uint8_t* p = row + size_t(b >> 3) * (FMT == kQ5_K ? 176 : 144);
        r.head[0] = *reinterpret_cast<const u4a4_t*>(p);
        r.q = *reinterpret_cast<const u4a4_t*>(p + (FMT == kQ5_K ? 48 : 16) + (g >> 1) * 32 + 16 * h);
        if constexpr (FMT == kQ5_K) r.h[0] = *reinterpret_cast<const u4a4_t*>(p + 16 + 16 * h);
    } else {
        const uint8_t* p = row + size_t(b >> 3) * 210;
        // the lane's elements: 8h..8h+7 and 16+8h..16+8h+7 of the line
        typedef uint32_t u2a2_t __attribute__((ext_vector_type(2), aligned(2)));
        const uint8_t* lo = p + (g >> 2) * 64 + (g & 1u) * 32 + 8 * h;
        const uint8_t* hi = p + 128 + (g >> 2) * 32 + 8 * h;
        const u2a2_t q0 = *reinterpret_cast<const u2a2_t*>(lo), q1 = *reinterpret_cast<const u2a2_t*>(lo + 16);
        const u2a2_t h0 = *reinterpret_cast<const u2a2_t*>(hi), h1 = *reinterpret_cast<const u2a2_t*>(hi + 16);
        r.q = u4_t{q0[0], q0[1], q1[0], q1[1]};
        r.h[0] = u4_t{h0[0], h0[1], h1[0], h1[1]};
        r.sc = *reinterpret_cast<const uint16_t*>(p + 192 + 2 * g);
        r.d = *reinterpret_cast<const uint16_t*>(p + 208);
    }
}
// The group's codes, its scale(s) -- per step for Q6_K -- and, of its offset,
// centre * scale and min.  flip (all bits of a uniform word, or none): codes and
// scales with their signs changed.  The bf16 products' sums are rounded down, not
// to nearest (measured: the mean of the errors of a long K is -0.4 of their
// spread), which scales of one sign would carry to every output alike, and a
// model's later layers feel that more than as much noise: with half of the
// groups flipped it cancels.  Q6_K's sub-block scales have either sign already.
template <int FMT>
__device__ __forceinline__ void decode_group(const Group<FMT>& r, uint32_t b, uint32_t h, uint32_t flip, b8_t (&w)[2],
                                             float (&s)[2], float& cds, float& min) {
    const uint32_t g = b & 7u;
    uint32_t c[4];
    cds = min = 0.0f;
    if constexpr (FMT == kQ8_0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) c[i] = r.q[i];
        s[0] = s[1] = bitsf(fbits(half_bits_to_float(r.d)) ^ (flip & 0x80000000u));
    } else if constexpr (FMT == kQ4_0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) c[i] = ((r.q[i] << (h ? 0 : 4)) & 0xF0F0F0F0u) ^ 0x80808080u;
        s[0] = s[1] = bitsf(fbits(half_bits_to_float(r.d) * 0.0625f) ^ (flip & 0x80000000u));
    } else if constexpr (kOffset<FMT>) {
        const uint32_t sh = 8 * (g & 3u);
        const u4_t& hd = r.head[0];
        const uint32_t sc = g < 4 ? (hd[1] >> sh) & 63u : ((hd[3] >> sh) & 15u) | ((hd[1] >> (sh + 2)) & 0x30u);
        const uint32_t mn = g < 4 ? (hd[2] >> sh) & 63u : ((hd[3] >> (sh + 4)) & 15u) | ((hd[2] >> (sh + 2)) & 0x30u);
        const float ds = half_bits_to_float(hd[0]) * float(sc);
        min = half_bits_to_float(hd[0] >> 16) * float(mn);  // exact
        // flipped: the code's complement, which is centred one lower
        constexpr uint32_t top = FMT == kQ4_K ? 0xF0F0F0F0u : 0xF8F8F8F8u;
        const uint32_t sign = 0x80808080u ^ (flip & top);
        cds = ((FMT == kQ4_K ? 8.0f : 16.0f) - (flip ? 1.0f : 0.0f)) * ds;
        s[0] = s[1] = ds * (FMT == kQ4_K ? 0.0625f : 0.125f) * (flip ? -1.0f : 1.0f);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t n = (r.q[i] << (4 * (1 - (g & 1u)))) & 0xF0F0F0F0u;  // the code in the upper nibble
            if constexpr (FMT == kQ4_K) c[i] = n ^ sign;
            else c[i] = ((n >> 1) | (((r.h[0][i] >> g) & 0x01010101u) << 7)) ^ sign;
        }
    } else {
        const float d = half_bits_to_float(r.d) * 0.25f;
#pragma unroll
        for (int q = 0; q < 2; ++q) s[q] = d * float(int(int8_t(uint8_t(r.sc >> (8 * q)))));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t n = (r.q[i] >> (4 * ((g >> 1) & 1u))) & 0x0F0F0F0Fu;
            c[i] = ((n << 2) | (((r.h[0][i] >> (2 * (g & 3u))) & 0x03030303u) << 6)) ^ 0x80808080u;
        }
    }
    w[0] = codes8(c[0], c[1], FMT == kQ8_0 || FMT == kQ4_0 ? flip & 0x80008000u : 0u);
    w[1] = codes8(c[2], c[3], FMT == kQ8_0 || FMT == kQ4_0 ? flip & 0x80008000u : 0u);
}

template <int FMT, int MT, int NW>
__global__ __launch_bounds__(64 * NW, MT == 1 ? 4 : 2) void gemm_skinny_f32_kernel(SkinnyTasks tasks, const float* X, uint32_t M,
                                                                                    uint32_t K) {
    // each wave's activations of one group, [MT * 32 rows][128 B], 16-byte units
    // XOR-swizzled by the row; the waves' sums at the end
    __shared__ __align__(16) float lds[NW][MT][16 * 64];
    const uint32_t tiles = tasks.tile[tasks.count];
    // blockIdx.x = (split * token tiles + token tile) * tiles + tile
    const uint32_t tile = blockIdx.x % tiles, token_tiles = (M + 32 * MT - 1) / (32 * MT);
    const uint32_t m0 = blockIdx.x / tiles % token_tiles * (32 * MT), split = blockIdx.x / tiles / token_tiles;
    int t = 0;
    while (t + 1 < tasks.count && tile >= tasks.tile[t + 1]) ++t;  // uniform
    const uint32_t N = tasks.rows[t], n0 = (tile - tasks.tile[t]) * 32;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t l32 = lane & 31, lh = lane >> 5;
    const uint32_t first = split * tasks.groups, end = min(K >> 5, first + tasks.groups);
    const uint32_t flip = (first + wave) & 1u ? ~0u : 0u;  // by wave: a wave's groups are NW apart
    // loads cover whole lines: 8 lanes a row's 128 bytes (a lane reading its own
    // operand row touched 32 lines an instruction and bound the kernel)
    struct Source {
        const uint8_t* row;
        const float* x[MT][4];
    };
    auto source = [&](uint32_t lane) {
        Source o;
        o.row = tasks.w[t] + size_t(min(n0 + (lane & 31), N - 1)) * row_bytes_dev(FMT, K);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                o.x[i][q] = X + size_t(min(m0 + 32 * i + 8 * q + (lane >> 3), M - 1)) * K + 4 * (lane & 7);
        return o;
    };
    float* stage = &lds[wave][0][0];
    const uint32_t st_w = (uint32_t(lane >> 3) * 8 + ((lane & 7) ^ ((lane >> 4) & 7))) * 4;  // + 8 rows: swizzle + 4 mod 8

    v16f acc[MT], zero;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        zero[v] = 0.0f;
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[i][v] = 0.0f;
    }
    // A group's weights and activations are loaded while the wave's group
    // before it is multiplied (the last one again, unused).
    struct Data {
        Group<FMT> w;
        f4_t x[MT][4];  // [token tile][8 rows]
    };
    auto load = [&](const Source& from, uint32_t b, Data& d) {
        load_group<FMT>(from.row, b, lh, d.w);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) d.x[i][q] = *reinterpret_cast<const f4_t*>(from.x[i][q] + 32 * b);
    };
    auto stage_x = [&](const Data& d) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q)  // row 8q + lane / 8 of the tile, unit lane % 8
                *reinterpret_cast<f4_t*>(stage + i * 1024 + q * 256 + (st_w ^ (q & 1 ? 16u : 0u))) = d.x[i][q];
    };
    auto read_x = [&](int i, int s, float (&e)[8]) {
#pragma unroll
        for (uint32_t q = 0; q < 2; ++q) {
            const uint32_t unit = step_k<FMT>(s, lh) / 4 + q;
            const f4_t f = *reinterpret_cast<const f4_t*>(stage + i * 1024 + l32 * 32 + ((unit ^ ((l32 >> 1) & 7)) * 4));
#pragma unroll
            for (int c = 0; c < 4; ++c) e[4 * q + c] = f[c];
        }
    };
    auto multiply = [&](uint32_t b, const Data& d) {
        stage_x(d);
        b8_t w[2];
        float sc[2], cds, min;
        decode_group<FMT>(d.w, b, lh, flip, w, sc, cds, min);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            v16f p = zero;
            float sum = 0.0f;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                float e[8];
                read_x(i, s, e);
                if constexpr (kOffset<FMT>) sum += ((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]));
                b8_t p0, p1, p2;
                split3(e, p0, p1, p2);
                p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p2, w[s], p, 0, 0, 0);
                p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p1, w[s], p, 0, 0, 0);
                p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p0, w[s], p, 0, 0, 0);
                if (FMT == kQ6_K || s == 1) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[i][v] = fmaf(p[v], sc[s], acc[i][v]);
                    p = zero;
                }
            }
            if constexpr (kOffset<FMT>) acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(sum, cds - min, acc[i], 0, 0, 0);
        }
    };
    if (first + wave < end) {
        const Source from = source(lane);
        Data d0, d1;
        load(from, first + wave, d0);
        for (uint32_t b = first + wave;;) {
            load(from, min(b + NW, end - 1), d1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(b, d0);
            if ((b += NW) >= end) break;
            load(from, min(b + NW, end - 1), d0);
            __builtin_amdgcn_sched_barrier(0);
            multiply(b, d1);
            if ((b += NW) >= end) break;
        }
    }
    // Sums that are not finite again, in fp32 with the dequantised weights: an
    // infinite activation is to give an infinity of the sign of the weight it meets
    // (a centred code and the group's offset can have opposite ones), and a code
    // times a huge one may have overflowed where the weight times it does not.
    float odd = 0.0f;  // NaN if one is not
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) odd = fmaf(acc[i][v], 0.0f, odd);
    if (__any(odd != 0.0f)) {
        uint32_t l = lane;  // opaque: the addresses are formed here again, not kept through the loop above
        asm volatile("" : "+v"(l));
        const Source from = source(l);
        v16f t[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) t[i] = zero;
        for (uint32_t b = first + wave; b < end; b += NW) {
            Data d;
            load(from, b, d);
            stage_x(d);
            b8_t w[2];
            float sc[2], cds, min;
            decode_group<FMT>(d.w, b, lh, flip, w, sc, cds, min);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    float e[8];
                    read_x(i, s, e);
#pragma unroll
                    for (int c = 0; c < 8; ++c) {
                        const float q = float(w[s][c]);
                        const float wd = kOffset<FMT> ? fmaf(sc[s], q, cds) - min : sc[s] * q;  // one rounding
                        t[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(e[c], wd, t[i], 0, 0, 0);
                    }
                }
        }
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (!(fabsf(acc[i][v]) < __builtin_inff())) acc[i][v] = t[i][v];
    }
    // the waves' sums, added in wave order (a wave's own region: no wait before)
    float* Y = split ? tasks.partial + size_t(split - 1) * M * N : tasks.y[t];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) lds[wave][i][v * 64 + lane] = acc[i][v];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int q = 0; q < 16 / NW; ++q) {
            const int v = 16 / NW * wave + q;
            float s = lds[0][i][v * 64 + lane];
#pragma unroll
            for (int w = 1; w < NW; ++w) s += lds[w][i][v * 64 + lane];
            const uint32_t m = m0 + 32 * i + 8 * (v >> 2) + 4 * lh + (v & 3), n = n0 + l32;
            if (m < M && n < N) Y[size_t(m) * N + n] = s;
        }
}

template <int FMT>
hipError_t launch_skinny_fmt(const SkinnyTasks& t, const float* X, uint32_t ks, uint32_t nw, uint32_t M, uint32_t K,
                             hipStream_t stream) {
    const dim3 grid(t.tile[t.count] * ks * (M <= 32 ? 1 : (M + 63) / 64));
    if (M <= 32) hipLaunchKernelGGL((gemm_skinny_f32_kernel<FMT, 1, 16>), grid, dim3(1024), 0, stream, t, X, M, K);
    else if (nw == 2) hipLaunchKernelGGL((gemm_skinny_f32_kernel<FMT, 2, 2>), grid, dim3(128), 0, stream, t, X, M, K);
    else if (nw == 4) hipLaunchKernelGGL((gemm_skinny_f32_kernel<FMT, 2, 4>), grid, dim3(256), 0, stream, t, X, M, K);
    else hipLaunchKernelGGL((gemm_skinny_f32_kernel<FMT, 2, 8>), grid, dim3(512), 0, stream, t, X, M, K);
    return hipGetLastError();
}

}  // namespace

// A CU spends the given time on a group of 32 k of one workgroup (VALU-bound:
// the three-way split of the activations and the conversion of the codes;
// measured at K = 8192, one workgroup per CU, 1..32 and 33..64 tokens).  K
// splits keep a workgroup to 128 groups, as far as the grid then still fits
// the chip at once; a split adds its planes' traffic and a launch.
SkinnyPlan plan_gemm_skinny_f32(int fmt, size_t M, size_t N, size_t K, size_t planes) {
    const bool wide = M > 32;
    const double group_us = fmt == kQ6_K   ? (wide ? 0.265 : 0.20)
                            : fmt == kQ5_K ? (wide ? 0.22 : 0.125)
                            : fmt == kQ4_K ? (wide ? 0.205 : 0.11)
                                           : (wide ? 0.18 : 0.137);
    const uint32_t nb = uint32_t(K / 32), cus = uint32_t(device_cu_count());
    const size_t wgs = (N + 31) / 32 * (wide ? (M + 63) / 64 : 1);
    const uint32_t most = uint32_t(std::min<size_t>({planes + 1, std::max<size_t>(1, cus / wgs), 32}));
    uint32_t ks = std::max(1u, std::min(most, (nb + 127) / 128));
    const uint32_t per = (nb + ks - 1) / ks;
    ks = (nb + per - 1) / per;  // no empty splits
    auto rounds = [&](uint32_t slots) { return double((wgs * ks + slots - 1) / slots); };
    double us = 3.0 + rounds(cus) * (per * group_us + 2.0);  // 2 us: a workgroup's start and its waves' sum
    // Fewer waves: two or four workgroups on a CU share its time, 15 % better, and
    // one start and end (which 3 us describes better here).  1000 x 14336 x 256 of
    // Q6_K 150 us with 8 waves, 81 with 4, 73 with 2; 1000 x 4096 x 1024 of Q8_0
    // 71, 55, 63; a grid of one round loses: 64 x 4096 x 1024 11.7, 12.8, 18.8.
    // Up to 32 groups, where the 128 x 128 tiles on the fp32 MFMA before this
    // kernel had been up to 1.7x faster than 8 waves.
    uint32_t nw = 8;
    double best = 3.0 + rounds(cus) * (per * group_us + 3.0);
    for (uint32_t n : {4u, 2u}) {
        const uint32_t share = 8 / n;
        const double t = 3.0 + rounds(cus * share) * (0.85 * share * per * group_us + 2.0);
        if (wide && per <= 32 && t < best) best = t, nw = n;
    }
    if (nw < 8) us = std::min(us, best);
    if (ks > 1) us += 3.0 + double(ks - 1) * double(M) * double(N) * 8.0 / 4.0e6;
    return SkinnyPlan{ks, nw, us};
}

hipError_t launch_gemm_skinny_f32(int fmt, const uint8_t* const* w, float* const* Y, const size_t* rows, size_t count,
                                  const float* X, float* partial, uint32_t ks, uint32_t nw, size_t M, size_t K,
                                  hipStream_t stream) {
    SkinnyTasks t{};
    t.count = int(count);
    for (size_t i = 0; i < count; ++i) {
        t.w[i] = w[i];
        t.y[i] = Y[i];
        t.rows[i] = uint32_t(rows[i]);
        t.tile[i + 1] = t.tile[i] + uint32_t((rows[i] + 31) / 32);
    }
    const uint32_t m = uint32_t(M), k = uint32_t(K), nb = k / 32;
    t.partial = partial;
    t.groups = (nb + ks - 1) / ks;
    hipError_t e = hipErrorInvalidValue;
    switch (fmt) {
    case kQ8_0: e = launch_skinny_fmt<kQ8_0>(t, X, ks, nw, m, k, stream); break;
    case kQ4_0: e = launch_skinny_fmt<kQ4_0>(t, X, ks, nw, m, k, stream); break;
    case kQ4_K: e = launch_skinny_fmt<kQ4_K>(t, X, ks, nw, m, k, stream); break;
    case kQ5_K: e = launch_skinny_fmt<kQ5_K>(t, X, ks, nw, m, k, stream); break;
    case kQ6_K: e = launch_skinny_fmt<kQ6_K>(t, X, ks, nw, m, k, stream); break;
    default: break;
    }
    return e != hipSuccess || ks <= 1 ? e : launch_splitk_add(partial, Y[0], M, rows[0], ks - 1, stream);
}

}  // namespace zq
