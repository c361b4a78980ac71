// zq_gemm_split.hip -- fp32-activation prefill GEMM on the f16 matrix cores.
//
// Y[t][n] = sum_k X[t][k] * W[n][k] with fp32 activations, for every weight
// format.  A GGML weight is a small whole code times a group scale (plus a
// group offset for Q4_K / Q5_K), and the codes are exact in binary16.  So:
//  * split_acts_kernel scales each activation row by a power of two and
//    stores it as f16 hi + lo (23 significant bits), 32 elements at a time;
//  * the GEMM multiplies codes by hi and lo on v_mfma_f32_32x32x16_f16 (exact
//    products, fp32 sums: two instructions where one fp32 MFMA of the same
//    size would take sixteen) and applies the group scales in fp32.
// Bound: the issue of what runs beside the MFMAs.  By the counters the matrix
// cores are busy 42 % of the chip's cycles with Q8_0 512 x 14336 x 4096 (0.88 PF
// of f16 products; 224 workgroups on 256 CUs), 54 % with Q6_K 1000 x 4096 x 14336
// (1.05 PF), at 1.9-2.0 GHz; a loop of these MFMAs alone reaches 1.6 PF on random
// data, where power takes the clock to 1.6 GHz, and 1.2 PF with 8 FMAs to each.
// A tile of 128 x 256 (128 x 128 for small grids, see plan_gemm_split) because the
// next operand reads, the staging and the scale FMAs of a stage then just fit
// between its MFMAs.  Measured, fp32-MFMA or three-product f16 kernel -> here:
//   Q8_0  512 x 14336 x 4096   555 -> 144-150 us (108 -> 400-417 TFLOP/s of the GEMM)
//   Q6_K 1000 x 4096 x 14336   534 -> 370-380 us; 512 tokens 0.32-0.37 -> 0.22 ms
//   Q4_K / Q5_K 512 x 14336 x 4096   0.29-0.32 -> 0.18 / 0.30-0.34 -> 0.19 ms
// and an error against 64 bits that is no larger in any format, of a single
// product (Q8_0 4e-7..1.2e-6 -> 1.1e-7..3.5e-7, Q4_K 2.0e-7..2.2e-7 ->
// 1.3e-7..2.1e-7) and of a decoder's logits.
#include "zq_device.hpp"
#include "zq_gemm_common.hpp"
#include "zq_internal.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace zq {
namespace {

constexpr int kThreads = 256;
// Word 3 of a raw buffer resource on gfx9-family parts (32-bit data format,
// no swizzle, stride 0): offsets are plain byte offsets from the base.
constexpr int kBufferWord3 = 0x00020000;

typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u4a2_t __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u4a4_t __attribute__((ext_vector_type(4), aligned(4)));

// ---------------------------------------------------- split activations ---
// Row r of X as f16 hi + lo of x * 2^e, e such that the row's largest finite
// magnitude lies in [2^14, 2^15): out[r][block] = 32 hi halves, 32 lo halves;
// ex[r] = e.  x - hi is exact in fp32, so hi + lo carries x to 2^-23 of
// itself (2^-40 of the row's maximum for elements so small that lo is
// subnormal).  A NaN reaches every output of its row.  A row with an infinity
// (whose products with a weight's parts can have opposite signs where the
// weight's own sign decides), or with so large a span that 2^-40 of its maximum
// shows where its largest elements meet zero codes, is marked instead: ex[r] =
// kExactRow, and exact_tile() multiplies it in fp32.  That is: the elements more
// than 2^20 below the maximum, `lost` of them, lose up to 2^-25 each (scaled), and
// this is set against fp32's rounding of the sum of those more than 2^8 below it
// (the others may meet zeros): marked if the sum of their squares is under lost /
// 16.  A row whose small elements are few, or that has others between, is not.
constexpr int kExactRow = 1 << 20;
__device__ __forceinline__ float finite_abs(float v) {
    const float a = fabsf(v);
    return a < __builtin_inff() ? a : 0.0f;
}
// SUMS (K % 256 == 0): also sums[r][super-block] = 8 hi then 8 lo halves of the
// groups' S / 32, S the sum of a group's 32 scaled elements.
template <bool SUMS>
__global__ __launch_bounds__(kThreads) void split_acts_kernel(const float* __restrict__ X, _Float16* __restrict__ out,
                                                              int* __restrict__ ex, _Float16* __restrict__ sums,
                                                              uint32_t K) {
    __shared__ float red[kThreads / 64];
    const float4* r = reinterpret_cast<const float4*>(X + size_t(blockIdx.x) * K);
    const uint32_t K4 = K / 4;
    float m = 0.0f;
    for (uint32_t i = threadIdx.x; i < K4; i += kThreads) {
        const float4 v = r[i];
        m = fmaxf(m, fmaxf(fmaxf(finite_abs(v.x), finite_abs(v.y)), fmaxf(finite_abs(v.z), finite_abs(v.w))));
    }
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    m = red[0];
#pragma unroll
    for (int w = 1; w < kThreads / 64; ++w) m = fmaxf(m, red[w]);
    const int e = m > 0.0f ? 15 - __builtin_amdgcn_frexp_expf(m) : 0;
    float lost = 0.0f;  // non-zero elements more than 2^20 below the maximum, 1e9 for an infinity
    float low = 0.0f;   // squares of those more than 2^8 below it, as far as looked at
    auto add_low = [&](float f) { low = fabsf(f) < 0x1p6f ? fmaf(f, f, low) : low; };
    _Float16* o = out + size_t(blockIdx.x) * K * 2;
    auto split = [](float f, _Float16& h, _Float16& l) {
        h = _Float16(f);
        const float rest = f - float(h);
        l = _Float16(fabsf(f) < __builtin_inff() ? rest : 0.0f);
    };
    for (uint32_t i = threadIdx.x; i < K4; i += kThreads) {
        const float4 v = r[i];
        const float f[4] = {ldexpf(v.x, e), ldexpf(v.y, e), ldexpf(v.z, e), ldexpf(v.w, e)};
        h4_t h, l;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            _Float16 a, b;
            split(f[k], a, b);
            h[k] = a;
            l[k] = b;
        }
        const float least = fminf(fminf(fabsf(f[0]), fabsf(f[1])), fminf(fabsf(f[2]), fabsf(f[3])));
        const float most = fmaxf(fmaxf(fabsf(f[0]), fabsf(f[1])), fmaxf(fabsf(f[2]), fabsf(f[3])));
        if (__any(least < 0x1p-6f || most == __builtin_inff())) {  // seldom
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float t = fabsf(f[k]);
                lost += t == __builtin_inff() ? 1e9f : t != 0.0f && t < 0x1p-6f ? 1.0f : 0.0f;
                add_low(f[k]);
            }
        }
        _Float16* d = o + size_t(i >> 3) * 64 + (i & 7u) * 4;
        *reinterpret_cast<h4_t*>(d) = h;
        *reinterpret_cast<h4_t*>(d + 32) = l;
        if constexpr (SUMS) {  // a group is the 8 lanes of an aligned octet; K / 4 is a multiple of 64
            const float t = group_sum<8>((f[0] + f[1]) + (f[2] + f[3])) * 0.03125f;
            if ((i & 7u) == 0) {
                _Float16 a, b;
                split(t, a, b);
                _Float16* g = sums + (size_t(blockIdx.x) * (K / 256) + (i >> 6)) * 16 + ((i >> 3) & 7u);
                g[0] = a;
                g[8] = b;
            }
        }
    }
    auto block_sum = [&](float v) {
        v = wave_sum(v);
        __syncthreads();
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
        __syncthreads();
        return (red[0] + red[1]) + (red[2] + red[3]);
    };
    lost = block_sum(lost);  // whole numbers below 2^24, or past 2^28
    bool exact = lost >= 1e9f;
    // the neighbours of the few lost elements of an ordinary row are enough
    if (lost > 0.0f && !exact && block_sum(low) < 0.0625f * lost) {
        low = 0.0f;
        for (uint32_t i = threadIdx.x; i < K4; i += kThreads) {
            const float4 v = r[i];
            add_low(ldexpf(v.x, e));
            add_low(ldexpf(v.y, e));
            add_low(ldexpf(v.z, e));
            add_low(ldexpf(v.w, e));
        }
        exact = block_sum(low) < 0.0625f * lost;
    }
    if (threadIdx.x == 0) ex[blockIdx.x] = exact ? kExactRow : e;
}

// ------------------------------------------------------------- decoders ---
// v, opaque to the optimiser at this point: keeps a lane offset 32-bit beside
// its scalar base (one register, no 64-bit add per load), where hoisting its
// extension out of the loop would take two and an add.
__device__ __forceinline__ uint32_t opaque(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}
// Four code bytes u0..u3 (0..255) as binary16 u - off (NEG: off - u), two per
// dword: a byte placed under 0x64 is the binary16 1024 + u.
template <bool NEG = false>
__device__ __forceinline__ void bytes_to_half(uint32_t u, _Float16 off, h2_t& a, h2_t& b) {
    const h2_t o = {off, off};
    a = __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u));
    b = __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u));
    a = NEG ? o - a : a - o;
    b = NEG ? o - b : b - o;
}

// A thread's share of one 32-element block: half h holds elements 16h..16h+15.
// In the MFMA's k order, step j (0, 1) and lane half h take elements
// 16h + 8j .. 16h + 8j + 7, for weights and activations alike.
template <int FMT>
struct Raw {
    u4_t q;
    uint32_t d;
};
// Byte of half h's codes within a block.
template <int FMT>
__device__ __forceinline__ uint32_t code_offset(uint32_t h) {
    return FMT == kQ8_0 ? 2 + 16 * h : 2;
}
// Block b's codes at base + co and scale at base + so, both for block 0.
template <int FMT>
__device__ __forceinline__ void load_raw(const uint8_t* base, uint32_t b, uint32_t co, uint32_t so, Raw<FMT>& r) {
    const uint8_t* p = base + size_t(b) * (FMT == kQ8_0 ? 34 : 18);
    r.q = *reinterpret_cast<const u4a2_t*>(p + opaque(co));
    r.d = *reinterpret_cast<const uint16_t*>(p + opaque(so));
}
// The 8 codes of step j, NEG: with their signs changed.
template <int FMT, bool NEG = false>
__device__ __forceinline__ h8_t decode_raw(const Raw<FMT>& r, uint32_t h, uint32_t j) {
    h8_t o;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t q = r.q[2 * j + i];
        h2_t a, b;
        if constexpr (FMT == kQ8_0) bytes_to_half<NEG>(q ^ 0x80808080u, _Float16(1152.0f), a, b);
        else bytes_to_half<NEG>((q >> (4 * h)) & 0x0F0F0F0Fu, _Float16(1032.0f), a, b);
        o[4 * i] = a[0];
        o[4 * i + 1] = a[1];
        o[4 * i + 2] = b[0];
        o[4 * i + 3] = b[1];
    }
    return o;
}

// A thread's 16 dequantised weights of block b, element order as above.
template <int FMT>
__device__ __forceinline__ void weights16(const uint8_t* base, uint32_t off, uint32_t b, uint32_t h, float (&w)[16]) {
    Raw<FMT> r;
    load_raw<FMT>(base, b, off + code_offset<FMT>(h), off, r);
    const float d = half_bits_to_float(r.d);
#pragma unroll
    for (uint32_t j = 0; j < 2; ++j) {
        const h8_t q = decode_raw<FMT>(r, h, j);
#pragma unroll
        for (int i = 0; i < 8; ++i) w[8 * j + i] = float(q[i]) * d;
    }
}

// The 32 x 32 outputs of a wave's activation rows (x: the lane's, from its
// first element of block 0) and weight rows (load(b, w): weights16 of the
// lane's), on the fp32 MFMA: what marked rows take.  A lane half holds 16 k of
// a block, one of each pair that an instruction multiplies.
template <class Load>
__device__ __forceinline__ v16f exact_tile(const float* x, uint32_t b_begin, uint32_t b_end, Load load) {
    v16f t;
#pragma unroll
    for (int v = 0; v < 16; ++v) t[v] = 0.0f;
    for (uint32_t b = b_begin; b < b_end; ++b) {
        float4 a[4];
        float w[16];
#pragma unroll
        for (int q = 0; q < 4; ++q) a[q] = reinterpret_cast<const float4*>(x + 32 * b)[q];
        load(b, w);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            t = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q].x, w[4 * q], t, 0, 0, 0);
            t = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q].y, w[4 * q + 1], t, 0, 0, 0);
            t = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q].z, w[4 * q + 2], t, 0, 0, 0);
            t = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q].w, w[4 * q + 3], t, 0, 0, 0);
        }
    }
    return t;
}
// The end of both kernels: a wave's 64 x 64 sums (from row m, column n) to Y,
// scaled back; marked rows from exact_tile.
template <class Load>
__device__ __forceinline__ void store_tile(v16f (&acc)[2][2], const int* __restrict__ ex, const float* __restrict__ X,
                                           float* __restrict__ Y, uint32_t m0, uint32_t n0, uint32_t M, uint32_t N,
                                           uint32_t K, uint32_t b_begin, uint32_t b_end, Load load) {
    uint32_t lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));  // opaque: nothing below is formed before the main loop
    const uint32_t l32 = lane & 31, lh = lane >> 5;
    // the exponents of rows l32 and 32 + l32, passed between lanes: one wait for them
    int er[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) er[i] = ex[min(m0 + i * 32 + l32, M - 1)];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        int ev[16];
#pragma unroll
        for (uint32_t v = 0; v < 16; ++v) ev[v] = __shfl(er[i], 8 * (v >> 2) + 4 * lh + (v & 3));
        if (__any(er[i] == kExactRow)) {
            const float* x = X + size_t(min(m0 + i * 32 + l32, M - 1)) * K + 16 * lh;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint32_t n = min(n0 + j * 32 + l32, N - 1);
                const v16f t = exact_tile(x, b_begin, b_end, [&](uint32_t b, float (&w)[16]) { load(n, lh, b, w); });
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    if (ev[v] == kExactRow) acc[i][j][v] = t[v];
            }
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (ev[v] == kExactRow) ev[v] = 0;
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const uint32_t m = m0 + i * 32 + 8 * (v >> 2) + 4 * lh + (v & 3);
            if (m >= M) continue;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint32_t n = n0 + j * 32 + l32;
                if (n < N) Y[size_t(m) * N + n] = ldexpf(acc[i][j][v], -ev[v]);
            }
        }
    }
}

// --------------------------------------------------------------- kernel ---
// One K stage of a tile in LDS: activations [BM][128 B] (the row's 32 hi and
// 32 lo halves), weight codes [BN][64 B] as f16, group scales [BN].  16-byte
// units are XOR-swizzled so the rows that an operand read touches together
// fall on distinct banks.
template <int BM, int BN>
struct SplitStage {
    static constexpr int A = BM * 128, W = BN * 64, S = BN * 4;
    static constexpr int LDS = 3 * (A + W + S);
};

// WM x WN waves of a 64 x 64 tile each.
template <int FMT, int WM, int WN>
__device__ __forceinline__ void gemm_split_body(const uint8_t* W, const uint8_t* XS,
                                                const int* __restrict__ ex, const float* __restrict__ X, float* __restrict__ Y, float* __restrict__ partial, uint32_t M,
                                                uint32_t N, uint32_t K, uint32_t tiles_m, uint32_t tiles_n,
                                                uint32_t blocks_per_split) {
    constexpr int BM = 64 * WM, BN = 64 * WN, TH = 64 * WM * WN;
    constexpr int AU = BM * 8 / TH;  // 16-byte activation units per thread
    static_assert(BN * 2 == TH, "a thread stages half a block of one row");
    using G = SplitStage<BM, BN>;
    extern __shared__ __align__(16) uint8_t lds[];
    uint8_t* As = lds;
    uint8_t* Bs = lds + 3 * G::A;
    float* Sw = reinterpret_cast<float*>(lds + 3 * (G::A + G::W));
    const uint32_t total_tiles = tiles_m * tiles_n;
    const uint32_t split = blockIdx.x / total_tiles;
    uint32_t tm, tn;
    tile_of(tiles_m, tiles_n, blockIdx.x % total_tiles, tm, tn);
    const uint32_t m0 = tm * BM, n0 = tn * BN;
    const uint32_t nb = K >> 5;
    const uint32_t b_begin = split * blocks_per_split;
    const uint32_t b_end = min(nb, b_begin + blocks_per_split);
    float* Yout = split ? partial + size_t(split - 1) * M * N : Y;
    const size_t rb = row_bytes_dev(FMT, K);
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int l32 = lane & 31, lh = lane >> 5;

    // loaders: activation units i * TH + tid (row unit / 8, 16 B unit % 8),
    // weight half block tid (row / 2, half % 2)
    // -- 32-bit offsets from the tile's first rows, so a load's address is a
    // scalar base and a fixed lane offset
    const __amdgpu_buffer_rsrc_t a_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(XS + size_t(m0) * K * 4), 0, -1, kBufferWord3);
    uint32_t a_off[AU];
#pragma unroll
    for (int i = 0; i < AU; ++i)
        a_off[i] = (min(m0 + uint32_t(i * (TH / 8) + (tid >> 3)), M - 1) - m0) * K * 4 + (tid & 7) * 16;
    const uint32_t a_dst = uint32_t(tid >> 3) * 128 + (((tid & 7) ^ ((tid >> 4) & 7)) * 16);
    const uint32_t w_half = tid & 1, w_row = tid >> 1, w_swz = (w_row >> 2) & 3;
    const uint8_t* w_base = W + size_t(n0) * rb;
    const uint32_t w_off = (min(n0 + w_row, N - 1) - n0) * uint32_t(rb);

    struct Stage {
        u4_t a[AU];
        Raw<FMT> w;
    };
    auto load_a = [&](uint32_t b, Stage& r, int i) {
        r.a[i] = __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, a_off[i], b * 128, 0);
    };
    auto load_w = [&](uint32_t b, Stage& r) {
        load_raw<FMT>(w_base, b, w_off + code_offset<FMT>(w_half), w_off, r.w);
    };
    auto store_a = [&](int buf, const Stage& r, int i) {
        *reinterpret_cast<u4_t*>(As + buf * G::A + i * (TH / 8) * 128 + a_dst) = r.a[i];
    };
    // Every other block is staged with the signs of its codes and scale changed
    // (PAR): the f16 products' sums are rounded down, not to nearest, which scales
    // of one sign would carry to every output alike (measured: the mean of the
    // errors -0.4 to -0.6 of their spread); so it cancels.
    auto store_w = [&](int buf, const Stage& r, uint32_t j, auto par_c) {  // step j's 8 codes
        *reinterpret_cast<h8_t*>(Bs + buf * G::W + w_row * 64 + (((2 * j + w_half) ^ w_swz) * 16)) =
            decode_raw<FMT, decltype(par_c)::value == 1>(r.w, w_half, j);
    };
    auto store_s = [&](int buf, const Stage& r, auto par_c) {
        const float d = half_bits_to_float(r.w.d);
        Sw[buf * BN + w_row] = decltype(par_c)::value == 1 ? -d : d;
    };

    v16f acc[2][2];
    v16f zero;
#pragma unroll
    for (int v = 0; v < 16; ++v) zero[v] = acc[0][0][v] = acc[0][1][v] = acc[1][0][v] = acc[1][1][v] = 0.0f;

    // operand readers: rows i of the wave's activations, columns j of its weights
    const uint32_t ar = uint32_t(wm * 64 + l32), br = uint32_t(wn * 64 + l32);
    const uint32_t a_swz = (ar >> 1) & 7, b_swz = (br >> 2) & 3;  // the same for row + 32
    h8_t w[2][2], ah[2][2], al[2][2];
    float dw[2];
    auto read_w = [&](int buf, int j) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
            w[j][s] = *reinterpret_cast<const h8_t*>(Bs + buf * G::W + (br + j * 32) * 64 + (((2 * s + lh) ^ b_swz) * 16));
        dw[j] = Sw[buf * BN + br + j * 32];
    };
    auto read_a = [&](int buf, int i, int s) {
        const uint8_t* r = As + buf * G::A + (ar + i * 32) * 128;
        al[i][s] = *reinterpret_cast<const h8_t*>(r + (((4 + 2 * lh + s) ^ a_swz) * 16));
        ah[i][s] = *reinterpret_cast<const h8_t*>(r + (((2 * lh + s) ^ a_swz) * 16));
    };

    // Stage b multiplies block b.  Three LDS buffers: while block b is read
    // from one, block b + 1 is complete in the next (so its first operands
    // are fetched before the stage's barrier) and block b + 2, loaded during
    // stage b - 1, is written to the third; each of its registers is reloaded
    // with block b + 3 once written out.
    // One barrier a stage.  Blocks past the end repeat the last one, unused.
    // The stage is 16 slots of one MFMA each (4 tiles x lo, hi x 2 k steps);
    // a tile's 16 scaled additions follow in the next tile's four slots, and
    // the staging is spread over the slots, because a wave's VALU work runs
    // under its own MFMAs only where it is issued between them (measured: an
    // MFMA with 4, 8, 16 FMAs behind it takes 38, 53, 89 cycles of a SIMD's one
    // wave, 33, 43, 66 with two).  PAR, the block's parity: the column order alternates so that the column read last is free first.
    v16f p[2];        // products of a tile; p[1] enters a stage with the previous stage's last tile
    float dc = 0.0f;  // ... its scale
    float dt = 0.0f;  // the scale of a stage's last but one tile (its column's is replaced early)
    p[1] = zero;
    Stage r;
    auto stage = [&](auto buf_c, auto par_c, uint32_t b) {
        constexpr int BUF = decltype(buf_c)::value, PAR = decltype(par_c)::value;
        constexpr int NB = (BUF + 1) % 3, WB = (BUF + 2) % 3;
        const uint32_t far = min(b + 3, b_end - 1);
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            // tiles (0, P), (0, 1-P), (1, 1-P), (1, P)
            const int t = s >> 2, i = t >> 1, j = (t == 0 || t == 3) ? PAR : 1 - PAR, k = s & 3;
            const h8_t& a = k < 2 ? al[i][k] : ah[i][k - 2];
            p[t & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, w[j][k & 1], k ? p[t & 1] : zero, 0, 0, 0);
            // the tile before: of this stage, or the last of the one before (1, 1-P)
            const int u = (t + 3) & 3, ui = u >> 1, uj = t == 0 ? 1 - PAR : (u == 0 ? PAR : 1 - PAR);
            const float d = t == 0 ? dc : t == 3 && k ? dt : dw[uj];
#pragma unroll
            for (int v = 4 * k; v < 4 * k + 4; ++v) acc[ui][uj][v] = fmaf(p[(t + 1) & 1][v], d, acc[ui][uj][v]);
            if (s == 0) read_w(BUF, 1 - PAR);
            if (s == 1) read_a(BUF, 1, 0);
            if (s == 2) read_a(BUF, 1, 1);
            if (s >= 3 && s < 3 + AU) store_a(WB, r, s - 3);
            if (s >= 4 && s < 4 + AU) load_a(far, r, s - 4);
            if (s == 9) store_w(WB, r, 0, par_c);  // block b + 2
            if (s == 11) store_w(WB, r, 1, par_c);
            if (s == 12) store_s(WB, r, par_c);
            if (s == 13) load_w(far, r);
            if (s == 8) read_a(NB, 0, 0);
            if (s == 10) read_a(NB, 0, 1);
            if (s == 12) dt = dw[1 - PAR], dc = dw[PAR], read_w(NB, 1 - PAR);
            __builtin_amdgcn_sched_barrier(0);
        }
        lds_barrier();
    };
    if (b_begin >= b_end) return;
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    auto fill = [&](int buf, uint32_t b, auto par_c) {
#pragma unroll
        for (int i = 0; i < AU; ++i) load_a(b, r, i);
        load_w(b, r);
#pragma unroll
        for (int i = 0; i < AU; ++i) store_a(buf, r, i);
        store_w(buf, r, 0, par_c);
        store_w(buf, r, 1, par_c);
        store_s(buf, r, par_c);
    };
    fill(0, b_begin, I0{});
    fill(1, min(b_begin + 1, b_end - 1), I1{});
#pragma unroll
    for (int i = 0; i < AU; ++i) load_a(min(b_begin + 2, b_end - 1), r, i);
    load_w(min(b_begin + 2, b_end - 1), r);
    lds_barrier();
    read_a(0, 0, 0);
    read_a(0, 0, 1);
    read_w(0, 0);
    int last = 0;  // the column order of the last stage
    for (uint32_t b = b_begin;;) {
        stage(I0{}, I0{}, b);
        if (last = 0, ++b >= b_end) break;
        stage(I1{}, I1{}, b);
        if (last = 1, ++b >= b_end) break;
        stage(I2{}, I0{}, b);
        if (last = 0, ++b >= b_end) break;
        stage(I0{}, I1{}, b);
        if (last = 1, ++b >= b_end) break;
        stage(I1{}, I0{}, b);
        if (last = 0, ++b >= b_end) break;
        stage(I2{}, I1{}, b);
        if (last = 1, ++b >= b_end) break;
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        if (last) acc[1][1][v] = fmaf(p[1][v], dc, acc[1][1][v]);
        else acc[1][0][v] = fmaf(p[1][v], dc, acc[1][0][v]);
    }
    store_tile(acc, ex, X, Yout, m0 + wm * 64, n0 + wn * 64, M, N, K, b_begin, b_end,
               [&](uint32_t n, uint32_t h, uint32_t b, float (&o)[16]) { weights16<FMT>(w_base, (n - n0) * uint32_t(rb), b, h, o); });
}
template <int FMT, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_split_kernel(
    const uint8_t* W, const uint8_t* XS, const int* __restrict__ ex, const float* __restrict__ X, float* __restrict__ Y,
    float* __restrict__ partial, uint32_t M, uint32_t N, uint32_t K, uint32_t tiles_m, uint32_t tiles_n, uint32_t blocks_per_split) {
    gemm_split_body<FMT, WM, WN>(W, XS, ex, X, Y, partial, M, N, K, tiles_m, tiles_n, blocks_per_split);
}


// ------------------------------------------------- super-block formats ---
// Q4_K / Q5_K: w = d*sc*q - dmin*m = d*(sc*(q - c)) + (c*sc*d - m*dmin) with c
// = 8 / 16.  sc*(q - c) is a whole number below 1024, exact in f16, so a
// super-block's products need no scaling inside (two MFMAs per 16 k): part
// is their sum, and acc += d * part.  The offsets multiply the group sums of
// x, carried as f16 hi + lo of S / 32 (8 groups x 2 = the 16 k of one MFMA):
// part += (32*c*sc) . (S/32), then acc -= dmin * ((32*m) . (S/32)).
// Q6_K: w = d*(sc*(q - 32)), the whole number below 2^13 carried as f16 hi +
// lo (three MFMAs per 16 k).
// The two-level sum keeps the rounding error that of K / 256 additions.
template <int FMT>
constexpr bool kOffsets = FMT == kQ4_K || FMT == kQ5_K;
template <int FMT>
constexpr int kPlanes = FMT == kQ6_K ? 2 : 1;
template <int FMT>
constexpr uint32_t kSuperBytes = FMT == kQ6_K ? 210 : FMT == kQ5_K ? 176 : 144;

template <int FMT>
struct RawK {
    u4_t q;
    u4_t h[FMT == kQ4_K ? 0 : 1];   // fifth bits / the codes' upper two bits
    u4_t head[kOffsets<FMT> ? 1 : 0];  // d, dmin, the 12 scale bytes
    uint32_t sc, d;                 // Q6_K: the half's int8 scale, d
};
// Group g, half h of the super-block at p + off (p and g uniform).
template <int FMT>
__device__ __forceinline__ void load_rawk(const uint8_t* p, uint32_t off, uint32_t g, uint32_t h, RawK<FMT>& r) {
    const uint32_t oh = opaque(off + 16 * h);
    if constexpr (kOffsets<FMT>) {
        r.head[0] = *reinterpret_cast<const u4a4_t*>(p + opaque(off));
        r.q = *reinterpret_cast<const u4a4_t*>(p + (FMT == kQ5_K ? 48 : 16) + (g >> 1) * 32 + oh);
        if constexpr (FMT == kQ5_K) r.h[0] = *reinterpret_cast<const u4a4_t*>(p + 16 + oh);
    } else {
        r.q = *reinterpret_cast<const u4a2_t*>(p + (g >> 2) * 64 + (g & 1) * 32 + oh);
        r.h[0] = *reinterpret_cast<const u4a2_t*>(p + 128 + (g >> 2) * 32 + oh);
        r.sc = *(p + 192 + 2 * g + opaque(off + h));
        r.d = *reinterpret_cast<const uint16_t*>(p + 208 + opaque(off));
    }
}
// Scale and min of group g from the three words of the scale bytes
// (src/quant.cpp:133-141 of the reference).
__device__ __forceinline__ uint32_t kq_scale(const u4_t& w, uint32_t g) {
    const uint32_t sh = 8 * (g & 3u);
    return g < 4 ? (w[1] >> sh) & 63u : ((w[3] >> sh) & 15u) | ((w[1] >> (sh + 2)) & 0x30u);
}
__device__ __forceinline__ uint32_t kq_min(const u4_t& w, uint32_t g) {
    const uint32_t sh = 8 * (g & 3u);
    return g < 4 ? (w[2] >> sh) & 63u : ((w[3] >> (sh + 4)) & 15u) | ((w[2] >> (sh + 2)) & 0x30u);
}
// The 8 scaled codes of step j (Q6_K: hi and lo), with their signs changed for
// flip = 0x80008000 (uniform; else 0).
template <int FMT>
__device__ __forceinline__ void decode_rawk(const RawK<FMT>& r, uint32_t g, uint32_t j, uint32_t flip, h8_t (&o)[kPlanes<FMT>]) {
    const _Float16 sc = kOffsets<FMT> ? _Float16(float(kq_scale(r.head[0], g))) : _Float16(float(int(int8_t(uint8_t(r.sc)))));
    const h2_t s = __builtin_bit_cast(h2_t, __builtin_bit_cast(uint32_t, h2_t{sc, sc}) ^ flip);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int e = 2 * j + i;
        uint32_t u;
        if constexpr (kOffsets<FMT>) {
            u = (r.q[e] >> (4 * (g & 1))) & 0x0F0F0F0Fu;
            if constexpr (FMT == kQ5_K) u |= ((r.h[0][e] >> g) & 0x01010101u) << 4;
        } else {
            u = ((r.q[e] >> (4 * ((g >> 1) & 1))) & 0x0F0F0F0Fu) | (((r.h[0][e] >> (2 * (g & 3))) & 0x03030303u) << 4);
        }
        h2_t c[2];
        bytes_to_half(u, _Float16(1024.0f + (FMT == kQ4_K ? 8.0f : FMT == kQ5_K ? 16.0f : 32.0f)), c[0], c[1]);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const h2_t hi = c[k] * s;
            o[0][4 * i + 2 * k] = hi[0];
            o[0][4 * i + 2 * k + 1] = hi[1];
            if constexpr (kPlanes<FMT> == 2) {
                const h2_t lo = __builtin_elementwise_fma(c[k], s, -hi);
                o[1][4 * i + 2 * k] = lo[0];
                o[1][4 * i + 2 * k + 1] = lo[1];
            }
        }
    }
}

// A thread's 16 dequantised weights of block b: its exact parts, rounded once
// as the reference's dequantisation is.
template <int FMT>
__device__ __forceinline__ void weights16k(const uint8_t* base, uint32_t off, uint32_t b, uint32_t h, float (&w)[16]) {
    const uint32_t g = b & 7u;
    RawK<FMT> r;
    load_rawk<FMT>(base + size_t(b >> 3) * kSuperBytes<FMT>, off, g, h, r);
#pragma unroll
    for (uint32_t j = 0; j < 2; ++j) {
        h8_t o[kPlanes<FMT>];
        decode_rawk<FMT>(r, g, j, 0u, o);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if constexpr (kOffsets<FMT>) {
                const float sq = float(o[0][i]) + (FMT == kQ4_K ? 8.0f : 16.0f) * float(kq_scale(r.head[0], g));
                w[8 * j + i] = fmaf(half_bits_to_float(r.head[0][0]), sq,
                                    -(half_bits_to_float(r.head[0][0] >> 16) * float(kq_min(r.head[0], g))));
            } else {
                w[8 * j + i] = half_bits_to_float(r.d) * (float(o[0][i]) + float(o[1][i]));
            }
        }
    }
}

template <int FMT, int BM, int BN>
struct SplitStageK {
    static constexpr int A = BM * 128, W = BN * 64 * kPlanes<FMT>;
    static constexpr int SA = kOffsets<FMT> ? BM * 32 : 0;   // group sums: 8 hi, 8 lo halves per row
    static constexpr int OF = kOffsets<FMT> ? BN * 32 : 0;   // 32*c*sc and 32*m: 8 halves each per column
    static constexpr int D = BN * 8;                         // d, dmin
    static constexpr int LDS = 3 * (A + W) + SA + OF + D;
    static_assert(LDS <= 160 * 1024, "one workgroup per CU");
};

template <int FMT, int WM, int WN>
__device__ __forceinline__ void gemm_split_kq_body(const uint8_t* W, const uint8_t* XS, const uint8_t* SS,
                                                   const int* __restrict__ ex, const float* __restrict__ X, float* __restrict__ Y, float* __restrict__ partial, uint32_t M,
                                                   uint32_t N, uint32_t K, uint32_t tiles_m, uint32_t tiles_n,
                                                   uint32_t blocks_per_split) {
    constexpr int BM = 64 * WM, BN = 64 * WN, TH = 64 * WM * WN, P = kPlanes<FMT>;
    constexpr int AU = BM * 8 / TH;  // 16-byte activation units per thread
    static_assert(BN * 2 == TH, "a thread stages half a block of one row");
    using G = SplitStageK<FMT, BM, BN>;
    extern __shared__ __align__(16) uint8_t lds[];
    uint8_t* As = lds;
    uint8_t* Bs = As + 3 * G::A;
    uint8_t* Sa = Bs + 3 * G::W;
    uint8_t* Of = Sa + G::SA;
    float* Ds = reinterpret_cast<float*>(Of + G::OF);
    const uint32_t total_tiles = tiles_m * tiles_n;
    const uint32_t split = blockIdx.x / total_tiles;
    uint32_t tm, tn;
    tile_of(tiles_m, tiles_n, blockIdx.x % total_tiles, tm, tn);
    const uint32_t m0 = tm * BM, n0 = tn * BN;
    const uint32_t nb = K >> 5;
    const uint32_t b_begin = split * blocks_per_split;  // whole super-blocks
    const uint32_t b_end = min(nb, b_begin + blocks_per_split);
    float* Yout = split ? partial + size_t(split - 1) * M * N : Y;
    const size_t rb = size_t(nb >> 3) * kSuperBytes<FMT>;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const int l32 = lane & 31, lh = lane >> 5;

    const __amdgpu_buffer_rsrc_t a_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(XS + size_t(m0) * K * 4), 0, -1, kBufferWord3);
    uint32_t a_off[AU];
#pragma unroll
    for (int i = 0; i < AU; ++i)
        a_off[i] = (min(m0 + uint32_t(i * (TH / 8) + (tid >> 3)), M - 1) - m0) * K * 4 + (tid & 7) * 16;
    const uint32_t a_dst = uint32_t(tid >> 3) * 128 + (((tid & 7) ^ ((tid >> 4) & 7)) * 16);
    const uint32_t w_half = tid & 1, w_row = tid >> 1, w_swz = (w_row >> 2) & 3;
    const uint8_t* w_base = W + size_t(n0) * rb;
    const uint32_t w_off = (min(n0 + w_row, N - 1) - n0) * uint32_t(rb);
    struct Stage {
        u4_t a[AU];
        RawK<FMT> w;
    };
    Stage r;
    auto load_a = [&](uint32_t b) {
#pragma unroll
        for (int i = 0; i < AU; ++i) r.a[i] = __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, a_off[i], b * 128, 0);
    };
    auto load_w = [&](uint32_t b) { load_rawk<FMT>(w_base + size_t(b >> 3) * kSuperBytes<FMT>, w_off, b & 7u, w_half, r.w); };
    auto store_a = [&](int buf, int i) {
        *reinterpret_cast<u4_t*>(As + buf * G::A + i * (TH / 8) * 128 + a_dst) = r.a[i];
    };
    // every other super-block with its signs changed, as in gemm_split_body
    auto flip_of = [&](uint32_t b) { return (b >> 3) & 1u ? 0x80008000u : 0u; };
    auto store_w = [&](int buf, uint32_t b, uint32_t j) {  // step j's 8 codes of block b
        h8_t o[P];
        decode_rawk<FMT>(r.w, b & 7u, j, flip_of(b), o);
#pragma unroll
        for (int q = 0; q < P; ++q)
            *reinterpret_cast<h8_t*>(Bs + buf * G::W + q * BN * 64 + w_row * 64 + (((2 * j + w_half) ^ w_swz) * 16)) = o[q];
    };
    // the super-block's d and dmin and its offset factors (half 0: scales, 1: mins)
    auto store_head = [&](uint32_t b) {
        int t = tid;  // opaque: the addresses below are not kept in registers around the loop
        asm volatile("" : "+v"(t));
        const uint32_t w_half = t & 1, w_row = t >> 1;
        const float sign = flip_of(b) ? -1.0f : 1.0f;
        if constexpr (kOffsets<FMT>) {
            const float f = sign * (w_half ? 32.0f : FMT == kQ4_K ? 256.0f : 512.0f);
            h8_t o;
#pragma unroll
            for (uint32_t g = 0; g < 8; ++g) {
                const uint32_t sc = kq_scale(r.w.head[0], g), mn = kq_min(r.w.head[0], g);
                o[g] = _Float16(f * float(w_half ? mn : sc));
            }
            *reinterpret_cast<h8_t*>(Of + w_half * BN * 16 + w_row * 16) = o;
            Ds[w_half * BN + w_row] = sign * half_bits_to_float(w_half ? r.w.head[0][0] >> 16 : r.w.head[0][0]);
        } else {
            Ds[w_row] = sign * half_bits_to_float(r.w.d);
        }
    };

    v16f acc[2][2], part[2][2];
    v16f zero;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        zero[v] = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t >> 1][t & 1][v] = part[t >> 1][t & 1][v] = 0.0f;
    }

    const uint32_t ar = uint32_t(wm * 64 + l32), br = uint32_t(wn * 64 + l32);
    const uint32_t a_swz = (ar >> 1) & 7, b_swz = (br >> 2) & 3;  // the same for row + 32
    // Operands of a phase: rows i of the activations' hi or lo plane (two k
    // steps; a[phase % 2]), and the weights' planes, all columns.
    h8_t a[2][2], wh[2][2], wl[2][2];
    auto read_w = [&](int buf, int q, h8_t (&o)[2][2]) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int s = 0; s < 2; ++s)
                o[j][s] = *reinterpret_cast<const h8_t*>(Bs + buf * G::W + q * BN * 64 + (br + j * 32) * 64 +
                                                         (((2 * s + lh) ^ b_swz) * 16));
    };
    auto read_a = [&](int buf, int f, int s) {  // phases (0, lo), (0, hi), (1, hi), (1, lo)
        const int unit = (f == 1 || f == 2 ? 0 : 4) + 2 * lh + s;
        a[f & 1][s] = *reinterpret_cast<const h8_t*>(As + buf * G::A + (ar + (f >> 1) * 32) * 128 + ((unit ^ a_swz) * 16));
    };
    // Closes a super-block: the offsets, the scales, and part back to 0.
    auto close = [&]() {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float d = Ds[br + j * 32];
            h8_t os, om;
            float dm = 0.0f;
            if constexpr (kOffsets<FMT>) {
                dm = -Ds[BN + br + j * 32];
                os = *reinterpret_cast<const h8_t*>(Of + (br + j * 32) * 16);
                om = *reinterpret_cast<const h8_t*>(Of + BN * 16 + (br + j * 32) * 16);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if constexpr (kOffsets<FMT>) {
                    const h8_t sa = *reinterpret_cast<const h8_t*>(Sa + (ar + i * 32) * 32 + lh * 16);
                    part[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sa, os, part[i][j], 0, 0, 0);
                    const v16f t = __builtin_amdgcn_mfma_f32_32x32x16_f16(sa, om, zero, 0, 0, 0);
                    // One addition to acc per super-block, since its rounding is
                    // the larger part of a long K's error; and the two products,
                    // which largely cancel, without that of t * dm.
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const float p = t[v] * dm;
                        acc[i][j][v] += fmaf(part[i][j][v], d, p) + fmaf(t[v], dm, -p);
                    }
                } else {
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[i][j][v] = fmaf(part[i][j][v], d, acc[i][j][v]);
                }
                part[i][j] = zero;
            }
        }
    };

    // The pipeline of gemm_split_body: three LDS buffers, block b + 2 staged
    // and block b + 3 loaded while block b is multiplied, the next block's
    // first operands read before the barrier.  A super-block's head is staged
    // with its third block (while its first is multiplied, after every wave
    // has closed the one before), its group sums one stage later.
    u4_t sums = {0, 0, 0, 0};
    auto sum_unit = [&]() {
        int t = tid;
        asm volatile("" : "+v"(t));
        return uint32_t(t) % (BM * 2);
    };
    auto stage = [&](auto buf_c, uint32_t b) {
        constexpr int BUF = decltype(buf_c)::value, NB = (BUF + 1) % 3, WB = (BUF + 2) % 3;
        const uint32_t g = b & 7u, far = min(b + 3, b_end - 1), nb2 = min(b + 2, b_end - 1);
        if (g == 0) {
            if constexpr (kOffsets<FMT>) {  // row su / 2, hi or lo su % 2 (threads past the tile repeat)
                const uint32_t su = sum_unit();
                sums = *reinterpret_cast<const u4_t*>(SS + (size_t(min(m0 + (su >> 1), M - 1)) * (nb >> 3) + (b >> 3)) * 32 +
                                                      (su & 1) * 16);
            }
            store_head(b);
        }
        if constexpr (kOffsets<FMT>)
            if (g == 1) *reinterpret_cast<u4_t*>(Sa + sum_unit() * 16) = sums;
        h8_t wn[2][2];
        int slot = 0;
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            const int i = f >> 1;
            const bool hi = f == 1 || f == 2;
#pragma unroll
            for (int s = 0; s < (hi ? 4 * P : 4); ++s, ++slot) {
                const int k = (s >> 1) & 1, j = s & 1;
                const h8_t& bw = hi && P == 2 && s < 4 ? wl[j][k] : wh[j][k];
                part[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[f & 1][k], bw, part[i][j], 0, 0, 0);
                if (s < 2) read_a(f == 3 ? NB : BUF, (f + 1) & 3, s);  // the next phase's rows
                if (f == 0 && s == 2 && P == 2) read_w(BUF, 1, wl);
                if (f == 3 && s == 1) read_w(NB, 0, wn);
                if (slot >= 2 && slot < 2 + AU) store_a(WB, slot - 2);
                if (slot == 2 + AU) load_a(far);
                if (slot == 6) store_w(WB, nb2, 0);
                if (slot == 9) store_w(WB, nb2, 1);
                if (slot == 10) load_w(far);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) wh[q >> 1][q & 1] = wn[q >> 1][q & 1];
        if (g == 7) close();
        lds_barrier();
    };
    if (b_begin >= b_end) return;
    auto fill = [&](int buf, uint32_t b) {
        load_a(b);
        load_w(b);
#pragma unroll
        for (int i = 0; i < AU; ++i) store_a(buf, i);
        store_w(buf, b, 0);
        store_w(buf, b, 1);
    };
    fill(0, b_begin);
    fill(1, b_begin + 1);
    load_a(b_begin + 2);
    load_w(b_begin + 2);
    lds_barrier();
    read_a(0, 0, 0);
    read_a(0, 0, 1);
    read_w(0, 0, wh);
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    for (uint32_t b = b_begin;;) {
        stage(I0{}, b);
        if (++b >= b_end) break;
        stage(I1{}, b);
        if (++b >= b_end) break;
        stage(I2{}, b);
        if (++b >= b_end) break;
    }
    store_tile(acc, ex, X, Yout, m0 + wm * 64, n0 + wn * 64, M, N, K, b_begin, b_end,
               [&](uint32_t n, uint32_t h, uint32_t b, float (&o)[16]) { weights16k<FMT>(w_base, (n - n0) * uint32_t(rb), b, h, o); });
}
template <int FMT, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN, WN == 4 ? 2 : 1) void gemm_split_kq_kernel(
    const uint8_t* W, const uint8_t* XS, const uint8_t* SS, const int* __restrict__ ex, const float* __restrict__ X, float* __restrict__ Y, float* __restrict__ partial, uint32_t M,
    uint32_t N, uint32_t K, uint32_t tiles_m, uint32_t tiles_n, uint32_t blocks_per_split) {
    gemm_split_kq_body<FMT, WM, WN>(W, XS, SS, ex, X, Y, partial, M, N, K, tiles_m, tiles_n, blocks_per_split);
}

}  // namespace

// Time in microseconds of `tiles` tiles of the 128 x (64 * wn) kernel with ks
// splits of `blocks` blocks: a CU runs its workgroups' stages one after the
// other at 1.17 us (256 columns) or 0.60 us (128 columns) each; 1.4 and 1.02
// us for the super-block formats, whose 128-column form holds one wave a SIMD
// (measured at 512 tokens of 14336x4096 and 1000 of 4096x14336).  A split
// adds its plane's write and read and the launch that adds the planes.
static double split_cost(bool super, int wn, uint32_t tiles, uint32_t ks, uint32_t blocks, size_t M, size_t N) {
    const double rounds = std::ceil(double(tiles) * ks / device_cu_count());
    const double t = rounds * blocks * (wn == 4 ? (super ? 1.4 : 1.17) : (super ? 1.02 : 0.60));
    return ks > 1 ? t + 3.0 + double(ks - 1) * double(M) * double(N) * 8.0 / 4.0e6 : t;
}
// The cheapest tile width and split with at most `planes` planes beside Y;
// splits are whole super-blocks where the format has them, and at least 8
// blocks.
SplitPlan plan_gemm_split(int fmt, size_t M, size_t N, size_t K, size_t planes) {
    const bool super = fmt != kQ8_0 && fmt != kQ4_0;
    const uint32_t unit = super ? 8 : 1, units = uint32_t(K / 32) / unit;
    const uint32_t most = uint32_t(std::min<size_t>({planes + 1, 32, std::max(1u, units * unit / 8)}));
    SplitPlan best;
    for (int wn : {4, 2}) {
        const uint32_t tiles = uint32_t(((M + 127) / 128) * ((N + 64 * wn - 1) / (64 * wn)));
        for (uint32_t ks = 1; ks <= most; ++ks) {
            const uint32_t ups = (units + ks - 1) / ks;
            if ((units + ups - 1) / ups != ks) continue;  // would leave empty splits
            const double t = split_cost(super, wn, tiles, ks, ups * unit, M, N);
            if (t < best.us) best = SplitPlan{wn, ks, ups * unit, t};
        }
    }
    return best;
}

namespace {
struct SplitArgs {
    const uint8_t *w, *xs, *ss;
    const int* ex;
    const float* X;
    float *Y, *partial;
    uint32_t m, n, k;
    hipStream_t stream;
};
}  // namespace

template <int FMT, int WN>
static hipError_t launch_tile(const SplitArgs& a, const SplitPlan& plan) {
    constexpr int BM = 128, BN = 64 * WN;
    const uint32_t tiles_m = (a.m + BM - 1) / BM, tiles_n = (a.n + BN - 1) / BN;
    const dim3 grid(tiles_m * tiles_n * plan.ks), block(128 * WN);
    if constexpr (FMT == kQ8_0 || FMT == kQ4_0)
        hipLaunchKernelGGL((gemm_split_kernel<FMT, 2, WN>), grid, block, (SplitStage<BM, BN>::LDS), a.stream, a.w, a.xs,
                           a.ex, a.X, a.Y, a.partial, a.m, a.n, a.k, tiles_m, tiles_n, plan.blocks);
    else
        hipLaunchKernelGGL((gemm_split_kq_kernel<FMT, 2, WN>), grid, block, (SplitStageK<FMT, BM, BN>::LDS), a.stream, a.w,
                           a.xs, a.ss, a.ex, a.X, a.Y, a.partial, a.m, a.n, a.k, tiles_m, tiles_n, plan.blocks);
    return hipGetLastError();
}
template <int FMT>
static hipError_t launch_fmt(const SplitArgs& a, const SplitPlan& plan) {
    return plan.wn == 4 ? launch_tile<FMT, 4>(a, plan) : launch_tile<FMT, 2>(a, plan);
}

bool gemm_split_supported(int fmt, size_t K) {
    // a tile's rows are addressed with 32-bit offsets from its first
    return K <= (size_t(1) << 21) && (fmt == kQ8_0 || fmt == kQ4_0
                                          ? K % 32 == 0
                                          : (fmt == kQ4_K || fmt == kQ5_K || fmt == kQ6_K) && K % 256 == 0);
}

// [M] rows of K hi + lo halves, the row exponents and, for Q4_K / Q5_K, the
// group sums; rounded up to 256 bytes.
size_t gemm_split_bytes(int fmt, size_t M, size_t K) {
    const size_t sums = fmt == kQ4_K || fmt == kQ5_K ? M * (K / 256) * 32 : 0;
    return (M * K * 4 + sums + M * sizeof(int) + 255) / 256 * 256;
}

// Tokens whose split activations the workspace holds: M, or whole tiles.
static size_t tokens_that_fit(int fmt, size_t M, size_t K, size_t ws_bytes) {
    if (gemm_split_bytes(fmt, M, K) <= ws_bytes) return M;
    size_t t = (M - 1) / 128 * 128;
    while (t && gemm_split_bytes(fmt, t, K) > ws_bytes) t -= 128;
    return t;
}
// The rest of the tokens after such a part: by the cheaper kernel, unsplit.
static bool rest_on_skinny(int fmt, size_t rest, size_t N, size_t K, const void* ws, size_t ws_bytes, SkinnyPlan& p) {
    p = plan_gemm_skinny_f32(fmt, rest, N, K, 0);
    const double us = gemm_split_us(fmt, rest, N, K, ws, ws_bytes);
    if (p.us <= us) return true;
    p.us = us;
    return false;
}

double gemm_split_us(int fmt, size_t M, size_t N, size_t K, const void* ws, size_t ws_bytes) {
    if (!gemm_split_supported(fmt, K) || !ws || (reinterpret_cast<uintptr_t>(ws) & 15u)) return 1e300;
    const size_t fit = tokens_that_fit(fmt, M, K, ws_bytes), sb = gemm_split_bytes(fmt, M, K);
    if (fit < M) {
        // (Q4_K / Q5_K at the asked-for size, which has no room for the group
        // sums: 97 of 100 tokens fit; less than half is not worth it)
        if (fit < (M + 1) / 2) return 1e300;
        SkinnyPlan rest;
        (void)rest_on_skinny(fmt, M - fit, N, K, ws, ws_bytes, rest);
        return gemm_split_us(fmt, fit, N, K, ws, ws_bytes) + rest.us;
    }
    // beside the GEMM: two launches and the activations read and written once
    return 8.0 + double(M) * double(K) * 8.0 / 4.0e6 +
           plan_gemm_split(fmt, M, N, K, (ws_bytes - sb) / (M * N * sizeof(float))).us;
}

hipError_t launch_gemm_split(int fmt, const uint8_t* w, const float* X, float* Y, void* ws, size_t ws_bytes, size_t M,
                             size_t N, size_t K, hipStream_t stream, uint32_t* launches) {
    const size_t sb = gemm_split_bytes(fmt, M, K);
    if (!gemm_split_supported(fmt, K) || !ws || (reinterpret_cast<uintptr_t>(ws) & 15u)) return hipErrorInvalidConfiguration;
    const size_t fit = tokens_that_fit(fmt, M, K, ws_bytes);
    if (fit < M) {
        if (fit < (M + 1) / 2) return hipErrorInvalidConfiguration;
        uint32_t n = 0, rest_n = 1;
        if (const hipError_t e = launch_gemm_split(fmt, w, X, Y, ws, ws_bytes, fit, N, K, stream, &n); e != hipSuccess) return e;
        const float* rx = X + fit * K;
        float* ry = Y + fit * N;
        SkinnyPlan p;
        const hipError_t e =
            rest_on_skinny(fmt, M - fit, N, K, ws, ws_bytes, p)
                ? launch_gemm_skinny_f32(fmt, &w, &ry, &N, 1, rx, nullptr, 1, p.nw, M - fit, K, stream)
                : launch_gemm_split(fmt, w, rx, ry, ws, ws_bytes, M - fit, N, K, stream, &rest_n);
        if (launches) *launches = n + rest_n;
        return e;
    }
    uint8_t* xs = static_cast<uint8_t*>(ws);
    uint8_t* ss = xs + M * K * 4;
    const bool sums = fmt == kQ4_K || fmt == kQ5_K;
    int* ex = reinterpret_cast<int*>(ss + (sums ? M * (K / 256) * 32 : 0));
    const SplitArgs a{w, xs, ss, ex, X, Y, reinterpret_cast<float*>(xs + sb), uint32_t(M), uint32_t(N), uint32_t(K), stream};
    const SplitPlan plan =
        plan_gemm_split(fmt, M, N, K, (ws_bytes - sb) / (M * N * sizeof(float)));
    if (sums)
        hipLaunchKernelGGL(split_acts_kernel<true>, dim3(a.m), dim3(kThreads), 0, stream, X,
                           reinterpret_cast<_Float16*>(xs), ex, reinterpret_cast<_Float16*>(ss), a.k);
    else
        hipLaunchKernelGGL(split_acts_kernel<false>, dim3(a.m), dim3(kThreads), 0, stream, X,
                           reinterpret_cast<_Float16*>(xs), ex, static_cast<_Float16*>(nullptr), a.k);
    if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    const hipError_t e = fmt == kQ8_0   ? launch_fmt<kQ8_0>(a, plan)
                         : fmt == kQ4_0 ? launch_fmt<kQ4_0>(a, plan)
                         : fmt == kQ4_K ? launch_fmt<kQ4_K>(a, plan)
                         : fmt == kQ5_K ? launch_fmt<kQ5_K>(a, plan)
                                        : launch_fmt<kQ6_K>(a, plan);
    if (launches) *launches = plan.ks > 1 ? 3 : 2;
    if (e != hipSuccess || plan.ks <= 1) return e;
    return launch_splitk_add(a.partial, Y, M, N, plan.ks - 1, stream);
}

}  // namespace zq
