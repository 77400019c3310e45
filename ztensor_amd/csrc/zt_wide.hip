// Wide-batch GEMMs on fp16 MFMA (gfx950): C[T, rows] = X[T, K] W[rows, K]^T
// for quantized W in the layout batch 1 reads and T tokens, X and C
// token-major (a prompt's prefill, or a wide decode batch).
//
// Two launches.  The pack kernel writes the activations once in MFMA operand
// order: per 16-token tile and 32-K step one 1 KB part (lane 16 g + i: the 8
// values of token i that lane group g multiplies in that step), so the GEMM
// stages them with direct global-to-LDS loads of 1 KB and reads them back
// with conflict-free ds_read_b128.  fp16 activations are one part, exact;
// fp32 activations are scaled by a power of two of their token (max |x| in
// [2^14, 2^15)) and split into fp16 hi + lo, |x - hi - lo| <= 2^-23 |x| +
// 2^-25 after scaling (zt_mfma.h).
//
// The GEMM's MFMA A operand is the activations (16 tokens) and the B operand
// the weights (16 rows), so D lane 16 g + i holds 4 tokens of weight row i:
// one register per lane scales the 4 values, and the lane that decodes a
// row's weights is the lane that uses the row's scale.  Weights go from
// global memory to registers and are decoded there to exact fp16 integers
// (q - 8, q - zero, q times a 6-bit scale, ...), so that only the activations'
// split and the fp32 sums round.  Two formats need parts: Q6_K's scale times q
// (hi + lo; the product of both second parts, at most 2^-22 of the whole, is
// left out) and IQ4_NL's float codebook (22 bits of it with fp16 activations,
// all 24 with fp32 ones).  A wave covers MT token tiles by NT row tiles, so
// that a decoded operand feeds MT x parts MFMAs; WN waves lie along the rows
// and WK along K (their sums meet through LDS at the end).
#include <type_traits>

#include "zt_common.h"
#include "zt_mfma.h"

namespace zt {
namespace {

// Weight formats (the ZT_WIDE_* values of zt_hip.h).
enum Fmt { W4A16, Q4_0, Q8_0, Q8_GGUF, Q5_0, Q4_K, Q5_K, Q6_K, IQ4_NL, kFmts };

// Element order of an operand's 8 slots, and which values a lane group takes.
//   kUnit:   the 128-K unit's 32 g + 8 s .. + 7 in step s, order 0 4 1 5 2 6 3 7;
//   kHalves: block s's 4 g .. + 3 and 16 + 4 g .. + 3, each in order 0 2 1 3;
//   kOctets: block s's 8 g .. + 7, order 0 2 4 6 1 3 5 7.
enum Order { kUnit, kHalves, kOctets };
constexpr Order order_of(Fmt f) { return f == W4A16 ? kUnit : f == IQ4_NL ? kOctets : kHalves; }
constexpr bool has_mins(Fmt f) { return f == Q4_K || f == Q5_K; }

// Load instructions of one row tile and 128-K unit (Weights::load).
constexpr int loads_of(Fmt f) { return f == Q6_K ? 5 : f == Q5_K ? 4 : f == Q5_0 || f == Q8_0 || f == Q8_GGUF ? 3 : 2; }

typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));

// x = p[0] + p[1] + p[2] in bf16 bits (the last two truncations are exact).
__device__ __forceinline__ void bf16_parts(float x, uint32_t (&p)[3]) {
    const float a = __uint_as_float(__float_as_uint(x) & 0xFFFF0000u), r = x - a;
    const float b = __uint_as_float(__float_as_uint(r) & 0xFFFF0000u);
    p[0] = __float_as_uint(a) >> 16;
    p[1] = __float_as_uint(r) >> 16;
    p[2] = __float_as_uint(r - b) >> 16;
}

// ---------------------------------------------------------- activation pack

// 32-K steps between two barriers of the GEMM: a stage.  The packed
// activations are [token tile][stage][part][token][4 KSU octets], so a
// token's octets of a stage are 256 (128) contiguous bytes in memory and in
// LDS; octet o of token i sits at position o ^ swz(i), which spreads the 16
// tokens of an operand read over all 16-byte bank slots.
constexpr int steps_of(int parts) { return parts == 2 ? 2 : 4; }
template <int KSU>
__device__ __forceinline__ int swz(int token) { return KSU == 4 ? token & 15 : (token & 15) >> 1; }

constexpr int kPackThreads = 512, kPackOctets = 8;  // K <= 32768

// One workgroup a token, its row held in registers between the max and the
// split.  sums: for the formats with block minima, the 32-element sums of the
// scaled token as three bf16 parts, [token tile][K / 1024][part]
// [lane 16 (block / 8 % 4) + token][block % 8].
template <Order O, class XT, bool SUMS, int NI>
__global__ void __launch_bounds__(kPackThreads) pack_kernel(const XT* __restrict__ x, uint4* __restrict__ xp,
                                                            float* __restrict__ inv, uint16_t* __restrict__ sums,
                                                            int K) {
    constexpr bool F32 = sizeof(XT) == 4;
    constexpr int P = F32 ? 2 : 1, KSU = steps_of(P);
    constexpr int perm[3][8] = {{0, 4, 1, 5, 2, 6, 3, 7}, {0, 2, 1, 3, 4, 6, 5, 7}, {0, 2, 4, 6, 1, 3, 5, 7}};
    __shared__ float wmax[kPackThreads / 64];
    const int tid = threadIdx.x, t = blockIdx.x;
    const XT* row = x + (long)t * K;
    const int nks = K / 32;
    // octet o: 32-K step, lane group and its first and fifth element
    auto where = [](int o, int& ks, int& g, int& k0, int& k1) {
        ks = O == kUnit ? (o >> 4) * 4 + (o & 3) : o >> 2;
        g = O == kUnit ? (o >> 2) & 3 : o & 3;
        k0 = O == kUnit ? 8 * o : O == kOctets ? 32 * ks + 8 * g : 32 * ks + 4 * g;
        k1 = O == kHalves ? k0 + 16 : k0 + 4;
    };
    uint4* dst = xp + (long)(t >> 4) * nks * P * 64 + (t & 15) * (4 * KSU);
    auto at = [&](int ks, int g, int part) {
        return (long)(ks / KSU) * (P * KSU * 64) + part * (KSU * 64) + ((4 * (ks % KSU) + g) ^ swz<KSU>(t));
    };
    if constexpr (F32) {
        float4v a[NI], b[NI];
        float m = 0.0f;
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int o = tid + i * kPackThreads;
            int ks, g, k0, k1;
            where(o, ks, g, k0, k1);
            a[i] = b[i] = (float4v){0.f, 0.f, 0.f, 0.f};
            if (o < K / 8) {
                a[i] = *reinterpret_cast<const float4v*>(row + k0);
                b[i] = *reinterpret_cast<const float4v*>(row + k1);
            }
        }
#pragma unroll
        for (int i = 0; i < NI; i++)
#pragma unroll
            for (int e = 0; e < 8; e++) m = fmaxf(m, fabsf(finite(e < 4 ? a[i][e & 3] : b[i][e & 3])));
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
        if ((tid & 63) == 0) wmax[tid >> 6] = m;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kPackThreads / 64; w++) m = fmaxf(m, wmax[w]);
        const int sh = scale_exponent(m);
        const float c = ldexpf(1.0f, sh);
        if (tid == 0) inv[t] = ldexpf(1.0f, -sh);
        const int no = SUMS ? (K / 8 + 127) & ~127 : K / 8;  // sums: whole 1024-K groups, zeros past K
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int o = tid + i * kPackThreads;
            if (o >= no) break;
            int ks, g, k0, k1;
            where(o, ks, g, k0, k1);
            float v[8], r[8];
            half8v h, l;
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = (e < 4 ? a[i][e & 3] : b[i][e & 3]) * c;
#pragma unroll
            for (int e = 0; e < 8; e++) r[e] = v[perm[O][e]];
            split_hi_lo(r, h, l);
            if (o < K / 8) {
                dst[at(ks, g, 0)] = __builtin_bit_cast(uint4, h);
                dst[at(ks, g, 1)] = __builtin_bit_cast(uint4, l);
            }
            if constexpr (SUMS) {
                float s = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
                s = single_step<1>(s);
                s = single_step<2>(s);
                if (g == 0) {
                    uint32_t p[3];
                    bf16_parts(s, p);
                    uint16_t* d = sums + ((long)(t >> 4) * ((nks + 31) / 32) + ks / 32) * 1536 +
                                  (16 * ((ks >> 3) & 3) + (t & 15)) * 8 + (ks & 7);
#pragma unroll
                    for (int q = 0; q < 3; q++) d[q * 512] = (uint16_t)p[q];
                }
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int o = tid + i * kPackThreads;
            if (o >= K / 8) break;
            int ks, g, k0, k1;
            where(o, ks, g, k0, k1);
            const uint2 a = *reinterpret_cast<const uint2*>(row + k0), b = *reinterpret_cast<const uint2*>(row + k1);
            uint4 w;
            if constexpr (O == kUnit) {
                w.x = __builtin_amdgcn_perm(b.x, a.x, 0x05040100u);
                w.y = __builtin_amdgcn_perm(b.x, a.x, 0x07060302u);
                w.z = __builtin_amdgcn_perm(b.y, a.y, 0x05040100u);
                w.w = __builtin_amdgcn_perm(b.y, a.y, 0x07060302u);
            } else if constexpr (O == kHalves) {
                w.x = __builtin_amdgcn_perm(a.y, a.x, 0x05040100u);
                w.y = __builtin_amdgcn_perm(a.y, a.x, 0x07060302u);
                w.z = __builtin_amdgcn_perm(b.y, b.x, 0x05040100u);
                w.w = __builtin_amdgcn_perm(b.y, b.x, 0x07060302u);
            } else {
                w.x = __builtin_amdgcn_perm(a.y, a.x, 0x05040100u);
                w.y = __builtin_amdgcn_perm(b.y, b.x, 0x05040100u);
                w.z = __builtin_amdgcn_perm(a.y, a.x, 0x07060302u);
                w.w = __builtin_amdgcn_perm(b.y, b.x, 0x07060302u);
            }
            dst[at(ks, g, 0)] = w;
        }
    }
}

// ------------------------------------------------------------------- GEMM

struct WideArgs {
    const uint8_t* w;   // the format's bulk data
    const uint8_t* s;   // scales (W4A16: packed (scale, zero) dwords; Q6_K: int8 scales)
    const uint8_t* e;   // Q5_0, Q6_K: fifth / high bits
    const uint8_t* d;   // Q6_K: super-block scales
    const char* xp;     // packed activations
    const float* inv;   // 1 / scale of each token (fp32 activations)
    const char* sums;   // block sums (formats with minima)
    float* c;
    int rows, K, T, gu;  // gu: 128-K units of a W4A16 group
    uint32_t wb, sb, eb, db;  // bytes of w, s, e, d: loads past them read zeros
};

// One wave's direct global -> LDS copy of 1 KB: lane l's 16 bytes at
// base + off go to lds + 16 l.  The caller waits for vmcnt before a barrier.
// (s_nop: 5 wait states between a vector write of the base's registers, which
// the compiler may have put right before, and the load's read of them.)
// m0, which the load takes its LDS address from, is a register the compiler
// reserves: it warns of the clobber that tells it of the write.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma_1k(const void* base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base)
                 : "memory", "m0");
}
#pragma clang diagnostic pop

__device__ __forceinline__ uint32_t and_or(uint32_t w, uint32_t mask, uint32_t base) { return (w & mask) | base; }

__device__ __forceinline__ half2v splat2(float v) { return (half2v){(_Float16)v, (_Float16)v}; }

__device__ __forceinline__ half8v join(half2v a, half2v b, half2v c, half2v d) {
    return (half8v){a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// 4 x 4 transpose over (register, lane group): w[b] of lane group g becomes w[g] of lane group b.
__device__ __forceinline__ void transpose4(u32x4& w) {
    auto a = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
    auto b = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
    auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    w = (u32x4){c[0], c[1], d[0], d[1]};
}

// One row tile's weights of a 128-K unit (4 blocks of 32), as loaded.
struct Raw {
    u32x4 a, b;       // bulk data
    uint32_t s[4];    // scales, or the super-block header
    uint32_t e[4];    // fifth / high bits
};

template <Fmt F>
struct Weights {
    __amdgpu_buffer_rsrc_t rw, rs, re, rd;
    int lg;
    __device__ __forceinline__ Weights(const WideArgs& p, int lg) : lg(lg) {
        rw = rsrc(p.w, p.wb);
        rs = rsrc(p.s, p.sb);
        re = rsrc(p.e, p.eb);
        rd = rsrc(p.d, p.db);
    }
    static __device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* b, uint32_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc((void*)b, (short)0, (int)bytes, 0x00020000);
    }
    // byte offsets of a row: bulk data (with the lane group's share), scales, bits
    struct Off {
        uint32_t w, s, e, d;
    };
    __device__ __forceinline__ Off row_offset(uint32_t row, const WideArgs& p) const {
        const uint32_t K = p.K;
        switch (F) {
            case W4A16: return {row * (K / 2) + 16 * lg, row * (K / 128 / p.gu) * 4, 0, 0};
            case Q4_0:
            case IQ4_NL: return {row * (K / 2) + 16 * lg, row * (K / 16), 0, 0};
            case Q8_0: return {row * K + 32 * lg, row * (K / 8), 0, 0};
            case Q8_GGUF: return {row * K + 32 * lg, row * (K / 16), 0, 0};
            case Q5_0: return {row * (K / 2) + 16 * lg, row * (K / 16), row * (K / 8), 0};
            case Q4_K: return {row * (K / 256 * 144) + 16 + 16 * lg, row * (K / 256 * 144), 0, 0};
            case Q5_K: return {row * (K / 256 * 176) + 16 + 16 * lg, row * (K / 256 * 176),
                               row * (K / 256 * 176) + 144 + 4 * lg, 0};
            default: return {row * (K / 2) + 16 * lg, row * (K / 16), row * (K / 4) + 4 * lg, row * (K / 128)};
        }
    }
    __device__ __forceinline__ void load(Raw& r, const Off& o, int u, int gu) const {
        u = __builtin_amdgcn_readfirstlane(u);  // a scalar offset, or the loads loop over the lanes
        const int sb = u >> 1, h = u & 1;
        if constexpr (F == W4A16) {
            r.a = __builtin_amdgcn_raw_buffer_load_b128(rw, o.w, 64 * u, 0);
            r.s[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, o.s, 4 * (u / gu), 0);
        } else if constexpr (F == Q4_0 || F == IQ4_NL || F == Q5_0) {
            r.a = __builtin_amdgcn_raw_buffer_load_b128(rw, o.w, 64 * u, 0);
            auto s = __builtin_amdgcn_raw_buffer_load_b64(rs, o.s, 8 * u, 0);
            r.s[0] = s[0];
            r.s[1] = s[1];
            if constexpr (F == Q5_0) {
                const u32x4 e = __builtin_amdgcn_raw_buffer_load_b128(re, o.e, 16 * u, 0);
#pragma unroll
                for (int b = 0; b < 4; b++) r.e[b] = e[b];
            }
        } else if constexpr (F == Q8_0 || F == Q8_GGUF) {
            r.a = __builtin_amdgcn_raw_buffer_load_b128(rw, o.w, 128 * u, 0);
            r.b = __builtin_amdgcn_raw_buffer_load_b128(rw, o.w + 16, 128 * u, 0);
            if constexpr (F == Q8_0) {
                const u32x4 s = __builtin_amdgcn_raw_buffer_load_b128(rs, o.s, 16 * u, 0);
#pragma unroll
                for (int b = 0; b < 4; b++) r.s[b] = s[b];
            } else {
                auto s = __builtin_amdgcn_raw_buffer_load_b64(rs, o.s, 8 * u, 0);
                r.s[0] = s[0];
                r.s[1] = s[1];
            }
        } else if constexpr (F == Q4_K || F == Q5_K) {
            const int sbb = sb * (F == Q4_K ? 144 : 176);
            r.a = __builtin_amdgcn_raw_buffer_load_b128(rw, o.w, sbb + 64 * h, 0);
            const u32x4 s = __builtin_amdgcn_raw_buffer_load_b128(rw, o.s, sbb, 0);
#pragma unroll
            for (int b = 0; b < 4; b++) r.s[b] = s[b];
            if constexpr (F == Q5_K) {
                r.e[0] = __builtin_amdgcn_raw_buffer_load_b32(rw, o.e, sbb, 0);
                r.e[1] = __builtin_amdgcn_raw_buffer_load_b32(rw, o.e + 16, sbb, 0);
            }
        } else {
            r.a = __builtin_amdgcn_raw_buffer_load_b128(rw, o.w, 64 * u, 0);
            r.e[0] = __builtin_amdgcn_raw_buffer_load_b32(re, o.e, 32 * u, 0);
            r.e[1] = __builtin_amdgcn_raw_buffer_load_b32(re, o.e + 16, 32 * u, 0);
            auto s = __builtin_amdgcn_raw_buffer_load_b64(rs, o.s, 8 * u, 0);
            r.s[0] = s[0];
            r.s[1] = s[1];
            r.s[2] = __builtin_amdgcn_raw_buffer_load_b16(rd, o.d, 2 * sb, 0);
        }
    }
    // the unit's lane-group transposes
    __device__ __forceinline__ void arrange(Raw& r) const {
        if constexpr (F != W4A16) transpose4(r.a);
        if constexpr (F == Q8_0 || F == Q8_GGUF) transpose4(r.b);
    }
};

// The 6-bit scale and minimum of block b (0-7) of a Q4_K / Q5_K super-block header (d, dmin, 12 bytes).
__device__ __forceinline__ uint32_t kq_byte(const uint32_t (&h)[4], int i) { return (h[1 + (i >> 2)] >> (8 * (i & 3))) & 0xffu; }
__device__ __forceinline__ uint32_t kq_scale(const uint32_t (&h)[4], int b) {
    return b < 4 ? kq_byte(h, b) & 63u : (kq_byte(h, b + 4) & 15u) | ((kq_byte(h, b - 4) >> 6) << 4);
}
__device__ __forceinline__ uint32_t kq_min(const uint32_t (&h)[4], int b) {
    return b < 4 ? kq_byte(h, b + 4) & 63u : (kq_byte(h, b + 4) >> 4) | ((kq_byte(h, b) >> 6) << 4);
}

// The float codebook of DequantizeIQ4NL, times 2^12, in fp16 parts: byte planes of 16 entries.
template <int PW>
struct IQ4Planes {
    uint32_t t[2 * PW][4];  // [part: its high byte, its low byte][entry / 4]
};
constexpr float kIQ4[16] = {-1.0f, -0.6961928f, -0.5250730f, -0.3947555f, -0.2831612f, -0.1790887f, -0.0805542f, 0.0f,
                            0.0805542f, 0.1790887f, 0.2831612f, 0.3947555f, 0.5250730f, 0.6961928f, 1.0f, 1.3312578f};
// fp16 bits of v, rounded to nearest even (|v| below 2^15, normal or subnormal)
constexpr uint32_t f16_bits(double v) {
    const uint32_t sign = v < 0 ? 0x8000u : 0u;
    double a = v < 0 ? -v : v;
    if (a == 0) return 0;
    int e = 0;
    while (a >= 2.0) { a /= 2; e++; }
    while (a < 1.0 && e > -14) { a *= 2; e--; }
    const double m = a * 1024;  // normal: [1024, 2048)
    uint32_t r = (uint32_t)m;
    const double f = m - r;
    if (f > 0.5 || (f == 0.5 && (r & 1))) r++;
    return sign | (((uint32_t)(e + 14) << 10) + r);  // r's bit 10 adds the exponent's last unit
}
constexpr double f16_value(uint32_t b) {
    const int e = (b >> 10) & 31;
    double m = (b & 1023) + (e ? 1024 : 0);
    for (int i = e ? e : 1; i < 25; i++) m /= 2;
    for (int i = 25; i < (e ? e : 1); i++) m *= 2;
    return b & 0x8000u ? -m : m;
}
// v rounded to 8 bits
constexpr double bits8(double v) {
    double u = 1;
    while (u * 256 <= (v < 0 ? -v : v)) u *= 2;
    while (u * 128 > (v < 0 ? -v : v) && v != 0) u /= 2;
    return (double)(long)(v / u + (v < 0 ? -0.5 : 0.5)) * u;
}
template <int PW>
constexpr IQ4Planes<PW> iq4_planes() {
    IQ4Planes<PW> p = {};
    for (int i = 0; i < 16; i++) {
        double v = 4096.0 * kIQ4[i];
        for (int z = 0; z < PW; z++) {
            const uint32_t h = f16_bits(PW == 3 && z == 0 ? bits8(v) : v);
            p.t[2 * z][i >> 2] |= (h >> 8) << (8 * (i & 3));
            p.t[2 * z + 1][i >> 2] |= (h & 255) << (8 * (i & 3));
            v -= f16_value(h);
        }
    }
    return p;
}
static_assert(f16_bits(1.0) == 0x3c00 && f16_bits(-0.5) == 0xb800 && f16_value(0x3c01) == 1.0009765625, "fp16");

// Four codebook entries (selectors 0-15 in a dword's bytes): two dwords of halves of each part.
template <int PW>
__device__ __forceinline__ void iq4_lookup(uint32_t sel, half2v (&o)[PW][2]) {
    constexpr IQ4Planes<PW> T = iq4_planes<PW>();
    const uint32_t s7 = sel & 0x07070707u;
    const uint32_t up = ((sel >> 3) & 0x01010101u) * 255u;  // byte mask of the entries 8-15
    uint32_t pl[2 * PW];
#pragma unroll
    for (int q = 0; q < 2 * PW; q++) {
        const uint32_t a = __builtin_amdgcn_perm(T.t[q][1], T.t[q][0], s7), b = __builtin_amdgcn_perm(T.t[q][3], T.t[q][2], s7);
        pl[q] = (b & up) | (a & ~up);
    }
#pragma unroll
    for (int z = 0; z < PW; z++) {
        o[z][0] = as_half2(__builtin_amdgcn_perm(pl[2 * z], pl[2 * z + 1], 0x05010400u));
        o[z][1] = as_half2(__builtin_amdgcn_perm(pl[2 * z], pl[2 * z + 1], 0x07030602u));
    }
}

// Decoded weights of one row tile and 32-K step: the exact value is the sum of the parts (P: the activations'), times
// the scale.  (IQ4_NL: 24 bits; to 22 with fp16 activations.)
constexpr int parts_of(Fmt f, int P) { return f == IQ4_NL ? P + 1 : f == Q6_K ? 2 : 1; }
constexpr bool unit_scaled(Fmt f) { return f == W4A16 || f == Q4_K || f == Q5_K || f == Q6_K; }  // one scale per 128-K unit

template <Fmt F, int PW>
__device__ __forceinline__ void decode(const Raw& r, int b, int u, int lg, half2v z1, half2v z2, half8v (&o)[PW]) {
    constexpr uint32_t M = 0x64006400u;  // 1024 in both halves: M | n is 1024 + n
    const half2v k16 = splat2(0.0625f);
    if constexpr (F == W4A16 || F == Q4_0) {
        // the low and high nibbles of bytes 0, 2 and 1, 3; a high nibble reads 1024 + 16 n
        const uint32_t w = r.a[b], w8 = w >> 8;
        const half2v lo02 = as_half2(and_or(w, 0x000F000Fu, M)) + z1, hi02 = as_half2(and_or(w, 0x00F000F0u, M)) * k16 + z2;
        const half2v lo13 = as_half2(and_or(w8, 0x000F000Fu, M)) + z1, hi13 = as_half2(and_or(w8, 0x00F000F0u, M)) * k16 + z2;
        // W4A16's interleaved nibbles: elements 0 4 1 5 2 6 3 7 of the dword's 8
        o[0] = F == W4A16 ? join(lo02, hi02, lo13, hi13) : join(lo02, lo13, hi02, hi13);
    } else if constexpr (F == Q5_0) {
        // the fifth bits of elements 4 lg .. + 3 (and 16 + 4 lg) to bit 4 of each byte
        const uint32_t q = r.e[b] >> (4 * lg);
        const uint32_t s0 = ((q & 15u) * 0x02040810u) & 0x10101010u, s1 = (((q >> 16) & 15u) * 0x02040810u) & 0x10101010u;
        const uint32_t w = (r.a[b] & 0x0F0F0F0Fu) | s0, v = ((r.a[b] >> 4) & 0x0F0F0F0Fu) | s1;
        const half2v k = splat2(-1040.0f);
        o[0] = join(as_half2(and_or(w, 0x00FF00FFu, M)) + k, as_half2(and_or(w >> 8, 0x00FF00FFu, M)) + k,
                    as_half2(and_or(v, 0x00FF00FFu, M)) + k, as_half2(and_or(v >> 8, 0x00FF00FFu, M)) + k);
    } else if constexpr (F == Q8_0 || F == Q8_GGUF) {
        const uint32_t w = r.a[b] ^ 0x80808080u, v = r.b[b] ^ 0x80808080u;  // q + 128
        const half2v k = splat2(-1152.0f);
        o[0] = join(as_half2(and_or(w, 0x00FF00FFu, M)) + k, as_half2(and_or(w >> 8, 0x00FF00FFu, M)) + k,
                    as_half2(and_or(v, 0x00FF00FFu, M)) + k, as_half2(and_or(v >> 8, 0x00FF00FFu, M)) + k);
    } else if constexpr (F == Q4_K || F == Q5_K) {
        // block b: the low (even b) or high nibbles of 32 bytes; lane group lg's bytes 4 lg .. + 3 and 16 + 4 lg .. + 3
        uint32_t w = r.a[2 * (b >> 1)], v = r.a[2 * (b >> 1) + 1];
        if (b & 1) {
            w >>= 4;
            v >>= 4;
        }
        // times the block's 6-bit scale: at most 31 x 63, exact
        const half2v c = splat2((float)((u & 1) ? kq_scale(r.s, 4 + b) : kq_scale(r.s, b))), k = c * splat2(-1024.0f);
        constexpr uint32_t B = F == Q5_K ? 0x00FF00FFu : 0x000F000Fu;
        if constexpr (F == Q5_K) {
            const int j = 4 * (u & 1) + b;  // the block's bit in every high-bit byte
            w = (w & 0x0F0F0F0Fu) | (((r.e[0] >> j) & 0x01010101u) << 4);
            v = (v & 0x0F0F0F0Fu) | (((r.e[1] >> j) & 0x01010101u) << 4);
        }
        auto scaled = [&](uint32_t q) { return __builtin_elementwise_fma(as_half2(and_or(q, B, M)), c, k); };  // c q
        o[0] = join(scaled(w), scaled(w >> 8), scaled(v), scaled(v >> 8));
    } else if constexpr (F == Q6_K) {
        // block b of a 128-value half: nibbles of bytes (b & 1) 32 + ..., low for b < 2, and bits 2 b of the high-bit bytes
        uint32_t w = r.a[2 * (b & 1)], v = r.a[2 * (b & 1) + 1];
        if (b >= 2) {
            w >>= 4;
            v >>= 4;
        }
        w = (w & 0x0F0F0F0Fu) | (((r.e[0] >> (2 * b)) & 0x03030303u) << 4);
        v = (v & 0x0F0F0F0Fu) | (((r.e[1] >> (2 * b)) & 0x03030303u) << 4);
        const half2v k = splat2(-1056.0f);
        const uint32_t sw = r.s[b >> 1] >> (16 * (b & 1));  // the scales of elements 0-15 and 16-31
        const half2v c0 = splat2((float)(int8_t)(sw & 0xff)), c1 = splat2((float)(int8_t)((sw >> 8) & 0xff));
        half2v q[4] = {as_half2(and_or(w, 0x00FF00FFu, M)) + k, as_half2(and_or(w >> 8, 0x00FF00FFu, M)) + k,
                       as_half2(and_or(v, 0x00FF00FFu, M)) + k, as_half2(and_or(v >> 8, 0x00FF00FFu, M)) + k};
        half2v h[4], l[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const half2v c = e < 2 ? c0 : c1;
            h[e] = q[e] * c;  // rounded to 11 bits
            l[e] = __builtin_elementwise_fma(q[e], c, -h[e]);  // the rest, exactly
        }
        o[0] = join(h[0], h[1], h[2], h[3]);
        o[1] = join(l[0], l[1], l[2], l[3]);
    } else {  // IQ4_NL: byte j's elements 2 j and 2 j + 1
        half2v e[PW][2], f[PW][2];
        iq4_lookup<PW>(r.a[b] & 0x0F0F0F0Fu, e);
        iq4_lookup<PW>((r.a[b] >> 4) & 0x0F0F0F0Fu, f);
#pragma unroll
        for (int z = 0; z < PW; z++) o[z] = join(e[z][0], e[z][1], f[z][0], f[z][1]);
    }
}

// The scale of block b (formats with one scale a block).
template <Fmt F>
__device__ __forceinline__ float block_scale(const Raw& r, int b, int u) {
    if constexpr (F == Q8_0) return __uint_as_float(r.s[b]);
    else return h2f((uint16_t)(r.s[b >> 1] >> (16 * (b & 1)))) * (F == IQ4_NL ? 0x1p-12f : 1.0f);
}

// The whole part of a W4A16 zero that goes into the operand q - zero (exact in fp16), 0 for large or non-finite zeros.
__device__ __forceinline__ float whole_zero(float z) { return fabsf(z) <= 960.0f ? rintf(z) : 0.0f; }

// fp32 sums of n terms of one size, added one by one, are off by sqrt(n / 2)
// roundings.  The terms are K / 32 scaled blocks (K / 128 units), over the
// waves along K.  Up to kChain values of K a wave adds them up as they come;
// past it roundings would exceed those of the tiled copies and the dequantized
// products, so more waves lie along K or (FAR) a wave's sums go to a second
// set of them every few units.  IQ4_NL and Q5_0, whose other paths are the
// most exact, always have the second set, at half the waves of their largest
// tiles.  Relative error against 64 bits, one chain and now, 1021 tokens of
// 4096 x 14336 (rows x K): Q4_0 4.0e-7 / 2.1e-7, Q5_0 3.9e-7 / 1.4e-7, Q4_K
// 3.0e-7 / 1.7e-7, IQ4_NL 2.8e-7 / 1.3e-7; us there: 314 / 338, 363 / 364, 361
// / 345, 333 / 298.
constexpr int kChain = 5120;
constexpr bool far_sums(Fmt f) { return f == IQ4_NL || f == Q5_0; }

// P: parts of the activations (2 for fp32).  FAR: sums in two steps.
template <Fmt F, int P, int MT, int NT, int WN, int WK, bool FAR>
__global__ void __launch_bounds__(64 * WN * WK, 2) wide_gemm_kernel(const WideArgs p) {
    constexpr int KSU = steps_of(P);
    constexpr int PW = parts_of(F, P);
    constexpr int UB = MT * KSU * P * 1024;  // bytes of one K group's stage
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = wave / WN, wn = wave % WN, li = lane & 15, lg = lane >> 4;
    const int ttiles = (p.T + 16 * MT - 1) / (16 * MT);
    // consecutive workgroups of an XCD take the token tiles of one row tile: its weights stay in that XCD's L2
    const int b = xcd_contiguous(blockIdx.x, gridDim.x);
    const int tt = b % ttiles, n0 = (b / ttiles) * (16 * NT * WN) + wn * 16 * NT;
    const int nu = p.K / 128, nsteps = (nu + WK - 1) / WK;
    const Weights<F> W(p, lg);
    typename Weights<F>::Off off[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) off[j] = W.row_offset((uint32_t)min(n0 + 16 * j + li, p.rows - 1), p);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    const long tstride = (long)(p.K / 32) * P * 1024;  // bytes of one token tile
    const char* xt = p.xp + (long)tt * MT * tstride;
    uint32_t xo[KSU];  // this lane's operand of step s inside a (token tile, part) of a stage
#pragma unroll
    for (int s = 0; s < KSU; s++) xo[s] = li * (KSU * 64) + (((4 * s + lg) ^ swz<KSU>(li)) * 16);

    // the K group's waves copy the activations of KSU steps, 1 KB a piece
    auto stage = [&](int u, int h, int buf) {
        constexpr int PC = KSU * P;  // pieces of a token tile, consecutive in memory
#pragma unroll
        for (int q = 0; q < (MT * PC + WN - 1) / WN; q++) {
            const int e = q * WN + wn;
            if ((MT * PC) % WN == 0 || e < MT * PC)
                dma_1k(xt + (long)(4 * u + KSU * h) * P * 1024 + (e / PC) * tstride + (e % PC) * 1024, 16u * lane,
                       lds0 + (buf * WK + kg) * UB + e * 1024);
        }
    };
    Raw next[NT];
    auto load_w = [&](int u) {
#pragma unroll
        for (int j = 0; j < NT; j++) W.load(next[j], off[j], u, p.gu);
    };

    float4v acc[MT][NT], sum[FAR ? MT : 1][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = sum[FAR ? i : 0][j] = (float4v){0.f, 0.f, 0.f, 0.f};

    if (kg < nu) {
        stage(kg, 0, 0);
        load_w(kg);
    }
    constexpr int H = 4 / KSU;  // barriers a unit
    bool odd = false;           // a W4A16 zero that is no whole number was seen
    auto add_up = [&] {
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++) {
                sum[FAR ? i : 0][j] += acc[i][j];
                acc[i][j] = (float4v){0.f, 0.f, 0.f, 0.f};
            }
    };
    const int per = !FAR ? nsteps : nsteps > 64 ? 5 : nsteps > 24 ? 3 : 2;  // both chains of about sqrt(4 nsteps) terms
    for (int t0 = 0; t0 < nsteps; t0 += per) {
    const int t1 = min(nsteps, t0 + per);
#pragma unroll 1
    for (int t = t0; t < t1; t++) {
        const int u = t * WK + kg;
        Raw cur[NT];
        float4v d[MT][NT];
        half2v z1[NT], z2[NT];
#pragma unroll
        for (int h = 0; h < H; h++) {
            const int buf = (t * H + h) & 1;
            // this stage's activations have landed, and the weights; the other buffer's readers are done
            // (a unit's later stages leave the next unit's weight loads, issued after their own, in flight)
            if (h > 0 && u + WK < nu) {
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NT * loads_of(F)) : "memory");
            } else {
                __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
                asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            }
            if (h + 1 < H) {
                if (u < nu) stage(u, h + 1, buf ^ 1);
            } else if (u + WK < nu) {
                stage(u + WK, 0, buf ^ 1);
            }
            if (h == 0) {
#pragma unroll
                for (int j = 0; j < NT; j++) cur[j] = next[j];
                if (u + WK < nu) load_w(u + WK);
                if (u < nu) {
#pragma unroll
                    for (int j = 0; j < NT; j++) W.arrange(cur[j]);
                    if constexpr (F == W4A16) {
#pragma unroll
                        for (int j = 0; j < NT; j++) {
                            // q - zero is exact for a whole zero; the rest of any other comes off at the end
                            const float z = h2f((uint16_t)(cur[j].s[0] >> 16));
                            const float zi = whole_zero(z);
                            z1[j] = splat2(-1024.0f - zi);
                            z2[j] = splat2(-64.0f - zi);
                            odd |= z != zi;
                        }
                    } else if constexpr (F == Q4_0) {
#pragma unroll
                        for (int j = 0; j < NT; j++) {
                            z1[j] = splat2(-1032.0f);
                            z2[j] = splat2(-72.0f);
                        }
                    }
                }
            }
            if (u < nu) {
                const char* xs = smem + (buf * WK + kg) * UB;
#pragma unroll
                for (int s = 0; s < KSU; s++) {
                    const int blk = KSU * h + s;
                    half8v bo[NT][PW];
                    float sc[NT];
#pragma unroll
                    for (int j = 0; j < NT; j++) {
                        decode<F>(cur[j], blk, u, lg, z1[j], z2[j], bo[j]);
                        if constexpr (!unit_scaled(F)) sc[j] = block_scale<F>(cur[j], blk, u);
                    }
#pragma unroll
                    for (int i = 0; i < MT; i++) {
                        half8v ao[P];
#pragma unroll
                        for (int q = 0; q < P; q++)
                            ao[q] = *reinterpret_cast<const half8v*>(xs + (i * P + q) * (KSU * 1024) + xo[s]);
#pragma unroll
                        for (int j = 0; j < NT; j++) {
                            auto times = [&](int q, int w, float4v c) {
                                return __builtin_amdgcn_mfma_f32_16x16x32_f16(ao[q < P ? q : 0], bo[j][w < PW ? w : 0], c, 0, 0, 0);
                            };
                            constexpr float4v none = {0.f, 0.f, 0.f, 0.f};
                            float4v v;
                            if constexpr (PW == 3) {
                                // 11 x 8 bits: sums of these are (nearly) exact, and the others, of 2^-8 of it and
                                // less, join them in one rounding
                                v = times(0, 0, none) + times(0, 1, times(1, 0, times(0, 2, times(1, 1, none))));
                            } else {
                                v = times(0, 0, unit_scaled(F) && blk > 0 ? d[i][j] : none);
                                if constexpr (P == 2) v = times(1, 0, v);
                                if constexpr (PW == 2) v = times(0, 1, v);
                            }
                            if constexpr (unit_scaled(F)) {
                                d[i][j] = v;
                            } else {
#pragma unroll
                                for (int r = 0; r < 4; r++) acc[i][j][r] = __builtin_fmaf(sc[j], v[r], acc[i][j][r]);
                            }
                        }
                    }
                }
                if constexpr (unit_scaled(F)) {
                    if (h == H - 1) {
#pragma unroll
                        for (int j = 0; j < NT; j++) {
                            const float s = h2f((uint16_t)(F == Q6_K ? cur[j].s[2] : cur[j].s[0]));
#pragma unroll
                            for (int i = 0; i < MT; i++)
#pragma unroll
                                for (int r = 0; r < 4; r++) acc[i][j][r] = __builtin_fmaf(s, d[i][j][r], acc[i][j][r]);
                        }
                    }
                }
            }
        }
    }
    if constexpr (FAR) add_up();
    }
    if constexpr (FAR) {
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++) acc[i][j] = sum[i][j];
    }
    if constexpr (F == W4A16) {
        // zeros that are no integers up to 960: s * zf * sum x off (all-ones B operands give a unit's sum x)
        if (__builtin_expect(__any(odd), 0)) {
            const half2v one = splat2(1.0f);
            const half8v ones = join(one, one, one, one);
            for (int u = kg; u < nu; u += WK) {
                float sz[NT];
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    const uint32_t v = __builtin_amdgcn_raw_buffer_load_b32(W.rs, off[j].s, 4 * (u / p.gu), 0);
                    const float z = h2f((uint16_t)(v >> 16));
                    sz[j] = -h2f((uint16_t)v) * (z - whole_zero(z));
                }
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    float4v v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int s = 0; s < 4; s++)
                        v = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            *reinterpret_cast<const half8v*>(xt + i * tstride + u * 4096 + xo[s]), ones, v, 0, 0, 0);
#pragma unroll
                    for (int j = 0; j < NT; j++)
#pragma unroll
                        for (int r = 0; r < 4; r++) acc[i][j][r] = __builtin_fmaf(sz[j], v[r], acc[i][j][r]);
                }
            }
        }
    }
    if constexpr (has_mins(F)) {
        // minus (dmin min_b) sum_b x over 32 blocks an MFMA step: both factors as three bf16 parts, the products
        // above 2^-24 of the whole kept
        const int ngrp = (p.K + 1023) / 1024, nsb = p.K / 256;
        const char* st = p.sums + (long)tt * MT * ngrp * 3072 + 16 * lane;
        for (int g = kg; g < ngrp; g += WK) {
            bf16x8v m[NT][3];
#pragma unroll
            for (int j = 0; j < NT; j++) {
                const int sb = 4 * g + lg;  // this lane group's super-block
                const u32x4 hv = __builtin_amdgcn_raw_buffer_load_b128(
                    W.rw, off[j].s + (uint32_t)min(sb, nsb - 1) * (F == Q4_K ? 144u : 176u), 0, 0);
                const uint32_t hd[4] = {hv[0], hv[1], hv[2], hv[3]};
                const float dmin = sb < nsb ? -h2f((uint16_t)(hv[0] >> 16)) : 0.0f;
                uint32_t q[3][4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    uint32_t x0[3], x1[3];
                    bf16_parts(dmin * (float)kq_min(hd, 2 * e), x0);
                    bf16_parts(dmin * (float)kq_min(hd, 2 * e + 1), x1);
#pragma unroll
                    for (int z = 0; z < 3; z++) q[z][e] = x0[z] | x1[z] << 16;
                }
#pragma unroll
                for (int z = 0; z < 3; z++) m[j][z] = __builtin_bit_cast(bf16x8v, (u32x4){q[z][0], q[z][1], q[z][2], q[z][3]});
            }
#pragma unroll
            for (int i = 0; i < MT; i++) {
                bf16x8v x[3];
#pragma unroll
                for (int z = 0; z < 3; z++)
                    x[z] = __builtin_bit_cast(bf16x8v, *reinterpret_cast<const u32x4*>(st + ((long)i * ngrp + g) * 3072 + z * 1024));
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    float4v v = {0.f, 0.f, 0.f, 0.f};
                    v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[2], m[j][0], v, 0, 0, 0);
                    v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[0], m[j][2], v, 0, 0, 0);
                    v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[1], m[j][1], v, 0, 0, 0);
                    v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[1], m[j][0], v, 0, 0, 0);
                    v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[0], m[j][1], v, 0, 0, 0);
                    v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[0], m[j][0], v, 0, 0, 0);
                    acc[i][j] += v;
                }
            }
        }
    }
    if constexpr (WK > 1) {
        // the K groups' sums meet through LDS, halving the groups
        float4v* red = reinterpret_cast<float4v*>(smem);
#pragma unroll
        for (int h = WK / 2; h >= 1; h >>= 1) {
            __syncthreads();
            if (kg >= h && kg < 2 * h) {
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < NT; j++) red[(((kg - h) * WN + wn) * MT * NT + i * NT + j) * 64 + lane] = acc[i][j];
            }
            __syncthreads();
            if (kg < h) {
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < NT; j++) acc[i][j] += red[((kg * WN + wn) * MT * NT + i * NT + j) * 64 + lane];
            }
        }
        if (kg != 0) return;
    }
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int tok = (tt * MT + i) * 16 + 4 * lg + r;
            if (tok >= p.T) continue;
            const float iv = P == 2 ? p.inv[tok] : 1.0f;
#pragma unroll
            for (int j = 0; j < NT; j++) {
                const int row = n0 + 16 * j + li;
                if (row < p.rows) p.c[(long)tok * p.rows + row] = P == 2 ? acc[i][j][r] * iv : acc[i][j][r];
            }
        }
}

// ------------------------------------------------------------ few tokens
//
// Up to 16 tokens of fp16 activations on 4-bit weights of 16 bytes a block,
// one launch on the upload layout.  Bound by memory: a wave needs many bytes
// in flight, in long runs (operands read straight from the rows, 16 rows of 64
// bytes an instruction, took 12.8 us where this takes 8.7 us, W4A16 1024 x
// 8192 rows x K, 16 tokens).  The waves of a workgroup lie along K and work
// alone up to the final sum.  A wave takes 512 values of K, a quad of units,
// at a time: a load instruction reads 256 bytes of each of 4 rows (or tokens),
// and a private LDS region turns rows into operands: lane l writes piece
// l % 16 of row 4 v + l / 16 at position piece ^ row, and lane 16 g + i reads
// piece 4 u + g of row i, both without bank conflicts.  A quad's registers are
// free once it is written to LDS, so the next quad's loads are in flight
// while this one is multiplied.
template <Fmt F, int NT, int WK>
__global__ void __launch_bounds__(64 * WK, 2) few_gemm_kernel(const WideArgs p) {
    static_assert(F == W4A16 || F == IQ4_NL, "16-byte blocks, fp16 activations");
    constexpr int PW = parts_of(F, 1), SD = F == W4A16 ? 1 : 2;  // 16-byte scale loads of a row and quad
    constexpr int RB = 4096 * (1 + NT);                       // LDS of a wave: one activation unit, NT weight quads
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63, kg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int n0 = blockIdx.x * 16 * NT, nu = p.K / 128, nq = (nu + 3) / 4;
    const __amdgpu_buffer_rsrc_t rw = Weights<F>::rsrc(p.w, p.wb), rs = Weights<F>::rsrc(p.s, p.sb),
                                 rx = Weights<F>::rsrc(p.xp, (uint32_t)p.T * (uint32_t)p.K * 2u);
    uint32_t wo[NT][4], so[NT], xo[4];
#pragma unroll
    for (int j = 0; j < NT; j++) {
#pragma unroll
        for (int v = 0; v < 4; v++)
            wo[j][v] = (uint32_t)min(n0 + 16 * j + 4 * v + lg, p.rows - 1) * (uint32_t)(p.K / 2) + 16u * li;
        so[j] = (uint32_t)min(n0 + 16 * j + li, p.rows - 1) * (uint32_t)(F == W4A16 ? p.K / 128 / p.gu * 4 : p.K / 16);
    }
#pragma unroll
    for (int v = 0; v < 4; v++) xo[v] = (uint32_t)min(4 * v + lg, p.T - 1) * (uint32_t)p.K * 2u + 16u * li;
    char* xs = smem + kg * RB;
    char* ws = xs + 4096;
    uint32_t put[4], get[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
        put[v] = (4 * v + lg) * 256 + ((li ^ (4 * v + lg)) * 16);
        get[v] = li * 256 + (((4 * v + lg) ^ li) * 16);
    }
    u32x4 w[NT][4], x[4][4], sn[NT][SD];
    // past the last unit the loads read other rows or zeros, and nothing uses them
    auto load_w = [&](int q) {
        q = __builtin_amdgcn_readfirstlane(q);
#pragma unroll
        for (int j = 0; j < NT; j++) {
#pragma unroll
            for (int v = 0; v < 4; v++) w[j][v] = __builtin_amdgcn_raw_buffer_load_b128(rw, wo[j][v], 256 * q, 2);  // nontemporal
            if (F == W4A16 && p.gu > 1) {
#pragma unroll
                for (int v = 0; v < 4; v++)
                    sn[j][0][v] = __builtin_amdgcn_raw_buffer_load_b32(rs, so[j], 4 * ((4 * q + v) / p.gu), 0);
            } else {
#pragma unroll
                for (int d = 0; d < SD; d++) sn[j][d] = __builtin_amdgcn_raw_buffer_load_b128(rs, so[j], 16 * (SD * q + d), 0);
            }
        }
    };
    auto load_x = [&](int q, int v) {
        const int u = __builtin_amdgcn_readfirstlane(4 * q + v);
#pragma unroll
        for (int t = 0; t < 4; t++) x[v][t] = __builtin_amdgcn_raw_buffer_load_b128(rx, xo[t], 256 * u, 0);
    };
    // between a wave's own LDS writes and reads: its LDS operations run in
    // order, so only the compiler has to keep theirs
    auto order = [] { asm volatile("" ::: "memory"); };
    // IQ4_NL adds a block at a time: two chains of sums, half as long each
    float4v acc[NT], ac2[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) acc[j] = ac2[j] = (float4v){0.f, 0.f, 0.f, 0.f};
    bool odd = false;  // a W4A16 zero that is no whole number was seen
    if (kg < nq) {
        load_w(kg);
#pragma unroll
        for (int v = 0; v < 4; v++) load_x(kg, v);
    }
    for (int q = kg; q < nq; q += WK) {
        u32x4 sc[NT][SD];
        order();
#pragma unroll
        for (int j = 0; j < NT; j++) {
#pragma unroll
            for (int v = 0; v < 4; v++) *reinterpret_cast<u32x4*>(ws + j * 4096 + put[v]) = w[j][v];
#pragma unroll
            for (int d = 0; d < SD; d++) sc[j][d] = sn[j][d];
        }
        const bool more = q + WK < nq;
        if (more) load_w(q + WK);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            order();
#pragma unroll
            for (int t = 0; t < 4; t++) *reinterpret_cast<u32x4*>(xs + put[t]) = x[v][t];
            order();
            if (more) load_x(q + WK, v);
            __builtin_amdgcn_sched_barrier(0);
            if (4 * q + v < nu) {
                half8v ao[4];
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    const u32x4 o = *reinterpret_cast<const u32x4*>(xs + get[b]);
                    const u32x4 e = F == W4A16
                        ? nibble_order(o)
                        : (u32x4){__builtin_amdgcn_perm(o[1], o[0], 0x05040100u), __builtin_amdgcn_perm(o[3], o[2], 0x05040100u),
                                  __builtin_amdgcn_perm(o[1], o[0], 0x07060302u), __builtin_amdgcn_perm(o[3], o[2], 0x07060302u)};
                    ao[b] = __builtin_bit_cast(half8v, e);
                }
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    Raw r;
                    r.a = *reinterpret_cast<const u32x4*>(ws + j * 4096 + get[v]);
                    transpose4(r.a);
                    half2v z1 = splat2(0.f), z2 = z1;
                    float s = 0.f;
                    if constexpr (F == W4A16) {
                        const float z = h2f((uint16_t)(sc[j][0][v] >> 16)), zi = whole_zero(z);
                        z1 = splat2(-1024.0f - zi);
                        z2 = splat2(-64.0f - zi);
                        s = h2f((uint16_t)sc[j][0][v]);
                        odd |= z != zi;
                    } else {
#pragma unroll
                        for (int d = 0; d < 2; d++) r.s[d] = sc[j][v >> 1][2 * (v & 1) + d];
                    }
                    float4v d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int b = 0; b < 4; b++) {
                        half8v bo[PW];
                        decode<F>(r, b, 0, lg, z1, z2, bo);
                        if constexpr (F == W4A16) {
                            d = __builtin_amdgcn_mfma_f32_16x16x32_f16(ao[b], bo[0], d, 0, 0, 0);
                        } else {
                            d = __builtin_amdgcn_mfma_f32_16x16x32_f16(ao[b], bo[0], (float4v){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                            d = __builtin_amdgcn_mfma_f32_16x16x32_f16(ao[b], bo[PW - 1], d, 0, 0, 0);
                            const float t = block_scale<F>(r, b, 0);
#pragma unroll
                            for (int e = 0; e < 4; e++) {
                                float4v& sum = b & 1 ? ac2[j] : acc[j];
                                sum[e] = __builtin_fmaf(t, d[e], sum[e]);
                            }
                        }
                    }
                    if constexpr (F == W4A16) {
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[j][e] = __builtin_fmaf(s, d[e], acc[j][e]);
                    }
                }
            }
        }
    }
    if constexpr (F == W4A16) {
        // (after the walk: a branch in it, between an MFMA and the first use of
        // its result, compiled to a read of the result before it was there)
        // the rests of such zeros: s * rest * sum x off, a unit at a time (all-ones B operands give sum x)
        if (__builtin_expect(__any(odd), 0)) {
            const half2v one = splat2(1.0f);
            const half8v ones = join(one, one, one, one);
            const uint32_t xr = (uint32_t)min(li, p.T - 1) * (uint32_t)p.K * 2u + 16u * lg;
            for (int q = kg; q < nq; q += WK)
                for (int u = 4 * q; u < min(4 * q + 4, nu); u++) {
                    const int us = __builtin_amdgcn_readfirstlane(u);
                    float4v sx = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int b = 0; b < 4; b++)
                        sx = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            __builtin_bit_cast(half8v, __builtin_amdgcn_raw_buffer_load_b128(rx, xr + 64 * b, 256 * us, 0)),
                            ones, sx, 0, 0, 0);
#pragma unroll
                    for (int j = 0; j < NT; j++) {
                        const uint32_t v = __builtin_amdgcn_raw_buffer_load_b32(rs, so[j], 4 * (us / p.gu), 0);
                        const float z = h2f((uint16_t)(v >> 16)), m = -h2f((uint16_t)v) * (z - whole_zero(z));
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[j][e] = __builtin_fmaf(m, sx[e], acc[j][e]);
                    }
                }
        }
    }
    // the waves' sums, over the whole stage: every wave is past its last read of it
    __syncthreads();
    float* red = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) red[(kg * NT + j) * 256 + e * 64 + lane] = acc[j][e] + ac2[j][e];
    __syncthreads();
    for (int o = threadIdx.x; o < NT * 256; o += 64 * WK) {
        float sum = 0.0f;
#pragma unroll
        for (int g = 0; g < WK; g++) sum += red[g * (NT * 256) + o];
        const int ln = o & 63, tok = 4 * (ln >> 4) + ((o >> 6) & 3), row = n0 + (o >> 8) * 16 + (ln & 15);
        if (tok < p.T && row < p.rows) p.c[(long)tok * p.rows + row] = sum;
    }
}

template <Fmt F, int NT, int WK>
hipError_t launch_few(const WideArgs& a, hipStream_t st) {
    constexpr int shm = WK * 4096 * (1 + NT);
    if constexpr (shm > 65536) {
        static std::atomic<uint64_t> done{0};
        const hipError_t rc = raise_lds(reinterpret_cast<const void*>(&few_gemm_kernel<F, NT, WK>), shm, done);
        if (rc != hipSuccess) return rc;
    }
    few_gemm_kernel<F, NT, WK><<<ceil_div(a.rows, 16 * NT), 64 * WK, shm, st>>>(a);
    return hipGetLastError();
}

template <Fmt F, int P, int MT, int NT, int WN, int WK, bool FAR = far_sums(F)>
hipError_t launch_tile(const WideArgs& a, hipStream_t st) {
    constexpr int xb = 2 * WK * MT * steps_of(P) * P * 1024, rb = WK > 1 ? WK / 2 * WN * MT * NT * 1024 : 0;
    constexpr int shm = xb > rb ? xb : rb;
    if constexpr (shm > 65536) {
        static std::atomic<uint64_t> done{0};
        const hipError_t rc =
            raise_lds(reinterpret_cast<const void*>(&wide_gemm_kernel<F, P, MT, NT, WN, WK, FAR>), shm, done);
        if (rc != hipSuccess) return rc;
    }
    const long grid = (long)ceil_div(a.T, 16 * MT) * ceil_div(a.rows, 16 * NT * WN);
    wide_gemm_kernel<F, P, MT, NT, WN, WK, FAR><<<(int)grid, 64 * WN * WK, shm, st>>>(a);
    return hipGetLastError();
}

// The tile.  While one round of workgroups covers the matrix, its time is
// the chain of loads and barriers along K, so the smallest tile whose
// workgroups still fit the 256 CUs wins, with as many waves along K as the
// registers and LDS allow (16 waves against 8 in 64 x 128 tiles, K = 4096 /
// 14336, 512 tokens of 4096 rows: Q4_0 54 / 159 us against 61 / 179, W4A16 35
// / 91 against 37 / 106; Q6_K's decode and the second sums of IQ4_NL and Q5_0
// would spill there and stay at 8 waves).  Past one round the tile that
// feeds most MFMAs a decoded weight and stage wins, as long as its last round
// is full enough: 128 x 256 in 8 waves (14336 x 4096 rows x K, us against 64
// x 128 in 4 waves: 512 tokens W4A16 76 / 104, Q4_0 147 / 152, Q6_K 183 /
// 239; 1024 tokens 144 / 179, 235 / 274, 356 / 415).
template <Fmt F, int P>
hipError_t launch_gemm(const WideArgs& a, hipStream_t st) {
    auto tiles = [&](int tokens, int rows) { return (long)ceil_div(a.T, tokens) * ceil_div(a.rows, rows); };
    auto fits = [&](int tokens, int rows) { return tiles(tokens, rows) <= 256; };
    // whether rounds of 256 workgroups are at least this full on average
    auto full = [&](int tokens, int rows, double share) {
        const long t = tiles(tokens, rows);
        return (double)t >= share * 256.0 * (double)((t + 255) / 256);
    };
    constexpr bool KQ = has_mins(F);
    if (a.T <= 16 && fits(16, 32)) return launch_tile<F, P, 1, 2, 1, 8>(a, st);
    if (fits(32, 16)) return launch_tile<F, P, 2, 1, 1, 8>(a, st);
    if (fits(32, 32)) return launch_tile<F, P, 2, 2, 1, 8>(a, st);
    if (fits(32, 64)) return launch_tile<F, P, 2, 2, 2, 8>(a, st);
    if (fits(64, 64)) return launch_tile<F, P, 4, 2, 2, 4>(a, st);
    constexpr bool FS = far_sums(F);
    if constexpr (F == IQ4_NL && P == 2) {  // as the column kernel that fp32 tokens had: short chains
        if (a.K > kChain) return launch_tile<F, P, 4, 2, 2, 4>(a, st);
        return launch_tile<F, P, 4, 2, 4, 2>(a, st);
    }
    if (fits(64, 128)) return launch_tile<F, P, 4, 2, 4, F == Q6_K || FS ? 2 : 4>(a, st);
    // (two parts without minima: 64 x 256 tiles, two workgroups a CU, hold their rate below 128 x 256)
    if constexpr (P == 1 || KQ || F == Q6_K) {
        if constexpr (KQ) {
            if (a.K > 2 * kChain && fits(128, 128)) return launch_tile<F, P, 8, 2, 4, 2, true>(a, st);
        }
        if (fits(128, 128)) return launch_tile<F, P, 8, 2, 4, 2>(a, st);
    }
    if (full(128, 256, P == 1 || F == Q6_K ? 0.65 : 0.85)) {
        if constexpr (F != W4A16 && F != Q6_K && !FS) {
            if (a.K > kChain) return launch_tile<F, P, 8, 2, 8, 1, true>(a, st);
        }
        return launch_tile<F, P, 8, 2, 8, 1>(a, st);
    }
    if constexpr (F == Q5_0) {
        if (full(64, 256, 0.8)) return launch_tile<F, P, 4, 2, 8, 1>(a, st);
    } else if constexpr (!FS && F != W4A16 && F != Q6_K) {
        // as many waves along K as keep to kChain
        if (a.K > (KQ ? 1 : 2) * kChain) return launch_tile<F, P, 4, 2, 4, 4>(a, st);
        if constexpr (!KQ) {
            if (full(64, 256, 0.8)) return launch_tile<F, P, 4, 2, 8, 2>(a, st);
            if (a.K > kChain) return launch_tile<F, P, 4, 2, 4, 2>(a, st);
        }
    }
    return launch_tile<F, P, 4, 2, 4, 1>(a, st);
}

// One 16-row tile a wave and 8 waves along K while that gives the CUs one
// workgroup each, two tiles up to 8192 rows (8192 x 8192, 16 tokens, W4A16:
// 15.2 us, 19.8 with one tile), then shorter workgroups, several a CU (18944 x
// 3584 rows x K, 8 tokens, IQ4_NL: 23.9 us with 4 waves, 30.8 with 8).
template <Fmt F>
hipError_t launch_few_gemm(const WideArgs& a, hipStream_t st) {
    if (a.rows <= 4096) return launch_few<F, 1, 8>(a, st);
    if (a.rows <= 8192) return launch_few<F, 2, 8>(a, st);
    if (F == W4A16 && a.rows > 24576) return launch_few<F, 2, 2>(a, st);
    return launch_few<F, 1, 4>(a, st);
}

// Bytes of the packed activations of T tokens (whole 128-token tiles: the
// largest tile's reads stay inside), of the token scales and of the block sums.
long padded(int T) { return (long)(T + 127) / 128 * 128; }
long pack_bytes(int T, int K, int P) { return padded(T) * K * 2 * P; }
long inv_bytes(int T) { return padded(T) * 4; }
long sums_bytes(int T, int K) { return padded(T) / 16 * ((K + 1023) / 1024) * 3072; }

template <Order O, class XT, bool S, int NI>
void launch_pack(const WideArgs& a, const XT* x, hipStream_t st) {
    pack_kernel<O, XT, S, NI><<<a.T, kPackThreads, 0, st>>>(x, (uint4*)a.xp, (float*)a.inv, (uint16_t*)a.sums, a.K);
}

template <Fmt F, int P>
hipError_t launch_fmt(const WideArgs& a, const void* X, hipStream_t st) {
    constexpr Order O = order_of(F);
    constexpr bool S = has_mins(F);
    using XT = std::conditional_t<P == 2, float, uint16_t>;
    const XT* x = static_cast<const XT*>(X);
    if constexpr (P == 1) {
        if (a.T <= 16) {  // the activations as they are
            WideArgs b = a;
            b.xp = reinterpret_cast<const char*>(x);
            return launch_few_gemm<F>(b, st);
        }
    }
    const int ni = ceil_div(S ? (a.K + 1023) & ~1023 : a.K, 8 * kPackThreads);
    if (ni <= 1) launch_pack<O, XT, S, 1>(a, x, st);
    else if (ni <= 2) launch_pack<O, XT, S, 2>(a, x, st);
    else if (ni <= 4) launch_pack<O, XT, S, 4>(a, x, st);
    else launch_pack<O, XT, S, kPackOctets>(a, x, st);
    const hipError_t rc = hipGetLastError();
    return rc != hipSuccess ? rc : launch_gemm<F, P>(a, st);
}

// Sizes the path takes: whole 128-K units (256 for the super-blocks), a
// token's row in one workgroup's registers, 31-bit byte offsets of the bulk
// data, and 32-bit grids.
bool wide_ok(int fmt, int x_fp16, int rows, int K, int T) {
    if (fmt < 0 || fmt >= kFmts || rows <= 0 || T <= 0 || K <= 0) return false;
    const bool kq = fmt == Q4_K || fmt == Q5_K || fmt == Q6_K;
    if (K % (kq ? 256 : 128) != 0 || K > kPackThreads * kPackOctets * 8) return false;
    if (x_fp16 ? fmt != W4A16 && fmt != IQ4_NL : fmt == W4A16) return false;
    const long n = (long)rows * K;
    const long bulk = fmt == Q8_0 || fmt == Q8_GGUF ? n : fmt == Q4_K ? n / 256 * 144 : fmt == Q5_K ? n / 256 * 176 : n / 2;
    return bulk < 0x7fffffffL && (long)ceil_div(T, 16) * ceil_div(rows, 16) < 0x7fffffffL;
}

}  // namespace
}  // namespace zt

using namespace zt;

ZT_EXPORT long zt_gemm_wide_workspace_bytes(int fmt, int x_fp16, int rows, int K, int T) {
    if (!wide_ok(fmt, x_fp16, rows, K, T)) return -1;
    return pack_bytes(T, K, x_fp16 ? 1 : 2) + inv_bytes(T) + (has_mins((Fmt)fmt) ? sums_bytes(T, K) : 0);
}

ZT_EXPORT int zt_gemm_wide_f32(int fmt, const void* W, long offset1, long offset2, const uint32_t* szr, int group_size,
                               const void* X, int x_fp16, float* C, int rows, int K, int T, void* workspace,
                               long workspace_bytes, hipStream_t stream) {
    if (rows < 0 || K < 0 || T < 0) return (int)hipErrorInvalidValue;
    if (rows == 0 || T == 0) return (int)hipSuccess;
    const long need = zt_gemm_wide_workspace_bytes(fmt, x_fp16, rows, K, T);
    if (need < 0 || workspace_bytes < need || W == nullptr || X == nullptr || C == nullptr || workspace == nullptr)
        return (int)hipErrorInvalidValue;
    if (((uintptr_t)W | (uintptr_t)X | (uintptr_t)workspace | (uintptr_t)offset1 | (uintptr_t)offset2) & 15 ||
        ((uintptr_t)C & 3) || offset1 < 0 || offset2 < 0)
        return (int)hipErrorInvalidValue;
    WideArgs a{};
    a.c = C;
    a.rows = rows;
    a.K = K;
    a.T = T;
    a.gu = 1;
    a.xp = static_cast<char*>(workspace);
    a.inv = reinterpret_cast<const float*>(a.xp + pack_bytes(T, K, x_fp16 ? 1 : 2));
    a.sums = reinterpret_cast<const char*>(a.inv) + inv_bytes(T);
    const uint8_t* w = static_cast<const uint8_t*>(W);
    const long n = (long)rows * K, nb = n / 32, tb = n / 256;
    auto data = [&](const uint8_t* p, long bytes) { a.w = p; a.wb = (uint32_t)bytes; };
    auto scales = [&](const void* p, long bytes) { a.s = static_cast<const uint8_t*>(p); a.sb = (uint32_t)bytes; };
    auto bits = [&](const uint8_t* p, long bytes) { a.e = p; a.eb = (uint32_t)bytes; };
    hipError_t rc = hipErrorInvalidValue;
    switch (fmt) {
        case W4A16:
            if (szr == nullptr || ((uintptr_t)szr & 3) || group_size <= 0 || group_size % 128 != 0 || K % group_size != 0) break;
            data(w, n / 2);
            scales(szr, n / group_size * 4);
            a.gu = group_size / 128;
            rc = launch_fmt<W4A16, 1>(a, X, stream);
            break;
        case Q4_0:
            data(w + offset1, n / 2);
            scales(w, nb * 2);
            rc = launch_fmt<Q4_0, 2>(a, X, stream);
            break;
        case Q8_0:
            data(w + offset1, n);
            scales(w, nb * 4);
            rc = launch_fmt<Q8_0, 2>(a, X, stream);
            break;
        case Q8_GGUF:
            data(w + offset1, n);
            scales(w, nb * 2);
            rc = launch_fmt<Q8_GGUF, 2>(a, X, stream);
            break;
        case Q5_0:
            data(w + offset2, n / 2);
            scales(w, nb * 2);
            bits(w + offset1, nb * 4);
            rc = launch_fmt<Q5_0, 2>(a, X, stream);
            break;
        case Q4_K:
            data(w, tb * 144);
            rc = launch_fmt<Q4_K, 2>(a, X, stream);
            break;
        case Q5_K:
            data(w, tb * 176);
            rc = launch_fmt<Q5_K, 2>(a, X, stream);
            break;
        case Q6_K:
            data(w, tb * 128);
            bits(w + 128 * tb, tb * 64);
            scales(w + 192 * tb, tb * 16);
            a.d = w + 208 * tb;
            a.db = (uint32_t)(tb * 2);
            rc = launch_fmt<Q6_K, 2>(a, X, stream);
            break;
        default:  // IQ4_NL
            data(w + offset1, n / 2);
            scales(w, nb * 2);
            rc = x_fp16 ? launch_fmt<IQ4_NL, 1>(a, X, stream) : launch_fmt<IQ4_NL, 2>(a, X, stream);
    }
    return (int)rc;
}
