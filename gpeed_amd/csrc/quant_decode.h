// Decoders of the GGUF block formats, shared by the raw-row kernels. The
// unit is a 32-weight sub-block: every format's scales are constant over 16
// or 32 weights, so one lane decodes 32 weights with two scales at most.
// Each decoder mirrors the reference's block function (quant.cpp:165-502)
// operation for operation with FP contraction off, so every dequantized
// value is bit-identical to the CPU decode. The codebooks are expanded at
// compile time and copied into LDS by each workgroup.
#pragma once

#include "iq3_common.h"
#include "quant_grids.h"

#include <type_traits>

namespace gpeed {

namespace {

constexpr int kDtF32 = 0, kDtF16 = 1, kDtQ8_0 = 8, kDtQ2_K = 10, kDtQ3_K = 11, kDtQ6_K = 14, kDtIQ3_XXS = 18,
              kDtIQ3_S = 21, kDtIQ2_S = 22, kDtIQ4_XS = 23, kDtBF16 = 30;

struct Iq2sGrid { uint64_t v[1024]; };
struct Iq3sGrid { uint32_t v[512]; };
constexpr uint16_t kIq2sPacked[1024] = {GPEED_IQ2S_PACKED};
constexpr uint16_t kIq3sPacked[512] = {GPEED_IQ3S_PACKED};
constexpr uint8_t kIq2sLevel[3] = {GPEED_IQ2S_LEVELS};
constexpr int8_t kIq4nl[16] = {GPEED_IQ4NL_VALUES};

constexpr Iq2sGrid expand_iq2s() {
    Iq2sGrid g{};
    for (int i = 0; i < 1024; ++i) {
        uint64_t e = 0;
        for (int j = 0; j < 8; ++j) e |= (uint64_t)kIq2sLevel[(kIq2sPacked[i] >> (2 * j)) & 3] << (8 * j);
        g.v[i] = e;
    }
    return g;
}
constexpr Iq3sGrid expand_iq3s() {
    Iq3sGrid g{};
    for (int i = 0; i < 512; ++i) {
        uint32_t e = 0;
        for (int j = 0; j < 4; ++j) e |= (2u * ((kIq3sPacked[i] >> (3 * j)) & 7u) + 1u) << (8 * j);
        g.v[i] = e;
    }
    return g;
}
constexpr Iq2sGrid kIq2sGrid = expand_iq2s();
constexpr Iq3sGrid kIq3sGrid = expand_iq3s();

// Geometry (quant.cpp:52-114): weights per block, bytes per block. Scalar
// types are handled in 32-weight runs.
template <int DT> struct Fmt;
template <> struct Fmt<kDtF32> { static constexpr int kElems = 32, kBytes = 128; };
template <> struct Fmt<kDtF16> { static constexpr int kElems = 32, kBytes = 64; };
template <> struct Fmt<kDtBF16> { static constexpr int kElems = 32, kBytes = 64; };
template <> struct Fmt<kDtQ8_0> { static constexpr int kElems = 32, kBytes = 34; };
template <> struct Fmt<kDtQ2_K> { static constexpr int kElems = 256, kBytes = 84; };
template <> struct Fmt<kDtQ3_K> { static constexpr int kElems = 256, kBytes = 110; };
template <> struct Fmt<kDtQ6_K> { static constexpr int kElems = 256, kBytes = 210; };
template <> struct Fmt<kDtIQ3_XXS> { static constexpr int kElems = 256, kBytes = 98; };
template <> struct Fmt<kDtIQ3_S> { static constexpr int kElems = 256, kBytes = 110; };
template <> struct Fmt<kDtIQ2_S> { static constexpr int kElems = 256, kBytes = 82; };
template <> struct Fmt<kDtIQ4_XS> { static constexpr int kElems = 256, kBytes = 136; };

// Codebook copies in LDS (only the one the format uses is sized).
template <int DT>
struct Tables {
    static constexpr int kN = DT == kDtIQ2_S ? 1024 : DT == kDtIQ3_S ? 512 : DT == kDtIQ3_XXS ? 256 : 16;
    using T = typename std::conditional<DT == kDtIQ2_S, uint64_t, uint32_t>::type;
    T v[kN];
    __device__ void load(int tid, int nthreads) {
        for (int i = tid; i < kN; i += nthreads) {
            if constexpr (DT == kDtIQ2_S) v[i] = kIq2sGrid.v[i];
            else if constexpr (DT == kDtIQ3_S) v[i] = kIq3sGrid.v[i];
            else if constexpr (DT == kDtIQ3_XXS) v[i] = kIq3xxsGrid[i];
            else v[i] = (uint32_t)(int32_t)kIq4nl[i];
        }
    }
};

// Loads of block fields: blocks sit at 2-byte-aligned addresses (every
// block size is even). From LDS, wider fields are assembled from 16-bit
// loads; from global memory (WIDE) they are one load at that alignment.
typedef uint32_t u32_a2_t __attribute__((aligned(2)));
typedef u32x4_t u32x4_a2_t __attribute__((aligned(2)));
__device__ __forceinline__ uint32_t u8(const uint8_t* p) { return *p; }
__device__ __forceinline__ uint32_t u16(const uint8_t* p) { return *reinterpret_cast<const uint16_t*>(p); }
template <bool WIDE>
__device__ __forceinline__ uint32_t ld32(const uint8_t* p) {
    if constexpr (WIDE) return *reinterpret_cast<const u32_a2_t*>(p);
    else return u16(p) | (u16(p + 2) << 16);
}
// N words (a multiple of 4) from a 2-byte-aligned address
template <bool WIDE, int N>
__device__ __forceinline__ void ldwords(const uint8_t* p, uint32_t* w) {
    if constexpr (WIDE) {
#pragma unroll
        for (int i = 0; i < N / 4; ++i) {
            const u32x4_t v = reinterpret_cast<const u32x4_a2_t*>(p)[i];
#pragma unroll
            for (int k = 0; k < 4; ++k) w[4 * i + k] = v[k];
        }
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) w[i] = ld32<false>(p + 4 * i);
    }
}
__device__ __forceinline__ uint32_t byte_of(const uint32_t* w, int i) { return (w[i >> 2] >> (8 * (i & 3))) & 255u; }

// byte i of w as a float, one instruction (an integer subtraction folded into
// the conversion would take three)
template <int I>
__device__ __forceinline__ float ubyte_f32(uint32_t w) {
    float f;
    if constexpr (I == 0) asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(f) : "v"(w));
    else if constexpr (I == 1) asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(f) : "v"(w));
    else if constexpr (I == 2) asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(f) : "v"(w));
    else asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(f) : "v"(w));
    return f;
}
// y[0..3] = s * (byte - off)
__device__ __forceinline__ void scaled_bytes(uint32_t w, float off, float s, float* y) {
#pragma clang fp contract(off)
    y[0] = s * (ubyte_f32<0>(w) - off);
    y[1] = s * (ubyte_f32<1>(w) - off);
    y[2] = s * (ubyte_f32<2>(w) - off);
    y[3] = s * (ubyte_f32<3>(w) - off);
}

// The fields of one 32-weight sub-block in registers (layouts below).
template <int DT>
struct Sub {
    static constexpr int kWords = DT == kDtF32 ? 32 : DT == kDtF16 || DT == kDtBF16 ? 16 : DT == kDtQ8_0 ? 9
                                  : DT == kDtQ6_K ? 17 : DT == kDtQ2_K ? 10 : DT == kDtQ3_K ? 18 : DT == kDtIQ3_XXS ? 4
                                  : DT == kDtIQ2_S ? 3 : DT == kDtIQ3_S ? 4 : 6;
    uint32_t w[kWords];
};

// Loads the fields of weights 32*sb .. 32*sb+31 of the block at blk.
template <int DT, bool WIDE>
__device__ __forceinline__ void load_sub(const uint8_t* __restrict__ blk, int sb, Sub<DT>& r) {
    if constexpr (DT == kDtF32) {
#pragma unroll
        for (int i = 0; i < 32; ++i) r.w[i] = reinterpret_cast<const uint32_t*>(blk)[i];
    } else if constexpr (DT == kDtF16 || DT == kDtBF16) {
        ldwords<WIDE, 16>(blk, r.w);
    } else if constexpr (DT == kDtQ8_0) {
        // d (fp16), 32 int8 codes
        ldwords<WIDE, 8>(blk + 2, r.w);
        r.w[8] = u16(blk);
    } else if constexpr (DT == kDtQ6_K) {
        // ql[128] qh[64] sc[16] d; half h = sb/4, quarter q = sb%4: the
        // nibbles ql[64h + 32(q&1) ..], the top bits qh[32h ..], the scales
        // sc[8h + 2q], sc[8h + 2q + 1]
        const int h = sb >> 2, q = sb & 3;
        ldwords<WIDE, 8>(blk + 64 * h + 32 * (q & 1), r.w);
        ldwords<WIDE, 8>(blk + 128 + 32 * h, r.w + 8);
        r.w[16] = u16(blk + 192 + 8 * h + 2 * q) | (u16(blk + 208) << 16);
    } else if constexpr (DT == kDtQ2_K) {
        // scales[16] qs[64] d dmin; half h = sb/4, plane j = sb%4: codes
        // qs[32h ..], scale bytes scales[8h + 2j], scales[8h + 2j + 1]
        const int h = sb >> 2, j = sb & 3;
        ldwords<WIDE, 8>(blk + 16 + 32 * h, r.w);
        r.w[8] = u16(blk + 8 * h + 2 * j);
        r.w[9] = ld32<WIDE>(blk + 80);
    } else if constexpr (DT == kDtQ3_K) {
        // hmask[32] qs[64] scales[12] d; h = sb/4, j = sb%4: codes qs[32h ..],
        // hmask; scales 8h + 2j and the next: low bits in bytes 2j, 2j + 1 of
        // the first eight, top bits in bytes 8 + (2j & 2) and the next
        const int h = sb >> 2, j = sb & 3;
        ldwords<WIDE, 8>(blk + 32 + 32 * h, r.w);
        ldwords<WIDE, 8>(blk, r.w + 8);
        r.w[16] = u16(blk + 96 + 2 * j) | (u16(blk + 104 + (2 * j & 2)) << 16);
        r.w[17] = u16(blk + 108);
    } else if constexpr (DT == kDtIQ3_XXS) {
        // d, qs[64] grid indices, 8 words of 4 x 7 sign bits + 4-bit scale
        r.w[0] = u16(blk);
        r.w[1] = ld32<WIDE>(blk + 66 + 4 * sb);
        r.w[2] = ld32<WIDE>(blk + 2 + 8 * sb);
        r.w[3] = ld32<WIDE>(blk + 6 + 8 * sb);
    } else if constexpr (DT == kDtIQ2_S) {
        // d, qs[32] grid low bytes, signs[32], qh[8], scales[8]
        r.w[0] = u16(blk) | (u8(blk + 66 + sb) << 16) | (u8(blk + 74 + sb) << 24);
        r.w[1] = ld32<WIDE>(blk + 2 + 4 * sb);
        r.w[2] = ld32<WIDE>(blk + 34 + 4 * sb);
    } else if constexpr (DT == kDtIQ3_S) {
        // d, qs[64], qh[8], signs[32], scales[4]
        r.w[0] = u16(blk) | (u8(blk + 66 + sb) << 16) | (u8(blk + 106 + (sb >> 1)) << 24);
        r.w[1] = ld32<WIDE>(blk + 2 + 8 * sb);
        r.w[2] = ld32<WIDE>(blk + 6 + 8 * sb);
        r.w[3] = ld32<WIDE>(blk + 74 + 4 * sb);
    } else if constexpr (DT == kDtIQ4_XS) {
        // d, scales_h (u16), scales_l[4], qs[128]
        r.w[0] = ld32<WIDE>(blk);
        r.w[1] = u8(blk + 4 + (sb >> 1));
        ldwords<WIDE, 4>(blk + 8 + 16 * sb, r.w + 2);
    }
}

// decode_sub: the 32 weights of a loaded sub-block (sb: its index in its
// block) into y. Each formula restates the reference's block function for
// those weights; the comment gives its lines. ds multiplies the block's
// scales: 1 gives the reference's values bit for bit, another power of two
// those values scaled by it (exactly, short of overflow and underflow).
template <int DT>
__device__ __forceinline__ void decode_sub(const Sub<DT>& r, int sb, const Tables<DT>& tb, float ds, float (&y)[32]) {
#pragma clang fp contract(off)
    if constexpr (DT == kDtF32) {
        // quant.cpp:528-531: a copy
#pragma unroll
        for (int i = 0; i < 32; ++i) y[i] = __uint_as_float(r.w[i]) * ds;
    } else if constexpr (DT == kDtF16 || DT == kDtBF16) {
        // quant.cpp:532-545 (f16_to_f32 :130-154, bf16_to_f32 :156-161); the
        // hardware fp16 conversion is exact (subnormals included)
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            const uint32_t h = (r.w[i >> 1] >> (16 * (i & 1))) & 0xFFFFu;
            y[i] = (DT == kDtF16 ? (float)__builtin_bit_cast(_Float16, (uint16_t)h) : __uint_as_float(h << 16)) * ds;
        }
    } else if constexpr (DT == kDtQ8_0) {
        // quant.cpp:165-184: y = d * q
        const float d = f16_bits_to_f32(r.w[8]) * ds;
#pragma unroll
        for (int i = 0; i < 32; ++i) y[i] = d * (float)(int8_t)byte_of(r.w, i);
    } else if constexpr (DT == kDtQ6_K) {
        // quant.cpp:212-306: weight l < 32 takes the low (q < 2) or high
        // nibble and bits 2q of the top-bit byte, scale l/16 of the two;
        // y = (d * sc) * (v - 32).
        const int q = sb & 3;
        const float d = f16_bits_to_f32(r.w[16] >> 16) * ds;
        const float ds0 = d * (float)(int8_t)(r.w[16] & 255u);
        const float ds1 = d * (float)(int8_t)((r.w[16] >> 8) & 255u);
        // (four codes a word; a byte converts to float32 in one instruction)
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const uint32_t c = ((r.w[k] >> (2 * q & 4)) & 0x0F0F0F0Fu) | (((r.w[8 + k] >> (2 * q)) & 0x03030303u) << 4);
            scaled_bytes(c, 32.0f, k < 4 ? ds0 : ds1, y + 4 * k);
        }
    } else if constexpr (DT == kDtQ2_K) {
        // quant.cpp:309-335: weight l < 32: code (qs[l] >> 2j) & 3, scale
        // byte l/16 of the two; y = (d * (sc & 15)) * code - dmin * (sc >> 4).
        const int j = sb & 3;
        const float d = f16_bits_to_f32(r.w[9] & 0xFFFFu) * ds;
        const float mn = f16_bits_to_f32(r.w[9] >> 16) * ds;
        const uint32_t s0 = r.w[8] & 255u, s1 = r.w[8] >> 8;
        const float dl0 = d * (float)(s0 & 15u), ml0 = mn * (float)(s0 >> 4);
        const float dl1 = d * (float)(s1 & 15u), ml1 = mn * (float)(s1 >> 4);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const uint32_t cw = (r.w[k] >> (2 * j)) & 0x03030303u;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float c = (float)((cw >> (8 * i)) & 255u);
                y[4 * k + i] = k < 4 ? dl0 * c - ml0 : dl1 * c - ml1;
            }
        }
    } else if constexpr (DT == kDtQ3_K) {
        // quant.cpp:337-370: weight l < 32: code (qs[l] >> 2j) & 3, minus 4
        // where bit 4h + j of hmask[l] is clear; 6-bit scale k = 8h + 2j +
        // l/16 (low nibble of byte k, or high nibble of byte k-8 for k >= 8;
        // top bits from byte 8 + k%4 at 2*(k/4)); y = (d * (scale - 32)) *
        // value.
        const int h = sb >> 2, j = sb & 3;
        const float d = f16_bits_to_f32(r.w[17]) * ds;
        float dl[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int k = 8 * h + 2 * j + s;
            const uint32_t lb = (r.w[16] >> (8 * s)) & 255u;
            const uint32_t low = h == 0 ? lb & 15u : lb >> 4;
            const uint32_t top = (((r.w[16] >> (16 + 8 * s)) & 255u) >> (2 * (k >> 2))) & 3u;
            dl[s] = d * (float)((int)(int8_t)(uint8_t)(low | (top << 4)) - 32);
        }
        // (code + 4 hmask bit, four a word, less 4 as floats: exact)
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const uint32_t c = ((r.w[k] >> (2 * j)) & 0x03030303u) | (((r.w[8 + k] >> (4 * h + j)) & 0x01010101u) << 2);
            scaled_bytes(c, 4.0f, dl[k >> 2], y + 4 * k);
        }
    } else if constexpr (DT == kDtIQ3_XXS) {
        // quant.cpp:186-210: the eighth sign of a group makes the parity
        // even. y = ((d * (0.5 + s)) * 0.5) * grid * sign.
        const float d = f16_bits_to_f32(r.w[0]) * ds;
        const uint32_t aux = r.w[1];
        const float db = d * (0.5f + (float)(aux >> 28)) * 0.5f;
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            const uint32_t qq = (r.w[2 + (l >> 1)] >> (16 * (l & 1))) & 0xFFFFu;
            const uint32_t s7 = (aux >> (7 * l)) & 127u;
            const uint32_t sg = s7 | ((__builtin_popcount(s7) & 1u) << 7);
            const uint32_t g1 = tb.v[qq & 255u], g2 = tb.v[qq >> 8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t gv = ((e < 4 ? g1 : g2) >> (8 * (e & 3))) & 255u;
                y[8 * l + e] = db * (float)gv * (((sg >> e) & 1u) ? -1.0f : 1.0f);
            }
        }
    } else if constexpr (DT == kDtIQ2_S) {
        // quant.cpp:373-418: group l < 4: index qs[4sb + l] | bits 2l, 2l+1
        // of qh[sb] as bits 8-9; scale nibble (low for l < 2) of scales[sb];
        // y = ((d * (0.5 + s)) * 0.25) * grid * sign, sign bit e of
        // signs[4sb + l].
        const float d = f16_bits_to_f32(r.w[0] & 0xFFFFu) * ds;
        const uint32_t qh = (r.w[0] >> 16) & 255u, sc = r.w[0] >> 24;
        const float db0 = d * (0.5f + (float)(sc & 15u)) * 0.25f;
        const float db1 = d * (0.5f + (float)(sc >> 4)) * 0.25f;
        const uint32_t qs = r.w[1], sg = r.w[2];
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            const uint32_t idx = ((qs >> (8 * l)) & 255u) | ((qh << (8 - 2 * l)) & 0x300u);
            const uint64_t g = tb.v[idx];
            const uint32_t s = sg >> (8 * l);
            const float dl = l < 2 ? db0 : db1;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                y[8 * l + e] = dl * (float)(uint32_t)((g >> (8 * e)) & 255u) * (((s >> e) & 1u) ? -1.0f : 1.0f);
        }
    } else if constexpr (DT == kDtIQ3_S) {
        // quant.cpp:421-482: group l < 4: indices qs[8sb + 2l], qs[8sb + 2l +
        // 1] with bit 8 from bits 2l and 2l+1 of qh[sb]; scale nibble of
        // scales[sb/2] (low for even sb); y = (d * (1 + 2s)) * grid * sign,
        // sign bit e of signs[4sb + l].
        const float d = f16_bits_to_f32(r.w[0] & 0xFFFFu) * ds;
        const uint32_t qh = (r.w[0] >> 16) & 255u;
        const uint32_t scb = r.w[0] >> 24;
        const float db = d * (1.0f + 2.0f * (float)((sb & 1) ? scb >> 4 : scb & 15u));
        const uint32_t sg = r.w[3];
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            const uint32_t qq = (r.w[1 + (l >> 1)] >> (16 * (l & 1))) & 0xFFFFu;
            const uint32_t i1 = (qq & 255u) | ((qh << (8 - 2 * l)) & 256u);
            const uint32_t i2 = (qq >> 8) | ((qh << (7 - 2 * l)) & 256u);
            const uint32_t g1 = tb.v[i1], g2 = tb.v[i2];
            const uint32_t s = sg >> (8 * l);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t gv = ((e < 4 ? g1 : g2) >> (8 * (e & 3))) & 255u;
                y[8 * l + e] = db * (float)gv * (((s >> e) & 1u) ? -1.0f : 1.0f);
            }
        }
    } else if constexpr (DT == kDtIQ4_XS) {
        // quant.cpp:485-502: 6-bit scale = nibble sb%2 of scales_l[sb/2] |
        // bits 2sb, 2sb+1 of scales_h << 4; weight i < 16 is the low nibble
        // of qs[16sb + i], weight 16 + i its high nibble;
        // y = (d * (ls - 32)) * level[code].
        const float d = f16_bits_to_f32(r.w[0] & 0xFFFFu) * ds;
        const uint32_t sh = r.w[0] >> 16;
        const int ls = (int)(((r.w[1] >> (4 * (sb & 1))) & 15u) | (((sh >> (2 * sb)) & 3u) << 4));
        const float dl = d * (float)(ls - 32);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const uint32_t b = (r.w[2 + (i >> 2)] >> (8 * (i & 3))) & 255u;
            y[i] = dl * (float)(int32_t)tb.v[b & 15u];
            y[16 + i] = dl * (float)(int32_t)tb.v[b >> 4];
        }
    }
}

// Weights 32*sb .. 32*sb+31 of the block at blk, as the reference decodes them.
template <int DT>
__device__ __forceinline__ void decode32(const uint8_t* __restrict__ blk, int sb, const Tables<DT>& tb, float (&y)[32]) {
    Sub<DT> r;
    load_sub<DT, false>(blk, sb, r);
    decode_sub<DT>(r, sb, tb, 1.0f, y);
}

// Sub-blocks per block and the sub-block's block address.
template <int DT>
__device__ __forceinline__ const uint8_t* sub_block(const uint8_t* row, long long sbi, int& sb) {
    constexpr int kSub = Fmt<DT>::kElems / 32;
    sb = (int)(sbi % kSub);
    return row + (size_t)(sbi / kSub) * Fmt<DT>::kBytes;
}

}  // namespace

}  // namespace gpeed
