// W4 weight decode shared by the GEMV engine (mdx_gemv.hip) and the many-row GEMM (mdx_gemm.hip): the code tables
// of a group scale and the table lookups of a chunk's code dwords (16 columns x 128 k, tile-major nibble order).
#pragma once

#include "mdx_common.hpp"

namespace mdx {

struct Lut {
    uint32_t w[4];
};

__device__ __forceinline__ Lut make_lut(float s, const float* cb) {
    Lut L;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        uint32_t v = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const float r = rintf(__fmul_rn(cb[d * 4 + b], s));
            const int q = (r != r) ? 0 : int(fminf(fmaxf(r, -127.f), 127.f));
            v |= (uint32_t(q) & 0xFFu) << (8 * b);
        }
        L.w[d] = v;
    }
    return L;
}

// The default codebook's 16-byte table from its magnitudes (make_lut_c8's bytes): byte reversal and
// a carry-free negation of four int8 at once (~b + 1 per byte; no byte is -128 after the clamp).
__device__ __forceinline__ Lut lut_from_q8(uint32_t qa, uint32_t qb) {
    auto neg4 = [](uint32_t b) {
        const uint32_t n = ~b;
        return ((n & 0x7F7F7F7Fu) + 0x01010101u) ^ (n & 0x80808080u);
    };
    Lut L;
    L.w[0] = neg4(__builtin_amdgcn_perm(0u, qb, 0x00010203u));  // -q8, -q7, -q6, -q5
    L.w[1] = neg4(__builtin_amdgcn_perm(0u, qa, 0x00010203u));  // -q4 .. -q1
    L.w[2] = __builtin_amdgcn_perm(0u, qa, 0x0201000Cu);        // 0, q1, q2, q3
    L.w[3] = __builtin_amdgcn_perm(qb, qa, 0x06050403u);        // q4 .. q7
    return L;
}

// The table of the default codebook (c - 8) from its eight magnitudes: rint and the clamp are odd
// functions and (-k) s = -(k s) exactly, so entry 8 - k is the negation of q(k s) = clamp(rint(k s),
// +-127) (NaN -> 0) and entry 8 is 0 (0 * s rounds to 0, or is NaN -> 0): eight products instead of
// sixteen, the same bytes as make_lut.
__device__ __forceinline__ Lut make_lut_c8(float s) {
    if (__builtin_amdgcn_ballot_w64(!(fabsf(s) <= 15.875f)) == 0) {
        // every |k s| of the active lanes at most 127 (no NaN): fl32(k s) + 1.5 2^23 rounds to an integer once more, to
        // nearest even as rint does, and holds it in its low byte: two instructions per magnitude and no clamp (the tables
        // that lanes build per chunk: f32 scales per 32, 8 rows, 12288 x 4096 15.0 -> 13.2 us, 4096 x 12288 15.5 -> 13.8)
        uint32_t u[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) u[k] = __float_as_uint(__fadd_rn(__fmul_rn(float(k + 1), s), 12582912.f));
        auto four = [](uint32_t b0, uint32_t b1, uint32_t b2, uint32_t b3) {
            return __builtin_amdgcn_perm(__builtin_amdgcn_perm(b3, b2, 0x0C0C0400u), __builtin_amdgcn_perm(b1, b0, 0x0C0C0400u), 0x05040100u);
        };
        return lut_from_q8(four(u[0], u[1], u[2], u[3]), four(u[4], u[5], u[6], u[7]));
    }
    int q[9];
    q[0] = 0;
#pragma unroll
    for (int k = 1; k <= 8; ++k) {
        const float r = rintf(__fmul_rn(float(k), s));
        q[k] = (r != r) ? 0 : int(fminf(fmaxf(r, -127.f), 127.f));
    }
    auto pk = [](int b0, int b1, int b2, int b3) {
        return (uint32_t(b0) & 0xFFu) | ((uint32_t(b1) & 0xFFu) << 8) | ((uint32_t(b2) & 0xFFu) << 16) | (uint32_t(b3) << 24);
    };
    Lut L;
    L.w[0] = pk(-q[8], -q[7], -q[6], -q[5]);
    L.w[1] = pk(-q[4], -q[3], -q[2], -q[1]);
    L.w[2] = pk(0, q[1], q[2], q[3]);
    L.w[3] = pk(q[4], q[5], q[6], q[7]);
    return L;
}

// The eight magnitudes q(k s), k = 1..8, of the default codebook's table as int8 bytes (q1..q4, q5..q8).
__device__ __forceinline__ uint2 make_q8(float s) {
    uint32_t w[2] = {0u, 0u};
#pragma unroll
    for (int k = 1; k <= 8; ++k) {
        const float r = rintf(__fmul_rn(float(k), s));
        const int q = (r != r) ? 0 : int(fminf(fmaxf(r, -127.f), 127.f));
        w[(k - 1) >> 2] |= (uint32_t(q) & 0xFFu) << (8 * ((k - 1) & 3));
    }
    return make_uint2(w[0], w[1]);
}

// make_q8 for an fp16 scale |s| <= 127 / 8 (bits & 0x7FFF <= 0x4BF0; every fp16-ratio GPTQ scale): four packed
// half-precision FMAs k s + 1536 (k = 1..8). Each forms k s exactly and rounds once; in [1024, 2048) the
// spacing of half precision is 1, so the result is 1536 + rint(k s) (ties to even, 1536 being even), and
// its low byte is rint(k s) as int8. |k s| <= 127: no clamp. Two byte permutes gather the eight bytes.
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
constexpr uint32_t F16_FAST_MAX = 0x4BF0u;  // fp16 15.875

__device__ __forceinline__ uint2 make_q8_f16(uint32_t sbits) {
    const half2_t s2 = __builtin_bit_cast(half2_t, sbits | (sbits << 16));
    const half2_t magic = {(_Float16)1536.0f, (_Float16)1536.0f};
    uint32_t r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const half2_t kk = {(_Float16)float(2 * i + 1), (_Float16)float(2 * i + 2)};
        r[i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(kk, s2, magic));
    }
    return make_uint2(__builtin_amdgcn_perm(r[1], r[0], 0x06040200u), __builtin_amdgcn_perm(r[3], r[2], 0x06040200u));
}

// four codes (one per byte, values 0..15) -> four int8 via the 16-byte table
__device__ __forceinline__ uint32_t lut4(const Lut& L, uint32_t c) {
    const uint32_t sel = c & 0x07070707u;
    const uint32_t lo = __builtin_amdgcn_perm(L.w[1], L.w[0], sel);
    const uint32_t hi = __builtin_amdgcn_perm(L.w[3], L.w[2], sel);
    const uint32_t pick = ((c >> 1) & 0x04040404u) | 0x03020100u;
    return __builtin_amdgcn_perm(hi, lo, pick);
}

// per-weight decode of one chunk's four code dwords (two scales: dwords 0-1 and 2-3; one when the
// group spans the lane's 32 k, `one`, uniform); cbdef (uniform): the default codebook c - 8
__device__ __forceinline__ void decode_exact(const uint32_t* wd, float s0, float s1, bool one, bool cbdef,
                                             const float* cb, uint32_t* lo, uint32_t* hi) {
    const Lut L0 = cbdef ? make_lut_c8(s0) : make_lut(s0, cb);
    Lut L1 = L0;
    if (!one) L1 = (__float_as_uint(s1) == __float_as_uint(s0)) ? L0 : (cbdef ? make_lut_c8(s1) : make_lut(s1, cb));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const Lut& L = j < 2 ? L0 : L1;
        lo[j] = lut4(L, wd[j] & 0x0F0F0F0Fu);
        hi[j] = lut4(L, (wd[j] >> 4) & 0x0F0F0F0Fu);
    }
}

// per-weight decode of one chunk's four code dwords through one table (a group spans the chunk)
// (q8: T holds the default codebook's eight magnitudes in .x, .y)
__device__ __forceinline__ void decode_tbl(const uint32_t* wd, const uint4 T, bool q8, uint32_t* lo, uint32_t* hi) {
    Lut L;
    if (q8) {
        L = lut_from_q8(T.x, T.y);
    } else {
        L.w[0] = T.x;
        L.w[1] = T.y;
        L.w[2] = T.z;
        L.w[3] = T.w;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        lo[j] = lut4(L, wd[j] & 0x0F0F0F0Fu);
        hi[j] = lut4(L, (wd[j] >> 4) & 0x0F0F0F0Fu);
    }
}

// The table-only decode of one chunk's four code dwords (tile-major nibble order: k 8j..8j+3 in the low
// nibbles of dword j, k 8j+4..8j+7 in the high ones). Per four codes: the byte selectors (c & 7) index
// both 8-byte halves of the table by v_perm_b32, and a third v_perm_b32 picks per byte by bit 3 of the
// code (selector i or 4 + i, built by one bitop3 from the shifted codes): 13 VALU per code dword.
// Q8: T.x, T.y hold the default codebook's eight magnitudes (expanded once per chunk).
template <bool Q8>
__device__ __forceinline__ void decode_tb(const uint4 w, const uint4 T, uint32_t* lo, uint32_t* hi) {
    Lut L;
    if (Q8) {
        L = lut_from_q8(T.x, T.y);
    } else {
        L.w[0] = T.x;
        L.w[1] = T.y;
        L.w[2] = T.z;
        L.w[3] = T.w;
    }
    const uint32_t wd[4] = {w.x, w.y, w.z, w.w};
    const uint32_t m4 = 0x04040404u, id = 0x03020100u;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t v = wd[j];
        const uint32_t sl = v & 0x07070707u, sh = (v >> 4) & 0x07070707u;
        // (a & b) | c: bitop3 truth table 0xEA (index 4 a + 2 b + c)
        const uint32_t pl = __builtin_amdgcn_bitop3_b32(v >> 1, m4, id, 0xEA);
        const uint32_t ph = __builtin_amdgcn_bitop3_b32(v >> 5, m4, id, 0xEA);
        lo[j] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(L.w[3], L.w[2], sl), __builtin_amdgcn_perm(L.w[1], L.w[0], sl), pl);
        hi[j] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(L.w[3], L.w[2], sh), __builtin_amdgcn_perm(L.w[1], L.w[0], sh), ph);
    }
}

// decode_tb with a table per half chunk (T0: the lane's first 16 k, dwords 0-1; T1: dwords 2-3)
__device__ __forceinline__ void decode_tb2(const uint4 w, const uint4 T0, const uint4 T1, uint32_t* lo, uint32_t* hi) {
    const uint32_t wd[4] = {w.x, w.y, w.z, w.w};
    const uint32_t m4 = 0x04040404u, id = 0x03020100u;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint4 T = j < 2 ? T0 : T1;
        const uint32_t v = wd[j];
        const uint32_t sl = v & 0x07070707u, sh = (v >> 4) & 0x07070707u;
        const uint32_t pl = __builtin_amdgcn_bitop3_b32(v >> 1, m4, id, 0xEA);  // (decode_tb)
        const uint32_t ph = __builtin_amdgcn_bitop3_b32(v >> 5, m4, id, 0xEA);
        lo[j] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(T.w, T.z, sl), __builtin_amdgcn_perm(T.y, T.x, sl), pl);
        hi[j] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(T.w, T.z, sh), __builtin_amdgcn_perm(T.y, T.x, sh), ph);
    }
}

template <int SDT>
__device__ __forceinline__ float rd_scale(const uint8_t* p) {
    if (SDT == MDX_DT_F32) return *reinterpret_cast<const float*>(p);
    if (SDT == MDX_DT_F16) return fp16_to_f32(*reinterpret_cast<const uint16_t*>(p));
    return fp8_to_f32(*p);
}

}  // namespace mdx
