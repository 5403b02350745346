// Weight units decoded in registers to f16 MFMA fragments, shared by the
// few-row kernel (skinny.hip) and the panel GEMM (panel.hip).
#pragma once
#include "formats.h"
#include "matmul.h"

namespace oco {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f16x2 f16_pair(uint32_t bits) {
    f16x2 h;
    __builtin_memcpy(&h, &bits, 4);
    return h;
}

// Two f32 as a pair of f16 (round to nearest even).  The empty asm keeps the
// compiler from folding a fused multiply-add and this conversion into the
// slower mixed-precision form; the conversion itself is left to the compiler,
// which then sees every register that feeds a matrix instruction.
__device__ __forceinline__ uint32_t pk_f16(float a, float b) {
    asm("" : "+v"(a));
    asm("" : "+v"(b));
    return f16_bits(a, b);
}
// Four f16 of a * code - m from the bytes of one dword (a * code exact in f32).
__device__ __forceinline__ void four_ub(uint32_t n, float a, float m, uint32_t &p01, uint32_t &p23) {
    const float f0 = __builtin_fmaf(a, ub(n, 0), -m), f1 = __builtin_fmaf(a, ub(n, 1), -m);
    const float f2 = __builtin_fmaf(a, ub(n, 2), -m), f3 = __builtin_fmaf(a, ub(n, 3), -m);
    p01 = pk_f16(f0, f1);
    p23 = pk_f16(f2, f3);
}

// Buffer loads at any byte offset, zero past the resource's range.
struct RowSrc {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ uint32_t u16(uint32_t o) const { return __builtin_amdgcn_raw_buffer_load_b16(r, o, 0, 0); }
    __device__ __forceinline__ uint32_t u32(uint32_t o) const { return __builtin_amdgcn_raw_buffer_load_b32(r, o, 0, 0); }
    __device__ __forceinline__ u32x2 u64(uint32_t o) const { return __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, 0); }
    __device__ __forceinline__ u32x4 u128(uint32_t o) const { return __builtin_amdgcn_raw_buffer_load_b128(r, o, 0, 0); }
};
constexpr uint32_t UNIT_OFF = 0x80000000u;  // past every range: reads zero without touching memory

// A lane's quarter q of one row's 256-column unit: 64 weights as eight runs
// of eight consecutive columns (col(q, i) within the unit).
//   UNIT   bytes of a whole unit; load(src, row offset + unit offset, columns
//          left in the row from the unit's start);
//   prep   once per unit; run(i) the i-th run as four dwords of f16.
template <int FMT>
struct WeightUnit;

template <int FMT>
struct WeightK4 {  // Q4_K, Q5_K: quarter q = sub-blocks 2q (runs 0-3) and 2q + 1 (runs 4-7)
    static constexpr bool Q5 = FMT == OCO_Q5_K;
    static constexpr uint32_t UNIT = Q5 ? 176 : 144;
    u32x4 hdr, c0, c1, h0, h1;
    float a0, m0, a1, m1;
    uint32_t q;
    __device__ __forceinline__ static uint32_t col(uint32_t q, int i) { return 64 * q + 8 * i; }
    __device__ __forceinline__ void load(const RowSrc &s, uint32_t o, uint32_t q_, uint32_t) {
        hdr = s.u128(o);
        c0 = s.u128(o + UNIT - 128 + 32 * q_);
        c1 = s.u128(o + UNIT - 128 + 32 * q_ + 16);
        if constexpr (Q5) {
            h0 = s.u128(o + 16);
            h1 = s.u128(o + 32);
        }
    }
    __device__ __forceinline__ void prep(uint32_t q_) {
        q = q_;
        const float d = half_bits_to_f32(hdr.x & 0xffffu), dmin = half_bits_to_f32(hdr.x >> 16);
        // bytes s0 .. s3 = hdr.y, s4 .. s7 = hdr.z, s8 .. s11 = hdr.w; sub-blocks 2q, 2q + 1
        const uint32_t sh = 16 * (q & 1);
        uint32_t sc, mn;
        if (q < 2) {
            sc = (hdr.y >> sh) & 0x3f3fu;
            mn = (hdr.z >> sh) & 0x3f3fu;
        } else {
            const uint32_t t = hdr.w >> sh;
            sc = (t & 0x0f0fu) | ((hdr.y >> sh) >> 2 & 0x3030u);
            mn = (t >> 4 & 0x0f0fu) | ((hdr.z >> sh) >> 2 & 0x3030u);
        }
        a0 = d * (float)(sc & 0xffu);
        a1 = d * (float)(sc >> 8);
        m0 = dmin * (float)(mn & 0xffu);
        m1 = dmin * (float)(mn >> 8);
    }
    __device__ __forceinline__ void run(int i, uint32_t *out) const {
        const u32x4 c = (i & 2) ? c1 : c0;
        const u32x4 h = (i & 2) ? h1 : h0;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t w = c[2 * (i & 1) + j];
            uint32_t n = (i < 4 ? w : w >> 4) & 0x0f0f0f0fu;
            const float a = i < 4 ? a0 : a1, m = i < 4 ? m0 : m1;
            if constexpr (Q5) {
                n |= ((h[2 * (i & 1) + j] >> (2 * q + (i >= 4))) & 0x01010101u) << 4;
                four_ub(n, a, m, out[2 * j], out[2 * j + 1]);
            } else {
                q4_four(n, a, m, out[2 * j], out[2 * j + 1]);
            }
        }
    }
};
template <>
struct WeightUnit<OCO_Q4_K> : WeightK4<OCO_Q4_K> {};
template <>
struct WeightUnit<OCO_Q5_K> : WeightK4<OCO_Q5_K> {};

// Q6_K: half h = q / 2, quarters p = q % 2 (runs 0-3, low nibbles) and p + 2
// (runs 4-7, high nibbles) of it.
template <>
struct WeightUnit<OCO_Q6_K> {
    static constexpr uint32_t UNIT = 210;
    u32x4 l0, l1, h0, h1;
    u32x2 sc;
    uint32_t db;
    float s[4];
    uint32_t p;
    __device__ __forceinline__ static uint32_t col(uint32_t q, int i) { return 128 * (q >> 1) + 32 * (q & 1) + 64 * (i >> 2) + 8 * (i & 3); }
    __device__ __forceinline__ void load(const RowSrc &r, uint32_t o, uint32_t q, uint32_t) {
        l0 = r.u128(o + 32 * q);
        l1 = r.u128(o + 32 * q + 16);
        h0 = r.u128(o + 128 + 32 * (q >> 1));
        h1 = r.u128(o + 128 + 32 * (q >> 1) + 16);
        sc = r.u64(o + 192 + 8 * (q >> 1));
        db = r.u16(o + 208);
    }
    __device__ __forceinline__ void prep(uint32_t q) {
        p = q & 1;
        const float d = 0.25f * half_bits_to_f32(db);  // run() takes four times the codes
        const uint32_t a = sc.x >> (16 * p), b = sc.y >> (16 * p);
        s[0] = d * (float)(int8_t)(a & 0xffu);
        s[1] = d * (float)(int8_t)(a >> 8 & 0xffu);
        s[2] = d * (float)(int8_t)(b & 0xffu);
        s[3] = d * (float)(int8_t)(b >> 8 & 0xffu);
    }
    __device__ __forceinline__ void run(int i, uint32_t *out) const {
        const u32x4 l = (i & 2) ? l1 : l0, h = (i & 2) ? h1 : h0;
        const float sv = s[i >> 1];  // 16 columns a scale
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t w = l[2 * (i & 1) + j], x = h[2 * (i & 1) + j];
            // 4 (code - 32) as signed bytes (the code's top bit inverted is
            // the sign), so that s / 4 times them is the reference's s * (code -
            // 32), exact in f32, an infinite scale included: s * code - 32 s
            // would be Inf - Inf there.
            const uint32_t lo = (i < 4 ? w << 2 : w >> 2) & 0x3c3c3c3cu;
            const uint32_t hi = (i < 4 ? x << (6 - 2 * p) : x << (2 - 2 * p)) & 0xc0c0c0c0u;
            const uint32_t c = (lo | hi) ^ 0x80808080u;
            out[2 * j] = pk_f16(sv * (float)(int8_t)c, sv * (float)(int8_t)(c >> 8));
            out[2 * j + 1] = pk_f16(sv * (float)(int8_t)(c >> 16), sv * (float)(int8_t)(c >> 24));
        }
    }
};

// 32-element blocks: quarter q = blocks 2q (runs 0-3) and 2q + 1 (runs 4-7).
// Every load stays inside one block, because a row may end with the first of
// the two and the tensor with the row; a block past the row reads as zero,
// and so does its scale.
template <>
struct WeightUnit<OCO_Q8_0> {
    static constexpr uint32_t UNIT = 272;
    u32x4 v0, v1, v2, v3;  // block 0 from its scale on, block 1 from its codes on
    uint32_t tail, d1b;    // block 0's last two codes, block 1's scale
    float d0, d1;
    __device__ __forceinline__ static uint32_t col(uint32_t q, int i) { return 64 * q + 8 * i; }
    __device__ __forceinline__ void load(const RowSrc &r, uint32_t o, uint32_t q, uint32_t left) {
        const uint32_t o0 = 64 * q < left ? o + 68 * q : UNIT_OFF, o1 = 64 * q + 32 < left ? o + 68 * q + 34 : UNIT_OFF;
        v0 = r.u128(o0);
        v1 = r.u128(o0 + 16);
        tail = r.u16(o0 + 32);
        d1b = r.u16(o1);
        v2 = r.u128(o1 + 2);
        v3 = r.u128(o1 + 18);
    }
    __device__ __forceinline__ void prep(uint32_t) {
        d0 = half_bits_to_f32(v0.x & 0xffffu);
        d1 = half_bits_to_f32(d1b);
    }
    __device__ __forceinline__ uint32_t word(int i) const { return i < 4 ? v0[i] : i < 8 ? v1[i - 4] : tail; }
    __device__ __forceinline__ void run(int i, uint32_t *out) const {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int b = 2 * (i & 3) + j;  // dword of the block's codes
            const uint32_t w = i < 4 ? __builtin_amdgcn_alignbyte(word(b + 1), word(b), 2) : b < 4 ? v2[b] : v3[b - 4];
            const float d = i < 4 ? d0 : d1;
            out[2 * j] = pk_f16(d * (float)(int8_t)w, d * (float)(int8_t)(w >> 8));
            out[2 * j + 1] = pk_f16(d * (float)(int8_t)(w >> 16), d * (float)(int8_t)(w >> 24));
        }
    }
};

// Q4_0 / Q4_1: a block's low nibbles are its columns 0-15, its high nibbles 16-31.
// Q4_0 is d * (code - 8): code - 8 is exact in f16 and the packed f16 product
// rounds once, as half(d * (code - 8)) does, an infinite scale included (d *
// code - 8 d would be Inf - Inf there).
template <int FMT>
struct WeightQ4 {
    static constexpr uint32_t B = FMT == OCO_Q4_0 ? 18 : 20, HEAD = B - 16, UNIT = 8 * B;
    u32x4 v0, v1;        // block 0 from its scale on, block 1's codes
    uint32_t tail, head;  // the rest of block 0, block 1's scale (and minimum)
    float d[2], m[2];    // Q4_1
    f16x2 dh[2];         // Q4_0
    __device__ __forceinline__ static uint32_t col(uint32_t q, int i) { return 64 * q + 8 * i; }
    __device__ __forceinline__ void load(const RowSrc &r, uint32_t o, uint32_t q, uint32_t left) {
        const uint32_t o0 = 64 * q < left ? o + 2 * B * q : UNIT_OFF, o1 = 64 * q + 32 < left ? o + 2 * B * q + B : UNIT_OFF;
        v0 = r.u128(o0);
        tail = FMT == OCO_Q4_0 ? r.u16(o0 + 16) : r.u32(o0 + 16);
        head = FMT == OCO_Q4_0 ? r.u16(o1) : r.u32(o1);
        v1 = r.u128(o1 + HEAD);
    }
    __device__ __forceinline__ void prep(uint32_t) {
        if constexpr (FMT == OCO_Q4_0) {
            dh[0] = f16_pair((v0.x & 0xffffu) * 0x10001u);
            dh[1] = f16_pair((head & 0xffffu) * 0x10001u);
        } else {
            d[0] = half_bits_to_f32(v0.x & 0xffffu);
            d[1] = half_bits_to_f32(head & 0xffffu);
            m[0] = -half_bits_to_f32(v0.x >> 16);
            m[1] = -half_bits_to_f32(head >> 16);
        }
    }
    __device__ __forceinline__ void run(int i, uint32_t *out) const {
        const int blk = i >> 2;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int b = 2 * (i & 1) + j;  // dword of the block's codes
            uint32_t w;
            if (blk)
                w = v1[b];
            else if constexpr (FMT == OCO_Q4_0)
                w = __builtin_amdgcn_alignbyte(b < 3 ? v0[b < 3 ? b + 1 : 0] : tail, v0[b], 2);
            else
                w = b < 3 ? v0[b < 3 ? b + 1 : 0] : tail;
            const uint32_t n = ((i & 2) ? w >> 4 : w) & 0x0f0f0f0fu;
            if constexpr (FMT == OCO_Q4_0) {
                // 0x6400 | code is 1024 + code.  The empty asm keeps the runs in
                // program order, each decode beside the matrix instructions of
                // the one before: without it 256 rows of 12288 x 4096 take 70.2
                // us, with it 64.0 (d * code - 8 d in f32: 67.2).
                const f16x2 c01 = f16_pair(__builtin_amdgcn_perm(0x64646464u, n, 0x04010400u));
                const f16x2 c23 = f16_pair(__builtin_amdgcn_perm(0x64646464u, n, 0x04030402u));
                const f16x2 mid = {(_Float16)1032.0f, (_Float16)1032.0f};
                f16x2 q01 = c01 - mid, q23 = c23 - mid;
                asm volatile("" : "+v"(q01), "+v"(q23));
                const f16x2 p01 = dh[blk] * q01, p23 = dh[blk] * q23;
                __builtin_memcpy(&out[2 * j], &p01, 4);
                __builtin_memcpy(&out[2 * j + 1], &p23, 4);
            } else {
                q4_four(n, d[blk], m[blk], out[2 * j], out[2 * j + 1]);
            }
        }
    }
};
template <>
struct WeightUnit<OCO_Q4_0> : WeightQ4<OCO_Q4_0> {};
template <>
struct WeightUnit<OCO_Q4_1> : WeightQ4<OCO_Q4_1> {};

// F16: run i at columns 32 i + 8 q.
template <>
struct WeightUnit<OCO_F16> {
    static constexpr uint32_t UNIT = 512;
    u32x4 v[8];
    __device__ __forceinline__ static uint32_t col(uint32_t q, int i) { return 32 * i + 8 * q; }
    __device__ __forceinline__ void load(const RowSrc &r, uint32_t o, uint32_t q, uint32_t left) {
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = r.u128(32u * i < left ? o + 64 * i + 16 * q : UNIT_OFF);
    }
    __device__ __forceinline__ void prep(uint32_t) {}
    __device__ __forceinline__ void run(int i, uint32_t *out) const {
        out[0] = v[i].x;
        out[1] = v[i].y;
        out[2] = v[i].z;
        out[3] = v[i].w;
    }
};

}  // namespace oco
