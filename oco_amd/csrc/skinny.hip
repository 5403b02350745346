// Y[m, n] = X[m, k] W[n, k]^T for a few activation rows (m <= 32): decode
// batches, draft verification, short prompts.  Replaces the small-m plans of
// DenseMatrix::apply (src/weights/compute/matrix.rs:130-379) on the same
// operands as the larger tiles here: half(w) and half(x), fp32 accumulation.
//
// Bound by the weight stream (28 MB for Q4_K 12288 x 4096).  A workgroup
// takes 16 NT weight rows and all of K: its eight wavefronts take every
// eighth 256-column unit of those rows and meet in LDS at the end, so at
// k = 4096 each wavefront requests everything it will read before its first
// product, and no barrier sits between loads and products.  Weights go from
// global memory to the lane whose MFMA fragment they fill and are decoded in
// registers; lane (row r = l % 16, group q = l / 16) holds a quarter of its
// row's unit in the format's own order, and the activations, converted to
// f16 once per wavefront and unit, are read back from a wavefront-private
// LDS buffer in that order.
// Q4_K 12288 x 4096, 8 rows: 52 us on the 64 x 64 LDS tiles (192 workgroups,
// every weight through LDS, a barrier per 128 columns) -> 14.7 us here.
#include "formats.h"
#include "matmul.h"
#include "skinny.h"

namespace oco {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct SkinnyArgs {
    const uint8_t *w;
    const void *x;
    uint32_t n, k, m, row_bytes;
    uint32_t x_f16, y_bf16;
    void *y;
    const float *bias;
    const float *inv;  // per-row factor of the result (1 / activation gain) or null
};

__device__ __forceinline__ uint32_t pk_f16(float a, float b) {
    uint32_t r;
    asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// Four f16 of a * code - m from the bytes of one dword (a * code exact in f32).
__device__ __forceinline__ void four_ub(uint32_t n, float a, float m, uint32_t &p01, uint32_t &p23) {
    const float f0 = __builtin_fmaf(a, ub(n, 0), -m), f1 = __builtin_fmaf(a, ub(n, 1), -m);
    const float f2 = __builtin_fmaf(a, ub(n, 2), -m), f3 = __builtin_fmaf(a, ub(n, 3), -m);
    p01 = pk_f16(f0, f1);
    p23 = pk_f16(f2, f3);
}
__device__ __forceinline__ void q4_four_s(uint32_t n, float a, float m, uint32_t &p01, uint32_t &p23) {
    const q4f32x2 c01 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(n, 512.0f, false);
    const q4f32x2 c23 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(n, 512.0f, true);
    p01 = pk_f16(__builtin_fmaf(a, c01[0], -m), __builtin_fmaf(a, c01[1], -m));
    p23 = pk_f16(__builtin_fmaf(a, c23[0], -m), __builtin_fmaf(a, c23[1], -m));
}

// Buffer loads at any byte offset, zero past the resource's range.
struct RowSrc {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ uint32_t u16(uint32_t o) const { return __builtin_amdgcn_raw_buffer_load_b16(r, o, 0, 0); }
    __device__ __forceinline__ uint32_t u32(uint32_t o) const { return __builtin_amdgcn_raw_buffer_load_b32(r, o, 0, 0); }
    __device__ __forceinline__ u32x2 u64(uint32_t o) const { return __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, 0); }
    __device__ __forceinline__ u32x4 u128(uint32_t o) const { return __builtin_amdgcn_raw_buffer_load_b128(r, o, 0, 0); }
};
constexpr uint32_t SKINNY_OFF = 0x80000000u;  // past every range: reads zero without touching memory

// A lane's quarter q of one row's 256-column unit: 64 weights as eight runs
// of eight consecutive columns (col(q, i) within the unit).
//   UNIT   bytes of a whole unit; load(src, row offset + unit offset, columns
//          left in the row from the unit's start);
//   prep   once per unit; run(i) the i-th run as four dwords of f16.
template <int FMT>
struct SkinnyUnit;

template <int FMT>
struct SkinnyK4 {  // Q4_K, Q5_K: quarter q = sub-blocks 2q (runs 0-3) and 2q + 1 (runs 4-7)
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
                q4_four_s(n, a, m, out[2 * j], out[2 * j + 1]);
            }
        }
    }
};
template <>
struct SkinnyUnit<OCO_Q4_K> : SkinnyK4<OCO_Q4_K> {};
template <>
struct SkinnyUnit<OCO_Q5_K> : SkinnyK4<OCO_Q5_K> {};

// Q6_K: half h = q / 2, quarters p = q % 2 (runs 0-3, low nibbles) and p + 2
// (runs 4-7, high nibbles) of it.
template <>
struct SkinnyUnit<OCO_Q6_K> {
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
        const float d = half_bits_to_f32(db);
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
            const uint32_t w = l[2 * (i & 1) + j];
            const uint32_t lo = (i < 4 ? w : w >> 4) & 0x0f0f0f0fu;
            const uint32_t hi = (h[2 * (i & 1) + j] >> (2 * p + (i < 4 ? 0 : 4))) & 0x03030303u;
            // s * (code - 32): both products are exact in f32, so the fused
            // form rounds once, to the value of the reference's multiply
            four_ub(lo | (hi << 4), sv, 32.0f * sv, out[2 * j], out[2 * j + 1]);
        }
    }
};

// 32-element blocks: quarter q = blocks 2q (runs 0-3) and 2q + 1 (runs 4-7).
// Every load stays inside one block, because a row may end with the first of
// the two and the tensor with the row; a block past the row reads as zero,
// and so does its scale.
template <>
struct SkinnyUnit<OCO_Q8_0> {
    static constexpr uint32_t UNIT = 272;
    u32x4 v0, v1, v2, v3;  // block 0 from its scale on, block 1 from its codes on
    uint32_t tail, d1b;    // block 0's last two codes, block 1's scale
    float d0, d1;
    __device__ __forceinline__ static uint32_t col(uint32_t q, int i) { return 64 * q + 8 * i; }
    __device__ __forceinline__ void load(const RowSrc &r, uint32_t o, uint32_t q, uint32_t left) {
        const uint32_t o0 = 64 * q < left ? o + 68 * q : SKINNY_OFF, o1 = 64 * q + 32 < left ? o + 68 * q + 34 : SKINNY_OFF;
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
template <int FMT>
struct SkinnyQ4 {
    static constexpr uint32_t B = FMT == OCO_Q4_0 ? 18 : 20, HEAD = B - 16, UNIT = 8 * B;
    u32x4 v0, v1;        // block 0 from its scale on, block 1's codes
    uint32_t tail, head;  // the rest of block 0, block 1's scale (and minimum)
    float d[2], m[2];
    __device__ __forceinline__ static uint32_t col(uint32_t q, int i) { return 64 * q + 8 * i; }
    __device__ __forceinline__ void load(const RowSrc &r, uint32_t o, uint32_t q, uint32_t left) {
        const uint32_t o0 = 64 * q < left ? o + 2 * B * q : SKINNY_OFF, o1 = 64 * q + 32 < left ? o + 2 * B * q + B : SKINNY_OFF;
        v0 = r.u128(o0);
        tail = FMT == OCO_Q4_0 ? r.u16(o0 + 16) : r.u32(o0 + 16);
        head = FMT == OCO_Q4_0 ? r.u16(o1) : r.u32(o1);
        v1 = r.u128(o1 + HEAD);
    }
    __device__ __forceinline__ void prep(uint32_t) {
        d[0] = half_bits_to_f32(v0.x & 0xffffu);
        d[1] = half_bits_to_f32(head & 0xffffu);
        if constexpr (FMT == OCO_Q4_0) {
            m[0] = 8.0f * d[0];  // d q - 8 d = d (q - 8): both exact in f32
            m[1] = 8.0f * d[1];
        } else {
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
            q4_four_s(((i & 2) ? w >> 4 : w) & 0x0f0f0f0fu, d[blk], m[blk], out[2 * j], out[2 * j + 1]);
        }
    }
};
template <>
struct SkinnyUnit<OCO_Q4_0> : SkinnyQ4<OCO_Q4_0> {};
template <>
struct SkinnyUnit<OCO_Q4_1> : SkinnyQ4<OCO_Q4_1> {};

// F16: run i at columns 32 i + 8 q.
template <>
struct SkinnyUnit<OCO_F16> {
    static constexpr uint32_t UNIT = 512;
    u32x4 v[8];
    __device__ __forceinline__ static uint32_t col(uint32_t q, int i) { return 32 * i + 8 * q; }
    __device__ __forceinline__ void load(const RowSrc &r, uint32_t o, uint32_t q, uint32_t left) {
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = r.u128(32u * i < left ? o + 64 * i + 16 * q : SKINNY_OFF);
    }
    __device__ __forceinline__ void prep(uint32_t) {}
    __device__ __forceinline__ void run(int i, uint32_t *out) const {
        out[0] = v[i].x;
        out[1] = v[i].y;
        out[2] = v[i].z;
        out[3] = v[i].w;
    }
};

constexpr int SK_WAVES = 8;
constexpr int SK_LD = 256 + 8;  // halves per staged activation row: rows 4 banks apart, reads of 16 rows conflict-free

// MT tiles of 16 activation rows, NT tiles of 16 weight rows.
template <int FMT, int MT, int NT>
__global__ __launch_bounds__(64 * SK_WAVES) void skinny_kernel(KPRE_PARAMS, SkinnyArgs a) {
    KPRE_APPLY(a);
    using U = SkinnyUnit<FMT>;
    constexpr uint32_t STAGE = SK_WAVES * MT * 16 * SK_LD * 2, PART = SK_WAVES * MT * NT * 1024;
    __shared__ __attribute__((aligned(16))) uint8_t smem[STAGE > PART ? STAGE : PART];
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const uint32_t n0 = blockIdx.x * 16 * NT, rows = min(a.n - n0, 16u * NT);
    RowSrc ws, xs;
    ws.r = uniform_rsrc(a.w + (uint64_t)n0 * a.row_bytes, rows * a.row_bytes);
    xs.r = uniform_rsrc(a.x, a.m * a.k * 2);
    uint32_t wrow[NT], xrow[MT];
#pragma unroll
    for (int t = 0; t < NT; t++) wrow[t] = min(16 * t + r, rows - 1) * a.row_bytes;
#pragma unroll
    for (int i = 0; i < MT; i++) xrow[i] = (16 * i + r) * a.k * 2;

    const uint32_t units = (a.k + 255) / 256;
    struct Buf {
        U w[NT];
        u32x4 x[MT][8];
    };
    auto load = [&](Buf &b, uint32_t u) {  // units past the last read nothing
        const uint32_t left = u < units ? a.k - 256 * u : 0;
        const uint32_t o = u < units ? u * U::UNIT : SKINNY_OFF;
#pragma unroll
        for (int t = 0; t < NT; t++) b.w[t].load(ws, u < units ? wrow[t] + o : SKINNY_OFF, q, left);
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const bool live = 16 * i + r < a.m && 32u * j + 8 * q < left;
                b.x[i][j] = xs.u128(live ? xrow[i] + 2 * (256 * u + 32 * j + 8 * q) : SKINNY_OFF);
            }
    };
    f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint16_t *xl = reinterpret_cast<uint16_t *>(smem) + (size_t)wave * MT * 16 * SK_LD;
    auto compute = [&](Buf &b) {
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < 8; j++) {
                u32x4 v = b.x[i][j];
                if (!a.x_f16)
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = pk_f16(__uint_as_float(v[e] << 16), __uint_as_float(v[e] & 0xffff0000u));
                *reinterpret_cast<u32x4 *>(xl + (16 * i + r) * SK_LD + 32 * j + 8 * q) = v;
            }
        // lanes read what other lanes of the wavefront wrote: the LDS is in
        // order, the fences keep the compiler from moving reads over writes
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int t = 0; t < NT; t++) b.w[t].prep(q);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            f16x8 xv[MT];
#pragma unroll
            for (int i = 0; i < MT; i++) xv[i] = *reinterpret_cast<const f16x8 *>(xl + (16 * i + r) * SK_LD + U::col(q, j));
#pragma unroll
            for (int t = 0; t < NT; t++) {
                uint32_t o[4];
                b.w[t].run(j, o);
                f16x8 wv;
                __builtin_memcpy(&wv, o, 16);
#pragma unroll
                for (int i = 0; i < MT; i++) acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv[i], wv, acc[i][t], 0, 0, 0);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    Buf b0, b1;
    load(b0, wave);
    load(b1, wave + SK_WAVES);
    for (uint32_t u = wave; u < units; u += 2 * SK_WAVES) {
        compute(b0);
        load(b0, u + 2 * SK_WAVES);
        if (u + SK_WAVES < units) compute(b1);
        load(b1, u + 3 * SK_WAVES);
    }
    // partial sums of the eight wavefronts: [wave][tile][lane] quads
    __syncthreads();
    f32x4 *part = reinterpret_cast<f32x4 *>(smem);
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int t = 0; t < NT; t++) part[(wave * MT * NT + i * NT + t) * 64 + lane] = acc[i][t];
    __syncthreads();
    for (uint32_t o = threadIdx.x; o < MT * NT * 64; o += 64 * SK_WAVES) {
        f32x4 s = part[o];
#pragma unroll
        for (int w = 1; w < SK_WAVES; w++) s += part[w * MT * NT * 64 + o];
        // lane: weight row l % 16, activation rows 4 (l / 16) .. + 4
        const uint32_t tile = o / 64, l = o % 64, col = n0 + 16 * (tile % NT) + (l & 15), row0 = 16 * (tile / NT) + 4 * (l >> 4);
        if (col >= a.n) continue;
        const float bias = a.bias ? round_bf16(a.bias[col]) : 0.f;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const uint32_t row = row0 + v;
            if (row >= a.m) break;
            const float f = s[v] * (a.inv ? a.inv[row] : 1.0f) + bias;
            const uint64_t at = (uint64_t)row * a.n + col;
            if (a.y_bf16)
                reinterpret_cast<uint16_t *>(a.y)[at] = f32_to_bf16_bits(f);
            else
                reinterpret_cast<float *>(a.y)[at] = f;
        }
    }
}

typedef void (*SkinnyFn)(u32x4, u32x4, u32x4, u32x2, SkinnyArgs);

template <int FMT>
static SkinnyFn skinny_pick(int mt, int nt) {
    if constexpr (FMT != OCO_F16) {
        if (mt == 1 && nt == 3) return skinny_kernel<FMT, 1, 3>;
        if (mt == 2 && nt == 2) return skinny_kernel<FMT, 2, 2>;
    }
    if (mt == 1) return nt == 2 ? skinny_kernel<FMT, 1, 2> : skinny_kernel<FMT, 1, 1>;
    return skinny_kernel<FMT, 2, 1>;
}

bool skinny_fits(uint32_t format, uint32_t m, uint32_t n, uint32_t k) {
    switch (format) {
    case OCO_Q4_0: case OCO_Q4_1: case OCO_Q8_0: case OCO_Q4_K: case OCO_Q5_K: case OCO_Q6_K: case OCO_F16: break;
    default: return false;
    }
    // 32-bit offsets into a workgroup's weight rows and into the activations
    return m >= 1 && m <= SKINNY_ROWS && 48ull * oco_row_bytes(format, k) < SKINNY_OFF && 2ull * m * k < SKINNY_OFF &&
           n <= 0x7fffffffu;
}

int skinny_launch(uint32_t format, const void *w, const void *x, bool x_f16, void *y, bool y_bf16, const float *bias,
                  const float *inv, uint32_t m, uint32_t n, uint32_t k, hipStream_t stream) {
    const int mt = m <= 16 ? 1 : 2;
    // Weight rows per workgroup: as many as leave about one workgroup per CU
    // (the activations are loaded and converted once per workgroup).
    const uint32_t tiles = (n + 15) / 16;
    int nt = tiles >= 640 ? 3 : tiles >= 384 ? 2 : 1;
    // registers: two units of weights and activations in flight
    const int most = (mt == 1 ? 3 : 2) - (format == OCO_F16 ? 1 : 0);
    nt = std::min(nt, most);
    SkinnyFn fn = nullptr;
    switch (format) {
#define CASE(F) case F: fn = skinny_pick<F>(mt, nt); break;
        CASE(OCO_Q4_0) CASE(OCO_Q4_1) CASE(OCO_Q8_0) CASE(OCO_Q4_K) CASE(OCO_Q5_K) CASE(OCO_Q6_K) CASE(OCO_F16)
#undef CASE
    }
    if (!fn) return fail(OCO_ERR_UNSUPPORTED, "oco_matmul: format %u", format);
    SkinnyArgs a = {};
    a.w = (const uint8_t *)w;
    a.x = x;
    a.n = n;
    a.k = k;
    a.m = m;
    a.row_bytes = (uint32_t)oco_row_bytes(format, k);
    a.x_f16 = x_f16;
    a.y_bf16 = y_bf16;
    a.y = y;
    a.bias = bias;
    a.inv = inv;
    hipLaunchKernelGGL(fn, dim3((tiles + nt - 1) / nt), dim3(64 * SK_WAVES), 0, stream, KPRE_ARGS(a), a);
    return launch_check("oco_matmul: few rows");
}

}  // namespace oco
