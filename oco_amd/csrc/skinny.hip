// Y[m, n] = X[m, k] W[n, k]^T for a few activation rows (m <= SKINNY_ROWS): decode
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
#include "skinny.h"
#include "units.h"

namespace oco {

struct SkinnyArgs {
    const uint8_t *w;
    const void *x;
    uint32_t n, k, m, row_bytes;
    uint32_t x_f16, y_bf16;
    void *y;
    const float *bias;
    const float *inv;  // per-row factor of the result (1 / activation gain) or null
};

constexpr int SK_WAVES = 8;
constexpr int SK_LD = 256 + 8;  // halves per staged activation row: rows 4 banks apart, reads of 16 rows conflict-free

// MT tiles of 16 activation rows, NT tiles of 16 weight rows.
template <int FMT, int MT, int NT>
__global__ __launch_bounds__(64 * SK_WAVES) void skinny_kernel(KPRE_PARAMS, SkinnyArgs a) {
    KPRE_APPLY(a);
    using U = WeightUnit<FMT>;
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
        const uint32_t o = u < units ? u * U::UNIT : UNIT_OFF;
#pragma unroll
        for (int t = 0; t < NT; t++) b.w[t].load(ws, u < units ? wrow[t] + o : UNIT_OFF, q, left);
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const bool live = 16 * i + r < a.m && 32u * j + 8 * q < left;
                b.x[i][j] = xs.u128(live ? xrow[i] + 2 * (256 * u + 32 * j + 8 * q) : UNIT_OFF);
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
    return m >= 1 && m <= SKINNY_ROWS && 48ull * oco_row_bytes(format, k) < UNIT_OFF && 2ull * m * k < UNIT_OFF &&
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
