// Y[m, n] = X[m, k] W[n, k]^T for a prompt chunk, weights decoded on the way
// into the matrix cores: the f16 operands of the dequantize pass (half(w),
// half(x)) and fp32 accumulation, without the pass's n x k x 2 bytes of f16
// weights to memory and back, and with the bias and the output type in the
// kernel.  Replaces the large tiles of DenseMatrix::apply
// (src/weights/compute/matrix.rs:130-379).
//
// A workgroup of four wavefronts, one per SIMD, covers 16 MT activation rows
// x 64 NT weight rows.  The wavefronts split the weight rows, so each weight
// is decoded once per workgroup, in the registers of the lane whose MFMA
// fragment it fills (units.h); the activations are shared: 256 columns of
// them per step go straight to LDS (global_load_lds), two steps of them, each
// row's 16-byte runs rotated by XOR with the row so that 16 rows read
// conflict-free.  One barrier per 256 columns; the next step's weights and
// activations are requested during a step's products.
// Bound by the SIMD's issue: per 32 columns and wavefront 16 MT NT clocks of
// MFMA and about 80 NT of decode (Q4_K), which do not overlap on one SIMD.
#include "panel.h"

#include "units.h"

namespace oco {

struct PanelArgs {
    const uint8_t *w;
    const uint16_t *x;  // f16 rows
    uint32_t n, k, m, row_bytes;
    uint32_t mtiles, splits;  // row tiles; K parts
    void *y;
    const float *bias;
    const float *inv;   // per-row factor of the result or null
    float *part;        // K parts: f32 [splits][m][n] (y, bias and inv unused)
    uint32_t y_bf16;
};

// s_waitcnt vmcnt(0) lgkmcnt(0), expcnt left at its maximum
__device__ __forceinline__ void panel_wait() { __builtin_amdgcn_s_waitcnt(7 << 4); }

template <int B, int E, typename F>
__device__ __forceinline__ void panel_for(F &&f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        panel_for<B + 1, E>(f);
    }
}

// Registers for two workgroups on a CU where the LDS holds two (up to 64 rows):
// Q4_K's 64 x 192 would take 264 and leave one, 512 rows of 12288 x 4096 97.6 us
// against 78.6.
template <int FMT, int MT, int NT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MT == 8 ? 1 : 2))) void panel_kernel(KPRE_PARAMS, PanelArgs a) {
    KPRE_APPLY(a);
    using U = WeightUnit<FMT>;
    constexpr int BM = 16 * MT, XL = BM / 8;  // 16-byte activation loads per lane and step
    // Separate arrays, so that the compiler can tell reads of one step's
    // activations from the asynchronous loads into the other.
    __shared__ __attribute__((aligned(16))) uint8_t xs0[BM * 512], xs1[BM * 512];
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    // workgroups that share weights (the row tiles of a column tile) run on one XCD
    const uint32_t lin = xcd_order(blockIdx.x, gridDim.x);
    const uint32_t mt = lin % a.mtiles, rest = lin / a.mtiles, part = rest % a.splits, ct = rest / a.splits;
    const uint32_t m0 = mt * BM, n0 = ct * 64 * NT, rows = min(a.n - n0, 64u * NT);
    const uint32_t all = a.k / 256, u0 = (uint32_t)((uint64_t)part * all / a.splits),
                   u1 = (uint32_t)((uint64_t)(part + 1) * all / a.splits);
    RowSrc ws;
    ws.r = uniform_rsrc(a.w + (uint64_t)n0 * a.row_bytes, rows * a.row_bytes);
    uint32_t wrow[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) wrow[t] = min((wave * NT + t) * 16 + r, rows - 1) * a.row_bytes;
    // activation load i of a step: LDS rows 2 (wave + 4 i), + 1; slot s of row
    // R holds run s ^ (R % 16)
    gbytes xsrc[XL];
#pragma unroll
    for (int i = 0; i < XL; i++) {
        const uint32_t R = 2 * (wave + 4 * i) + (lane >> 5), run = (lane & 31) ^ (R & 15);
        xsrc[i] = gp(reinterpret_cast<const uint8_t *>(a.x)) + (uint64_t)min(m0 + R, a.m - 1) * a.k * 2 + 16 * run;
    }
    f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    // The requests for step u: NT weight units, then XL activation loads.
    // Past the last step the weights read nothing and the activations repeat it.
    auto item = [&](auto kk, uint32_t u, uint8_t *xs, U *w) __attribute__((always_inline)) {
        constexpr int K = decltype(kk)::value;
        if constexpr (K < NT) {
            w[K].load(ws, u < u1 ? wrow[K] + u * U::UNIT : UNIT_OFF, q, 256);
        } else {
            constexpr int i = K - NT;
            __builtin_amdgcn_global_load_lds((const GLOBAL void *)(xsrc[i] + (uint64_t)min(u, u1 - 1) * 512),
                                             (__attribute__((address_space(3))) void *)(xs + (wave + 4 * i) * 1024), 16, 0, 0);
        }
    };
    constexpr int ITEMS = NT + XL, RUNS = 6;  // spread over the first six of a step's eight runs
    auto step = [&](uint32_t u, const uint8_t *xs, U *w, uint8_t *xn, U *wn) __attribute__((always_inline)) {
        // This step's activations are in LDS and its weights here, and the last
        // step's LDS reads are done: their buffer is overwritten after the barrier.
        panel_wait();
        asm volatile("s_barrier" ::: "memory");
#pragma unroll
        for (int t = 0; t < NT; t++) w[t].prep(q);
        panel_for<0, 8>([&](auto cc) __attribute__((always_inline)) {
            constexpr int C = decltype(cc)::value;
            if constexpr (C < RUNS)
                panel_for<C * ITEMS / RUNS, (C + 1) * ITEMS / RUNS>([&](auto kk) { item(kk, u + 1, xn, wn); });
            f16x8 xv[MT];
#pragma unroll
            for (int i = 0; i < MT; i++)
                xv[i] = *reinterpret_cast<const f16x8 *>(xs + (16 * i + r) * 512 + 16 * ((U::col(q, C) / 8) ^ r));
#pragma unroll
            for (int t = 0; t < NT; t++) {
                uint32_t o[4];
                w[t].run(C, o);
                f16x8 wv;
                __builtin_memcpy(&wv, o, 16);
#pragma unroll
                for (int i = 0; i < MT; i++) acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv, xv[i], acc[i][t], 0, 0, 0);
            }
        });
    };
    U w0[NT], w1[NT];
    panel_for<0, ITEMS>([&](auto kk) { item(kk, u0, xs0, w0); });
    for (uint32_t u = u0; u < u1; u += 2) {
        step(u, xs0, w0, xs1, w1);
        if (u + 1 < u1) step(u + 1, xs1, w1, xs0, w0);  // uniform
    }
    panel_wait();  // no load into LDS outlives the workgroup

    // lane: activation row l % 16 of its tile, weight rows 4 (l / 16) .. + 4
    const bool quads = a.n % 4 == 0 && ((uintptr_t)(a.part ? (void *)a.part : a.y) & 15) == 0;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const uint32_t c = n0 + (wave * NT + t) * 16 + 4 * q;
        if (c >= a.n) continue;
        float b[4] = {0.f, 0.f, 0.f, 0.f};
        if (a.bias && !a.part)
#pragma unroll
            for (int v = 0; v < 4; v++) b[v] = c + v < a.n ? round_bf16(a.bias[c + v]) : 0.f;
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const uint32_t row = m0 + 16 * i + r;
            if (row >= a.m) continue;
            const uint64_t at = (uint64_t)row * a.n + c;
            f32x4 v = acc[i][t];
            if (a.part) {
                float *o = a.part + (uint64_t)part * a.m * a.n + at;
                if (quads)
                    *reinterpret_cast<GLOBAL f32x4 *>(gp(o)) = v;
                else
                    for (int e = 0; e < 4; e++)
                        if (c + e < a.n) o[e] = v[e];
                continue;
            }
            const float g = a.inv ? a.inv[row] : 1.0f;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = v[e] * g + b[e];
            if (a.y_bf16) {
                uint16_t *o = reinterpret_cast<uint16_t *>(a.y) + at;
                const uint32_t h[4] = {f32_to_bf16_bits(v[0]), f32_to_bf16_bits(v[1]), f32_to_bf16_bits(v[2]), f32_to_bf16_bits(v[3])};
                if (quads)
                    *reinterpret_cast<GLOBAL u32x2 *>(gp(o)) = u32x2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
                else
                    for (int e = 0; e < 4; e++)
                        if (c + e < a.n) o[e] = (uint16_t)h[e];
            } else {
                float *o = reinterpret_cast<float *>(a.y) + at;
                if (quads)
                    *reinterpret_cast<GLOBAL f32x4 *>(gp(o)) = v;
                else
                    for (int e = 0; e < 4; e++)
                        if (c + e < a.n) o[e] = v[e];
            }
        }
    }
}

typedef void (*PanelFn)(u32x4, u32x4, u32x4, u32x2, PanelArgs);

// The tiles in use: (16-row activation tiles, 16-row weight tiles per
// wavefront).  Wider ones at eight activation tiles (128 x 128, 128 x 192)
// leave one wavefront per SIMD with nothing to cover its waits and measured
// slower than 64 x 192 at every size; 128 x 64 pays for the largest decode
// only (Q6_K 12288 x 4096 at 128 rows 48.0 us, 64 x 64 55.8).
template <int FMT>
static PanelFn panel_pick(int mt, int nt) {
    if constexpr (FMT == OCO_Q6_K)
        if (mt == 8) return panel_kernel<FMT, 8, 1>;
    if constexpr (FMT == OCO_Q4_K || FMT == OCO_Q4_0 || FMT == OCO_Q4_1) {
        if (nt == 3) return panel_kernel<FMT, 4, 3>;
        if (nt == 2) return panel_kernel<FMT, 4, 2>;
    }
    return mt == 4 ? panel_kernel<FMT, 4, 1> : panel_kernel<FMT, 2, 1>;
}

// What a tile takes, in us: once per call (launches included), once more per
// workgroup that a CU runs, and per 256 columns for a workgroup alone on its
// CU and for two that share it (zero: not built for the format).  A CU that
// runs three takes a pair's time and one alone's, and so on: 64 x 192 of Q4_K
// steps at 2.8, 4.2-4.6, 6.2, 7.8 for one to four.  Fitted, with the estimates
// below, to 2900 timings of 83 matrices (256 to 151936 rows, K 256 to 28672) at
// 32 to 1000 rows, with weights streamed from HBM, in long runs; they miss them by
// 8% (root mean square).
struct PanelTile {
    int mt, nt;
    double start, more;
    struct {
        double alone, pair;
    } step[4];  // by panel_class
};
static const PanelTile PANEL_TILES[] = {{4, 3, 8.2, 0.0, {{2.05, 3.55}, {3.1, 4.4}, {}, {}}},
                                        {4, 2, 6.7, 0.4, {{1.55, 2.55}, {2.1, 3.2}, {}, {}}},
                                        {8, 1, 4.5, 2.5, {{}, {}, {}, {2.4, 4.7}}},
                                        {4, 1, 5.0, 0.7, {{1.0, 1.48}, {1.37, 2.1}, {1.53, 2.2}, {1.84, 2.85}}},
                                        {2, 1, 5.1, 0.1, {{0.76, 1.07}, {1.13, 1.43}, {1.2, 1.82}, {1.68, 2.58}}}};

// Formats of about the same decode; below zero: not decoded here.
static int panel_class(uint32_t format) {
    switch (format) {
    case OCO_Q4_K: return 0;
    case OCO_Q4_0: case OCO_Q4_1: return 1;
    case OCO_Q8_0: case OCO_Q5_K: return 2;
    case OCO_Q6_K: return 3;
    }
    return -1;
}

static uint64_t panel_workgroups(int mt, int nt, uint64_t s, uint32_t m, uint32_t n) {
    return (uint64_t)((n + 64 * nt - 1) / (64 * nt)) * ((m + 16 * mt - 1) / (16 * mt)) * s;
}

bool panel_fits(uint32_t format, const PanelPlan &pl, uint32_t m, uint32_t n, uint32_t k) {
    const int cls = panel_class(format);
    if (cls < 0 || k == 0 || k % 256 || m == 0 || n == 0 || m > 0x3fffffffu || n > 0x3fffffffu) return false;
    bool built = false;
    for (const PanelTile &t : PANEL_TILES) built = built || (t.mt == pl.mt && t.nt == pl.nt && t.step[cls].alone > 0);
    if (!built || 64ull * pl.nt * oco_row_bytes(format, k) >= UNIT_OFF) return false;
    const uint64_t s = pl.splits;
    if (s == 0 || s > k / 256 || (s > 1 && s * m * 2 > k)) return false;  // the parts lie where the pass's f16 weights would
    return panel_workgroups(pl.mt, pl.nt, s, m, n) < 0x80000000ull;
}

// The tile and the K parts by estimated time, and whether that beats the
// dequantize pass + GEMM + epilogue, whose time depends on the kernel the
// library takes and is not monotone in the rows (Q4_K 14336 x 4096 at 192,
// 224 and 352 rows: 80, 73 and 86 us): its estimate lies low, 0.76 to 1.13 times
// the measured (5th and 95th percentile), so that the panel kernel is taken
// where its lead holds, and a few percent are asked for on top.  Of 985 streamed
// products three are more than 2% slower here than on the GEMM, at most 7%, and the
// choice is 1.014 times the fastest of all on average.  Q4_K 12288 x 4096,
// bf16 out, us, pass and GEMM against this: 32 rows 51, 19; 64 rows 50, 25; 128
// rows 66, 35; 256 rows 74, 51; 512 rows 85, 81; 14336 x 4096 at 448 rows 87
// against 94 to 106 on the tiles here, which are not taken.
PanelPlan panel_plan(uint32_t format, uint32_t m, uint32_t n, uint32_t k, bool direct) {
    PanelPlan best = {};
    const int cls = panel_class(format);
    if (!panel_fits(format, {2, 1, 1}, m, n, k)) return best;
    const double mn = 1e-6 * m * n, mk = 1e-6 * m * k, nk = 1e-6 * n * k;
    // us per 10^6 weights of the pass
    const double pass = format == OCO_Q5_K ? 1.75 : cls == 1 ? 0.98 : 0.72;
    const double epilogue = direct ? 0 : 1.5 + 1.2 * mn;
    const double gemm = 7.5 + 1.25e-3 * k + pass * nk + (1.4 + 2.6 * std::min(k, 8192u) / 4096) * mn + 2 * mk + epilogue;
    const double stream = 1e-6 * n * oco_row_bytes(format, k) / 5.1;  // the weights at the rate of a copy
    double least = 0.96 * gemm;
    for (const PanelTile &t : PANEL_TILES)
        for (uint32_t s = 1; s <= 8; s *= 2) {
            if (!panel_fits(format, {t.mt, t.nt, s}, m, n, k)) break;
            const uint64_t load = (panel_workgroups(t.mt, t.nt, s, m, n) + 255) / 256;  // on the fullest CU
            const double step = (load % 2) * t.step[cls].alone + (load / 2) * t.step[cls].pair;
            const double us = t.start + t.more * load + std::max((k / 256 + s - 1) / s * step, stream) + 0.95 * mk + 0.9 * mn +
                              (s > 1 ? 1.2 + 0.32 * s + 1.4 * s * mn : 0);  // the parts and their sum
            if (us < least) {
                least = us;
                best = {t.mt, t.nt, s};
            }
        }
    return best;
}

int panel_launch(uint32_t format, const PanelPlan &pl, const void *w, const uint16_t *x, void *y, bool y_bf16,
                 const float *bias, const float *inv, float *part, uint32_t m, uint32_t n, uint32_t k, hipStream_t stream) {
    PanelFn fn = nullptr;
    switch (format) {
#define CASE(F) case F: fn = panel_pick<F>(pl.mt, pl.nt); break;
        CASE(OCO_Q4_0) CASE(OCO_Q4_1) CASE(OCO_Q8_0) CASE(OCO_Q4_K) CASE(OCO_Q5_K) CASE(OCO_Q6_K)
#undef CASE
    }
    if (!fn) return fail(OCO_ERR_UNSUPPORTED, "oco_matmul: format %u", format);
    PanelArgs a = {};
    a.w = (const uint8_t *)w;
    a.x = x;
    a.n = n;
    a.k = k;
    a.m = m;
    a.row_bytes = (uint32_t)oco_row_bytes(format, k);
    a.mtiles = (m + 16 * pl.mt - 1) / (16 * pl.mt);
    a.splits = pl.splits;
    a.y = y;
    a.bias = bias;
    a.inv = inv;
    a.part = pl.splits > 1 ? part : nullptr;
    a.y_bf16 = y_bf16;
    const uint32_t grid = (n + 64 * pl.nt - 1) / (64 * pl.nt) * a.mtiles * pl.splits;
    hipLaunchKernelGGL(fn, dim3(grid), dim3(256), 0, stream, KPRE_ARGS(a), a);
    return launch_check("oco_matmul: panel");
}

}  // namespace oco
