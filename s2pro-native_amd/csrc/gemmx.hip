/* s2pro MI355X — the GEMM of the batched rows (16 < M <= 128: verify batches,
 * draft trees, prefill chunks) over INT4-g32, INT8 and bf16 weights.
 *
 * Replaces the reference's M > 16 path (dequant + cuBLAS, gemm.c:467-490, or
 * the WMMA kernel int8_gemv.cu:535-618).
 *
 * What bounds it: the activations.  A workgroup that owns few weight rows
 * reads all M x K of them through its L1, so N is dealt out in blocks of up to
 * 96 rows (two row groups of three 16-row tiles) and K is split over
 * workgroups where the blocks alone would not cover the CUs; k_gmx_merge, the
 * next launch, sums the splits in order and runs the epilogue.
 *   - k_gmx_pack first lays the activations out as MFMA operands: 1 KB per 16
 *     rows x 32 k, so that an operand is one contiguous load of the wave.
 *     From the row-major rows an operand load takes 64 bytes of 16 rows whose
 *     strides (5, 8 and 19 KB) fall on a quarter or fewer of the L2's
 *     channels.  The pass also applies an input RMSNorm (the rule's
 *     roundings) once, and the INT4 k-slot order;
 *   - the workgroup's 8 waves are KW K slices x RG row groups x MG groups of
 *     activation rows; a wave holds T weight tiles x MTW activation tiles: a
 *     loaded weight is dequantised once for MTW products, a loaded activation
 *     operand serves T;
 *   - neither goes through LDS, so waves run without barriers until their
 *     partial tiles meet there, where one thread per four outputs sums the K
 *     slices in order (deterministic).  K advances in chunks of 128, operands
 *     one chunk ahead.  Up to 39 of the tiles' scalar bases and trip counts sit
 *     in lanes of a vector register (INT4, T = 2, MTW = 4); nothing is in scratch.
 * INT4 weights become 1.5 + w / 16 (exact), the bias -1.5 sum x of a group is
 * an MFMA against a constant and the C operand of the group's products. */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemv_dev.h"

#define GX_WAVES 8
#define GX_CK 128 /* k values a chunk */
#define GX_MIN_ROWS 12288 /* six 16-row tiles on half the CUs: K needs no split */

struct GmxArgs {
    const uint8_t* w;
    const void* s;
    const uint16_t* x; /* packed: [K / 128][mt][4 operands][64 lanes][8] */
    uint16_t* y;
    float* part;       /* K splits: [splits][M][np] */
    float* ssq_out;    /* RESID: [ceil(N / 16)][GEMV_MAX_M] sums of squares, or NULL */
    int ldy, M, N, K, epi;
    int rpt;           /* output rows a tile (<= 16) */
    int groups;        /* tile groups, one a workgroup and round */
    int kw, rg, mg;    /* wave grid: K slices, row groups, activation groups */
    int mt;            /* 16-row activation tiles of x: ceil(M / 16) */
    int splits, np;    /* K splits over workgroups; columns of a partial row */
};

/* bytes of a weight row per chunk, and 16-byte loads of it */
static __host__ __device__ constexpr int gx_cb(int wfmt) {
    return wfmt == GEMV_W_INT4 ? 64 : wfmt == GEMV_W_INT8 ? 128 : 256;
}
template <int WFMT>
struct GxW {
    s2p_u32x4 w[gx_cb(WFMT) / 64];
};
template <>
struct GxW<GEMV_W_INT4> {
    s2p_u32x4 w[1];
    s2p_u32x2 s; /* the chunk's four f16 group scales of the lane's row */
};

/* every argument in one round of scalar loads */
S2P_DEV void gx_args(const GmxArgs& a) {
    asm volatile("" ::"s"(a.w), "s"(a.s), "s"(a.x), "s"(a.y), "s"(a.part), "s"(a.ssq_out), "s"(a.ldy), "s"(a.M),
                 "s"(a.N), "s"(a.K), "s"(a.epi), "s"(a.rpt), "s"(a.groups), "s"(a.kw), "s"(a.rg),
                 "s"(a.mg), "s"(a.mt), "s"(a.splits), "s"(a.np));
}

template <int WFMT, int T, int MTW>
__global__ __launch_bounds__(64 * GX_WAVES) void k_gmx(GmxArgs a) {
#pragma clang fp contract(off)
    constexpr int NL = gx_cb(WFMT) / 64;
    gx_args(a);
    extern __shared__ __align__(16) unsigned char gx_smem[];
    LDS(float)* red = (LDS(float)*)gx_smem; /* [kw][rg][T][mg][MTW][64 lanes][4] */
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, r = lane & 15;
    const int kw = wave % a.kw, wr = wave / a.kw, rg = wr % a.rg, mg = wr / a.rg;
    const bool sw = a.epi == GEMV_EPI_SWIGLU;
    const int F = sw ? a.N >> 1 : a.N;
    const int ntp = sw ? T : T * a.rg; /* output tiles a group */
    /* chunks of split blockIdx.y, then of this wave's slice of it */
    const int sp = blockIdx.y, nall = a.K / GX_CK;
    const int s0 = nall * sp / a.splits, nck = nall * (sp + 1) / a.splits - s0;
    const int kb = nck / a.kw, krem = nck - kb * a.kw;
    const int c0 = s0 + kw * kb + min(kw, krem), nc = kb + (kw < krem ? 1 : 0);
    const uint32_t rb = (uint32_t)(a.K / GX_CK * gx_cb(WFMT)); /* bytes of a weight row */

    /* activation operands: tile c of this wave (past the last: it again, its
     * outputs are dropped), 4 KB a chunk and tile */
    GblPtr xb[MTW];
#pragma unroll
    for (int c = 0; c < MTW; c++)
        xb[c] = gbl_base(a.x, ((uint64_t)c0 * a.mt + min(mg * MTW + c, a.mt - 1)) * 4096u);
    const uint32_t xs = (uint32_t)a.mt * 4096u, xl = 16u * lane;

    for (int g = blockIdx.x; g < a.groups; g += gridDim.x) {
        /* tiles: scalar base of the first row, lane offset of row r (past the
         * end: the last row again) */
        GblPtr wb[T], sb[T];
        uint32_t wl[T], sl[T];
#pragma unroll
        for (int t = 0; t < T; t++) {
            const int ot = sw ? g * T + t : (g * a.rg + rg) * T + t;
            const int n0 = min(ot * a.rpt, F - 1);
            const uint32_t rl = (uint32_t)min(r, min(a.rpt, F - n0) - 1);
            const uint64_t row0 = (uint64_t)(n0 + (sw && rg ? F : 0));
            wb[t] = gbl_base(a.w, row0 * rb + (uint64_t)c0 * gx_cb(WFMT));
            wl[t] = rl * rb + 16u * q;
            if constexpr (WFMT == GEMV_W_INT4) {
                sb[t] = gbl_base(a.s, row0 * (uint32_t)(a.K >> 4) + (uint64_t)c0 * 8);
                sl[t] = rl * (uint32_t)(a.K >> 4);
            }
        }
        GxW<WFMT> w0[T], w1[T];
        s2p_u32x4 x0[MTW][4], x1[MTW][4];
        auto load = [&](GxW<WFMT>(&w)[T], s2p_u32x4(&x)[MTW][4], int ck)
            __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < T; t++) {
#pragma unroll
                for (int l = 0; l < NL; l++)
                    w[t].w[l] = gbl_at<s2p_u32x4>(wb[t] + ck * gx_cb(WFMT) + l * 64, wl[t]);
                if constexpr (WFMT == GEMV_W_INT4)
                    w[t].s = gbl_at<s2p_u32x2>(sb[t] + ck * 8, sl[t]);
            }
#pragma unroll
            for (int c = 0; c < MTW; c++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    x[c][i] = gbl_at<s2p_u32x4>(xb[c] + (size_t)ck * xs + i * 1024, xl);
        };
        s2p_f32x4 acc[T][MTW];
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int c = 0; c < MTW; c++) acc[t][c] = (s2p_f32x4){0.f, 0.f, 0.f, 0.f};
        auto mul = [&](GxW<WFMT>(&w)[T], s2p_u32x4(&x)[MTW][4]) __attribute__((always_inline)) {
            if constexpr (WFMT == GEMV_W_INT4) {
                const s2p_u32x4 k15 = {0xBFC0BFC0u, 0xBFC0BFC0u, 0xBFC0BFC0u, 0xBFC0BFC0u};
                uint32_t kmask = 0x00780078u, kone = 0x3F803F80u;
                asm volatile("" : "+v"(kmask), "+v"(kone));
                uint32_t d[T][4];
#pragma unroll
                for (int t = 0; t < T; t++) {
#pragma unroll
                    for (int i = 0; i < 4; i++) d[t][i] = w[t].w[0][i];
                    xpose4(d[t][0], d[t][1], d[t][2], d[t][3]);
                }
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    s2p_u32x4 wv[T];
                    float sf[T];
#pragma unroll
                    for (int t = 0; t < T; t++) {
                        wv[t] = deq_int4(d[t][i], kmask, kone);
                        const uint32_t sp = w[t].s[i >> 1];
                        sf[t] = (float)__builtin_bit_cast(
                            _Float16, (uint16_t)((i & 1) ? (sp >> 16) : (sp & 0xFFFFu)));
                    }
#pragma unroll
                    for (int c = 0; c < MTW; c++) {
                        const s2p_f32x4 cb = mfma16x16x32(x[c][i], k15, (s2p_f32x4){0.f, 0.f, 0.f, 0.f});
#pragma unroll
                        for (int t = 0; t < T; t++) {
                            const s2p_f32x4 raw = mfma16x16x32(x[c][i], wv[t], cb);
#pragma unroll
                            for (int e = 0; e < 4; e++)
                                acc[t][c][e] = fmaf(sf[t], raw[e], acc[t][c][e]);
                        }
                    }
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int t = 0; t < T; t++) {
                        s2p_u32x4 wv;
                        if constexpr (WFMT == GEMV_W_INT8) {
                            const s2p_u32x2 lo = deq_s8(w[t].w[i >> 1][2 * (i & 1)]);
                            const s2p_u32x2 hi = deq_s8(w[t].w[i >> 1][2 * (i & 1) + 1]);
                            wv = (s2p_u32x4){lo.x, lo.y, hi.x, hi.y};
                        } else {
                            wv = w[t].w[i];
                        }
#pragma unroll
                        for (int c = 0; c < MTW; c++) acc[t][c] = mfma16x16x32(x[c][i], wv, acc[t][c]);
                    }
            }
        };
        if (nc > 0) {
            load(w0, x0, 0);
            int c = 0;
            for (; c + 2 < nc; c += 2) {
                load(w1, x1, c + 1);
                mul(w0, x0);
                load(w0, x0, c + 2);
                mul(w1, x1);
            }
            if (c + 1 < nc) {
                load(w1, x1, c + 1);
                mul(w0, x0);
                mul(w1, x1);
            } else {
                mul(w0, x0);
            }
        }
        if (g != (int)blockIdx.x) __syncthreads(); /* the last round's sums are read */
        const int slots = a.rg * T * a.mg * MTW; /* partial tiles of a K slice */
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int c = 0; c < MTW; c++)
                *(LDS(s2p_f32x4)*)(red + ((size_t)(kw * slots + (rg * T + t) * (a.mg * MTW) +
                                                   mg * MTW + c) * 64 + lane) * 4) = acc[t][c];
        __syncthreads();
        /* item: four activation rows m = 16 ct + 4 q .. + 3 of weight row r of
         * an output tile */
        const int mtn = a.mg * MTW, items = ntp * mtn * 64;
        for (int it = tid; it < items; it += 64 * GX_WAVES) { /* whole waves */
            const int l = it & 63, tc = it >> 6, j = tc / mtn, ct = tc - j * mtn;
            const int lr = l & 15, m0 = 16 * ct + 4 * (l >> 4);
            const int n = (g * ntp + j) * a.rpt + lr;
            const bool resid = a.epi == GEMV_EPI_RESID;
            const bool ok = m0 < a.M && lr < a.rpt && n < F;
            if (!ok && !resid) continue; /* a residual's 16 lanes stay together */
            const int live = ok ? min(4, a.M - m0) : 0;
            auto total = [&](int tile) __attribute__((always_inline)) {
                s2p_f32x4 v = {0.f, 0.f, 0.f, 0.f};
                for (int k = 0; k < a.kw; k++) {
                    const s2p_f32x4 p = *(const LDS(s2p_f32x4)*)(
                        red + ((size_t)(k * slots + tile * mtn + ct) * 64 + l) * 4);
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] += p[e];
                }
                return v;
            };
            s2p_f32x4 v = total(j), u = v;
            if (sw) u = total(T + j);
            if (a.splits > 1) { /* k_gmx_merge scales and finishes */
                float* pp = a.part + ((size_t)sp * a.M + m0) * a.np + n; /* live rows only */
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (e < live) pp[(size_t)e * a.np] = v[e];
                continue;
            }
            float f = WFMT == GEMV_W_INT4 ? 16.0f : 1.0f, fu = f;
            if constexpr (WFMT == GEMV_W_INT8) {
                f = ((const float*)a.s)[min(n, F - 1)];
                if (sw) fu = ((const float*)a.s)[F + min(n, F - 1)];
            }
            uint16_t* yp = a.y + (size_t)m0 * a.ldy + n;
            uint16_t yo[4] = {0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (resid && e < live) yo[e] = yp[(size_t)e * a.ldy];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float sq = 0.f;
                if (e < live) {
                    const uint16_t b = f2bf(v[e] * f);
                    uint16_t o = b;
                    if (sw) o = silu_mul_bf16(b, f2bf(u[e] * fu));
                    else if (resid) o = f2bf(__fadd_rn(bf2f(yo[e]), bf2f(b)));
                    yp[(size_t)e * a.ldy] = o;
                    sq = bf2f(o) * bf2f(o);
                }
                if (resid && a.ssq_out) { /* rpt is 16: a tile is one block of columns */
                    sq = sum_lanes16(sq);
                    if (lr == 0 && e < live)
                        a.ssq_out[(size_t)(n >> 4) * GEMV_MAX_M + m0 + e] = sq;
                }
            }
        }
    }
}

/* the K splits of a launch, summed in split order, and the epilogue: a thread
 * takes four adjacent outputs of row blockIdx.y */
__global__ __launch_bounds__(256) void k_gmx_merge(GmxArgs a, int wfmt) {
#pragma clang fp contract(off)
    const int m = blockIdx.y, n0 = ((int)blockIdx.x * 256 + (int)threadIdx.x) * 4;
    const int live = min(4, max(0, a.N - n0)); /* 0: past the row, kept for the lane sums */
    const float* p = a.part + (size_t)m * a.np + min(n0, a.np - 4);
    const size_t stride = (size_t)a.M * a.np;
    uint16_t* yp = a.y + (size_t)m * a.ldy + n0;
    uint16_t yo[4] = {0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (a.epi == GEMV_EPI_RESID && e < live) yo[e] = yp[e];
    s2p_f32x4 v = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < a.splits; k0 += 8) {
        s2p_f32x4 t[8];
#pragma unroll
        for (int k = 0; k < 8; k++)
            t[k] = *(const s2p_f32x4*)(p + (size_t)min(k0 + k, a.splits - 1) * stride);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            if (k0 + k >= a.splits) break;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] += t[k][e];
        }
    }
    uint16_t o[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        float f = 1.0f;
        if (wfmt == GEMV_W_INT4) f = 16.0f;
        if (wfmt == GEMV_W_INT8) f = ((const float*)a.s)[min(n0 + e, a.N - 1)];
        o[e] = f2bf(v[e] * f);
        if (a.epi == GEMV_EPI_RESID) o[e] = f2bf(__fadd_rn(bf2f(yo[e]), bf2f(o[e])));
    }
    if (live == 4 && ((uintptr_t)yp & 7) == 0) {
        *(uint64_t*)yp = (uint64_t)o[0] | ((uint64_t)o[1] << 16) | ((uint64_t)o[2] << 32) |
                         ((uint64_t)o[3] << 48);
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (e < live) yp[e] = o[e];
    }
    if (a.epi == GEMV_EPI_RESID && a.ssq_out) { /* 16 columns are four lanes */
        float sq = 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (e < live) sq += bf2f(o[e]) * bf2f(o[e]);
        sq = quad_sum(sq);
        if ((threadIdx.x & 3) == 0 && live > 0) a.ssq_out[(size_t)(n0 >> 4) * GEMV_MAX_M + m] = sq;
    }
}

/* activations into the operand layout: workgroup (ct, part) takes rows 16 ct
 * .. + 15 (past M: the last row) and its share of the chunks.  NORM: the rows
 * become bf16(x * inv_rms(x) * w), the rule's roundings; every part sums the
 * squares of its 16 whole rows itself.  Lane (q, r) of operand i of a chunk
 * holds row r's k values 32 i + 8 q .. + 7 (INT4 in the k-slot order), INT8
 * 64 (i / 2) + 16 q + 8 (i % 2) .. + 7: what the lane's weight bytes pair with */
template <int WFMT, bool NORM>
__global__ __launch_bounds__(512) void k_gmx_pack(const uint16_t* __restrict__ x, int ldx,
                                                  const uint16_t* __restrict__ w,
                                                  uint16_t* __restrict__ xp, int M, int K, int mt,
                                                  float eps) {
#pragma clang fp contract(off)
    __shared__ float s_inv[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ct = blockIdx.x;
    if constexpr (NORM) {
        /* the wave's two rows, every load of up to 2560 k values in flight */
        constexpr int NB = 5;
        const uint16_t* xr[2];
        float s[2] = {0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 2; j++) xr[j] = x + (size_t)min(16 * ct + 2 * wave + j, M - 1) * ldx;
        for (int k0 = 0; k0 < K; k0 += 512 * NB) {
            s2p_u32x4 v[2][NB];
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int b = 0; b < NB; b++)
                    v[j][b] = *(const s2p_u32x4*)(xr[j] + min(k0 + 512 * b + 8 * lane, K - 8));
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int b = 0; b < NB; b++) {
                    if (k0 + 512 * b + 8 * lane >= K) continue;
#pragma unroll
                    for (int d = 0; d < 4; d++) {
                        s[j] = fmaf(bf2f_lo(v[j][b][d]), bf2f_lo(v[j][b][d]), s[j]);
                        s[j] = fmaf(bf2f_hi(v[j][b][d]), bf2f_hi(v[j][b][d]), s[j]);
                    }
                }
        }
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const float t = wave_sum_down(s[j]);
            if (lane == 0) s_inv[2 * wave + j] = rsqrt_rule(t / (float)K + eps);
        }
        __syncthreads();
    }
    const int nck = K / GX_CK, parts = gridDim.y;
    const int ca = nck * (int)blockIdx.y / parts, ce = nck * ((int)blockIdx.y + 1) / parts;
    for (int it = ca * 256 + tid; it < ce * 256; it += 512) {
        const int ck = it >> 8, i = (it >> 6) & 3, q = (it >> 4) & 3, r = it & 15;
        const int k = ck * GX_CK +
                      (WFMT == GEMV_W_INT8 ? 64 * (i >> 1) + 16 * q + 8 * (i & 1) : 32 * i + 8 * q);
        s2p_u32x4 v = *(const s2p_u32x4*)(x + (size_t)min(16 * ct + r, M - 1) * ldx + k);
        if constexpr (NORM) {
            const s2p_u32x4 wv = *(const s2p_u32x4*)(w + k);
            const float inv = s_inv[r];
#pragma unroll
            for (int d = 0; d < 4; d++)
                v[d] = (uint32_t)f2bf(__fmul_rn(__fmul_rn(bf2f_lo(v[d]), inv), bf2f_lo(wv[d]))) |
                       ((uint32_t)f2bf(__fmul_rn(__fmul_rn(bf2f_hi(v[d]), inv), bf2f_hi(wv[d])))
                        << 16);
        }
        if constexpr (WFMT == GEMV_W_INT4) v = int4_order(v);
        *(s2p_u32x4*)(xp + (((size_t)ck * mt + ct) * 256 + (it & 255)) * 8) = v;
    }
}

template <int WFMT, int T, int MTW>
static hipError_t gx_run(const GmxArgs& a, dim3 grid, hipStream_t st) {
    const size_t lds = (size_t)a.kw * a.rg * T * a.mg * MTW * 1024; /* 8 T MTW KB */
    /* once per instantiation (thread-safe static initialisation) */
    static const hipError_t attr =
        hipFuncSetAttribute((const void*)k_gmx<WFMT, T, MTW>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, 8 * T * MTW * 1024);
    (void)attr;
    hipLaunchKernelGGL((k_gmx<WFMT, T, MTW>), grid, dim3(64 * GX_WAVES), lds, st, a);
    return hipGetLastError();
}
template <int WFMT, int T>
static hipError_t gx_mtw(const GmxArgs& a, int mtw, dim3 grid, hipStream_t st) {
    switch (mtw) {
        case 1: return gx_run<WFMT, T, 1>(a, grid, st);
        case 2: return gx_run<WFMT, T, 2>(a, grid, st);
        case 3: return gx_run<WFMT, T, 3>(a, grid, st);
        default: break;
    }
    if constexpr (T < 3) return gx_run<WFMT, T, 4>(a, grid, st);
    return hipErrorInvalidValue;
}
template <int WFMT>
static hipError_t gx_launch(const GmxArgs& a, const GemvArgs& g, int t, int mtw, dim3 grid,
                            hipStream_t st) {
    uint16_t* xp = (uint16_t*)a.x;
    const int nck = a.K / GX_CK;
    /* a workgroup a chunk and 16 rows: the pass is a round trip, not bandwidth.
     * A norm reads its rows once a workgroup: two chunks, a piece a thread
     * (M = 40, K = 2560: 4.5 us; in eight parts with row sums load by load 6.7) */
    const bool norm = g.xmode == GEMV_X_NORM;
    const dim3 pg((unsigned)a.mt, (unsigned)(norm ? (nck + 1) / 2 : (nck < 32 ? nck : 32)));
    if (norm)
        hipLaunchKernelGGL((k_gmx_pack<WFMT, true>), pg, dim3(512), 0, st, g.x, g.ldx, g.norm_w, xp,
                           a.M, a.K, a.mt, g.norm_eps);
    else
        hipLaunchKernelGGL((k_gmx_pack<WFMT, false>), pg, dim3(512), 0, st, g.x, g.ldx, nullptr, xp,
                           a.M, a.K, a.mt, 0.f);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (t == 1) e = gx_mtw<WFMT, 1>(a, mtw, grid, st);
    else if (t == 2) e = gx_mtw<WFMT, 2>(a, mtw, grid, st);
    else if constexpr (WFMT != GEMV_W_BF16) e = gx_mtw<WFMT, 3>(a, mtw, grid, st);
    else return hipErrorInvalidValue;
    if (e != hipSuccess || a.splits == 1) return e;
    hipLaunchKernelGGL(k_gmx_merge, dim3((unsigned)((a.N + 1023) / 1024), (unsigned)a.M), dim3(256),
                       0, st, a, WFMT);
    return hipGetLastError();
}

/* shapes in reach of this GEMM that another engine runs faster (M from 17 on,
 * weights not resident, merges and packing included) */
static bool gx_other(const GemvArgs& g) {
    const int64_t km = (int64_t)g.K * g.M;
    if (g.wfmt == GEMV_W_BF16) /* one launch of k_gemv3 against two and the merge: N = K = 1024,
                                * M = 17 8.1 us against 10.2, M = 32 10.0 and 10.3; N = 6144,
                                * M = 17 11.2 and 10.9; K = 512, N = 4096, M = 17 7.8 and 8.3 */
        return g.N <= 4096 && g.K >= 512 && g.K <= 1024 && g.M <= (g.K > 512 ? 32 : 20);
    if (g.wfmt != GEMV_W_INT4 || g.M > 96) return false;
    /* INT4 at M <= 96: k_gemm4, which stages the row-major activations itself.
     * Few rows, whose K both split: at M = 40 wqkv 16 us against 18, w2 20.4
     * against 20.5 (with the merges; gate_up 33.5 against 27.8) */
    if (g.N < GX_MIN_ROWS) return true;
    /* little K: the packing launch shows (K = 512, N = 19456, M = 17: 7.0 against
     * 9.0; M = 64: 12.7 and 11.9; K = 1024, N = 18742, M = 17: 10.1 against 11.1) */
    if (km <= 512 * 24 || (g.N > 16384 && km <= 1024 * 33)) return true;
    /* k_gemm4 still in one round where six tiles a CU are two here (K = 2560, N =
     * 30000: M = 17 21.5 us against 27.0, M = 96 48.1 and 48.0), in two where they
     * are three (N = 60000: M = 17 40.6 against 46.5, M = 80 87.4 and 91.0, M = 96
     * 94.5 and 90.9), and with two activation tiles in five where they are seven
     * (the head's 155776 rows: M = 17 97.9 against 102.7) */
    const int cus = s2p_cu_count();
    const int r = (g.N + 96 * cus - 1) / (96 * cus), r4 = (g.N + 128 * cus - 1) / (128 * cus);
    return r > r4 && (r == 2 || (r == 3 && g.M <= 80) || (5 * r >= 7 * r4 && g.M <= 24));
}

/* the calls that this GEMM takes: 16 < M <= 128, K a multiple of 128, room for
 * the packed activations (16 ceil(M / 16) x K bf16) in part */
extern "C" int s2p_gmx_takes(const GemvArgs* g) {
    return g->M > 16 && g->M <= GEMV_MAX_M && !(g->K & 127) && g->N > 0 && g->part &&
           (int64_t)((g->M + 15) / 16) * 8 * g->K <= g->part_cap && !gx_other(*g);
}

/* hipErrorNotSupported where it does not; part holds the packed activations and
 * then the K splits' partials */
extern "C" hipError_t s2p_gmx_launch(const GemvArgs* ap, hipStream_t st) {
    const GemvArgs& g = *ap;
    if (!s2p_gmx_takes(ap)) return hipErrorNotSupported;
    const bool swiglu = g.epi == GEMV_EPI_SWIGLU;
    GmxArgs a = {};
    a.w = g.w;
    a.s = g.s;
    a.y = g.y;
    a.ldy = g.ldy;
    a.M = g.M;
    a.N = g.N;
    a.K = g.K;
    a.epi = g.epi;
    a.ssq_out = g.ssq_out;
    a.mt = (g.M + 15) / 16;
    a.x = (const uint16_t*)g.part;
    const int64_t xf = (int64_t)a.mt * 8 * g.K; /* floats of the packed activations */
    a.part = g.part + xf;
    const int cus = s2p_cu_count(), nck = g.K / GX_CK;
    const int rows = swiglu ? g.N >> 1 : g.N;
    const int tiles16 = (rows + 15) / 16;
    /* tiles a wave: up to three (bf16: two) */
    const int tmax = g.wfmt == GEMV_W_BF16 ? 2 : 3;
    a.rg = 2;
    int t;
    int rounds = 1;
    /* activation tiles: up to four a wave (three beside three weight tiles),
     * else in groups of waves; the waves left over are K slices */
    auto wave_grid = [&]() {
        const int mw = t == 3 ? 3 : 4;
        a.mg = a.mt <= mw ? 1 : a.mt <= 2 * mw ? 2 : 4;
        a.kw = GX_WAVES / (a.rg * a.mg);
    };
    if (swiglu || tiles16 >= tmax * cus) {
        /* enough rows: one round of workgroups over the whole of K, dealt out
         * evenly, or as few rounds as the tiles allow */
        const int per_cu = (tiles16 + cus - 1) / cus, most = swiglu ? tmax : 2 * tmax;
        rounds = (per_cu + most - 1) / most;
        int ot = (per_cu + rounds - 1) / rounds;
        t = swiglu ? ot : (ot + a.rg - 1) / a.rg;
        ot = swiglu ? t : t * a.rg;
        a.rpt = g.epi == GEMV_EPI_RESID /* tiles of the sums' 16 columns */
                    ? 16
                    : ((rows + cus * rounds - 1) / (cus * rounds) + ot - 1) / ot;
        a.splits = 1;
        wave_grid();
    } else {
        /* few rows: blocks of 2 t tiles, K split over the remaining workgroups */
        t = tiles16 >= 256 ? tmax : 2;
        a.rpt = 16;
        wave_grid();
        const int blocks = (tiles16 + 2 * t - 1) / (2 * t);
        int sp = cus / blocks;
        if (sp > nck / a.kw) sp = nck / a.kw; /* a chunk for each of a workgroup's K slices: INT8, 17
                                           * rows, N = 512, K = 4096 in 8 splits 11.2 us, in 32 17.0 */
        if (sp < 1) sp = 1;
        a.np = (g.N + 3) & ~3;
        while (sp > 1 && xf + (int64_t)sp * g.M * a.np > g.part_cap) sp--;
        a.splits = sp;
    }
    const int ot = swiglu ? t : t * a.rg;
    const int tiles = (rows + a.rpt - 1) / a.rpt;
    a.groups = (tiles + ot - 1) / ot;
    const int mtw = (a.mt + a.mg - 1) / a.mg;
    const dim3 grid((unsigned)(a.groups < cus ? a.groups : cus), (unsigned)a.splits);
    switch (g.wfmt) {
        case GEMV_W_INT4: return gx_launch<GEMV_W_INT4>(a, g, t, mtw, grid, st);
        case GEMV_W_INT8: return gx_launch<GEMV_W_INT8>(a, g, t, mtw, grid, st);
        default: return gx_launch<GEMV_W_BF16>(a, g, t, mtw, grid, st);
    }
}
