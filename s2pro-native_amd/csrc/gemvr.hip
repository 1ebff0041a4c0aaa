/* s2pro MI355X — the M <= 16 GEMV of the quantised and bf16 linears: weights
 * straight from HBM into MFMA operands, all of a workgroup's loads in flight
 * at once.
 *
 * What bounds it: the weight stream (25 MB for an INT8 w2, 50 MB for its
 * gate/up) and, below ~10 MB, the launch itself.  So nothing stands between a
 * load and its multiply and no round trip is exposed but the first:
 *   - one workgroup a CU; its waves split K, every wave streams its slice of
 *     all rows of the workgroup's tiles;
 *   - one 16-byte load of a wave covers 128 bytes (a full cache line) of 8
 *     rows; 64 bytes of 16 rows, the MFMA's own shape, streamed 50 MB in 12.2
 *     us where this takes 9.1.  Lane (q, r) = (lane / 16, lane % 16) holds row
 *     r % 8, 16-byte chunk 2 q + r / 8;
 *   - M <= 8: a tile is 8 rows.  As the B operand, columns r < 8 carry the
 *     even chunks of the 8 rows and columns r >= 8 the odd ones; the A operand
 *     holds the up to 8 activation rows the same way (rows < 8 at the even
 *     chunks, rows >= 8 the same rows at the odd ones), so the two diagonal
 *     quadrants of one MFMA are the products of 8 x 8 (row, activation) pairs
 *     over all 8 chunks; they are added at the end;
 *   - M > 8 (WIDE): a tile is 16 rows, two loads; a rotation by 8 lanes
 *     exchanges their halves into an operand of all rows' even chunks and one
 *     of the odd ones;
 *   - K is permuted alike on both sides.  INT8: the 16 codes of a chunk feed
 *     two MFMAs.  BF16: 8 weights feed one.  INT4: a chunk is one 32-k scale
 *     group; four permlane swaps exchange the lane quarters, so each of the
 *     load's four MFMAs covers one group a column;
 *   - the activations go from L2 to registers once per workgroup (k_gvr), or
 *     stream beside the weights (K > 4096: k_gvs);
 *   - RMSNorm: the rows' sums of squares come from the same registers, one
 *     exchange through LDS.  Only the first tile's weights are issued before
 *     it: behind all of them the activations arrive late and the multiplies
 *     start when the stream is nearly over (INT8 gate/up at M = 4: 14.1 us with
 *     all ten tiles first, 12.7 with one to six; wqkv 6.9 with all three, 6.2
 *     with one);
 *   - INT8 codes convert exactly (signed byte -> f32 -> bf16, no bias term);
 *     INT4 nibbles become 1.5 + w / 16, and the bias -1.5 sum x of a group is
 *     an MFMA against a constant, the C operand of the group's product;
 *   - the waves' partial tiles meet in LDS and are summed in wave order by
 *     one thread per output (deterministic), which runs the epilogue. */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemv_dev.h"

struct GvrArgs {
    const uint8_t* w;
    const void* s;
    const uint16_t* x;
    uint16_t* y;
    const uint16_t* norm_w;
    float* ssq_out;
    int ldx, ldy, M, N, K, epi;
    float norm_eps;
    int rpt;    /* output rows a tile, at most its 8 (WIDE: 16) */
    int groups; /* tile groups, one a workgroup and round */
};

static __host__ __device__ constexpr int gr_rows(bool wide) { return wide ? 16 : 8; }
/* k values per unit (128 bytes of a row) and MFMAs, i.e. 16-byte activation
 * operands, per unit */
static __host__ __device__ constexpr int gr_uk(int wfmt) {
    return wfmt == GEMV_W_INT4 ? 256 : wfmt == GEMV_W_INT8 ? 128 : 64;
}
static __host__ __device__ constexpr int gr_nx(int wfmt, bool wide) {
    return gr_uk(wfmt) / (wide ? 32 : 64);
}

/* one unit of one tile: the lane's chunk (WIDE: of rows r % 8 and
 * 8 + r % 8), INT4 also the 8 group scales of row r % 8 (WIDE: r) */
template <int WFMT, bool WIDE>
struct GvrUnit {
    s2p_u32x4 w[WIDE ? 2 : 1];
};
template <bool WIDE>
struct GvrUnit<GEMV_W_INT4, WIDE> {
    s2p_u32x4 w[WIDE ? 2 : 1];
    s2p_u32x4 s;
};

/* a tile: scalar bases of its first row (at unit u0), and the lane's byte
 * offsets: weight rows (one a load) and the row of its INT4 scales */
template <int WFMT, bool WIDE>
struct GvrTile {
    GblPtr w, s;
    uint32_t wl[WIDE ? 2 : 1], sl;
};

/* unit u (past the tile's u0) of tile t */
template <int WFMT, bool WIDE>
S2P_DEV void gr_load(GvrUnit<WFMT, WIDE>& b, const GvrTile<WFMT, WIDE>& t, int u) {
#pragma unroll
    for (int i = 0; i < (WIDE ? 2 : 1); i++)
        b.w[i] = gbl_at<s2p_u32x4, true>(t.w + u * 128, t.wl[i]);
    if constexpr (WFMT == GEMV_W_INT4) b.s = gbl_at<s2p_u32x4>(t.s + u * 16, t.sl);
}

/* activation operand j of unit u: the k values its MFMA pairs with the
 * chunk's.  gr_klane: the lane's byte offset inside a unit */
template <int WFMT, bool WIDE>
S2P_DEV uint32_t gr_klane(int q, int hi) {
    if (WIDE) hi = 0;
    return WFMT == GEMV_W_INT4   ? 64u * hi + 16u * q
           : WFMT == GEMV_W_INT8 ? 32u * (2 * q + hi)
                                 : 16u * (2 * q + hi);
}
/* WIDE: operands 0 .. NX / 2 - 1 go with the even chunks, the rest with the
 * odd; u: units past the base */
template <int WFMT, bool WIDE>
S2P_DEV s2p_u32x4 gr_ldx(GblPtr x, uint32_t xl, int u, int j) {
    constexpr int H = gr_nx(WFMT, false), ODD = WFMT == GEMV_W_INT4 ? 64 : WFMT == GEMV_W_INT8 ? 32 : 16;
    const int jj = WIDE ? j % H : j, odd = WIDE ? j / H : 0;
    return gbl_at<s2p_u32x4>(
        x + u * (2 * gr_uk(WFMT)) + jj * (WFMT == GEMV_W_INT4 ? 128 : 16) + odd * ODD, xl);
}
/* lanes r < 8 of a, lanes r >= 8 from lanes r - 8 of b; and lanes r < 8 from
 * lanes r + 8 of a, lanes r >= 8 of b (DPP row_ror:8 on half the banks) */
S2P_DEV uint32_t gr_lo(uint32_t a, uint32_t b) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)a, (int)b, 0x128, 0xF, 0xC, false);
}
S2P_DEV uint32_t gr_hi(uint32_t a, uint32_t b) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)b, (int)a, 0x128, 0xF, 0x3, false);
}

/* acc += activations . one 16-byte chunk a lane against operands x[0 ..
 * NX - 1].  INT4: acc holds 1/16 of the sum, cb is the bias MFMA of each
 * group, and the scale of MFMA j sits at bit sh of s[j]. */
template <int WFMT>
S2P_DEV void gr_chunk(s2p_u32x4 w, const s2p_u32x4* x, const s2p_f32x4* cb, s2p_u32x4 s,
                      uint32_t sh, s2p_f32x4& acc) {
    if constexpr (WFMT == GEMV_W_INT4) {
        uint32_t kmask = 0x00780078u, kone = 0x3F803F80u;
        asm volatile("" : "+v"(kmask), "+v"(kone));
        uint32_t d0 = w.x, d1 = w.y, d2 = w.z, d3 = w.w;
        xpose4(d0, d1, d2, d3);
        const uint32_t dj[4] = {d0, d1, d2, d3};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float sf = (float)__builtin_bit_cast(_Float16, (uint16_t)(s[j] >> sh));
            const s2p_f32x4 raw = mfma16x16x32(x[j], deq_int4(dj[j], kmask, kone), cb[j]);
#pragma unroll
            for (int i = 0; i < 4; i++) acc[i] = fmaf(sf, raw[i], acc[i]);
        }
    } else if constexpr (WFMT == GEMV_W_INT8) {
        const s2p_u32x2 a0 = deq_s8(w.x), a1 = deq_s8(w.y), a2 = deq_s8(w.z), a3 = deq_s8(w.w);
        acc = mfma16x16x32(x[0], (s2p_u32x4){a0.x, a0.y, a1.x, a1.y}, acc);
        acc = mfma16x16x32(x[1], (s2p_u32x4){a2.x, a2.y, a3.x, a3.y}, acc);
    } else {
        acc = mfma16x16x32(x[0], w, acc);
    }
}
/* acc += activations . unit; hi: the lane holds odd chunks */
template <int WFMT, bool WIDE>
S2P_DEV void gr_mul(const GvrUnit<WFMT, WIDE>& b, const s2p_u32x4 (&x)[gr_nx(WFMT, WIDE)],
                    const s2p_f32x4 (&cb)[gr_nx(WFMT, WIDE)], int hi, s2p_f32x4& acc) {
    s2p_u32x4 s = {0u, 0u, 0u, 0u};
    if constexpr (WFMT == GEMV_W_INT4) s = b.s;
    if constexpr (!WIDE) {
        gr_chunk<WFMT>(b.w[0], x, cb, s, 16u * hi, acc);
    } else {
        constexpr int H = gr_nx(WFMT, false);
        s2p_u32x4 e, o;
#pragma unroll
        for (int d = 0; d < 4; d++) {
            e[d] = gr_lo(b.w[0][d], b.w[1][d]);
            o[d] = gr_hi(b.w[0][d], b.w[1][d]);
        }
        gr_chunk<WFMT>(e, x, cb, s, 0u, acc);
        gr_chunk<WFMT>(o, x + H, cb + H, s, 16u, acc);
    }
}

/* the bias operands of a unit (INT4): -1.5 x the groups' activation sums,
 * already in the C layout */
template <int WFMT, int NX>
S2P_DEV void gr_bias(const s2p_u32x4 (&x)[NX], s2p_f32x4 (&cb)[NX]) {
    if constexpr (WFMT == GEMV_W_INT4) {
        const s2p_u32x4 k15 = {0xBFC0BFC0u, 0xBFC0BFC0u, 0xBFC0BFC0u, 0xBFC0BFC0u};
#pragma unroll
        for (int j = 0; j < NX; j++)
            cb[j] = mfma16x16x32(x[j], k15, (s2p_f32x4){0.f, 0.f, 0.f, 0.f});
    }
}

/* a streaming wave's units [u0, u0 + nu): the remainder goes to the first waves, so
 * that a SIMD (waves w, w + 4, ..) gets its share of it */
template <int NW>
S2P_DEV void gr_split(int units, int wave, int& u0, int& nu) {
    const int base = units / NW, rem = units - base * NW;
    nu = base + (wave < rem ? 1 : 0);
    u0 = wave * base + min(wave, rem);
}

/* tile j of group g (ntp output tiles a group, then SWIGLU's up tiles) from
 * unit u0 on; rows past the end repeat the last one, their outputs are
 * dropped */
template <int WFMT, bool WIDE>
S2P_DEV GvrTile<WFMT, WIDE> gr_tile(const GvrArgs& a, int g, int j, int ntp, int u0, int r, int q) {
    const bool sw = a.epi == GEMV_EPI_SWIGLU;
    const int F = sw ? a.N >> 1 : a.N;
    const int up = j >= ntp ? 1 : 0;
    const int n0 = min((g * ntp + (up ? j - ntp : j)) * a.rpt, F - 1);
    const int last = min(a.rpt, F - n0) - 1;
    const uint64_t row0 = (uint64_t)(n0 + (up ? F : 0));
    const uint32_t rb = (uint32_t)(WFMT == GEMV_W_INT4   ? a.K >> 1
                                   : WFMT == GEMV_W_INT8 ? a.K
                                                         : a.K * 2); /* bytes of a row */
    const uint32_t ch = 16u * (2 * q + (r >> 3));
    GvrTile<WFMT, WIDE> t;
    t.w = gbl_base(a.w, row0 * rb + (uint64_t)u0 * 128);
    t.wl[0] = (uint32_t)min(r & 7, last) * rb + ch;
    if constexpr (WIDE) t.wl[1] = (uint32_t)min(8 + (r & 7), last) * rb + ch;
    if constexpr (WFMT == GEMV_W_INT4) {
        const uint32_t sb = (uint32_t)(a.K >> 4);
        t.s = gbl_base(a.s, row0 * sb + (uint64_t)u0 * 16);
        t.sl = (uint32_t)min(WIDE ? r : (r & 7), last) * sb;
    }
    return t;
}

/* a wave's partial tile into red, element i of lane (q, r) in 16-byte slots.
 * WIDE: (m, n) = (4 q + i, r) at slot [q][r]; narrow: the two diagonal
 * quadrants, q < 2 with r < 8 and q >= 2 with r >= 8, at slot [q][r % 8]: two
 * halves of 8 x 8, 64 floats apart, that the epilogue adds */
static __host__ __device__ constexpr int gr_ts(bool wide) { return wide ? 256 : 128; }
template <bool WIDE>
S2P_DEV void gr_put(LDS(float)* red, s2p_f32x4 v, int lane) {
    const int q = lane >> 4, r = lane & 15;
    if constexpr (WIDE) *(LDS(s2p_f32x4)*)(red + (q * 16 + r) * 4) = v;
    else if ((q >> 1) == (r >> 3)) *(LDS(s2p_f32x4)*)(red + (q * 8 + (r & 7)) * 4) = v;
}

/* (tile of the group, m, row of the tile) of item idx: tile by tile, or, for
 * a residual output, with the 16 columns of a sum of squares (a WIDE tile, a
 * pair of narrow ones) in adjacent lanes */
template <bool WIDE>
S2P_DEV void gr_item(const GvrArgs& a, int idx, int& j, int& m, int& c) {
    if (WIDE || a.epi == GEMV_EPI_RESID) {
        const int t = (idx >> 4) / a.M;
        m = (idx >> 4) - t * a.M;
        j = WIDE ? t : 2 * t + ((idx >> 3) & 1);
        c = idx & (WIDE ? 15 : 7);
    } else {
        j = (idx >> 3) / a.M;
        m = (idx >> 3) - j * a.M;
        c = idx & 7;
    }
}

/* the waves' partials red [NT][NW][tile] -> outputs of group g; yold: the
 * residual value of the thread's first item */
template <int WFMT, int NW, bool WIDE, bool SW>
S2P_DEV void gr_epilogue(const GvrArgs& a, const LDS(float)* red, int g, int ntp, int tid,
                         uint16_t yold) {
#pragma clang fp contract(off)
    constexpr int ROWS = gr_rows(WIDE), TS = gr_ts(WIDE);
    const bool sw = SW && a.epi == GEMV_EPI_SWIGLU;
    const int F = sw ? a.N >> 1 : a.N;
    const int items = ntp * ROWS * a.M;
    for (int i0 = 0; i0 < items; i0 += 64 * NW) {
        int j, m, c;
        gr_item<WIDE>(a, i0 + tid, j, m, c);
        const int n = (g * ntp + j) * a.rpt + c;
        const bool ok = i0 + tid < items && c < a.rpt && n < F;
        const int src = ((m >> 2) * ROWS + c) * 4 + (m & 3);
        auto total = [&](int t) __attribute__((always_inline)) {
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < NW; w++) {
                const LDS(float)* p = red + (t * NW + w) * TS + src;
                v += WIDE ? p[0] : p[0] + p[64];
            }
            return WFMT == GEMV_W_INT4 ? 16.0f * v : v;
        };
        uint16_t* yp = a.y + (size_t)m * a.ldy + n;
        if (sw) {
            if (!ok) continue;
            float gv = total(j), uv = total(ntp + j);
            if (WFMT == GEMV_W_INT8) {
                gv *= ((const float*)a.s)[n];
                uv *= ((const float*)a.s)[F + n];
            }
            *yp = silu_mul_bf16(f2bf(gv), f2bf(uv));
            continue;
        }
        float sq = 0.f;
        if (ok) {
            float v = total(j);
            if (WFMT == GEMV_W_INT8) v *= ((const float*)a.s)[n];
            const uint16_t yb = f2bf(v);
            if (a.epi == GEMV_EPI_RESID) {
                const uint16_t xo = f2bf(__fadd_rn(bf2f(i0 == 0 ? yold : *yp), bf2f(yb)));
                *yp = xo;
                sq = bf2f(xo) * bf2f(xo);
            } else {
                *yp = yb;
            }
        }
        if (a.epi == GEMV_EPI_RESID && a.ssq_out) {
            const float tot = sum_lanes16(sq);
            if ((tid & 15) == 0 && ok) a.ssq_out[(size_t)(n >> 4) * GEMV_MAX_M + m] = tot;
        }
    }
}

/* the residual value of the thread's first output of group g: loaded
 * unconditionally (a clamped address, not used otherwise), so that its wait
 * stays with its use and not behind the weights */
template <bool WIDE>
S2P_DEV uint16_t gr_yold(const GvrArgs& a, int g, int ntp, int tid) {
    const int F = a.epi == GEMV_EPI_SWIGLU ? a.N >> 1 : a.N;
    int j, m, c;
    gr_item<WIDE>(a, tid, j, m, c);
    return a.y[(size_t)min(m, a.M - 1) * a.ldy + min((g * ntp + j) * a.rpt + c, F - 1)];
}

/* every argument in one round of scalar loads: left to itself the compiler
 * issues them next to their first uses, several dependent round trips before
 * the first weight load */
S2P_DEV void gr_args(const GvrArgs& a) {
    asm volatile("" ::"s"(a.w), "s"(a.s), "s"(a.x), "s"(a.y), "s"(a.norm_w), "s"(a.ssq_out),
                 "s"(a.ldx), "s"(a.ldy), "s"(a.M), "s"(a.N), "s"(a.K), "s"(a.epi), "s"(a.norm_eps),
                 "s"(a.rpt), "s"(a.groups));
}

/* the activations stay in registers (U units a wave), NT tiles a round, the
 * next round's loads issued as this round's tiles are consumed */
template <int WFMT, int NW, int U, int NT, bool WIDE, bool NORM, bool TAIL>
__global__ __launch_bounds__(64 * NW) void k_gvr(GvrArgs a) {
#pragma clang fp contract(off)
    constexpr int NX = gr_nx(WFMT, WIDE), TS = gr_ts(WIDE);
    gr_args(a);
    extern __shared__ __align__(16) unsigned char gr_smem[];
    LDS(float)* red = (LDS(float)*)gr_smem; /* [2 if rounds > 1][NT][NW][TS] */
    __shared__ float s_ssq[NORM ? NW : 1][16];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, r = lane & 15, hi = r >> 3;
    /* K is NW x U units; TAIL: NW x (U - 1) and some more, one of which waves
     * < rem take (the others load their own last unit again and skip it) */
    int u0 = wave * U, nu = U;
    if constexpr (TAIL) gr_split<NW>(a.K / gr_uk(WFMT), wave, u0, nu);
    auto ui = [&](int u) __attribute__((always_inline)) {
        return TAIL && u == U - 1 ? nu - 1 : u;
    };
    const int ntp = a.epi == GEMV_EPI_SWIGLU ? NT / 2 : NT;

    /* activations first (the loads return in order); lanes past M hold
     * zeros and load nothing */
    s2p_u32x4 x[U][NX], wn[NORM ? U : 1][NX];
    const uint32_t kl = gr_klane<WFMT, WIDE>(q, hi);
    const int mrow = WIDE ? r : (r & 7);
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
        for (int j = 0; j < NX; j++) x[u][j] = (s2p_u32x4){0u, 0u, 0u, 0u};
    if (mrow < a.M) {
        const GblPtr xb = gbl_base(a.x, (uint64_t)u0 * (2 * gr_uk(WFMT)));
        const uint32_t xl = (uint32_t)mrow * (uint32_t)a.ldx * 2u + kl;
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int j = 0; j < NX; j++) x[u][j] = gr_ldx<WFMT, WIDE>(xb, xl, ui(u), j);
    }
    if constexpr (NORM) {
        const GblPtr nb = gbl_base(a.norm_w, (uint64_t)u0 * (2 * gr_uk(WFMT)));
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int j = 0; j < NX; j++) wn[u][j] = gr_ldx<WFMT, WIDE>(nb, kl, u, j);
    }
    int g = blockIdx.x;
    uint16_t yold = gr_yold<WIDE>(a, g, ntp, tid);
    GvrUnit<WFMT, WIDE> b[NT][U];
    auto load = [&](int gg, int j) __attribute__((always_inline)) {
        const GvrTile<WFMT, WIDE> t = gr_tile<WFMT, WIDE>(a, gg, j, ntp, u0, r, q);
#pragma unroll
        for (int u = 0; u < U; u++) gr_load<WFMT, WIDE>(b[j][u], t, ui(u));
    };
    constexpr int PRE = NORM ? 1 : NT;
#pragma unroll
    for (int j = 0; j < PRE; j++) load(g, j);
    /* these loads are out before anything waits for the activations (the
     * scheduler puts the first instructions on x, and their wait, between) */
    __builtin_amdgcn_sched_barrier(0);

    if constexpr (NORM) {
        /* sums of squares of the rows over this wave's slice, then the waves */
        float s = 0.f;
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int j = 0; j < NX; j++)
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    const float lo = bf2f_lo(x[u][j][d]), up = bf2f_hi(x[u][j][d]);
                    s = fmaf(lo, lo, s);
                    s = fmaf(up, up, s);
                }
        if constexpr (!WIDE) s += dpp_f<0x128>(s); /* row_ror:8: the other chunks of the row */
        s += __shfl_xor(s, 16, 64);
        s += __shfl_xor(s, 32, 64);
        if (lane < 16) s_ssq[wave][lane] = s;
        __syncthreads();
#pragma unroll
        for (int j = PRE; j < NT; j++) load(g, j);
        __builtin_amdgcn_sched_barrier(0);
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < NW; w++) t += s_ssq[w][r];
        const float inv = rsqrt_rule(t / (float)a.K + a.norm_eps);
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int j = 0; j < NX; j++)
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    const uint32_t v = x[u][j][d], w = wn[u][j][d];
                    const uint32_t lo = f2bf(__fmul_rn(__fmul_rn(bf2f_lo(v), inv), bf2f_lo(w)));
                    const uint32_t up = f2bf(__fmul_rn(__fmul_rn(bf2f_hi(v), inv), bf2f_hi(w)));
                    x[u][j][d] = lo | (up << 16);
                }
    }
    s2p_f32x4 cb[U][NX];
#pragma unroll
    for (int u = 0; u < U; u++) {
#pragma unroll
        for (int j = 0; j < NX; j++) x[u][j] = WFMT == GEMV_W_INT4 ? int4_order(x[u][j]) : x[u][j];
        if constexpr (!TAIL) gr_bias<WFMT, NX>(x[u], cb[u]);
    }

    auto mul = [&](int j, LDS(float)* rd) __attribute__((always_inline)) {
        s2p_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < U; u++)
            gr_mul<WFMT, WIDE>(b[j][u], x[u], cb[u], hi, acc);
        gr_put<WIDE>(rd + (j * NW + wave) * TS, acc, lane);
    };
    constexpr bool SW = (NT & 1) == 0;
    int par = 0;
    if constexpr (!TAIL)
    for (; g + (int)gridDim.x < a.groups; g += gridDim.x) {
        LDS(float)* rd = red + par * (NT * NW * TS);
        const uint16_t ynext = gr_yold<WIDE>(a, g + (int)gridDim.x, ntp, tid);
#pragma unroll
        for (int j = 0; j < NT; j++) {
            mul(j, rd);
            load(g + gridDim.x, j);
        }
        __syncthreads();
        gr_epilogue<WFMT, NW, WIDE, SW>(a, rd, g, ntp, tid, yold);
        yold = ynext;
        par ^= 1;
    }
    LDS(float)* rd = red + par * (NT * NW * TS);
    if constexpr (!TAIL) {
#pragma unroll
        for (int j = 0; j < NT; j++) mul(j, rd);
    } else { /* one round; unit by unit, its bias operands for all tiles */
        s2p_f32x4 acc[NT];
#pragma unroll
        for (int j = 0; j < NT; j++) acc[j] = (s2p_f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (u >= nu) break; /* uniform */
            gr_bias<WFMT, NX>(x[u], cb[u]);
#pragma unroll
            for (int j = 0; j < NT; j++) gr_mul<WFMT, WIDE>(b[j][u], x[u], cb[u], hi, acc[j]);
        }
#pragma unroll
        for (int j = 0; j < NT; j++) gr_put<WIDE>(rd + (j * NW + wave) * TS, acc[j], lane);
    }
    __syncthreads();
    gr_epilogue<WFMT, NW, WIDE, SW>(a, rd, g, ntp, tid, yold);
}

/* streamed kernel: waves, 16 rows a round, and units per chunk (three chunks
 * of weights and their activations in registers) */
#define GS_WAVES 8
static __host__ __device__ constexpr int gs_nt(bool wide) { return wide ? 1 : 2; }
static __host__ __device__ constexpr int gs_cu(int wfmt) {
    return wfmt == GEMV_W_INT4 ? 1 : wfmt == GEMV_W_INT8 ? 2 : 3;
}
template <int WFMT, bool WIDE>
struct GvrChunk {
    GvrUnit<WFMT, WIDE> b[gs_cu(WFMT)][gs_nt(WIDE)];
    s2p_u32x4 x[gs_cu(WFMT)][gr_nx(WFMT, WIDE)];
};

/* any K, 16 rows a round, plain activations: chunks of weights and their
 * activations, two chunks in flight behind the one that is multiplied */
template <int WFMT, bool WIDE>
__global__ __launch_bounds__(64 * GS_WAVES) void k_gvs(GvrArgs a) {
#pragma clang fp contract(off)
    constexpr int NX = gr_nx(WFMT, WIDE), C = gs_cu(WFMT), NW = GS_WAVES, NT = gs_nt(WIDE);
    constexpr int TS = gr_ts(WIDE);
    gr_args(a);
    __shared__ __align__(16) float s_red[2][NT * NW * TS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, r = lane & 15, hi = r >> 3;
    int u0, nu;
    gr_split<NW>(a.K / gr_uk(WFMT), wave, u0, nu);
    const int nch = (nu + C - 1) / C;
    const int rounds = (a.groups - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
    /* rows past M repeat the last one, their outputs are dropped */
    const uint32_t xl = (uint32_t)min(WIDE ? r : (r & 7), a.M - 1) * (uint32_t)a.ldx * 2u +
                        gr_klane<WFMT, WIDE>(q, hi);
    const GblPtr xb = gbl_base(a.x, (uint64_t)u0 * (2 * gr_uk(WFMT)));

    /* chunk t of the current round (past the slice: its last unit again) */
    GvrTile<WFMT, WIDE> tl[NT];
    auto at_group = [&](int g) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NT; j++) tl[j] = gr_tile<WFMT, WIDE>(a, g, j, NT, u0, r, q);
    };
    auto load = [&](GvrChunk<WFMT, WIDE>& c, int t) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < C; i++) {
            const int u = min(t * C + i, nu - 1);
#pragma unroll
            for (int j = 0; j < NT; j++) gr_load<WFMT, WIDE>(c.b[i][j], tl[j], u);
#pragma unroll
            for (int j = 0; j < NX; j++) c.x[i][j] = gr_ldx<WFMT, WIDE>(xb, xl, u, j);
        }
    };
    s2p_f32x4 acc[NT];
    auto step = [&](const GvrChunk<WFMT, WIDE>& c, int t) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < C; i++) {
            if (t * C + i >= nu) break; /* uniform */
            s2p_u32x4 x[NX];
            s2p_f32x4 cb[NX];
#pragma unroll
            for (int j = 0; j < NX; j++) x[j] = WFMT == GEMV_W_INT4 ? int4_order(c.x[i][j]) : c.x[i][j];
            gr_bias<WFMT, NX>(x, cb);
#pragma unroll
            for (int j = 0; j < NT; j++) gr_mul<WFMT, WIDE>(c.b[i][j], x, cb, hi, acc[j]);
            __builtin_amdgcn_sched_barrier(0); /* one unit's operands live at a time */
        }
    };
    GvrChunk<WFMT, WIDE> c0, c1, c2;
    int g = blockIdx.x;
    uint16_t yold = gr_yold<WIDE>(a, g, NT, tid);
    at_group(g);
    load(c0, 0);
    load(c1, 1);
    load(c2, 2);
    for (int rd = 0; rd < rounds; rd++, g += (int)gridDim.x) {
#pragma unroll
        for (int j = 0; j < NT; j++) acc[j] = (s2p_f32x4){0.f, 0.f, 0.f, 0.f};
        int t = 0;
        for (; t + 5 < nch; t += 3) {
            step(c0, t);
            load(c0, t + 3);
            step(c1, t + 1);
            load(c1, t + 4);
            step(c2, t + 2);
            load(c2, t + 5);
        }
        /* at most 5 chunks left, the first three loaded or loading */
        step(c0, t);
        if (t + 3 < nch) load(c0, t + 3);
        step(c1, t + 1);
        if (t + 4 < nch) load(c1, t + 4);
        step(c2, t + 2);
        step(c0, t + 3);
        step(c1, t + 4);
        uint16_t ynext = 0;
        if (rd + 1 < rounds) { /* the next rows' first chunks, in flight over the epilogue */
            ynext = gr_yold<WIDE>(a, g + (int)gridDim.x, NT, tid);
            at_group(g + (int)gridDim.x);
            load(c0, 0);
            load(c1, 1);
            load(c2, 2);
        }
        LDS(float)* red = (LDS(float)*)s_red[rd & 1];
#pragma unroll
        for (int j = 0; j < NT; j++) gr_put<WIDE>(red + (j * NW + wave) * TS, acc[j], lane);
        __syncthreads();
        gr_epilogue<WFMT, NW, WIDE, false>(a, red, g, NT, tid, yold);
        yold = ynext;
    }
}

template <int WFMT, int NW, int U, int NT, bool WIDE, bool NORM, bool TAIL = false>
static hipError_t gr_run(const GvrArgs& a, int grid, hipStream_t st) {
    constexpr int one = NT * NW * gr_ts(WIDE) * 4;
    /* once per instantiation (thread-safe static initialisation) */
    static const hipError_t attr =
        hipFuncSetAttribute((const void*)k_gvr<WFMT, NW, U, NT, WIDE, NORM, TAIL>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, 2 * one);
    (void)attr;
    hipLaunchKernelGGL((k_gvr<WFMT, NW, U, NT, WIDE, NORM, TAIL>), dim3((unsigned)grid), dim3(64 * NW),
                       a.groups > grid ? 2 * one : one, st, a);
    return hipGetLastError();
}

/* NT tiles a round, at most NTMAX of 1, 2, 3, 4, 6, 10 (hipErrorInvalidValue:
 * not built) */
template <int WFMT, int NW, int U, int NTMAX, bool WIDE, bool NORM>
static hipError_t gr_nt(const GvrArgs& a, int nt, int grid, hipStream_t st) {
    if constexpr (WIDE)
        if (nt == 1) return gr_run<WFMT, NW, U, 1, WIDE, NORM>(a, grid, st);
    if constexpr (NTMAX >= 2)
        if (nt == 2) return gr_run<WFMT, NW, U, 2, WIDE, NORM>(a, grid, st);
    if constexpr (NTMAX >= 3)
        if (nt == 3) return gr_run<WFMT, NW, U, 3, WIDE, NORM>(a, grid, st);
    if constexpr (NTMAX >= 4)
        if (nt == 4) return gr_run<WFMT, NW, U, 4, WIDE, NORM>(a, grid, st);
    if constexpr (NTMAX >= 6)
        if (nt == 6) return gr_run<WFMT, NW, U, 6, WIDE, NORM>(a, grid, st);
    if constexpr (NTMAX >= 10)
        if (nt == 10) return gr_run<WFMT, NW, U, 10, WIDE, NORM>(a, grid, st);
    return hipErrorInvalidValue;
}

/* resident classes, the model's widths (every wave the same number U of whole
 * units, no checks between the tiles' multiplies): 1: K = 2560 on 10 waves;
 * 2: K = 4096 on 8.  A longer K streams.  NT / NTW / NTN: most tiles a round that
 * the registers hold, narrow / WIDE / WIDE with a norm (a fourth INT4 WIDE tile
 * spills: a layer of 10 rows 2.2 us longer, the full head at 9 rows 50.1 us
 * instead of 48.5).  U3: units a wave of 16 waves that hold a longer K (w2's
 * 9728) whole, two tiles, one round */
template <int WFMT>
struct GvrClass;
template <>
struct GvrClass<GEMV_W_INT4> {
    static constexpr int U1 = 1, NT1 = 10, NTW1 = 3, NTN1 = 3, U2 = 2, NT2 = 6, NTW2 = 2, U3 = 3;
};
template <>
struct GvrClass<GEMV_W_INT8> {
    static constexpr int U1 = 2, NT1 = 10, NTW1 = 4, NTN1 = 3, U2 = 4, NT2 = 6, NTW2 = 2, U3 = 5;
};
template <>
struct GvrClass<GEMV_W_BF16> {
    static constexpr int U1 = 4, NT1 = 6, NTW1 = 2, NTN1 = 1, U2 = 8, NT2 = 3, NTW2 = 1, U3 = 0;
};

/* streamed calls that another engine runs faster (weights not resident) */
template <int WFMT>
static bool gr_other(const GemvArgs& g, const GvrArgs& a, int cus) {
    const int64_t kq = a.K >> 8;
    const bool few = WFMT != GEMV_W_BF16 && a.groups <= 16 && kq >= 38 && kq * kq * a.M >= 16000;
    const bool many = WFMT == GEMV_W_INT4 && a.K <= 8192 &&
                      (a.groups + cus - 1) / cus * a.M >= 16;
    if (!few && !many) return false;
    GemvArgs t = g;
    dim3 grid, block;
    size_t lds;
    const bool staged = s2p_gemv3_plan(&t, &grid, &block, &lds) == hipSuccess;
    /* few workgroups, each with a long K to itself, where k_gemv3 does not hold
     * the activations either: the split-K engine (INT8, N = 64: K = 12288, M = 8
     * 12.6 us against 13.6, M = 16 15.1 and 18.7; K = 9728, M = 16 14.6 and 16.0) */
    if (few && !staged) return true;
    /* several rounds of 16 INT4 rows and many activation rows, whose loads come
     * again with each round, while k_gemv3 keeps them in LDS, one chunk of K a
     * wave (K = 5120: N = 20000, M = 9 26.8 us against 33.5, M = 4 24.7 and 26.7;
     * N = 8192, M = 8 13.7 and 13.9, M = 4 12.6 and 11.8) */
    return many && staged;
}

template <int WFMT, bool WIDE>
static hipError_t gr_launch(const GemvArgs& g, GvrArgs& a, bool norm, hipStream_t st) {
    typedef GvrClass<WFMT> Cl;
    const int units = a.K / gr_uk(WFMT), cus = s2p_cu_count();
    const bool swiglu = a.epi == GEMV_EPI_SWIGLU;
    const int cls = units == 10 * Cl::U1 ? 1 : units == 8 * Cl::U2 ? 2 : 0;
    /* only a long K streams: at K = 1024 its rounds of 16 rows took 18 us where
     * the staged engine takes 8 (INT4, 18742 rows, M = 2) */
    if ((norm && cls != 1) || (cls == 0 && (swiglu || a.K <= 4096))) return hipErrorNotSupported;
    const int per = swiglu ? 2 : 1; /* weight tiles per output tile */
    const int rows = swiglu ? a.N >> 1 : a.N, trows = gr_rows(WIDE);
    int most = (cls == 1   ? (!WIDE ? Cl::NT1 : norm ? Cl::NTN1 : Cl::NTW1)
                      : cls == 2 ? (WIDE ? Cl::NTW2 : Cl::NT2)
                                 : gs_nt(WIDE)) / per;
    if (most < 1) return hipErrorNotSupported;
    /* output tiles a round: as many as cover the rows in as few rounds of
     * workgroups as the registers allow, the rows dealt out evenly (38
     * gate/up pairs a workgroup are 13 + 13 + 12); 16 rows for a residual
     * output, the columns of its sums of squares */
    int ot = gs_nt(WIDE);
    a.rpt = trows;
    if (a.epi != GEMV_EPI_RESID && cls != 0) {
        const int tpc = ((rows + trows - 1) / trows + cus - 1) / cus;
        /* several rounds: four tiles each (the head at M = 4: 60 us, with ten
         * 62 us INT4, 67 INT8) */
        if (tpc > most && most > 4 / per) most = 4 / per;
        const int rounds = (tpc + most - 1) / most;
        ot = (tpc + rounds - 1) / rounds;
        if (swiglu) ot = ot <= 3 ? ot : 5; /* 2, 4, 6 or 10 weight tiles */
        else ot = !WIDE && ot < 2 ? 2 : ot <= 4 ? ot : ot <= 6 ? 6 : 10;
        a.rpt = ((rows + cus * rounds - 1) / (cus * rounds) + ot - 1) / ot;
    }
    const int tiles = (rows + a.rpt - 1) / a.rpt;
    a.groups = (tiles + ot - 1) / ot;
    const int grid = a.groups < cus ? a.groups : cus, nt = ot * per;
    if (cls == 0 && gr_other<WFMT>(g, a, cus)) return hipErrorNotSupported;
    if constexpr (!WIDE && Cl::U3 > 0) /* 16 rows a workgroup, one round */
        if (cls == 0 && units > 16 * (Cl::U3 - 1) && units <= 16 * Cl::U3 && a.groups == grid)
            return gr_run<WFMT, 16, Cl::U3, 2, false, false, true>(a, grid, st);
    if (cls == 0) {
        hipLaunchKernelGGL((k_gvs<WFMT, WIDE>), dim3((unsigned)grid), dim3(64 * GS_WAVES), 0, st, a);
        return hipGetLastError();
    }
    if (cls == 2) return gr_nt<WFMT, 8, Cl::U2, WIDE ? Cl::NTW2 : Cl::NT2, WIDE, false>(a, nt, grid, st);
    return norm ? gr_nt<WFMT, 10, Cl::U1, WIDE ? Cl::NTN1 : Cl::NT1, WIDE, true>(a, nt, grid, st)
                : gr_nt<WFMT, 10, Cl::U1, WIDE ? Cl::NTW1 : Cl::NT1, WIDE, false>(a, nt, grid, st);
}

template <int WFMT>
static hipError_t gr_launch_m(const GemvArgs& g, GvrArgs& a, bool norm, hipStream_t st) {
    return a.M <= 8 ? gr_launch<WFMT, false>(g, a, norm, st) : gr_launch<WFMT, true>(g, a, norm, st);
}

extern "C" hipError_t s2p_gvr_launch(const GemvArgs* ap, hipStream_t st) {
    const GemvArgs& g = *ap;
    /* whole units only; the INT4 scales of a unit are one 16-byte load */
    const int uk = gr_uk(g.wfmt);
    if (g.M < 1 || g.M > 16 || g.K % uk || g.N <= 0 ||
        (g.wfmt == GEMV_W_INT4 && ((uintptr_t)g.s & 15)))
        return hipErrorNotSupported;
    GvrArgs a = {};
    a.w = g.w;
    a.s = g.s;
    a.x = g.x;
    a.y = g.y;
    a.norm_w = g.norm_w;
    a.ssq_out = g.ssq_out;
    a.ldx = g.ldx;
    a.ldy = g.ldy;
    a.M = g.M;
    a.N = g.N;
    a.K = g.K;
    a.epi = g.epi;
    a.norm_eps = g.norm_eps;
    const bool norm = g.xmode == GEMV_X_NORM;
    switch (g.wfmt) {
        case GEMV_W_INT4: return gr_launch_m<GEMV_W_INT4>(g, a, norm, st);
        case GEMV_W_INT8: return gr_launch_m<GEMV_W_INT8>(g, a, norm, st);
        default: return gr_launch_m<GEMV_W_BF16>(g, a, norm, st);
    }
}
