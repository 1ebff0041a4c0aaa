/* s2pro MI355X — lockstep decode attention: one query row per session over
 * its own bf16, INT8 or INT4 cache (s2pk_attention_decode and
 * s2pk_attention8_decode, reference kernels.cu:491-508, 751-946), four query
 * heads a kv head.
 *
 * What bounds it: the K/V stream (4,096 / 2,176 / 1,152 bytes a token).  A row
 * has four query vectors a kv head, so the MFMA's 16 columns are mostly empty
 * and the codes' conversion, not the products, is the vector work:
 *   - a block is (row, kv head, split) with 4 waves, each wave on its own
 *     32-slot tiles with its own softmax state;
 *   - scores on the MFMA, S = K Q^T: lane (q, r) loads 16 bytes of slot r; for
 *     the quantised caches lane quarters are exchanged so that every MFMA
 *     covers one 32-dim scale group, whose product takes the slot's f16 scale
 *     in f32.  INT8 codes convert exactly; INT4 nibbles become 1.5 + c / 16,
 *     the bias -1.5 sum q of the group being the C operand;
 *   - P V in f32 on the vector unit: V is loaded as it lies (a wave load is 1
 *     KB of whole rows), a lane owns 8 or 16 dims of its slot for the four
 *     heads, and p (times the V group scale) comes from LDS.  On the MFMA the
 *     codes would have to be gathered byte by byte across slots, and the scale
 *     folded into P one group at a time;
 *     Planes need no alignment: global vector loads take any address;
 *   - bf16 planes are loaded past the caches (nontemporal): each byte is read
 *     once a call.  16 sessions at 8,192 tokens (537 MB) take 84 us, 97 with
 *     cached loads; 64 at 2,048 83 against 96;
 *   - the lanes' sums fold once at the end (lane swaps that halve the values
 *     each step), the waves' states merge through LDS, the splits in
 *     k_attn_combine.
 * Measured (kernel + combine), caches not resident: 12 bf16 sessions of 512 to
 * 4,096 tokens 31 us (113 MB; the verify kernel with one row a segment 40), of
 * 4,096 each 38 (44); 8 INT8 sessions of 1,024 to 8,192 tokens 35 us (the
 * slot-a-thread kernel of kv8.hip 208). */
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "attn_dev.h"
#include "gemv_dev.h"

#define AD_WAVES 4
#define AD_TILE 32 /* slots a wave takes at a time */

struct AdArgs {
    const uint16_t* q;
    const void* const* kcs;
    const void* const* vcs;
    const uint16_t* const* kss; /* f16 scales (quantised caches) */
    const uint16_t* const* vss;
    uint16_t* out;
    const int32_t* pos;
    float* part;
    int rows, qh, kvh_n, max_seq, nsplit, split_pos;
};

template <class T>
S2P_DEV T ad_ld(const void* p) {
    return *(GBL(T)*)p;
}

/* a.hi half wave <-> b.lo; odd 16-lane rows of a <-> even rows of b */
S2P_DEV void ad_swap32(uint32_t& a, uint32_t& b) {
    auto s = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = s[0];
    b = s[1];
}
S2P_DEV float ad_fold32(float a, float b) {
    auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
S2P_DEV float ad_fold16(float a, float b) {
    auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

/* one tile of a wave in registers.  K: 16-byte loads, NK a 16-slot half; V:
 * NI loads of NS slots */
template <int BW>
struct AdTile {
    static constexpr int NK = BW == 16 ? 4 : BW == 8 ? 2 : 1;
    static constexpr int NS = BW == 16 ? 4 : 8, NI = AD_TILE / NS;
    s2p_u32x4 k[2][NK];
    s2p_u32x2 ks[2][4];           /* quantised: the 4 group scales of slots 4 q .. + 3 */
    uint32_t v[NI][BW == 4 ? 2 : 4];
    uint16_t vs[NI];              /* quantised: the lane's slot and group */
};

template <int BW>
__global__ __launch_bounds__(64 * AD_WAVES) __attribute__((amdgpu_waves_per_eu(BW == 16 ? 4 : 3))) void k_attn_dec(AdArgs a) {
#pragma clang fp contract(off)
    typedef AdTile<BW> Tile;
    constexpr int EL = BW == 16 ? 256 : BW == 8 ? 128 : 64; /* bytes of a slot */
    constexpr int ND = BW == 16 ? 8 : 16;                   /* dims of a lane's V piece */
    constexpr int LPS = 128 / ND;                           /* lanes a slot */
    __shared__ __align__(16) float s_p[AD_WAVES][AD_TILE][4];
    __shared__ __align__(16) float s_c[AD_WAVES][4];
    __shared__ __align__(16) float s_o[AD_WAVES][4][128];
    __shared__ float s_m[AD_WAVES][4], s_l[AD_WAVES][4];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, r = lane & 15;
    const int kvh = blockIdx.x % a.kvh_n, row = blockIdx.x / a.kvh_n, sp = blockIdx.y;
    const int ps_ = ad_ld<int32_t>(a.pos + row);
    const int len = ps_ >= 0 && ps_ < a.max_seq ? ps_ + 1 : 0;
    const int p_begin = sp * a.split_pos, p_end = min(p_begin + a.split_pos, len);
    const size_t pi0 = ((size_t)row * a.qh + 4 * kvh) * a.nsplit + sp; /* head h: + h nsplit */
    float* const po = a.part + (size_t)a.rows * a.qh * a.nsplit * 2;
    if (p_begin >= p_end) { /* uniform: an empty split */
        if (BW == 16 && a.nsplit == 1) return; /* a position outside the cache: no output */
        for (int i = tid; i < 512; i += 64 * AD_WAVES) {
            if (a.nsplit == 1)
                a.out[((size_t)row * a.qh + 4 * kvh) * 128 + i] = f2bf(NAN); /* nothing visible: 0 / 0 */
            else
                po[(pi0 + (size_t)(i >> 7) * a.nsplit) * 128 + (i & 127)] = 0.f;
        }
        if (tid < 4 && a.nsplit > 1) {
            a.part[(pi0 + (size_t)tid * a.nsplit) * 2] = -INFINITY;
            a.part[(pi0 + (size_t)tid * a.nsplit) * 2 + 1] = 0.f;
        }
        return;
    }
    const uint64_t plane = (uint64_t)kvh * a.max_seq;
    const GblPtr kb = gbl_base(a.kcs[row], plane * EL), vb = gbl_base(a.vcs[row], plane * EL);
    const GblPtr ksb = BW == 16 ? kb : gbl_base(a.kss[row], plane * 8);
    const GblPtr vsb = BW == 16 ? vb : gbl_base(a.vss[row], plane * 8);

    auto load = [&](Tile& t, int tb) __attribute__((always_inline)) {
        const uint32_t last = (uint32_t)p_end - 1;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t slot = min((uint32_t)(tb + 16 * h + r), last);
#pragma unroll
            for (int i = 0; i < Tile::NK; i++)
                t.k[h][i] = gbl_at<s2p_u32x4, BW == 16>(kb + 64 * i, slot * EL + 16u * q);
            if constexpr (BW != 16) { /* the lane's four slots of the scores */
#pragma unroll
                for (int i = 0; i < 4; i++)
                    t.ks[h][i] = gbl_at<s2p_u32x2>(
                        ksb, min((uint32_t)(tb + 16 * h + 4 * q + i), last) * 8u);
            }
        }
#pragma unroll
        for (int i = 0; i < Tile::NI; i++) {
            const uint32_t slot = min((uint32_t)(tb + i * Tile::NS + lane / LPS), last);
            if constexpr (BW == 4) {
                const s2p_u32x2 w = gbl_at<s2p_u32x2>(vb, slot * EL + 8u * (lane % LPS));
                t.v[i][0] = w.x;
                t.v[i][1] = w.y;
            } else {
                const s2p_u32x4 w = gbl_at<s2p_u32x4, BW == 16>(vb, slot * EL + 16u * (lane % LPS));
#pragma unroll
                for (int d = 0; d < 4; d++) t.v[i][d] = w[d];
            }
            if constexpr (BW != 16)
                t.vs[i] = gbl_at<uint16_t>(vsb, slot * 8u + 2u * ((lane % LPS) >> 1));
        }
    };

    /* Q operand (B, column r = head r; zeros past the four): group g holds
     * the dims that the lane's K bytes of its MFMA pair with */
    s2p_u32x4 qb[4];
    {
        const uint16_t* qr = a.q + ((size_t)row * a.qh + 4 * kvh + (r & 3)) * 128;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            /* INT8, after the half-wave exchange: quarters 0, 1 hold the low 8
             * of 16-dim pieces 2 g, 2 g + 1, quarters 2, 3 their high 8 */
            const int d = BW == 8 ? 32 * g + 16 * (q & 1) + 8 * (q >> 1) : 32 * g + 8 * q;
            s2p_u32x4 w = ad_ld<s2p_u32x4>(qr + d);
            if (BW == 4) /* the k-slot order of deq_int4 */
                w = int4_order(w);
            qb[g] = r < 4 ? w : (s2p_u32x4){0u, 0u, 0u, 0u};
        }
    }
    s2p_f32x4 cb[4]; /* INT4: -1.5 x the group sums of q */
    if constexpr (BW == 4) {
        const s2p_u32x4 k15 = {0xBFC0BFC0u, 0xBFC0BFC0u, 0xBFC0BFC0u, 0xBFC0BFC0u};
#pragma unroll
        for (int g = 0; g < 4; g++) cb[g] = mfma16x16x32(k15, qb[g], (s2p_f32x4){0.f, 0.f, 0.f, 0.f});
    }
    float m = -INFINITY, l = 0.f; /* of head r (lanes r < 4) */
    float acc[4][ND];
#pragma unroll
    for (int h = 0; h < 4; h++)
#pragma unroll
        for (int e = 0; e < ND; e++) acc[h][e] = 0.f;

    auto step = [&](Tile& t, int tb) __attribute__((always_inline)) {
        /* scores of slots tb + 16 h + 4 q + i, head r */
        float s[2][4];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            s2p_f32x4 sc = {0.f, 0.f, 0.f, 0.f};
            if constexpr (BW == 16) {
#pragma unroll
                for (int g = 0; g < 4; g++) sc = mfma16x16x32(t.k[h][g], qb[g], sc);
            } else {
                uint32_t kd[4][2];
                if constexpr (BW == 8) {
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        uint32_t d0 = t.k[h][i].x, d1 = t.k[h][i].y, d2 = t.k[h][i].z, d3 = t.k[h][i].w;
                        ad_swap32(d0, d2);
                        ad_swap32(d1, d3);
                        kd[2 * i][0] = d0;
                        kd[2 * i][1] = d1;
                        kd[2 * i + 1][0] = d2;
                        kd[2 * i + 1][1] = d3;
                    }
                } else {
                    uint32_t d0 = t.k[h][0].x, d1 = t.k[h][0].y, d2 = t.k[h][0].z, d3 = t.k[h][0].w;
                    xpose4(d0, d1, d2, d3);
                    kd[0][0] = d0;
                    kd[1][0] = d1;
                    kd[2][0] = d2;
                    kd[3][0] = d3;
                }
                uint32_t kmask = 0x00780078u, kone = 0x3F803F80u;
                asm volatile("" : "+v"(kmask), "+v"(kone));
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    s2p_f32x4 raw;
                    if constexpr (BW == 8) {
                        const s2p_u32x2 lo = deq_s8(kd[g][0]), hi = deq_s8(kd[g][1]);
                        raw = mfma16x16x32((s2p_u32x4){lo.x, lo.y, hi.x, hi.y}, qb[g],
                                           (s2p_f32x4){0.f, 0.f, 0.f, 0.f});
                    } else {
                        raw = mfma16x16x32(deq_int4(kd[g][0], kmask, kone), qb[g], cb[g]);
                    }
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const uint32_t w = t.ks[h][i][g >> 1];
                        const float ks = (float)__builtin_bit_cast(
                            _Float16, (uint16_t)((g & 1) ? (w >> 16) : (w & 0xFFFFu)));
                        sc[i] = fmaf(ks, raw[i], sc[i]);
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
                s[h][i] = tb + 16 * h + 4 * q + i < p_end
                              ? sc[i] * (BW == 4 ? 16.0f * 0.08838834764831845f : 0.08838834764831845f)
                              : -INFINITY;
            __builtin_amdgcn_sched_barrier(0);
        }
        /* online softmax: the head's 8 slots of the lane, then lanes r + 16 G */
        float tm = s[0][0];
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int i = 0; i < 4; i++) tm = fmaxf(tm, s[h][i]);
        tm = xg_max(tm);
        const float mn = fmaxf(m, tm);
        const float ms = mn == -INFINITY ? 0.f : mn; /* every score so far -inf: weights 0 */
        const float corr = __expf(m - ms);
        float ls = 0.f;
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float p = __expf(s[h][i] - ms);
                ls += p;
                if (r < 4) s_p[wave][16 * h + 4 * q + i][r] = p;
            }
        l = l * corr + ls;
        m = mn;
        if (lane < 4) s_c[wave][lane] = corr;
        wave_lds_sync();
        if (__any(corr != 1.0f)) {
            const s2p_f32x4 c4 = *(const LDS(s2p_f32x4)*)&s_c[wave][0];
#pragma unroll
            for (int h = 0; h < 4; h++)
#pragma unroll
                for (int e = 0; e < ND; e++) acc[h][e] *= c4[h];
        }
#pragma unroll
        for (int i = 0; i < Tile::NI; i++) {
            s2p_f32x4 p4 = *(const LDS(s2p_f32x4)*)&s_p[wave][i * Tile::NS + lane / LPS][0];
            if constexpr (BW != 16) {
                const float vs = h2f(t.vs[i]);
#pragma unroll
                for (int h = 0; h < 4; h++) p4[h] *= vs;
            }
#pragma unroll
            for (int e = 0; e < ND; e++) {
                float v;
                if constexpr (BW == 16) v = (e & 1) ? bf2f_hi(t.v[i][e >> 1]) : bf2f_lo(t.v[i][e >> 1]);
                else if constexpr (BW == 8) v = (float)(int8_t)(t.v[i][e >> 2] >> (8 * (e & 3)));
                else v = (float)((int32_t)(t.v[i][e >> 3] << (28 - 4 * (e & 7))) >> 28);
#pragma unroll
                for (int h = 0; h < 4; h++) acc[h][e] = fmaf(p4[h], v, acc[h][e]);
            }
            __builtin_amdgcn_sched_barrier(0); /* one V piece's values live at a time */
        }
        wave_lds_sync(); /* s_p is rewritten by the next tile */
    };

    /* this wave's tiles: w, w + 4, ... of the split */
    constexpr int STEP = AD_TILE * AD_WAVES;
    const int tb = p_begin + wave * AD_TILE;
    const int n = tb < p_end ? (p_end - tb + STEP - 1) / STEP : 0; /* uniform per wave */
    if (n > 0) {
        /* one tile in registers: three or four waves a SIMD keep loads in
         * flight (a second tile costs the third wave, or spills) */
        Tile t;
        for (int c = 0; c < n; c++) {
            load(t, tb + c * STEP);
            step(t, tb + c * STEP);
        }
    }
    /* fold the lanes' sums: lane row q ends with head q, the lane's dims */
    float f[ND];
#pragma unroll
    for (int e = 0; e < ND; e++) {
        f[e] = ad_fold16(ad_fold32(acc[0][e], acc[2][e]), ad_fold32(acc[1][e], acc[3][e]));
        if constexpr (LPS == 8) f[e] += dpp_f<0x128>(f[e]); /* row_ror:8: the other slots */
    }
    l = xg_sum(l);
    if (lane < 4) {
        s_m[wave][lane] = m;
        s_l[wave][lane] = l;
    }
    if (LPS == 16 || r < 8) {
#pragma unroll
        for (int e = 0; e < ND; e += 4)
            *(LDS(s2p_f32x4)*)&s_o[wave][q][(lane % LPS) * ND + e] =
                (s2p_f32x4){f[e], f[e + 1], f[e + 2], f[e + 3]};
    }
    __syncthreads();
    /* merge the waves: two outputs a thread */
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int h = (tid + 256 * i) >> 7, d = tid & 127;
        float M = s_m[0][h];
#pragma unroll
        for (int w = 1; w < AD_WAVES; w++) M = fmaxf(M, s_m[w][h]);
        const float Ms = M == -INFINITY ? 0.f : M;
        float lt = 0.f, o = 0.f;
#pragma unroll
        for (int w = 0; w < AD_WAVES; w++) { /* a wave without tiles has m = -inf: weight 0 */
            const float e = __expf(s_m[w][h] - Ms);
            lt = fmaf(s_l[w][h], e, lt);
            o = fmaf(s_o[w][h][d], e, o);
        }
        if (a.nsplit == 1) {
            a.out[((size_t)row * a.qh + 4 * kvh + h) * 128 + d] = f2bf(o / lt);
        } else {
            const size_t pi = pi0 + (size_t)h * a.nsplit;
            po[pi * 128 + d] = o;
            if (d == 0) {
                a.part[pi * 2] = M;
                a.part[pi * 2 + 1] = lt;
            }
        }
    }
}

/* Rounds a split of `units` rounds of (row, kv head) pairs, at most four
 * blocks a CU (what fits at once).
 * bf16: a tick's bytes are spread evenly when the CU with the most blocks has
 * few rounds to do; a block costs about half a round besides, the combine a
 * round and a twentieth a split, and one block a CU streams no faster than two
 * do together.  The least such cost, of equals the fewest splits.  With four
 * blocks a CU always, 64 sessions of 200 tokens took 15.5 us instead of 11.6
 * and one of 32,768 took 50 instead of 36; with two, 24 sessions of 4,096 took
 * 77 instead of 67.
 * Quantised: about four blocks a CU, so that ragged lengths even out (32 INT4
 * sessions of 512 to 4,096 tokens: 39 us, in two blocks a CU 49). */
static int ad_rounds(int pairs, int units, bool bf16) {
    const int cus = s2p_cu_count(), most = 4 * cus / pairs;
    if (!bf16) {
        const int ns = most < 1 ? 1 : most < units ? most : units;
        return (units + ns - 1) / ns;
    }
    int best = units;
    int64_t least = INT64_MAX;
    for (int n = 1; n <= most || n == 1;) { /* the split counts that whole rounds give */
        const int ups = (units + n - 1) / n;
        int64_t per_cu = ((int64_t)n * pairs + cus - 1) / cus;
        if (per_cu < 2) per_cu = 2;
        const int64_t cost = per_cu * (20 * (int64_t)ups + 10) + (n > 1 ? 20 + n : 0);
        if (cost < least) {
            least = cost;
            best = ups;
        }
        if (ups == 1) break;
        const int u = (units - 1) / n; /* the most rounds a split of the next count */
        n = (units + u - 1) / u;
    }
    return best;
}

extern "C" hipError_t s2p_attn_dec_launch(const uint16_t* q, const void* const* kcs,
                                          const void* const* vcs, const uint16_t* const* kss,
                                          const uint16_t* const* vss, uint16_t* out, int rows,
                                          int kv_heads, const int32_t* pos, int max_seq,
                                          int max_len, float* part, int bw, hipStream_t st) {
    AdArgs a = {};
    a.q = q;
    a.kcs = kcs;
    a.vcs = vcs;
    a.kss = kss;
    a.vss = vss;
    a.out = out;
    a.pos = pos;
    a.part = part;
    a.rows = rows;
    a.qh = 4 * kv_heads;
    a.kvh_n = kv_heads;
    a.max_seq = max_seq;
    /* splits of whole rounds of the block's tiles (128 slots) */
    const int units = (max_len + AD_TILE * AD_WAVES - 1) / (AD_TILE * AD_WAVES);
    const int ups = ad_rounds(rows * kv_heads, units, bw == 16);
    a.split_pos = ups * AD_TILE * AD_WAVES;
    a.nsplit = (units + ups - 1) / ups;
    const dim3 grid((unsigned)(rows * kv_heads), (unsigned)a.nsplit);
    if (bw == 16) hipLaunchKernelGGL(k_attn_dec<16>, grid, dim3(64 * AD_WAVES), 0, st, a);
    else if (bw == 8) hipLaunchKernelGGL(k_attn_dec<8>, grid, dim3(64 * AD_WAVES), 0, st, a);
    else hipLaunchKernelGGL(k_attn_dec<4>, grid, dim3(64 * AD_WAVES), 0, st, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || a.nsplit == 1) return e;
    return s2p_attn_combine_launch(part, out, rows, a.qh, a.nsplit, st);
}
