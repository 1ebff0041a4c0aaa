/* s2pro MI355X — fast-AR attention: RoPE, K/V append and attention over the at
 * most S2P_FA_SEQ slots of a frame (reference src/fastar/fastar.cu:647-789).
 *
 * What bounds it: one round trip to memory and the launch; a session's cache
 * is 11 slots.  So there are no tiles, no MFMA and no LDS: a wave is one query
 * head of one row, every load (the q, k, v of the row, the RoPE row, all
 * earlier slots) is issued at once, the scores are wave sums, and the four
 * waves of a kv head each rope the new key for themselves.  Measured 4.0 us
 * where a block of the verify attention took 7.1 (4 rows): its segment table,
 * LDS hand-over and wave merge were round trips of their own.
 * Values: q and k rounded to bf16 after RoPE; scores, weights and P V in f32. */
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "attn_dev.h"
#include "s2pro/fastar.h"

#define FAA_QKV 6144
#define FAA_OLD (S2P_FA_SEQ - 1) /* most earlier slots */

/* all lanes get lane 0's total */
S2P_DEV float faa_sum(float v) {
    v = xg_sum(sum16(v));
    return __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(v)));
}

/* block = (row, kv head); rows s * nn .. + nn - 1 of session s sit at slots
 * p0 .. p0 + nn - 1 (nn 1 or 2); rope: row of position p at p * rope_stride */
__global__ __launch_bounds__(256) void k_fa_attn(const uint16_t* __restrict__ qkv,
                                                 const float* __restrict__ rope, int rope_stride,
                                                 uint16_t* kv, int64_t sess_stride,
                                                 uint16_t* __restrict__ out, int p0, int nn) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kvh = blockIdx.x & 7, row = blockIdx.x >> 3;
    const int s = nn == 2 ? row >> 1 : row, i = nn == 2 ? row & 1 : 0;
    const int h = 4 * kvh + wave;
    uint16_t* kc = kv + s * sess_stride + (size_t)kvh * S2P_FA_SEQ * 128;
    uint16_t* vc = kc + (size_t)8 * S2P_FA_SEQ * 128;
    const uint16_t* x = qkv + (size_t)row * FAA_QKV;
    const uint16_t* xk = x + 4096 + kvh * 128;
    const uint16_t* xp = i ? xk - FAA_QKV : xk; /* the session's row before */
    const float* cs = rope + (size_t)(p0 + i) * rope_stride + (lane >> 1) * 2;
    const float* cp = i ? cs - rope_stride : cs;

    const uint16_t q0 = x[h * 128 + lane], q1 = x[h * 128 + lane + 64];
    const uint16_t k0 = xk[lane], k1 = xk[lane + 64];
    const uint16_t v0 = xk[1024 + lane], v1 = xk[1024 + lane + 64];
    const uint16_t kp0 = xp[lane], kp1 = xp[lane + 64];
    const uint16_t vp0 = xp[1024 + lane], vp1 = xp[1024 + lane + 64];
    const float2 c0 = *(const float2*)cs, c1 = *(const float2*)(cs + 64);
    const float2 d0 = *(const float2*)cp, d1 = *(const float2*)(cp + 64);
    uint16_t ok[FAA_OLD][2], ov[FAA_OLD][2];
#pragma unroll
    for (int t = 0; t < FAA_OLD; t++)
        if (t < p0) { /* uniform */
            ok[t][0] = kc[t * 128 + lane];
            ok[t][1] = kc[t * 128 + lane + 64];
            ov[t][0] = vc[t * 128 + lane];
            ov[t][1] = vc[t * 128 + lane + 64];
        }

    float a, b;
    qkrope_math(bf2f(q0), bf2f(q1), 0, 0, c0.x, c0.y, c1.x, c1.y, 0.f, lane, &a, &b, false);
    const float qa = bf2f(f2bf(a)), qb = bf2f(f2bf(b));
    qkrope_math(bf2f(k0), bf2f(k1), 0, 0, c0.x, c0.y, c1.x, c1.y, 0.f, lane, &a, &b, false);
    const uint16_t ka = f2bf(a), kb = f2bf(b);
    if (wave == 0) {
        const int slot = (p0 + i) * 128;
        kc[slot + lane] = ka;
        kc[slot + lane + 64] = kb;
        vc[slot + lane] = v0;
        vc[slot + lane + 64] = v1;
    }
    qkrope_math(bf2f(kp0), bf2f(kp1), 0, 0, d0.x, d0.y, d1.x, d1.y, 0.f, lane, &a, &b, false);
    const float pa = bf2f(f2bf(a)), pb = bf2f(f2bf(b));

    constexpr float scale = 0.08838834764831845f;
    float sc[FAA_OLD + 2], m = -INFINITY;
#pragma unroll
    for (int t = 0; t < FAA_OLD + 2; t++) sc[t] = -INFINITY;
#pragma unroll
    for (int t = 0; t < FAA_OLD; t++)
        if (t < p0) sc[t] = faa_sum(fmaf(qa, bf2f(ok[t][0]), qb * bf2f(ok[t][1]))) * scale;
    if (i) sc[FAA_OLD] = faa_sum(fmaf(qa, pa, qb * pb)) * scale;
    sc[FAA_OLD + 1] = faa_sum(fmaf(qa, bf2f(ka), qb * bf2f(kb))) * scale;
#pragma unroll
    for (int t = 0; t < FAA_OLD + 2; t++) m = fmaxf(m, sc[t]);
    const float ms = m == -INFINITY ? 0.f : m;
    float l = 0.f, o0 = 0.f, o1 = 0.f;
    auto add = [&](float st, uint16_t w0, uint16_t w1) __attribute__((always_inline)) {
        const float p = __expf(st - ms);
        l += p;
        o0 = fmaf(p, bf2f(w0), o0);
        o1 = fmaf(p, bf2f(w1), o1);
    };
#pragma unroll
    for (int t = 0; t < FAA_OLD; t++)
        if (t < p0) add(sc[t], ov[t][0], ov[t][1]);
    if (i) add(sc[FAA_OLD], vp0, vp1);
    add(sc[FAA_OLD + 1], v0, v1);
    const float inv = 1.0f / l;
    uint16_t* y = out + (size_t)row * 4096 + h * 128;
    y[lane] = f2bf(o0 * inv);
    y[lane + 64] = f2bf(o1 * inv);
}

extern "C" hipError_t s2p_fa_attn_launch(const void* qkv, const float* rope, int rope_stride,
                                         void* kv, int64_t sess_stride, void* out, int n_sess,
                                         int p0, int nn, hipStream_t st) {
    if (n_sess <= 0) return hipSuccess;
    if (nn < 1 || nn > 2 || p0 < 0 || p0 + nn > S2P_FA_SEQ) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_fa_attn, dim3((unsigned)(n_sess * nn * 8)), dim3(256), 0, st,
                       (const uint16_t*)qkv, rope, rope_stride, (uint16_t*)kv, sess_stride,
                       (uint16_t*)out, p0, nn);
    return hipGetLastError();
}
