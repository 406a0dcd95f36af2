// kq_dev.h -- superblock terms of the Q4_K / Q6_K kernels and the Q8_K of h,
// shared by batch-1 decode (moe_kq.hip) and small batches (moe_grouped_kq.hip).
#pragma once
#include "moe_common.h"
#include "moe_kq.h"

namespace cpb {

constexpr int kXsPad = 272;      // LDS bytes per 256-activation superblock (256 + 16: bank spread)

// Q4_K superblock term of one row (engine_qwen2.rs:84-114).  u: the 9 units
// (u[0] = d, dmin, 12 packed scale/min bytes; u[1..8] = qs[128]); xs: the 256
// int8 activations of the superblock (LDS, 16-aligned); xsum8: their 8 int32
// sums per 32; ys: their scale.  sums (TRACE): {sumi, mint}.
template <bool TRACE>
CPB_DEV float q4k_term(const u32x4 (&u)[kQ4Units], const int8_t* xs, const int32_t* xsum8, float ys, int32_t* sums) {
    const float d = half_bits(u[0][0] & 0xffffu), dmin = half_bits(u[0][0] >> 16);
    // scale bytes q[0..11] = bytes 4..15 of unit 0 (ggml get_scale_min_k4, :59-74)
    const uint32_t q03 = u[0][1], q47 = u[0][2], q811 = u[0][3];
    int sc[8], mn[8];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        sc[j] = (q03 >> (8 * j)) & 63;
        mn[j] = (q47 >> (8 * j)) & 63;
        const uint32_t qj4 = (q811 >> (8 * j)) & 0xff;      // q[j + 8]
        sc[4 + j] = (qj4 & 0xf) | (((q03 >> (8 * j + 6)) & 3) << 4);
        mn[4 + j] = (qj4 >> 4) | (((q47 >> (8 * j + 6)) & 3) << 4);
    }
    const u32x4* xv = (const u32x4*)xs;
    int sumi = 0;
#pragma unroll
    for (int jj = 0; jj < 4; jj++) {
        const u32x4 w0 = u[1 + 2 * jj], w1 = u[2 + 2 * jj];
        const uint32_t w[8] = {w0[0], w0[1], w0[2], w0[3], w1[0], w1[1], w1[2], w1[3]};
        const u32x4 a0 = xv[4 * jj + 0], a1 = xv[4 * jj + 1];   // sub-block 2jj   (32 B)
        const u32x4 b0 = xv[4 * jj + 2], b1 = xv[4 * jj + 3];   // sub-block 2jj+1 (32 B)
        const uint32_t xa[8] = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
        const uint32_t xb[8] = {b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]};
        int s0 = 0, s1 = 0;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            s0 = sdot4(w[i] & 0x0F0F0F0Fu, xa[i], s0);
            s1 = sdot4((w[i] >> 4) & 0x0F0F0F0Fu, xb[i], s1);
        }
        sumi += mul24(s0, sc[2 * jj]) + mul24(s1, sc[2 * jj + 1]);
    }
    int mint = 0;
#pragma unroll
    for (int j = 0; j < 8; j++) mint += mul24(mn[j], xsum8[j]);
    if (TRACE) { sums[0] = sumi; sums[1] = mint; }
    return ys * d * (float)sumi - ys * dmin * (float)mint;
}

// Q6_K superblock term of one row (engine_qwen2.rs:164-200).  u: 14 units in registers
// (ql[128] = u[0..7], qh[64] = u[8..11], int8 scales[16] = u[12], fp16 d in
// u[13]); xs: 256 int8 activations; xs16: their 16 int32 sums per 16.
// q - 32 is folded as dot(q, x) - 32 * sum(x) (an exact integer identity).
template <bool TRACE>
CPB_DEV float q6k_term(const u32x4 (&u)[kQ6Units], const int8_t* xs, const int32_t* xs16, float ys, int32_t* sums) {
    const float d = half_bits(u[13][0] & 0xffffu);
    const uint32_t* ql = (const uint32_t*)&u[0];
    const uint32_t* qh = (const uint32_t*)&u[8];
    const uint32_t* scw = (const uint32_t*)&u[12];
    const uint32_t* xw = (const uint32_t*)xs;
    int s[16];
#pragma unroll
    for (int g = 0; g < 16; g++) s[g] = 0;
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int l4 = 0; l4 < 8; l4++) {
            const uint32_t A = ql[h * 16 + l4], B = ql[h * 16 + 8 + l4], H = qh[h * 8 + l4];
            const uint32_t t0 = (A & 0x0F0F0F0Fu) | ((H & 0x03030303u) << 4);
            const uint32_t t1 = (B & 0x0F0F0F0Fu) | (((H >> 2) & 0x03030303u) << 4);
            const uint32_t t2 = ((A >> 4) & 0x0F0F0F0Fu) | (((H >> 4) & 0x03030303u) << 4);
            const uint32_t t3 = ((B >> 4) & 0x0F0F0F0Fu) | (((H >> 6) & 0x03030303u) << 4);
            const int hi = l4 >= 4 ? 1 : 0;          // element l = 4*l4 lies in the second 16 of its 32
            const int e0 = h * 128 + 4 * l4;         // first element of t0's 4
            s[h * 8 + 0 + hi] = sdot4(t0, xw[(e0 + 0) / 4], s[h * 8 + 0 + hi]);
            s[h * 8 + 2 + hi] = sdot4(t1, xw[(e0 + 32) / 4], s[h * 8 + 2 + hi]);
            s[h * 8 + 4 + hi] = sdot4(t2, xw[(e0 + 64) / 4], s[h * 8 + 4 + hi]);
            s[h * 8 + 6 + hi] = sdot4(t3, xw[(e0 + 96) / 4], s[h * 8 + 6 + hi]);
        }
    }
    int acc = 0;
#pragma unroll
    for (int g = 0; g < 16; g++) {
        const int sc = (int)(int8_t)(scw[g / 4] >> (8 * (g % 4)));
        acc += mul24(s[g] - 32 * xs16[g], sc);
    }
    if (TRACE) sums[0] = acc;
    return ys * d * (float)acc;
}

// Q8_K of the workgroup's h vectors into LDS (engine_qwen2.rs:288-300, amax
// seeded 1e-12): chunk c = 32 values of slot c / cps (hv, thread c's, c < nch);
// a 256-block is 8 chunks.  Pass 1: the chunk's amax, the chunk to hst (k-major:
// consecutive threads' 16-byte accesses fall on consecutive banks).  Pass 2: the
// scale per 256, round, sums per 32 and 16 (two q8_round16: one rarely taken
// branch per 16 values; sums from the packed bytes, a signed dot with ones).
// Ends with a workgroup barrier; every access is to LDS, so it runs while
// earlier global loads are in flight.
CPB_DEV void quant_h_chunks(float4 (&hv)[8], int c, int nch, int cps, int hstride, float4* hst, float* cmax, int8_t* hql,
                            int32_t* h32, int32_t* h16, float* hsl) {
    if (c < nch) {
        float m = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float4 v = hv[k];
            m = fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        }
        cmax[c] = m;
#pragma unroll
        for (int k = 0; k < 8; k++) hst[k * nch + c] = hv[k];
    }
    __syncthreads();
    if (c < nch) {
        const int blk = c / 8;
        float amax = 1e-12f;
#pragma unroll
        for (int k = 0; k < 8; k++) amax = fmaxf(amax, cmax[blk * 8 + k]);
        const float sc = amax / 127.0f;
#pragma unroll
        for (int k = 0; k < 8; k++) hv[k] = hst[k * nch + c];
        const int slot = c / cps, cc = c % cps;                     // slot, chunk within it
        int8_t* dst = hql + slot * hstride + (cc / 8) * kXsPad + (cc % 8) * 32;
        float hf[32];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            hf[4 * k] = hv[k].x; hf[4 * k + 1] = hv[k].y; hf[4 * k + 2] = hv[k].z; hf[4 * k + 3] = hv[k].w;
        }
        uint32_t qp[8];
        q8_round16(hf, sc, qp);
        q8_round16(hf + 16, sc, qp + 4);
        int s16[2] = {0, 0};
#pragma unroll
        for (int k = 0; k < 8; k++) s16[k / 4] = sdot4(qp[k], 0x01010101u, s16[k / 4]);
        ((u32x4*)dst)[0] = u32x4{qp[0], qp[1], qp[2], qp[3]};
        ((u32x4*)dst)[1] = u32x4{qp[4], qp[5], qp[6], qp[7]};
        h32[c] = s16[0] + s16[1];
        h16[2 * c] = s16[0];
        h16[2 * c + 1] = s16[1];
        if (c % 8 == 0) hsl[blk] = sc;
    }
    __syncthreads();
}

}  // namespace cpb
