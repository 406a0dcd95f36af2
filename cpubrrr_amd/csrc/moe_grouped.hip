// moe_grouped.hip -- batched / prefill gpt-oss MoE layer (gfx950).
//
// Reference: the tile path engine_gpt2.rs:1120-1239, whose contract is
// "bit-identical to per-token decode" (expert-major subscriber lists, weight
// quads reused across tokens).  Here the tokens' (token, slot) pairs are
// grouped by expert and each expert's gate/up and down products run on the
// matrix cores, exactly:
//
//   v_mfma_scale_f32_32x32x64_f8f6f4, A = weights (fp4 e2m1, 32 rows x 64 K),
//   B = activations (fp8 e4m3, 64 K x 32 tokens), one MXFP4 block per
//   instruction.  A's two K halves both carry the block's 32 raw codes (the
//   16 GGUF bytes as they are: no decode), B's first half carries 16*h and the
//   second half l of each int8 activation x = 16*h + l (h = x >> 4, l in
//   [0, 15]; both exact in e4m3), and the block's e8m0 byte is A's hardware
//   scale.  Every product and partial sum is exact in fp32, so
//       D = sum_i E2M1(c_i) * x_i * 2^(e-127) = S * 2^(e-128)
//   with S the reference's int32 block sum (engine_gpt2.rs:194-228).  The
//   epilogue then does what the decode kernels do with S: per 15-block k-part
//   acc = fma(D, xsb, acc) (the same exact product S * 2^(e-128) * xsb, one
//   rounding), parts added in order, bias, SwiGLU-OAI + Q8 (gate/up) or the
//   slot-ordered combine (down).  Results are therefore the decode path's bit
//   for bit.  Blocks with e8m0 < 32 or == 255 (tbl[0] = 0 and NaN in
//   hardware, subnormal scales) are not exact this way: the caller routes
//   such layers to the per-token kernels.
//
// Operand layouts (measured on gfx950): A lane l = (row l%32, K half l/32),
// nibble n <-> K 32*half + n; B lane l = (token l%32, half hb = l/32), bytes
// 0-15 <-> K 16*hb + j, bytes 16-31 <-> K 32 + 16*hb + j; D lane l register i
// = (row 8*(i/4) + 4*(l/32) + i%4, token l%32); scale_a lane l = row l%32.
// An MXFP4 block's nibble n is element n/2 (n even) or 16 + n/2 (n odd), so
// the activation "image" of a block (64 B) puts element e's 16*h at byte
// 32*(K/16) + K%16 and its l 16 bytes later, K = 2e (e < 16) or 2(e-16)+1.
//
// The weights are read in the decode kernels' stream layout (moe_mx.hip), so
// both paths share one copy in HBM.
#include "moe_common.h"
#include "moe_grouped.h"
#include "moe_mx.h"
#include "mx_dev.h"
#include "route_dev.h"
#include "select.h"

#include <algorithm>
#include <type_traits>

namespace cpb {

typedef int v8i_g __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

typedef __attribute__((address_space(3))) void lds_void_g;

constexpr int kImg = 64;          // image bytes per 32-block


// ---- 1. per token: rmsnorm, Q8 per 32, fp8 image ----
__global__ __launch_bounds__(256) void k_prep_batch(GroupedArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int t = blockIdx.x, d = a.d, tid = threadIdx.x, nth = blockDim.x;
    float* xs = (float*)smem;
    float* xnl = xs + d;
    float* scratch = xnl + d;
    norm_into(a.x + (size_t)t * d, a.norm_w, d, a.eps, a.norm, a.norm_nt, a.apply_norm, xs, xnl, scratch);
    // Q8 per 32-block (engine_gpt2.rs:691-699), four threads per block:
    // thread c owns elements 8p + 4h .. +3 and 16 + 8p + 4h .. +3 (p = c >> 1,
    // h = c & 1), so its share of xq is two whole dwords and its share of the
    // 64-byte image two whole 8-byte runs.  Image byte K of a part (K < 16:
    // bytes 0-15, 16h; bytes 16-31, l; then the same for K 16..31 at 32-63)
    // holds element K / 2 (K even) or 16 + (K - 1) / 2 (K odd): dword w of part
    // p packs elements 8p + 2w, 8p + 2w + 16, 8p + 2w + 1, 8p + 2w + 17.  The
    // e4m3 codes come from the hardware conversion, exact for these integers;
    // the block maximum from two lane exchanges; the exact division only
    // near a rounding tie.
    for (int i = tid; i < a.nb * 4; i += nth) {
        const int bk = i >> 2, c = i & 3, p = c >> 1, h = c & 1;
        const int e0 = 8 * p + 4 * h;
        const float4 f0 = ((const float4*)(xnl + bk * 32 + e0))[0];
        const float4 f1 = ((const float4*)(xnl + bk * 32 + 16 + e0))[0];
        const float v[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
        float m = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; k++) m = fmaxf(m, fabsf(v[k]));
        m = fmaxf(m, __shfl_xor(m, 1));
        m = fmaxf(m, __shfl_xor(m, 2));
        const float sc = fmaxf(1e-12f, m) / 127.0f;
        int q[8];
        {
            const float rs = __builtin_amdgcn_rcpf(sc);
            float r[8];
            bool near = false;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const float y = v[k] * rs;
                r[k] = __builtin_rintf(y);
                near = near || q8_near_half(y);
            }
            if (near) {
#pragma unroll
                for (int k = 0; k < 8; k++)
                    if (q8_near_half(v[k] * rs)) r[k] = roundf(v[k] / sc);
            }
#pragma unroll
            for (int k = 0; k < 8; k++) q[k] = q8_clamp(r[k]);
        }
        uint32_t qw[2] = {0u, 0u};
#pragma unroll
        for (int k = 0; k < 8; k++) qw[k >> 2] |= ((uint32_t)q[k] & 0xffu) << (8 * (k & 3));
        float* xo = a.xn + (size_t)t * d + bk * 32;
        *(float4*)(xo + e0) = f0;
        *(float4*)(xo + 16 + e0) = f1;
        uint32_t* qo = (uint32_t*)(a.xq + (size_t)t * d + bk * 32);
        qo[e0 >> 2] = qw[0];
        qo[(16 + e0) >> 2] = qw[1];
        if (c == 0) a.xsb[(size_t)t * a.nb + bk] = sc;
        // elements e0 + j (k = j) and 16 + e0 + j (k = 4 + j), j < 4: dwords
        // w = 2h and 2h + 1 of part p pack (e0 + 2(w - 2h), its +16, +1, +17)
        float fh[8], fl[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int hh = q[k] >> 4;
            fh[k] = (float)(16 * hh);
            fl[k] = (float)(q[k] - 16 * hh);
        }
        uint32_t hi[2], lo[2];
#pragma unroll
        for (int w = 0; w < 2; w++) {
            const int j = 2 * w;             // elements e0 + j, 16 + e0 + j, e0 + j + 1, 16 + e0 + j + 1
            hi[w] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(fh[j + 1], fh[4 + j + 1],
                                                               __builtin_amdgcn_cvt_pk_fp8_f32(fh[j], fh[4 + j], 0, false), true);
            lo[w] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(fl[j + 1], fl[4 + j + 1],
                                                               __builtin_amdgcn_cvt_pk_fp8_f32(fl[j], fl[4 + j], 0, false), true);
        }
        uint8_t* img = a.ximg + ((size_t)t * a.nb + bk) * kImg + 32 * p + 8 * h;
        *(uint2*)img = make_uint2(hi[0], hi[1]);
        *(uint2*)(img + 16) = make_uint2(lo[0], lo[1]);
    }
}

// ---- 2. router logits, exactly: workgroup = (8 experts, 8 tokens) ----
// Every (token, expert) logit as the reference computes it
// (engine_gpt2.rs:849-852, engine_qwen2.rs:395-400): acc = b; acc += W[j] *
// xn[j] for j = 0 .. d-1, fp32, each product and each sum rounded once, in
// order.  A chain cannot be split, but a batch has n_tok * ne of them: lane
// (tl, el) of the wave runs the chain of token 8 ty + tl and expert 8 ex + el,
// the products one step ahead of the adds.  The 8 tokens' xn and the 8
// experts' router rows stream through LDS in chunks of kChainChunk (the next
// chunk requested into registers while the current one is summed).  The
// selection ranks these values, and the weights are the softmax of the
// reference's own fp32 logits.
constexpr int kChainChunk = 128;
constexpr int kChainStride = kChainChunk + 4;     // floats per LDS row (spreads the 8 rows over the banks)
__global__ __launch_bounds__(64) void k_router_exact(GroupedArgs a) {
    __shared__ __align__(16) float xs[2][8][kChainStride];
    __shared__ __align__(16) float wsh[2][8][kChainStride];
    const int lane = threadIdx.x, d = a.d;
    const int tl = lane >> 3, el = lane & 7;
    const int t = blockIdx.y * 8 + tl, e = blockIdx.x * 8 + el;
    // staging: lane moves 16-byte pieces c = lane + 64 i (i < 4) of the
    // 8 x 128-float chunk: row c / 32, floats 4 (c % 32) ..
    const int nt = a.n_tok, ne = a.ne;
    const __amdgpu_buffer_rsrc_t rx = buf_rsrc(a.xn, (uint32_t)((size_t)nt * d * 4));
    const __amdgpu_buffer_rsrc_t rw = buf_rsrc(a.router_w, (uint32_t)((size_t)ne * d * 4));
    auto fetch = [&](int j0, u32x4 (&xr)[4], u32x4 (&wr)[4]) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int c = lane + 64 * i, row = c >> 5, j = j0 + 4 * (c & 31);
            const int tt = blockIdx.y * 8 + row, ee = blockIdx.x * 8 + row;
            xr[i] = __builtin_amdgcn_raw_buffer_load_b128(rx, tt < nt && j < d ? (uint32_t)(((size_t)tt * d + j) * 4) : kOffNone, 0, 0);
            wr[i] = __builtin_amdgcn_raw_buffer_load_b128(rw, ee < ne && j < d ? (uint32_t)(((size_t)ee * d + j) * 4) : kOffNone, 0, 0);
        }
    };
    auto put = [&](int buf, const u32x4 (&xr)[4], const u32x4 (&wr)[4]) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int c = lane + 64 * i, row = c >> 5, f = 4 * (c & 31);
            *(u32x4*)&xs[buf][row][f] = xr[i];
            *(u32x4*)&wsh[buf][row][f] = wr[i];
        }
    };
    float acc = (a.router_b && e < ne) ? a.router_b[e] : 0.0f;
    u32x4 xr[4], wr[4];
    fetch(0, xr, wr);
    put(0, xr, wr);
    const int nch = (d + kChainChunk - 1) / kChainChunk;
    for (int ch = 0; ch < nch; ch++) {
        const int buf = ch & 1;
        if (ch + 1 < nch) fetch((ch + 1) * kChainChunk, xr, wr);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int n = min(kChainChunk, d - ch * kChainChunk);   // a multiple of 32 (d % 32 == 0)
        const float* xp = &xs[buf][tl][0];
        const float* wp = &wsh[buf][el][0];
        for (int j = 0; j < n; j += 32) {
            f32x4 xv[8], wv[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                xv[u] = *(const f32x4*)(xp + j + 4 * u);
                wv[u] = *(const f32x4*)(wp + j + 4 * u);
            }
#pragma unroll
            for (int u = 0; u < 8; u++) {
#pragma unroll
                for (int c = 0; c < 4; c++) acc = __fadd_rn(acc, __fmul_rn(wv[u][c], xv[u][c]));
            }
        }
        if (ch + 1 < nch) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            put(buf ^ 1, xr, wr);
        }
    }
    if (t < nt && e < ne) a.logits[(size_t)t * ne + e] = acc;
}

// The same for batches that leave most of the chip idle, where a chain's
// length is the kernel's time: workgroup = 16 experts x 4 tokens, whose 64
// chains are wave 0's lanes (lane 16 r + i: expert 16 ex + i, token 4 ty + r).
// Wave 0 only adds; two producer waves form the products a chunk of CHUNK steps
// ahead, in LDS as wave 0 reads them ([4 steps][lane], 16 bytes).  A
// producer's unit is 16 steps: its lane 16 r + i holds expert i's row at steps
// 4 r .. 4 r + 3 (one 1 KB load of the transposed copy, nothing twice) and
// token c >> 2's xn at step 4 r + (c & 3) in lane 16 r + c, which the product
// takes by a row broadcast (DPP row_newbcast).  Of three LDS buffers one is
// being summed, one is complete (so that the reads of the next steps cross
// into it without a wait) and one is being filled: one barrier per chunk.
// Bound by the chain: 3.0 ns per step here (a lone wave's dependent add alone
// takes 1.8, a multiply beside it as much again), behind ~5 us of launch and
// first loads.  3 tokens x 32 experts x 2880 steps 23.4 -> 14.0 us, 512 tokens
// 26.5 -> 17.1, 11 tokens x 128 experts x 2048 17.3 -> 11.5 us against
// k_router_exact.  Every lane reading its own 16 bytes of both operands
// instead (no exchange) was bound by the L1: four lanes in four read the same.
constexpr int kPcProducers = 2, kPcSteps = 768;   // steps requested ahead
template <int S>
CPB_DEV float row_bcast(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x150 + S, 0xf, 0xf, true));
}
template <int CHUNK>
__global__ __launch_bounds__(64 * (1 + kPcProducers)) void k_router_exact_small(GroupedArgs a) {
    constexpr int kPcAhead = kPcSteps / CHUNK, kPcQ = CHUNK / 4;      // chunks requested ahead; 16-byte units of a chain's chunk
    constexpr int UP = CHUNK / 16 / kPcProducers;     // a producer's units per chunk
    constexpr int B = CHUNK / 32;                     // its blocks of 8 units
    static_assert(kPcAhead % 3 == 0, "the register sets and the LDS buffers turn together");
    __shared__ __align__(16) f32x4 prod[3][kPcQ][64];
    const int lane = threadIdx.x & 63, w = uniform((int)(threadIdx.x >> 6)), d = a.d, nt = a.n_tok, ne = a.ne;
    const int i = lane & 15, r = lane >> 4, e = blockIdx.x * 16 + i, t = blockIdx.y * 4 + r;
    // whole rounds of the register sets (the barriers of every wave; chunks past
    // the row's end are formed from other values or zeros and not summed)
    const int nch = (d + kPcAhead * CHUNK - 1) / (kPcAhead * CHUNK) * kPcAhead;
    if (w) {
        const __amdgpu_buffer_rsrc_t rx = buf_rsrc(a.xn, (uint32_t)((size_t)nt * d * 4));
        const __amdgpu_buffer_rsrc_t rw = buf_rsrc(a.router_t, (uint32_t)((size_t)router_t_rows(ne) * d * 4));
        const uint32_t u0 = UP * (w - 1);         // units u0 .. of every chunk
        const uint32_t wo = (uint32_t)(blockIdx.x * 16 * d) * 4 + u0 * 1024 + lane * 16;
        const int tx = blockIdx.y * 4 + (i >> 2);
        const uint32_t xo = tx < nt ? (uint32_t)tx * d * 4 + u0 * 64 + (4 * r + (i & 3)) * 4 : kOffNone;
        f32x4 wv[kPcAhead][UP];
        float xv[kPcAhead][UP];
        // (the whole offset in the vector offset: the scalar one is not part
        // of the buffer's range check)
        auto load = [&](int s, int ch) {
            const uint32_t wc = wo + (uint32_t)ch * (CHUNK * 64), xc = xo + (uint32_t)ch * (CHUNK * 4);
#pragma unroll
            for (int u = 0; u < UP; u++) {
                wv[s][u] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, wc + u * 1024, 0, 0));
                xv[s][u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, xc + u * 64, 0, 0));
            }
            __builtin_amdgcn_sched_barrier(0);    // one order of requests everywhere: exact waits
        };
        auto emit = [&](int s, int buf) {         // the chunk in register set s
#pragma unroll
            for (int u = 0; u < UP; u++) {
                auto token = [&](auto T) {
                    constexpr int k = decltype(T)::value;
                    prod[buf][4 * (u0 + u) + r][16 * k + i] =
                        f32x4{__fmul_rn(wv[s][u][0], row_bcast<4 * k>(xv[s][u])), __fmul_rn(wv[s][u][1], row_bcast<4 * k + 1>(xv[s][u])),
                              __fmul_rn(wv[s][u][2], row_bcast<4 * k + 2>(xv[s][u])), __fmul_rn(wv[s][u][3], row_bcast<4 * k + 3>(xv[s][u]))};
                };
                token(std::integral_constant<int, 0>{});
                token(std::integral_constant<int, 1>{});
                token(std::integral_constant<int, 2>{});
                token(std::integral_constant<int, 3>{});
            }
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int s = 0; s < kPcAhead; s++) load(s, s);
        emit(0, 0);
        load(0, kPcAhead);
        emit(1, 1);
        load(1, kPcAhead + 1);
        for (int k = 0; k < nch; k += kPcAhead) {
#pragma unroll
            for (int j = 0; j < kPcAhead; j++) {
                // the products written so far, and nothing else, before the barrier
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
                __builtin_amdgcn_s_barrier();     // chunk k + j - 1 is summed, its buffer free
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
                emit((j + 2) % kPcAhead, (j + 2) % 3);            // chunk k + j + 2
                load((j + 2) % kPcAhead, k + j + 2 + kPcAhead);
            }
        }
        return;
    }
    // a chunk's reads are waited for before its sums, so the barrier after them
    // needs no wait of its own (reads of the next, complete chunk stay in flight)
    auto arrive = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
    };
    float acc = (a.router_b && e < ne) ? a.router_b[e] : 0.0f;
    const int nb = d / 32;                        // blocks of 8 units (d % 32 == 0), B per chunk
    f32x4 v[8];
    auto block = [&](const f32x4* nx) {           // sums the 8 units in v, reads the next 8
#pragma unroll
        for (int h = 0; h < 8; h += 4) {
            asm volatile("" : "+v"(v[h + 3]));    // one wait for the four units
#pragma unroll
            for (int u = h; u < h + 4; u++) {
#pragma unroll
                for (int c = 0; c < 4; c++) acc = __fadd_rn(acc, v[u][c]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = h; u < h + 4; u++) v[u] = nx[u * 64];
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // block m's successor in buffer j: this chunk's, or the first of the next chunk, which is complete
    auto next = [&](int j, int m) { return m < B - 1 ? &prod[j][8 * (m + 1)][lane] : &prod[(j + 1) % 3][0][lane]; };
    int k = 0;
    arrive();
#pragma unroll
    for (int u = 0; u < 8; u++) v[u] = prod[0][u][lane];
    // (short of the end, so that the last three chunks' barriers are counted below:
    // nch in all, as the producers')
    for (; B * (k + 3) < nb; k += 3) {
#pragma unroll
        for (int j = 0; j < 3; j++) {
#pragma unroll
            for (int m = 0; m < B; m++) block(next(j, m));
            arrive();                             // of the next chunk
        }
    }
#pragma unroll
    for (int j = 0; j < 3; j++) {
#pragma unroll
        for (int m = 0; m < B; m++)
            if (B * (k + j) + m < nb) block(next(j, m));
        if (k + j + 1 < nch) arrive();
    }
    for (k += 4; k < nch; k++) arrive();          // the producers' last rounds
    if (t < nt && e < ne) a.logits[(size_t)t * ne + e] = acc;
}

// router_w [ne][d] -> router_t [router_t_rows(ne) / 16][d / 4][16][4] (load time; rows past ne zero)
__global__ __launch_bounds__(256) void k_router_transpose(const float* __restrict__ w, float* __restrict__ out, int ne, int d) {
    const int i = blockIdx.x * 256 + threadIdx.x;                    // 16-byte unit of the copy
    if (i >= router_t_rows(ne) * (d / 4)) return;
    const int j4 = i / 16 % (d / 4), e = i / (16 * (d / 4)) * 16 + i % 16;
    ((float4*)out)[i] = e < ne ? ((const float4*)w)[(size_t)e * (d / 4) + j4] : float4{0, 0, 0, 0};
}
int launch_router_transpose(const float* w, float* out, int ne, int d, hipStream_t s) {
    hipLaunchKernelGGL(k_router_transpose, dim3((router_t_rows(ne) * (d / 4) + 255) / 256), dim3(256), 0, s, w, out, ne, d);
    return hipGetLastError() == hipSuccess ? 0 : -19;
}


// ---- 3. top-k + softmax of a token's exact logits, one wavefront ----
// The reference selects by descending value with the lowest index winning ties
// (engine_gpt2.rs:852-867 insertion with strict comparisons;
// engine_qwen2.rs:403-410 stable sort), then takes a softmax over the k
// selected.  The logits are the reference's own, so the order is exact on
// them: lane l holds experts l + 64 j as order-preserving 32-bit keys, K
// rounds of a wave maximum, the lowest index by ballot.  A NaN ranks last (a
// strict comparison never lets one in), as -inf.
// Bound by the rounds' chain in the wave, so four tokens share a workgroup to
// put all of them in flight at once (kernel traces, against decode's selector
// with its intervals and certificate): 512 tokens x 32 experts 6.2 -> 5.0 us, 2049
// x 128 22 -> 5.
struct TokenLogits {
    float v[4];
};
CPB_DEV TokenLogits load_logits(const GroupedArgs& a, int t) {
    TokenLogits l;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int e = (int)(threadIdx.x & 63) + 64 * j;
        l.v[j] = e < a.ne && t < a.n_tok ? a.logits[(size_t)t * a.ne + e] : 0.0f;
    }
    return l;
}
// rank i's expert in lane i < k (the softmax weights go to a.wts)
CPB_DEV int select_exact(const GroupedArgs& a, const TokenLogits& l, int t) {
    const int lane = threadIdx.x & 63, K = a.k;
    uint32_t key[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float v = l.v[j] + 0.0f;                   // -0 and +0 are equal
        key[j] = lane + 64 * j < a.ne ? (v == v ? float_key(v) : 1u) : 0u;      // float_key(-inf) > 1
    }
    int my_e = 0;
    uint32_t my_k = 0u;
    for (int i = 0; i < K; i++) {
        const uint32_t m = wave_max_u32(max(max(key[0], key[1]), max(key[2], key[3])));
        int e = 0;
#pragma unroll
        for (int j = 3; j >= 0; j--) {
            const uint64_t b = __ballot(key[j] == m);
            if (b) e = 64 * j + (int)__builtin_ctzll(b);
        }
        if (lane == i) { my_e = e; my_k = m; }
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (lane + 64 * j == e) key[j] = 0u;         // taken
    }
    const float my_l = my_k > 1u ? key_float(my_k) : -__builtin_inff();
    // softmax over the k selected, reference order: ex_i = exp(l_i - l_0)
    // (lane i), then the serial sum ex_0 + ex_1 + ...
    const float l0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, my_l), 0));
    const float ex = expf(my_l - l0);
    float wsum = 0.0f;
    for (int i = 0; i < K; i++) wsum += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ex), i));
    if (lane < K) a.wts[(size_t)t * K + lane] = ex / wsum;
    return my_e;
}

__global__ __launch_bounds__(256) void k_select_batch(GroupedArgs a) {
    const int lane = threadIdx.x & 63, t = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (t >= a.n_tok) return;
    const int e = select_exact(a, load_logits(a, t), t);
    if (lane < a.k) a.ids[(size_t)t * a.k + lane] = e;
}

// ---- 4. grouping by expert ----
// One workgroup of 1024 threads, thread tid holding the experts of pairs tid +
// 1024 u (u < PER; -1: none): each pair takes its place among its expert's
// pairs from an LDS counter (arrival order: any order serves, a pair's outputs
// do not depend on its tile or on the other pairs there), then the exclusive
// prefix of the counts (pairs and tiles of a.tile pairs), each pair written at
// its expert's offset + its place, and the tile list.  The caller's config
// check bounds n_expert <= 256 (the LDS tables).
template <int PER>
CPB_DEV void group_pairs(const GroupedArgs& a, const int (&ex)[PER]) {
    __shared__ int cnt_l[256], off_l[256], toff_l[256];
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, ne = a.ne;
    for (int e = tid; e < ne; e += blockDim.x) cnt_l[e] = 0;
    int rk[PER];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PER; u++)
        rk[u] = ex[u] >= 0 ? __hip_atomic_fetch_add(cnt_l + ex[u], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) : 0;
    __syncthreads();
    if (w == 0) {
        int o = 0, to = 0;
        for (int base = 0; base < ne; base += 64) {
            const int e = base + lane;
            const int c = e < ne ? cnt_l[e] : 0;
            const int tl = (c + a.tile - 1) / a.tile;
            int ic = c, it = tl;
#pragma unroll
            for (int s2 = 1; s2 < 64; s2 <<= 1) {
                const int uc = __shfl_up(ic, s2), ut = __shfl_up(it, s2);
                if (lane >= s2) { ic += uc; it += ut; }
            }
            if (e < ne) { off_l[e] = o + ic - c; toff_l[e] = to + it - tl; }
            o += __shfl(ic, 63);
            to += __shfl(it, 63);
        }
        if (lane == 0) *a.ntiles = to;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PER; u++)
        if (ex[u] >= 0) a.sorted[off_l[ex[u]] + rk[u]] = tid + u * 1024;
    for (int e = w; e < ne; e += 16) {
        const int c = cnt_l[e], nt = (c + a.tile - 1) / a.tile;
        for (int j = lane; j < nt; j += 64) a.tiles[toff_l[e] + j] = int4{e, off_l[e] + a.tile * j, min(a.tile, c - a.tile * j), 0};
    }
}
// n_tok * k <= 16384 = kScanPer * 1024 (the caller's config check)
constexpr int kScanPer = 16;                   // pairs per thread held in registers
__global__ __launch_bounds__(1024) void k_group_scan(GroupedArgs a) {
    const int np = a.n_tok * a.k;
    int ex[kScanPer];                          // every pair's expert requested before the first wait
#pragma unroll
    for (int u = 0; u < kScanPer; u++) {
        const int p = (int)threadIdx.x + u * 1024;
        ex[u] = p < np ? a.ids[p] : -1;
    }
    group_pairs<kScanPer>(a, ex);
}
// Small batches: selection and grouping in one launch, a wave per kSelTok
// tokens (16 waves; np <= 1024).  One workgroup's four rounds of selection cost
// less than a launch and its gap at few tokens (3 tokens 9.3 -> 4.0 us) and the
// same at 64 (whole layer of 32 experts, 128.3 us at 64 tokens fused, 127.4 at 65
// in two launches); beyond, its waves would rank more tokens in turn while the
// chip stands idle.
constexpr int kSelTok = 4, kSelMax = 16 * kSelTok;
__global__ __launch_bounds__(1024) void k_select_group(GroupedArgs a) {
    __shared__ int ids_l[kSelMax * 8];
    const int lane = threadIdx.x & 63, w = uniform((int)(threadIdx.x >> 6)), np = a.n_tok * a.k;
    TokenLogits l[kSelTok];
#pragma unroll
    for (int i = 0; i < kSelTok; i++) l[i] = load_logits(a, w + 16 * i);
#pragma unroll
    for (int i = 0; i < kSelTok; i++) {
        const int t = w + 16 * i;
        if (t < a.n_tok) {
            const int e = select_exact(a, l[i], t);
            if (lane < a.k) ids_l[t * a.k + lane] = e;
        }
    }
    __syncthreads();
    const int ex[1] = {(int)threadIdx.x < np ? ids_l[threadIdx.x] : -1};
    group_pairs<1>(a, ex);
}

// One block of the grouped product: A = 16 raw code bytes (both K halves),
// B = the 32-byte half-image, hardware scale = the block's e8m0 byte.
// SEL: which byte of the word ew is the block's e8m0 (the instruction's
// scale operand select), so four blocks share one scale register
template <int SEL>
CPB_DEV v16f mx_block_mfma(const u32x4& w, const u32x4& x0, const u32x4& x1, uint32_t ew) {
    const v8i_g A = {(int)w[0], (int)w[1], (int)w[2], (int)w[3], 0, 0, 0, 0};
    const v8i_g B = {(int)x0[0], (int)x0[1], (int)x0[2], (int)x0[3], (int)x1[0], (int)x1[1], (int)x1[2], (int)x1[3]};
    const v16f Z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A, B, Z, 4, 0, SEL, (int)ew, 0, 127);
}
// the same with the byte index a value that is constant once the caller's
// loop is unrolled
CPB_DEV v16f mx_block_mfma_b(const u32x4& w, const u32x4& x0, const u32x4& x1, uint32_t ew, int sel) {
    switch (sel & 3) {
        case 0: return mx_block_mfma<0>(w, x0, x1, ew);
        case 1: return mx_block_mfma<1>(w, x0, x1, ew);
        case 2: return mx_block_mfma<2>(w, x0, x1, ew);
        default: return mx_block_mfma<3>(w, x0, x1, ew);
    }
}

// A k-part's two chains (blocks 0-7 and 8-14) are staged and multiplied as two
// sub-parts.  LDS staging of one sub-part's activations for a 32-token tile:
// per block i < 8 and token ti a 64-byte slot whose four 16-byte chunks are
// XOR-swizzled by the token (chunk c at position c ^ swz(ti)), then the 8 x 32
// scales; the staging's last rounds fill up to whole rounds of NW waves.  The
// swizzle puts the reads (lane ti reads chunk 2hb or 2hb + 1 of slot ti) on
// distinct banks in every group of 8 and of 16 lanes (80-byte padded slots had
// 2.75 M conflict cycles per gate/up launch).
constexpr int kSlot = 64;
constexpr int kSub = kSubUnits;               // blocks of a sub-part (the second has 7)
static_assert(kSub == 8 && kBlkPerPart == 15, "sub-parts of 8 and 7 blocks");
CPB_DEV_HOST_INLINE int stage_swz(int ti) { return ((ti >> 1) ^ (ti >> 2)) & 3; }
// image loads of 1 KB (half a block's tokens) and scale loads of 64 per wave and sub-part
constexpr int stage_img(int nw) { return (2 * kSub + nw - 1) / nw; }
constexpr int stage_sc(int nw) { return (kSub / 2 + nw - 1) / nw; }
constexpr int stage_bytes(int nw) { return nw * (stage_img(nw) * 1024 + stage_sc(nw) * 256); }
// Waves per workgroup, each with two 32-row tiles
constexpr int kGemmWaves = 4;

// The two staging buffers (a k-part's first and second sub-part): separate
// objects, so that the compiler can tell the buffer being filled from the one
// being read (it would otherwise wait for every direct load before each read)
constexpr int kStageBytes = stage_bytes(kGemmWaves);
__shared__ __align__(16) unsigned char g_stage0[kStageBytes];
__shared__ __align__(16) unsigned char g_stage1[kStageBytes];

// Direct global-to-LDS staging (no staging registers): each wavefront
// instruction writes 1 KB of LDS, lane L at byte 16 L, so lane L fetches the
// chunk the swizzled layout puts there (token h*16 + L/4 of the block, chunk
// (L & 3) ^ swz(token)); the scales take 64 per instruction.
// An offset beyond both buffers (at most 16384 rows x 120 blocks x 64 bytes),
// twice of which is beyond them too:
constexpr uint32_t kStageNone = 0x40000000u;
struct DmaPlan {
    __amdgpu_buffer_rsrc_t ri, rs;
    uint32_t vbase0, vbase1, sbase;  // bytes: block 0 of the lane's chunk in token half 0 / 1, its scale
};
CPB_DEV DmaPlan dma_plan(const uint8_t* img, const float* sc, size_t rows, int nbk, const int* src) {
    const int L = threadIdx.x & 63;
    DmaPlan p;
    p.ri = buf_rsrc(img, (uint32_t)(rows * nbk * kImg));
    p.rs = buf_rsrc(sc, (uint32_t)(rows * nbk * 4));
    const int t0 = L >> 2, t1 = 16 + (L >> 2), r0 = src[t0], r1 = src[t1];
    p.vbase0 = r0 >= 0 ? (uint32_t)r0 * nbk * kImg + (uint32_t)(((L & 3) ^ stage_swz(t0)) << 4) : kStageNone;
    p.vbase1 = r1 >= 0 ? (uint32_t)r1 * nbk * kImg + (uint32_t)(((L & 3) ^ stage_swz(t1)) << 4) : kStageNone;
    const int rs_ = src[L & 31];
    p.sbase = rs_ >= 0 ? (uint32_t)rs_ * nbk * 4 : kStageNone;
    return p;
}
// Sub-part sp (k-part sp / 2, its blocks 0-7 or 8-14) into st.  Every wave
// issues the same number of loads whatever the sub-part: the pieces past its
// last block, past the last k-part and past the last round read nothing and
// write zeros.  So a wave's loads are counted exactly, and the wait for these
// does not wait for what is requested after them.
template <int NW>
CPB_DEV void stage_dma(const DmaPlan& p, int nbk, int sp, unsigned char* st) {
    // the wave index as a scalar: every condition and LDS address below is
    // then scalar work
    const int w = uniform((int)(threadIdx.x >> 6)), L = threadIdx.x & 63;
    const int b0 = (sp >> 1) * kBlkPerPart + (sp & 1) * kSub;
    const int lim = min(kSub - (sp & 1), nbk - b0);
#pragma unroll
    for (int k = 0; k < stage_img(NW); k++) {
        const int m = w + k * NW, i = m >> 1, h = m & 1;
        const uint32_t add = (uint32_t)(b0 + i) * kImg + (i < lim ? 0u : kStageNone);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(p.ri, (lds_void_g*)(st + m * 1024), 16, (h ? p.vbase1 : p.vbase0) + add, 0, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < stage_sc(NW); k++) {
        const int n = w + k * NW, i = 2 * n + (L >> 5);
        const uint32_t off = p.sbase + (uint32_t)(b0 + i) * 4 + (i < lim ? 0u : kStageNone);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(p.rs, (lds_void_g*)(st + NW * stage_img(NW) * 1024 + n * 256), 4, off, 0, 0, 0);
    }
}

// Weight operands of the lane's two rows (one in each of the wave's two row
// tiles): a row's units (16 per k-part: the e8m0 bytes, then 15 blocks) follow
// each other at ustride bytes from off in the expert's stream; rs covers the
// expert's whole stream (out-of-range offsets read 0).
struct WeightStream {
    __amdgpu_buffer_rsrc_t rs;
    uint32_t off[2], ustride;
};
// Both K halves of the instruction's A operand (both lane halves) take the same
// 16 bytes of a row.  So that no byte is loaded twice, one load brings two
// units, lanes 0-31 unit 2 j + 1 and lanes 32-63 unit 2 j + 2 (a k-part's last
// pair: block 14 and the next k-part's e8m0 bytes), and each goes to both
// halves by v_permlane32_swap, which works in place: the pair's registers hold
// y until the odd block has used it.  Half the L1 traffic and half the
// registers of a load per unit.
CPB_DEV void split_pair(const u32x4& v, u32x4& x, u32x4& y) {
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const auto r = __builtin_amdgcn_permlane32_swap(v[c], v[c], false, false);
        x[c] = r[0];
        y[c] = r[1];
    }
}

// The loop shared by the two grouped GEMMs: two row tiles x one token tile per
// wave, whose activations both tiles' products read from LDS once (a b128 read
// takes the LDS 16 cycles, so at one tile per read the four SIMDs' reads took
// 61 ns per block and tile against 28 of matrix-core and 27 of VALU work: two,
// three and four waves per SIMD all ran at that rate).  512 tokens x 32
// experts: gate/up 161 -> 149 us, down 87 -> 76; 2049 x 128: 574 -> 496 and
// 298 -> 255 (kernel traces of one layer called again and again).  Now VALU
// issue comes first: by the counters at 512 tokens it takes 56 % of the
// gate/up's time (30 instructions per MFMA: 16 fmas, 4 exchanges of split_pair, 2
// chain adds, the MFMA and an address in the loop, 5 before and after it), the
// matrix cores 30 % and the LDS reads about as much.  Per block, D = A(rows) x B(tokens) on the matrix cores and acc = fma(D, xsb, acc)
// in block order, in two chains per k-part (its sub-parts, as the decode
// kernels' two wavefronts per k-part), the chains added to the total in order.
//
// Software pipeline: the two tiles' MFMAs and the other tile's sixteen fmas
// alternate, so the matrix core and the VALU run side by side; each weight pair
// is requested again, a k-part ahead, right after it has been taken apart.  Two
// LDS buffers alternate: right after the barrier that opens a sub-part the
// direct loads of the next go into the buffer that every wave has finished
// reading.  Before that barrier a wave waits for its own direct loads and not
// for the weight pairs requested since (a full fence there, which drained
// them, exposed a memory latency per k-part).
// TRACE writes the int32 block sums S = D * 2^(128 - e) of valid rows (tb, per
// row tile; null: none).
constexpr uint32_t s_waitcnt_vm(int n) { return (uint32_t)((n & 15) | 0x70 | 0xF00 | ((n >> 4) << 14)); }   // vmcnt(n) only
template <bool TRACE, int NW>
CPB_DEV void grouped_parts(const WeightStream& ws, int P, const uint8_t* img, const float* sc, size_t rows, int nbk,
                           const int* src, int lane, int32_t* const (&tb)[2], v16f (&tot)[2]) {
    const int ti = lane & 31, hb = lane >> 5;
    // the lane's two 16-byte chunks (2hb, 2hb + 1) of its token's slot
    const int o0 = ti * kSlot + (((2 * hb) ^ stage_swz(ti)) << 4), o1 = ti * kSlot + (((2 * hb + 1) ^ stage_swz(ti)) << 4);
    const int os = NW * stage_img(NW) * 1024 + ti * 4;
    const DmaPlan dp = dma_plan(img, sc, rows, nbk, src);
    auto wload = [&](int m, uint32_t unit) {
        return __builtin_amdgcn_raw_buffer_load_b128(ws.rs, ws.off[m] + unit * ws.ustride, 0, 0);
    };
    u32x4 ex[2], wp[2][8];
    ex[0] = wload(0, 0);
    ex[1] = wload(1, 0);
    __builtin_amdgcn_sched_barrier(0);
    stage_dma<NW>(dp, nbk, 0, g_stage0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 8; j++) {
        wp[0][j] = wload(0, 2 * j + 1 + hb);
        wp[1][j] = wload(1, 2 * j + 1 + hb);
        __builtin_amdgcn_sched_barrier(0);   // in the loop's order: exact waits there
    }
    tot[0] = tot[1] = v16f{};
    for (int q = 0; q < P; q++) {
#pragma unroll
        for (int half = 0; half < 2; half++) {
            const int sp = 2 * q + half, nblk = kSub - half;
            // the sub-part's activations have landed: the wave's own (all but
            // the 2 x 4 weight pairs requested since), then every wave's
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(s_waitcnt_vm(8));
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("" ::: "memory");
            const unsigned char* st = half ? g_stage1 : g_stage0;
            stage_dma<NW>(dp, nbk, sp + 1, half ? g_stage0 : g_stage1);
            __builtin_amdgcn_sched_barrier(0);
            const unsigned char* x0 = st + o0;
            const unsigned char* x1 = st + o1;
            const unsigned char* sl = st + os;
            v16f acc[2] = {}, D[2];
            u32x4 xa[2][2], X[2], Y[2];
            float sa[2], sd = 0.0f;
            auto xread = [&](int j) {
                xa[j & 1][0] = *(const u32x4*)(x0 + j * 32 * kSlot);
                xa[j & 1][1] = *(const u32x4*)(x1 + j * 32 * kSlot);
                sa[j & 1] = *(const float*)(sl + j * 128);
            };
            auto trace = [&](int m, int i) {
                const int bl = half * kSub + i, b = q * kBlkPerPart + bl;
                const uint32_t eb = (ex[m][bl >> 2] >> (8 * (bl & 3))) & 0xffu;
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int rl = 8 * (r >> 2) + 4 * hb + (r & 3);
                    const int e_r = __shfl((int)eb, rl);
                    if (tb[m] && b < nbk) tb[m][rl * (size_t)nbk + b] = (int)ldexpf(D[m][r], 128 - e_r);
                }
            };
            auto add = [&](int m, int i, float s) {
                if (TRACE) trace(m, i);
                else mfma_result(D[m]);
#pragma unroll
                for (int r = 0; r < 16; r++) acc[m][r] = fmaf(D[m][r], s, acc[m][r]);
            };
            // block i of tile m: an even block's pair is taken apart first (in
            // place), and requested again once the odd one has used its half
            auto refill = [&](int m, int i) { wp[m][half * 4 + (i >> 1)] = wload(m, 16 * (q + 1) + half * 8 + (i & ~1) + 1 + hb); };
            auto mul = [&](int m, int i) {
                const int bl = half * kSub + i;
                if (!(i & 1)) split_pair(wp[m][half * 4 + (i >> 1)], X[m], Y[m]);
                D[m] = mx_block_mfma_b(i & 1 ? Y[m] : X[m], xa[i & 1][0], xa[i & 1][1], ex[m][bl >> 2], bl);
                if (TRACE) mfma_result_now(D[m]);        // these kernels spill, results among what they spill
                if (i & 1) refill(m, i);
            };
            xread(0);
            xread(1);
#pragma unroll
            for (int i = 0; i < nblk; i++) {
                mul(0, i);
                // keep the order as written
                __builtin_amdgcn_sched_barrier(0);
                if (i) add(1, i - 1, sd);
                __builtin_amdgcn_sched_barrier(0);
                mul(1, i);
                sd = sa[i & 1];
                if (i + 2 < nblk) xread(i + 2);
                __builtin_amdgcn_sched_barrier(0);
                add(0, i, sd);
                __builtin_amdgcn_sched_barrier(0);
            }
            add(1, nblk - 1, sd);
            // the chains into the totals, in order
#pragma unroll
            for (int m = 0; m < 2; m++) {
#pragma unroll
                for (int r = 0; r < 16; r++) tot[m][r] += acc[m][r];
                if (half == 1) {
                    ex[m] = Y[m];                // the next k-part's e8m0 bytes
                    refill(m, nblk - 1);
                }
            }
        }
    }
    // the last direct loads (past the last k-part: zeros) land before the wave
    // can end and its LDS be given away
    __builtin_amdgcn_s_waitcnt(s_waitcnt_vm(0));
}

// ---- 5. grouped gate/up + SwiGLU-OAI + Q8 (+ image of h) ----
// one workgroup per (token tile, group of kGemmWaves row tiles)
// (grouped_item); wave w: gate and up of row tile w of the group, so SwiGLU, the
// Q8 and the image of a row tile finish in its wave.
template <bool TRACE>
__global__ __launch_bounds__(64 * kGemmWaves) __attribute__((amdgpu_waves_per_eu(2))) void k_gateup_grouped(GroupedArgs a) {
    constexpr int NW = kGemmWaves;
    __shared__ int src[32];
    const int T = a.dff / 32, P = a.parts_gu, nb = a.nb;
    int tile, grp;
    if (!grouped_item(uniform(*a.ntiles), (T + NW - 1) / NW, &tile, &grp)) return;
    const int4 tl = a.tiles[tile];
    const int e = uniform(tl.x), start = uniform(tl.y), cnt = uniform(tl.z);
    const int lane = threadIdx.x & 63, w = uniform((int)(threadIdx.x >> 6));
    const int rt = grp * NW + w;
    const bool live = rt < T;
    const int ti = lane & 31, hb = lane >> 5;
    const bool valid = ti < cnt;
    const int pair = valid ? a.sorted[start + ti] : 0;
    if (threadIdx.x < 32) src[threadIdx.x] = valid ? pair / a.k : -1;
    // the biases of the row tile's 32 gate and 32 up rows, requested now and
    // kept in one register until the epilogue (a load issued after the GEMM
    // would wait a full loaded-memory latency)
    __shared__ float bias_s[NW][64];
    const float* bp = hb ? a.up_b : a.gate_b;
    const float bias_v = bp && live ? bp[(size_t)e * a.dff + rt * 32 + ti] : 0.0f;
    __syncthreads();
    WeightStream ws;
    {
        const size_t ex_units = (size_t)T * P * kUnits * 64;         // one expert's gate/up stream
        ws.rs = buf_rsrc(a.gu + (size_t)e * ex_units, (uint32_t)(ex_units * 16));
        ws.off[0] = (uint32_t)((((size_t)(live ? rt : T) * P) * kUnits * 64 + ti) * 16);
        ws.off[1] = ws.off[0] + 32 * 16;
        ws.ustride = 64 * 16;
    }
    int32_t* tb[2] = {nullptr, nullptr};
    if (TRACE && valid && live) {
        tb[0] = a.gu_sums + ((size_t)pair * 2 * a.dff + rt * 32) * nb;
        tb[1] = tb[0] + (size_t)a.dff * nb;
    }
    v16f tot[2];
    grouped_parts<TRACE, NW>(ws, P, a.ximg, a.xsb, (size_t)a.n_tok, nb, src, lane, tb, tot);
    bias_s[w][lane] = bias_v;
    wave_lds_order();                                                  // the wave's own row
    if (!live) return;
    // the lane's rows 8 g + 4 hb + c (g, c < 4): whole hq words, and with rows
    // 16 apart (groups g and g + 2) whole 8-byte image runs
    float hv[16], m = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int rr = 8 * (r >> 2) + 4 * hb + (r & 3);
        const float vg = tot[0][r] + bias_s[w][rr], vu = tot[1][r] + bias_s[w][32 + rr];   // zeros without biases
        const float xg = fminf(vg, a.limit);                           // engine_gpt2.rs:887-906
        const float yu = fminf(fmaxf(vu, -a.limit), a.limit);
        hv[r] = (xg / (1.0f + expf(-a.alpha * xg))) * (yu + 1.0f);
        m = fmaxf(m, fabsf(hv[r]));
    }
    m = fmaxf(m, __shfl_xor(m, 32));
    const float sc = fmaxf(1e-12f, m) / 127.0f;
    if (!valid) return;
    uint8_t* img = a.himg + ((size_t)pair * a.nbf + rt) * kImg;
    // Q8 of the values (the exact division only when some lane's quotient lies
    // near a rounding tie), then the bytes: qw[g] byte c = value 4 g + c; elements
    // e and e + 16 sit at adjacent K (2e, 2e + 1), so groups g and g + 2 fill the
    // 8 bytes K = 16 g + 8 hb .. +7 (g < 2) of each half: byte 2 (c & 1) + (0 for
    // g, 1 for g + 2) of word c >> 1 holds the value's 16h (hi) and l (lo) as
    // e4m3, whose hardware conversion is exact for these integers (|16h| <= 128, 0
    // <= l <= 15)
    int qv[16];
    {
        const float rs = __builtin_amdgcn_rcpf(sc);
        float r[16];
        bool near = false;
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const float y = hv[j] * rs;
            r[j] = __builtin_rintf(y);
            near = near || q8_near_half(y);
        }
        if (near) {
#pragma unroll
            for (int j = 0; j < 16; j++)
                if (q8_near_half(hv[j] * rs)) r[j] = roundf(hv[j] / sc);
        }
#pragma unroll
        for (int j = 0; j < 16; j++) qv[j] = q8_clamp(r[j]);
    }
    uint32_t* hqw = (uint32_t*)(a.hq + (size_t)pair * a.dff + rt * 32 + 4 * hb);
#pragma unroll
    for (int g = 0; g < 4; g++) {
        uint32_t qw = 0u;
#pragma unroll
        for (int c = 0; c < 4; c++) qw |= ((uint32_t)qv[4 * g + c] & 0xffu) << (8 * c);
        hqw[2 * g] = qw;
    }
    float fh[16], fl[16];
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const int h = qv[j] >> 4;
        fh[j] = (float)(16 * h);
        fl[j] = (float)(qv[j] - 16 * h);
    }
#pragma unroll
    for (int g = 0; g < 2; g++) {
        uint32_t hi[2], lo[2];
#pragma unroll
        for (int w2 = 0; w2 < 2; w2++) {
            // word w2: values (g, c0), (g + 2, c0), (g, c0 + 1), (g + 2, c0 + 1), c0 = 2 w2
            const int j0 = 4 * g + 2 * w2, j1 = j0 + 8;
            hi[w2] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(fh[j0 + 1], fh[j1 + 1], __builtin_amdgcn_cvt_pk_fp8_f32(fh[j0], fh[j1], 0, false), true);
            lo[w2] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(fl[j0 + 1], fl[j1 + 1], __builtin_amdgcn_cvt_pk_fp8_f32(fl[j0], fl[j1], 0, false), true);
        }
        *(uint2*)(img + 32 * g + 8 * hb) = make_uint2(hi[0], hi[1]);
        *(uint2*)(img + 32 * g + 8 * hb + 16) = make_uint2(lo[0], lo[1]);
    }
    if (hb == 0) a.hsb[(size_t)pair * a.nbf + rt] = sc;
}

// ---- 6. grouped down (+ bias) into dnout ----
// one workgroup per (token tile, group of 2 kGemmWaves row tiles of 32 rows)
// (grouped_item); wave w: row tiles 2 w and 2 w + 1 of the group.
template <bool TRACE>
__global__ __launch_bounds__(64 * kGemmWaves) __attribute__((amdgpu_waves_per_eu(2))) void k_down_grouped(GroupedArgs a) {
    constexpr int NW = kGemmWaves;
    __shared__ int src[32];
    int tile, grp;
    const int T = a.d / 32;
    if (!grouped_item(uniform(*a.ntiles), (T + 2 * NW - 1) / (2 * NW), &tile, &grp)) return;
    const int4 tl = a.tiles[tile];
    const int e = uniform(tl.x), start = uniform(tl.y), cnt = uniform(tl.z);
    const int lane = threadIdx.x & 63, w = uniform((int)(threadIdx.x >> 6));
    const int RTv = mx_down_rt(a.k), Tv = a.d / RTv, P = a.parts_dn, nbf = a.nbf;
    const int rt = grp * 2 * NW + 2 * w;
    const int ti = lane & 31, hb = lane >> 5;
    const bool valid = ti < cnt;
    const int pair = valid ? a.sorted[start + ti] : 0;
    if (threadIdx.x < 32) src[threadIdx.x] = valid ? pair : -1;
    // the biases of the wave's 64 rows, requested now (one register until the
    // epilogue)
    __shared__ float bias_s[NW][64];
    const float bias_v = a.down_b && rt * 32 + lane < a.d ? a.down_b[(size_t)e * a.d + rt * 32 + lane] : 0.0f;
    __syncthreads();
    WeightStream ws;
    {
        const size_t ex_units = (size_t)Tv * P * kUnits * RTv;      // one expert's down stream
        ws.rs = buf_rsrc(a.dn + (size_t)e * ex_units, (uint32_t)(ex_units * 16));
#pragma unroll
        for (int m = 0; m < 2; m++) {
            const int row_l = (rt + m) * 32 + ti;                    // the lane's A row
            ws.off[m] = rt + m < T ? (uint32_t)(((size_t)(row_l / RTv) * P * kUnits * RTv + row_l % RTv) * 16) : kOffNone;
        }
        ws.ustride = RTv * 16;
    }
    int32_t* tb[2] = {nullptr, nullptr};
    if (TRACE && valid) {
#pragma unroll
        for (int m = 0; m < 2; m++)
            if (rt + m < T) tb[m] = a.dn_sums + ((size_t)pair * a.d + (rt + m) * 32) * nbf;
    }
    v16f tot[2];
    grouped_parts<TRACE, NW>(ws, P, a.himg, a.hsb, (size_t)a.n_tok * a.k, nbf, src, lane, tb, tot);
    bias_s[w][lane] = bias_v;
    wave_lds_order();                                                // the wave's own row
    if (!valid) return;
#pragma unroll
    for (int m = 0; m < 2; m++) {
        if (rt + m >= T) break;
        float* out = a.dnout + (size_t)pair * a.d + (rt + m) * 32 + 4 * hb;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            float4 v;
            float* vp = (float*)&v;
#pragma unroll
            for (int c = 0; c < 4; c++) vp[c] = tot[m][4 * g + c] + bias_s[w][m * 32 + 8 * g + 4 * hb + c];   // zeros without biases
            *(float4*)(out + 8 * g) = v;
        }
    }
}

// ---- 7. per token: x += sum over slots (ascending) of wts * (down + bias) ----
// one thread per 4 consecutive elements (d % 4 == 0), the same fp32 operations
// in the same order as a scalar loop
__global__ __launch_bounds__(256) void k_combine_batch(GroupedArgs a) {
    const int d4 = a.d / 4, K = a.k;
    const size_t n4 = (size_t)a.n_tok * d4;
    const float4* __restrict__ dn = (const float4*)a.dnout;
    float4* __restrict__ x = (float4*)a.x;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n4; i += (size_t)gridDim.x * blockDim.x) {
        const size_t t = i / d4, r4 = i % d4;
        float4 v[8];
        float wk[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            v[k] = k < K ? dn[(t * K + k) * d4 + r4] : float4{0, 0, 0, 0};
            wk[k] = k < K ? a.wts[t * K + k] : 0.0f;
        }
        float4 s = x[i];                                     // engine_gpt2.rs:911-921
#pragma unroll
        for (int k = 0; k < 8; k++) {
            if (k < K) {
                s.x += wk[k] * v[k].x;
                s.y += wk[k] * v[k].y;
                s.z += wk[k] * v[k].z;
                s.w += wk[k] * v[k].w;
            }
        }
        x[i] = s;
    }
}

int launch_grouped_layer(const GroupedArgs& a, bool trace, hipStream_t s, const LaunchEvents* ev) {
    const int nt = a.n_tok;
    if (a.kq) {
        if (launch_prep_kq(a, s)) return -19;
    } else {
        launch(k_prep_batch, dim3(nt), dim3(256), sizeof(float) * (2 * a.d + 64), s, a);
    }
    const int et = router_t_rows(a.ne) / 16, rt = (nt + 3) / 4;
    // One workgroup of 96 KB LDS per CU; up to two per CU with chunks of half
    // the length (48 KB, twice the barriers; whole layer, 128 experts top-8: 132
    // tokens 174.9 -> 170.7 us, 256 tokens 184.2 -> 179.5; 32 experts: 600 tokens
    // 273.3 -> 266.7, 1000 tokens 373.1 -> 367 us against k_router_exact).  Three
    // per CU share the SIMDs' issue: 384 x 128 207.2 -> 206.0, 1536 x 32 514.8 ->
    // 518, so k_router_exact takes those and the larger.
    if (et * rt <= 256) launch(k_router_exact_small<128>, dim3(et, rt), dim3(64 * (1 + kPcProducers)), 0, s, a);
    else if (et * rt <= 512) launch(k_router_exact_small<64>, dim3(et, rt), dim3(64 * (1 + kPcProducers)), 0, s, a);
    else launch(k_router_exact, dim3((a.ne + 7) / 8, (nt + 7) / 8), dim3(64), 0, s, a);
    if (nt <= kSelMax) {
        launch(k_select_group, dim3(1), dim3(1024), 0, s, a);
    } else {
        launch(k_select_batch, dim3((nt + 3) / 4), dim3(256), 0, s, a);
        launch(k_group_scan, dim3(1), dim3(1024), 0, s, a);
    }
    if (a.kq) {
        if (launch_kq_gemms(a, trace, s, ev)) return -19;
        launch(k_combine_batch, dim3((unsigned)std::min<size_t>(((size_t)nt * (a.d / 4) + 255) / 256, 2048)), dim3(256), 0, s, a);
        return hipGetLastError() == hipSuccess ? 0 : -19;
    }
    // one workgroup per (token tile, row group), dealt out by grouped_item:
    // 8 slots per XCD round, enough for the largest tile count
    const int ngu = a.max_tiles * ((a.dff / 32 + kGemmWaves - 1) / kGemmWaves);
    const int ndn = a.max_tiles * ((a.d / 32 + 2 * kGemmWaves - 1) / (2 * kGemmWaves));
    const dim3 ggu((ngu + 7) / 8 * 8), gdn((ndn + 7) / 8 * 8);
    if (ev) armed_events() = ev[0];
    if (trace) launch(k_gateup_grouped<true>, ggu, dim3(64 * kGemmWaves), 0, s, a);
    else launch(k_gateup_grouped<false>, ggu, dim3(64 * kGemmWaves), 0, s, a);
    if (ev) armed_events() = ev[1];
    if (trace) launch(k_down_grouped<true>, gdn, dim3(64 * kGemmWaves), 0, s, a);
    else launch(k_down_grouped<false>, gdn, dim3(64 * kGemmWaves), 0, s, a);
    launch(k_combine_batch, dim3((unsigned)std::min<size_t>(((size_t)nt * (a.d / 4) + 255) / 256, 2048)), dim3(256), 0, s, a);
    return hipGetLastError() == hipSuccess ? 0 : -19;
}

}  // namespace cpb
