// Routing side of the MoE expert path: router GEMV + top-k softmax + Q8_0
// activation quantization (one fused kernel), token->expert dispatch, the
// weighted combine, and the one-time weight repack.
#include <algorithm>

#include "jxmoe_device.h"
#include "jxmoe_dispatch.h"
#include "jxmoe_gemm.h"
#include "jxmoe_kernels.h"

namespace jx {

// Q8_0 of one 32-block held one value per lane of a half-wave (q8_block_vals),
// stored to o8 when ok: the int8 quants and (scale, block sum of q).  Returns q.
__device__ __forceinline__ int quant_block(float v, int l32, bool ok, const ActQ8& o8, size_t row, int b,
                                           float2* scale_out = nullptr) {
    float2 sv;
    const int q = q8_block_vals(v, sv);
    if (ok) {
        o8.q[row * o8.K + b * 32 + l32] = (int8_t)q;
        if (l32 == 0) {
            o8.s[row * (o8.K / 32) + b] = sv;
            if (scale_out) *scale_out = sv;
        }
    }
    return q;
}

// Matrix-core form (ActH) of Q8_0 rows, the down GEMM's operand: one
// exponent per row, E = exponent(max block scale of the row) - 7, so every
// dx * q * 2^-E (exact in fp32: an 11-bit scale times |q| <= 127) is below
// 2^15 and rounds to fp16 once.  The K-quant
// min-term values dx * sum(q) are stored times 2^-E as well; pe holds 2^E
// for every half-unit of the row.
// Row exponent of the matrix-core form from the row's largest block scale M.
__device__ __forceinline__ int acth_exponent(float M) {
    return (M > 0.0f) ? (int)((__float_as_uint(M) >> 23) & 0xFF) - 127 - 7 : 0;
}

// Elements 8c .. 8c+7 of one row (all in one 32-block): one 16-byte store, plus the row's pe entry
// and the block's min-term pieces when the chunk opens them.
// qq: the chunk's 8 quants, sb: its block's (scale, sum).
__device__ __forceinline__ void acth_chunk_v(uint2 qq, float2 sb, int K, const ActH& o, size_t row, int c, int E) {
    const int KH = K / 128;
    const int i = 8 * c, b = i >> 5, hh = i >> 7;
    const float dn = __uint_as_float((uint32_t)(127 - E) << 23), up = __uint_as_float((uint32_t)(127 + E) << 23);
    const float s = sb.x * dn;  // exact: power-of-two scaling
    uint32_t hw[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const uint32_t word = u < 2 ? qq.x : qq.y;
        const int q0 = (int)(int8_t)(word >> (16 * (u & 1))), q1 = (int)(int8_t)(word >> (16 * (u & 1) + 8));
        const _Float16 h0 = (_Float16)(s * (float)q0), h1 = (_Float16)(s * (float)q1);  // products exact
        hw[u] = (uint32_t)__builtin_bit_cast(uint16_t, h0) | ((uint32_t)__builtin_bit_cast(uint16_t, h1) << 16);
    }
    *reinterpret_cast<uint4*>(o.hl + row * (size_t)K + i) = make_uint4(hw[0], hw[1], hw[2], hw[3]);
    if ((i & 127) == 0) o.pe[row * (size_t)KH + hh] = up;
    if ((i & 31) == 0)  // exact: 11-bit scale x |sum| < 2^12, times 2^-E
        store_pieces3(o.xm + row * (size_t)o.KU * 24 + (b / 8) * 24 + (b % 8), sb.x * sb.y * dn);
}

// One row by one wave (all 64 lanes): the row exponent from a wave maximum of
// the block scales, then four chunks per lane per pass with every load issued
// before the first store.
__device__ void write_acth_row(const int8_t* q, const float2* sc, int K, const ActH& o, size_t row, int lane) {
    const int KB = K / 32;
    float M = 0.0f;
    for (int b = lane; b < KB; b += 64) M = fmaxf(M, sc[b].x);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) M = fmaxf(M, __shfl_xor(M, off, 64));
    const int E = acth_exponent(M);
    constexpr int U = 4;
    const int nc = K / 8;
    for (int c0 = lane; c0 < nc; c0 += U * 64) {
        uint2 qq[U];
        float2 sb[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = min(c0 + u * 64, nc - 1);
            qq[u] = *reinterpret_cast<const uint2*>(q + 8 * c);
            sb[u] = sc[c >> 2];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (c0 + u * 64 < nc) acth_chunk_v(qq[u], sb[u], K, o, row, c0 + u * 64, E);
    }
}

int chain_stride(int d) { return chain_stride_of(d); }

void chain_rows(const float* rows, int nrows, int d, float* out) {
    const int S = chain_stride_of(d);
    std::fill(out, out + (size_t)nrows * 16 * S, 0.0f);
    for (int r = 0; r < nrows; ++r)
        for (int e = 0; e < d; ++e) out[(size_t)r * 16 * S + (e & 15) * S + (e >> 4)] = rows[(size_t)r * d + e];
}

// Routing for many tokens.  A block takes T tokens (T <= RT_TMAX, fewer when
// d is large or n small) and a split of the router rows (RPB rows; a single
// split when the rows fit one block's 16 lane groups):
//  1. the block's token rows -> LDS, chain-major.
//  2. (row split 0) Q8_0 of x, one thread per 32-block (quantize_row_q8_0,
//     src/quant.cpp:1029-1045): amax, d = amax/127 (IEEE division), id = 1/d,
//     q = clamp(round-half-away(x*id)), stored scale = truncated fp16 of d; the
//     block sum of q rides along for the Q4_0 (-8 offset) and Q4_K (min)
//     terms.  With a matrix-core consumer the rows' ActH form follows.
//  3. Router logits in vec_dot_f32's exact fp32 order (src/quant.cpp:2756-2778):
//     16 lanes per router row, lane j runs the FMA chain over elements 16i+j
//     (lanes 0-7 are the reference's acc0, 8-15 its acc1), then acc0+acc1 and
//     the sequential sum of the 8 lanes (d % 32 == 0: no tails).  One router
//     load (four chain steps, chain-major copy) feeds every token of the block,
//     whose chains are independent.  The shared-expert gate vector
//     (transformer.cpp:2748-2751) is one more row.
//  4. Top-k by rank counting (descending logit, ties by index) and softmax over
//     the k selected logits (select_experts_cache_aware, src/tier.cpp:144-188):
//     in the block with a single row split, else in k_route_topk once every
//     split has written its logits.
#ifndef JX_RT_TMAX
#define JX_RT_TMAX 4
#endif
#ifndef JX_RT_LDS_KB
#define JX_RT_LDS_KB 80
#endif
#ifndef JX_RT_UNROLL
#define JX_RT_UNROLL 4
#endif
constexpr int RT_THREADS = 256;
constexpr int RT_GROUPS = RT_THREADS / 16;  // router rows in flight per block
constexpr int RT_UNROLL = JX_RT_UNROLL;     // router loads in flight per lane (four chain steps each)
constexpr int RT_TMAX = JX_RT_TMAX;
constexpr size_t RT_LDS_TARGET = JX_RT_LDS_KB * 1024;  // two blocks per CU

static size_t route_lds(int T, int d, int E) {
    return ((size_t)T * 16 * rs_stride(d) + (size_t)T * E) * sizeof(float);
}

struct RouteShape {
    int T, RS, RPB;
};

// Rows R = E (+1 shared gate): up to 16 rows one split (fused top-k), more in
// splits of 16.  Tokens per block: a fused Mixtral-sized router measured best
// at 2, split routers (61 and 128 rows, d 2048) at 4 (1, 2 and 6-8 slower);
// small batches take one token per block for parallelism.
static RouteShape route_shape(const RouteArgs& a) {
    const int R = a.E + (a.shgate ? 1 : 0);
    RouteShape r;
    r.RS = R <= RT_GROUPS ? 1 : (R + RT_GROUPS - 1) / RT_GROUPS;
    r.RPB = r.RS == 1 ? R : RT_GROUPS;
    int T = r.RS == 1 ? 2 : RT_TMAX;
    if (a.n < 64 * T) T = std::max(1, a.n / 64);
    while (T > 1 && route_lds(T, a.d, a.E) > RT_LDS_TARGET) --T;
    r.T = T;
    return r;
}

// rpb = 0: only steps 1-2 (the quantized and matrix-core forms of x), for k_route_mfma.
template <int T>
__global__ void __launch_bounds__(RT_THREADS) k_route(RouteArgs a, int nsplit, int rpb) {
    extern __shared__ __align__(16) float lds[];
    __shared__ int sel[T][MAX_K];
    __shared__ float shl[T];
    const int d = a.d, E = a.E, S = rs_stride(d), RS = 16 * S, KB = d / 32;
    const int split = blockIdx.x % nsplit;
    const int t0 = (blockIdx.x / nsplit) * T, nt = min(T, a.n - t0);
    const int tid = threadIdx.x;
    float* xs = lds;                                       // [T][16][S] chain-major rows
    float* lg = xs + T * RS;                               // [T][E] logits
    // every selection slot holds a valid expert even if NaN logits break the ranking
    for (int i = tid; i < T * MAX_K; i += RT_THREADS) sel[i / MAX_K][i % MAX_K] = i % MAX_K;

    // -- 1. rows -> LDS, four loads in flight per thread before their stores
    {
        const int c4 = d / 4, tot = nt * c4;
        for (int i0 = 0; i0 < tot; i0 += 4 * RT_THREADS) {
            float4 v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = min(i0 + u * RT_THREADS + tid, tot - 1);
                const int t = i / c4, c = i - t * c4;
                v[u] = *reinterpret_cast<const float4*>(a.x + (size_t)(t0 + t) * d + 4 * c);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = min(i0 + u * RT_THREADS + tid, tot - 1);  // clamped duplicates store the same values
                const int t = i / c4, c = i - t * c4;
                float* dst = xs + t * RS + 4 * (c & 3) * S + (c >> 2);  // elements 4c..4c+3: j = 4(c%4)+q, i = c/4
                dst[0] = v[u].x;
                dst[S] = v[u].y;
                dst[2 * S] = v[u].z;
                dst[3 * S] = v[u].w;
            }
        }
    }
    __syncthreads();

    if (split == 0) {  // block-uniform
        // -- 2. Q8_0 of x: one thread per 32-block (its max and integer sum are order-free)
        for (int i = tid; i < nt * KB; i += RT_THREADS) {
            const int t = i / KB, b = i - t * KB;
            const float* xr = xs + t * RS + 2 * b;  // element 32b + u at (u % 16) * S + 2b + u / 16
            float v[32];
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                const float2 p = *reinterpret_cast<const float2*>(xr + u * S);
                v[u] = p.x;
                v[16 + u] = p.y;
            }
            float amax = 0.0f;
#pragma unroll
            for (int u = 0; u < 32; ++u) amax = fmaxf(amax, __builtin_fabsf(v[u]));
            const float dd = amax / 127.0f;
            const float id = (dd != 0.0f) ? 1.0f / dd : 0.0f;
            int sum = 0;
            uint32_t w[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int u = 0; u < 32; ++u) {
                float r = round_away(v[u] * id);
                r = fminf(fmaxf(r, -127.0f), 127.0f);
                const int q = (int)r;
                sum += q;
                w[u >> 2] |= ((uint32_t)q & 0xFFu) << (8 * (u & 3));
            }
            const float2 sv = make_float2(f16_to_f32(f32_to_f16_trunc(dd)), (float)sum);
            const uint4 w0 = make_uint4(w[0], w[1], w[2], w[3]), w1 = make_uint4(w[4], w[5], w[6], w[7]);
            uint4* gq = reinterpret_cast<uint4*>(a.xq.q + (size_t)(t0 + t) * a.xq.K + 32 * b);
            gq[0] = w0;
            gq[1] = w1;
            a.xq.s[(size_t)(t0 + t) * KB + b] = sv;
            if (a.xh.q6)
                for (int part = 0; part < 2; ++part) {
                    const uint32_t w4[4] = {w[4 * part], w[4 * part + 1], w[4 * part + 2], w[4 * part + 3]};
                    write_q6_part(w4, sv, a.xh, (size_t)(t0 + t), b, part);
                }
            if (a.xh.xp) q8_pieces(sv, a.xh, (size_t)(t0 + t), b);
        }
    }

    if (rpb == 0) return;  // block-uniform
    // -- 3. router chains of this split's rows, exact vec_dot_f32 order
    {
        const int grp = tid >> 4, j = tid & 15;
        const int R = E + (a.shgate ? 1 : 0);
        const int r1 = min(R, (split + 1) * rpb);
        const int m = d / 16, m4 = m & ~3, Sg = chain_stride_of(d);
        for (int r = split * rpb + grp; r < r1; r += RT_GROUPS) {
            // F16 / BF16 router rows: vec_dot_{f16,bf16}_f32's order (src/quant.cpp:3015-3055), one chain
            // per lane jc < 8 over elements 8 i + jc, i.e. chain-major columns jc and jc + 8 interleaved
            // step by step (lanes 8-15 repeat lanes 0-7); the shared gate row stays fp32
            const bool c8 = a.chain8 && r < E;
            const int jc = c8 ? (j & 7) : j;
            const float* wr = a.router_cm + (size_t)r * 16 * Sg + jc * Sg;
            // token rows of the chains: tokens past nt (last block) repeat the last one, results dropped,
            // so the loop has no branches and the router loads can run ahead
            const float* xr[T];
#pragma unroll
            for (int t = 0; t < T; ++t) xr[t] = xs + min(t, nt - 1) * RS + jc * S;
            float acc[T];
#pragma unroll
            for (int t = 0; t < T; ++t) acc[t] = 0.0f;
            if (c8) {
                const float* wr8 = wr + 8 * Sg;
                for (int i = 0; i < m4; i += 4) {
                    const float4 w4 = *reinterpret_cast<const float4*>(wr + i);
                    const float4 w8 = *reinterpret_cast<const float4*>(wr8 + i);
#pragma unroll
                    for (int t = 0; t < T; ++t) {
                        const float4 x4 = *reinterpret_cast<const float4*>(xr[t] + i);
                        const float4 x8 = *reinterpret_cast<const float4*>(xr[t] + 8 * S + i);
                        acc[t] = __builtin_fmaf(w4.x, x4.x, acc[t]);
                        acc[t] = __builtin_fmaf(w8.x, x8.x, acc[t]);
                        acc[t] = __builtin_fmaf(w4.y, x4.y, acc[t]);
                        acc[t] = __builtin_fmaf(w8.y, x8.y, acc[t]);
                        acc[t] = __builtin_fmaf(w4.z, x4.z, acc[t]);
                        acc[t] = __builtin_fmaf(w8.z, x8.z, acc[t]);
                        acc[t] = __builtin_fmaf(w4.w, x4.w, acc[t]);
                        acc[t] = __builtin_fmaf(w8.w, x8.w, acc[t]);
                    }
                }
                for (int i = m4; i < m; ++i) {
#pragma unroll
                    for (int t = 0; t < T; ++t) {
                        acc[t] = __builtin_fmaf(wr[i], xr[t][i], acc[t]);
                        acc[t] = __builtin_fmaf(wr8[i], xr[t][8 * S + i], acc[t]);
                    }
                }
            } else {
#pragma unroll RT_UNROLL
                for (int i = 0; i < m4; i += 4) {
                    const float4 w4 = *reinterpret_cast<const float4*>(wr + i);
#pragma unroll
                    for (int t = 0; t < T; ++t) {
                        const float4 x4 = *reinterpret_cast<const float4*>(xr[t] + i);
                        acc[t] = __builtin_fmaf(w4.x, x4.x, acc[t]);
                        acc[t] = __builtin_fmaf(w4.y, x4.y, acc[t]);
                        acc[t] = __builtin_fmaf(w4.z, x4.z, acc[t]);
                        acc[t] = __builtin_fmaf(w4.w, x4.w, acc[t]);
                    }
                }
                for (int i = m4; i < m; ++i) {
                    const float wv = wr[i];
#pragma unroll
                    for (int t = 0; t < T; ++t) acc[t] = __builtin_fmaf(wv, xr[t][i], acc[t]);
                }
            }
#pragma unroll
            for (int t = 0; t < T; ++t) {
                if (t < nt) {
                    const float s = chain_sum(acc[t], c8);
                    if (j == 0) {
                        const size_t tok = (size_t)(t0 + t);
                        if (r < E) {
                            const float l = a.bias ? s + a.bias[r] : s;
                            if (nsplit == 1) lg[t * E + r] = l;
                            else a.logits[tok * E + r] = l;
                        } else if (nsplit == 1) {
                            shl[t] = s;
                        } else {
                            a.shscale[tok] = s;  // raw shared-gate logit; k_route_topk applies the sigmoid
                        }
                    }
                }
            }
        }
    }
    if (nsplit > 1) return;  // block-uniform
    __syncthreads();

    // -- 4. top-k by rank, softmax over the selected logits
    for (int i = tid; i < nt * E; i += RT_THREADS) {
        const int t = i / E, e = i - t * E;
        const float* lt = lg + t * E;
        const int rank = rank_of(lt, E, e);
        if (rank < a.k) sel[t][rank] = e;
        if (a.logits) a.logits[(size_t)(t0 + t) * E + e] = lt[e];
    }
    __syncthreads();
    static_assert(32 * T <= RT_THREADS, "one half-wave per token");
    if (tid < 32 * nt) {
        const int t = tid >> 5, i = tid & 31, k = a.k;
        const size_t o = (size_t)(t0 + t) * k;
        softmax_selected(lg + t * E, sel[t], k, i, a.ids + o, a.probs + o);
        if (i == 0 && a.shscale) a.shscale[t0 + t] = a.shgate ? 1.0f / (1.0f + expf(-shl[t])) : 1.0f;
    }
}

// Router logits for many tokens against a router of more than 16 rows, on the matrix cores: a step of a
// vec_dot_f32 chain (src/quant.cpp:2756-2778) for 64 tokens x 16 rows is one v_mfma_f32_16x16x1_4b_f32, an
// inner length of 1, so each result is one fused multiply-add rounded once: the chains' own arithmetic, in
// their order, at twice the vector unit's rate and from one operand register a side.  (Register-resident
// router rows against tokens from LDS, a 16-byte LDS read per four multiply-adds, were LDS-bound.)  A block
// owns 64 tokens and 16 rows, wave q the chains 4q .. 4q + 3 (a row's elements 16 i + 4q ..: one 16-byte LDS read
// of each operand per step).  Chunks of 4 steps come by DMA, three in flight (16-byte pieces XOR-swizzled by row
// against bank conflicts).
// Qwen3-shaped 2048 tokens (128 x 2048): 46 -> 24 us.
constexpr int RM_T = 64, RM_R = 16, RM_C = 64, RM_NB = 4;  // tokens, rows, floats per chunk, buffers

__global__ void __launch_bounds__(RT_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_route_mfma(RouteArgs a) {
    __shared__ __align__(16) float lds[RM_NB][RM_T + RM_R][RM_C];  // row r, piece c at piece c ^ (r % 16)
    const int tid = threadIdx.x, lane = tid & 63, q = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t0 = (int)blockIdx.y * RM_T, r0 = (int)blockIdx.x * RM_R;  // the row splits of a token block in a row
    const int d = a.d, E = a.E, R = E + (a.shgate ? 1 : 0), nc = d / RM_C;
    // a wave's DMAs of a chunk: tokens 16 q .. 16 q + 15 and rows 4 q .. 4 q + 3 (past the last: repeated, dropped below)
    const int l4 = lane >> 4, c16 = lane & 15;
    uint32_t xoff[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = 16 * q + 4 * u + l4;
        xoff[u] = (uint32_t)(min(t0 + r, a.n - 1) - t0) * (uint32_t)(d * 4) + (uint32_t)((c16 ^ (r & 15)) << 4);
    }
    const int rw = 4 * q + l4, rr = min(r0 + rw, R - 1);
    const uint8_t* wsrc = reinterpret_cast<const uint8_t*>(rr < E ? a.router + (size_t)rr * d : a.shgate) + ((c16 ^ rw) << 4);
    const uint8_t* xsrc = uniform_ptr(a.x + (size_t)t0 * d);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr)&lds[0][0][0];
    auto stage = [&](int c) {  // 5 DMAs, also past the last chunk (a buffer nothing reads any more)
        const uint32_t b = lds0 + (uint32_t)(c % RM_NB) * (uint32_t)sizeof(lds[0]);
        const size_t o = (size_t)min(c, nc - 1) * (RM_C * 4);
        gbyte* base = dma_base(xsrc + o);
#pragma unroll
        for (int u = 0; u < 4; ++u) dma16g(base, xoff[u], b + (16 * q + 4 * u) * (RM_C * 4));
        dma16v(wsrc + o, b + (RM_T + 4 * q) * (RM_C * 4));
    };
    v16f acc[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) acc[k] = v16f{};
    for (int c = 0; c < RM_NB - 1; ++c) stage(c);
    for (int c = 0; c < nc; ++c) {
        // chunk c is in (two younger ones are not), and every wave has read chunk c - 1
        asm volatile("s_waitcnt vmcnt(10) lgkmcnt(0)" ::: "memory");
        static_assert(RM_NB == 4, "two chunks of 5 DMAs younger than the one waited for");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        stage(c + RM_NB - 1);
        const float(*buf)[RM_C] = lds[c % RM_NB];
#pragma unroll
        for (int i = 0; i < RM_C / 16; ++i) {
            const int at = ((4 * i + q) ^ c16) * 4;  // both rows are lane % 16 modulo 16
            const float4 x4 = *reinterpret_cast<const float4*>(&buf[lane][at]);
            const float4 w4 = *reinterpret_cast<const float4*>(&buf[RM_T + c16][at]);
            acc[0] = __builtin_amdgcn_mfma_f32_16x16x1f32(x4.x, w4.x, acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_16x16x1f32(x4.y, w4.y, acc[1], 0, 0, 0);
            acc[2] = __builtin_amdgcn_mfma_f32_16x16x1f32(x4.z, w4.z, acc[2], 0, 0, 0);
            acc[3] = __builtin_amdgcn_mfma_f32_16x16x1f32(x4.w, w4.w, acc[3], 0, 0, 0);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the buffers are reused: no DMA may still land
    // acc0[j] + acc1[j] (chains j and j + 8: waves 0 and 2, 1 and 3), then their sum from j = 0 on
    __syncthreads();
    float* red = &lds[0][0][0];  // [2 waves][4 chains][16][64]
    static_assert(2 * 4 * 16 * 64 <= RM_NB * (RM_T + RM_R) * RM_C, "the chains' sums fit the staging buffers");
    if (q >= 2)
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int v = 0; v < 16; ++v) red[(((q - 2) * 4 + k) * 16 + v) * 64 + lane] = acc[k][v];
    __syncthreads();
    float sum[16];
    if (q < 2) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[k][v] += red[((q * 4 + k) * 16 + v) * 64 + lane];
            sum[v] = 0.0f;
            if (q == 0)
#pragma unroll
                for (int k = 0; k < 4; ++k) sum[v] += acc[k][v];
        }
    }
    __syncthreads();
    if (q == 0)
#pragma unroll
        for (int v = 0; v < 16; ++v) red[v * 64 + lane] = sum[v];
    __syncthreads();
    if (q != 1) return;
    const int r = r0 + (lane & 15);
    if (r >= R) return;
    const float bias = r < E && a.bias ? a.bias[r] : 0.0f;
#pragma unroll
    for (int v = 0; v < 16; ++v) {  // result of tokens 16 (v / 4) + 4 (lane / 16) + v % 4, row lane % 16
        float s = red[v * 64 + lane];
#pragma unroll
        for (int k = 0; k < 4; ++k) s += acc[k][v];
        const int tok = t0 + 16 * (v >> 2) + 4 * (lane >> 4) + (v & 3);
        if (tok >= a.n) continue;
        if (r < E) a.logits[(size_t)tok * E + r] = a.bias ? s + bias : s;
        else a.shscale[tok] = s;  // raw shared-gate logit; k_route_topk applies the sigmoid
    }
}

// Top-k and softmax once every split has written its logits (raw shared-gate
// logits in shscale): one wave per token, four tokens per block.
template <int NC>
__global__ void __launch_bounds__(256) k_route_topk(RouteArgs a) {
    const size_t t = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= (size_t)a.n) return;  // wave-uniform
    uint64_t msk[NC];
    (void)topk_token_wave<NC>(a, a.logits + t * a.E, t, a.shgate ? a.shscale : nullptr, msk);
}

static void launch_route_topk(const RouteArgs& a, hipStream_t st) {
    const dim3 grid((a.n + 3) / 4);
    const int nc = (a.E + 63) / 64;
    if (nc <= 1) hipLaunchKernelGGL(k_route_topk<1>, grid, dim3(256), 0, st, a);
    else if (nc <= 2) hipLaunchKernelGGL(k_route_topk<2>, grid, dim3(256), 0, st, a);
    else if (nc <= 4) hipLaunchKernelGGL(k_route_topk<4>, grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL(k_route_topk<MAX_E / 64>, grid, dim3(256), 0, st, a);
}

// The matrix-core router: more than 16 rows (fewer leave most of a result's 16 columns empty) in the fp32 chain
// order (F16 / BF16 rows have another), whole chunks, and from 512 tokens on (below, the split
// k_route, one token per block, fills more CUs).  x comes by 16-byte DMA, so a caller's x off that alignment stays with
// k_route's ordinary loads.
static bool route_mfma_fits(const RouteArgs& a) {
    return reinterpret_cast<uintptr_t>(a.x) % 16 == 0 && a.E + (a.shgate ? 1 : 0) > RT_GROUPS && a.d % RM_C == 0 && a.n >= 512 && a.n <= 65535 * RM_T && !a.chain8;
}

void launch_route(const RouteArgs& a, hipStream_t st) {
    if (route_mfma_fits(a)) {
        // quantized / matrix-core forms of x, then the logits, then top-k
        const int T = route_lds(4, a.d, a.E) <= RT_LDS_TARGET ? 4 : route_lds(2, a.d, a.E) <= RT_LDS_TARGET ? 2 : 1;
        const size_t lq = route_lds(T, a.d, a.E);
        auto forms = T == 4 ? k_route<4> : T == 2 ? k_route<2> : k_route<1>;
        if (lq > 65536)
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(forms), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lq);
        hipLaunchKernelGGL(forms, dim3((a.n + T - 1) / T), dim3(RT_THREADS), lq, st, a, 1, 0);
        const int R = a.E + (a.shgate ? 1 : 0), RS = (R + RM_R - 1) / RM_R;
        hipLaunchKernelGGL(k_route_mfma, dim3(RS, (a.n + RM_T - 1) / RM_T), dim3(RT_THREADS), 0, st, a);
        launch_route_topk(a, st);
        return;
    }
    RouteShape r = route_shape(a);
    r.T = r.T >= 4 ? 4 : r.T >= 2 ? 2 : 1;  // instantiated token counts
    const size_t lds = route_lds(r.T, a.d, a.E);
    const int tb = (a.n + r.T - 1) / r.T;
    auto go = [&](auto kern) {
        if (lds > 65536)
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int)lds);
        hipLaunchKernelGGL(kern, dim3(tb * r.RS), dim3(RT_THREADS), lds, st, a, r.RS, r.RPB);
    };
    switch (r.T) {
        case 4: go(k_route<4>); break;
        case 2: go(k_route<2>); break;
        default: go(k_route<1>); break;
    }
    if (r.RS > 1) launch_route_topk(a, st);
}

// The routing into the caller's device buffers (each may be null), in one launch: three device-to-device copies
// of a few KB cost a launch and its hand-over each.  Qwen3-shaped 37 tokens, residual form, routing kept: per
// step 119.0 -> 115.3 us.
__global__ void __launch_bounds__(256) k_copy_routing(const int* ids, const float* w, const int* counts, int* ids_out,
                                                      float* w_out, int* counts_out, int nk, int E) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < nk) {
        if (ids_out) ids_out[i] = ids[i];
        if (w_out) w_out[i] = w[i];
    }
    if (counts_out && i < E) counts_out[i] = counts[i];
}

void launch_copy_routing(const int* ids, const float* w, const int* counts, int* ids_out, float* w_out, int* counts_out,
                         int nk, int E, hipStream_t st) {
    hipLaunchKernelGGL(k_copy_routing, dim3((std::max(nk, E) + 255) / 256), dim3(256), 0, st, ids, w, counts, ids_out, w_out,
                       counts_out, nk, E);
}

// Matrix-core form of Q8_0 activations already in global memory, one wave per row.
__global__ void __launch_bounds__(256) k_q8_to_acth(ActQ8 in, int rows, ActH out) {
    const size_t row = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= (size_t)rows) return;  // wave-uniform
    write_acth_row(in.q + row * in.K, in.s + row * (in.K / 32), in.K, out, row, threadIdx.x & 63);
}

__device__ __forceinline__ uint32_t comp4(const uint4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// The same, one wave per row:
// every quant and scale load of the row is in flight before the first conversion (16 quants per lane
// and chunk, NC chunks per lane), and the row exponent comes from the scales already loaded.  The
// values are those of acth_chunk_v: fp16(dx * 2^-E * q), 2^E per half-unit, the min-term pieces of
// dx * sum(q) * 2^-E.
template <int NC>
__global__ void __launch_bounds__(256) k_q8_to_acth_hi(ActQ8 in, int rows, ActH o) {
    const size_t row = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= (size_t)rows) return;  // wave-uniform
    const int lane = threadIdx.x & 63, K = in.K, n16 = K / 16, KH = K / 128;
    const int8_t* q = in.q + row * K;
    const float2* sc = in.s + row * (K / 32);
    uint4 qv[NC];
    float2 sv[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int i = min(lane + 64 * c, n16 - 1);  // clamped duplicates are loaded, not stored
        qv[c] = ld16(q + 16 * i);
        sv[c] = sc[i >> 1];
    }
    float M = 0.0f;  // chunks 2b and 2b + 1 carry block b's scale, so this covers every block
#pragma unroll
    for (int c = 0; c < NC; ++c) M = fmaxf(M, sv[c].x);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) M = fmaxf(M, __shfl_xor(M, off, 64));
    const int E = acth_exponent(M);
    const float dn = __uint_as_float((uint32_t)(127 - E) << 23), up = __uint_as_float((uint32_t)(127 + E) << 23);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int i = lane + 64 * c;
        if (i >= n16) break;
        const int e = 16 * i, b = e >> 5, hh = e >> 7;
        const float s = sv[c].x * dn;  // exact: power-of-two scaling
        uint32_t hw[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const uint32_t word = comp4(qv[c], u >> 1);
            const int q0 = (int)(int8_t)(word >> (16 * (u & 1))), q1 = (int)(int8_t)(word >> (16 * (u & 1) + 8));
            const _Float16 h0 = (_Float16)(s * (float)q0), h1 = (_Float16)(s * (float)q1);  // products exact
            hw[u] = (uint32_t)__builtin_bit_cast(uint16_t, h0) | ((uint32_t)__builtin_bit_cast(uint16_t, h1) << 16);
        }
        uint4* hl = reinterpret_cast<uint4*>(o.hl + row * (size_t)K + e);
        hl[0] = make_uint4(hw[0], hw[1], hw[2], hw[3]);
        hl[1] = make_uint4(hw[4], hw[5], hw[6], hw[7]);
        if ((e & 127) == 0) o.pe[row * (size_t)KH + hh] = up;
        if ((e & 31) == 0)  // exact: 11-bit scale x |sum| < 2^12, times 2^-E
            store_pieces3(o.xm + row * (size_t)o.KU * 24 + (b / 8) * 24 + (b % 8), sv[c].x * sv[c].y * dn);
    }
}

void launch_q8_to_acth(const ActQ8& in, int rows, ActH out, hipStream_t st) {
    const int nc = (in.K / 16 + 63) / 64;
    if (in.K % 128 == 0 && nc <= 16) {
        const dim3 grid((rows + 3) / 4);
        if (nc <= 1) hipLaunchKernelGGL(k_q8_to_acth_hi<1>, grid, dim3(256), 0, st, in, rows, out);
        else if (nc <= 2) hipLaunchKernelGGL(k_q8_to_acth_hi<2>, grid, dim3(256), 0, st, in, rows, out);
        else if (nc <= 4) hipLaunchKernelGGL(k_q8_to_acth_hi<4>, grid, dim3(256), 0, st, in, rows, out);
        else if (nc <= 8) hipLaunchKernelGGL(k_q8_to_acth_hi<8>, grid, dim3(256), 0, st, in, rows, out);
        else hipLaunchKernelGGL(k_q8_to_acth_hi<16>, grid, dim3(256), 0, st, in, rows, out);
        return;
    }
    hipLaunchKernelGGL(k_q8_to_acth, dim3((rows + 3) / 4), dim3(256), 0, st, in, rows, out);
}

// The block GEMM's forms of Q8_0 rows already in global memory, one thread per half 32-block.
__global__ void __launch_bounds__(256) k_q8_to_block(ActQ8 in, int rows, ActH out) {
    const int KP = in.K / 16;
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x, row = i / KP;
    if (row >= (size_t)rows) return;
    const float2 sv = in.s[i / 2];
    const int b = (int)(i - row * KP) / 2, part = (int)(i & 1);
    if (out.q6) {
        const uint4 a = ld16(in.q + i * 16);
        const uint32_t w[4] = {a.x, a.y, a.z, a.w};
        write_q6_part(w, sv, out, row, b, part);
    }
    if (out.xp && part == 0) q8_pieces(sv, out, row, b);
}

void launch_q8_to_block(const ActQ8& in, int rows, const ActH& out, hipStream_t st) {
    const size_t n = (size_t)rows * (in.K / 16);
    hipLaunchKernelGGL(k_q8_to_block, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, in, rows, out);
}

// Matrix-core form (fp16 hi only) of fp32 activation rows h [rows][ld], out.K
// a multiple of 128 (K-quants: 256, zero padding past the real columns) -- the
// reference's fp32-activation products (vec_dot_quant_f32, src/quant.cpp:3269-3305)
// for a down projection without a Q8_0 form (Q5_0, or a K-quant whose K is not
// a multiple of 256).  One block per
// row: E = exponent(max |h|) - 14 so every h * 2^-E is below 2^15; hi =
// fp16(h * 2^-E) (relative error <= 2^-12 per value, as the Q8_0 down operand);
// the min-term value of each 32-block is its fp32 sum times 2^-E, split into
// three exact bf16 pieces.
__global__ void __launch_bounds__(256) k_f32_to_acth(const float* h, int ld, ActH o) {
    __shared__ float wmax[4];
    const size_t row = blockIdx.x;
    const int tid = threadIdx.x, K = o.K, KH = K / 128;
    const float* hr = h + row * (size_t)ld;
    float M = 0.0f;
    for (int i = tid; i < K / 4; i += 256) {
        const float4 v = *reinterpret_cast<const float4*>(hr + 4 * i);
        M = fmaxf(M, fmaxf(fmaxf(__builtin_fabsf(v.x), __builtin_fabsf(v.y)), fmaxf(__builtin_fabsf(v.z), __builtin_fabsf(v.w))));
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) M = fmaxf(M, __shfl_xor(M, off, 64));
    if ((tid & 63) == 0) wmax[tid >> 6] = M;
    __syncthreads();
    M = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    const int E = (M > 0.0f) ? (int)((__float_as_uint(M) >> 23) & 0xFF) - 127 - 14 : 0;
    const float dn = __uint_as_float((uint32_t)(127 - E) << 23), up = __uint_as_float((uint32_t)(127 + E) << 23);
    // eight consecutive values per thread; the four threads of a 32-block are consecutive lanes
    for (int c = tid; c < K / 8; c += 256) {
        const int i = 8 * c, b = i >> 5, hh = i >> 7;
        const float4 v0 = *reinterpret_cast<const float4*>(hr + i), v1 = *reinterpret_cast<const float4*>(hr + i + 4);
        const float f[8] = {v0.x * dn, v0.y * dn, v0.z * dn, v0.w * dn, v1.x * dn, v1.y * dn, v1.z * dn, v1.w * dn};
        uint32_t hw[4];
        float sum = 0.0f;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const _Float16 h0 = (_Float16)f[2 * u], h1 = (_Float16)f[2 * u + 1];
            hw[u] = (uint32_t)__builtin_bit_cast(uint16_t, h0) | ((uint32_t)__builtin_bit_cast(uint16_t, h1) << 16);
            sum += f[2 * u] + f[2 * u + 1];
        }
        *reinterpret_cast<uint4*>(o.hl + row * (size_t)K + i) = make_uint4(hw[0], hw[1], hw[2], hw[3]);
        if ((i & 127) == 0) o.pe[row * (size_t)KH + hh] = up;
        sum += __shfl_xor(sum, 1, 64);
        sum += __shfl_xor(sum, 2, 64);
        if ((i & 31) == 0) {
            const uint32_t bh = __float_as_uint(sum) & 0xFFFF0000u;
            const float r1 = sum - __uint_as_float(bh);
            const uint32_t bm = __float_as_uint(r1) & 0xFFFF0000u;
            const float r2 = r1 - __uint_as_float(bm);
            uint16_t* xm = o.xm + row * (size_t)o.KU * 24 + (b / 8) * 24 + (b % 8);
            xm[0] = (uint16_t)(bh >> 16);
            xm[8] = (uint16_t)(bm >> 16);
            xm[16] = (uint16_t)(__float_as_uint(r2) >> 16);
        }
    }
}

void launch_f32_to_acth(const float* h, int ld, int rows, ActH out, hipStream_t st) {
    hipLaunchKernelGGL(k_f32_to_acth, dim3(rows), dim3(256), 0, st, h, ld, out);
}

// ---------------------------------------------------------------- few tokens
// Decode routing: a one-block-per-token kernel would serialise every router
// row behind one CU's load latency.  Here block r owns router row r (expert r,
// or the shared-expert gate vector as row E): it stages that row and the n
// tokens in LDS with all loads in flight, then 16 lanes per token run the
// vec_dot_f32 chains from LDS.  Blocks also split the Q8_0 quantization of x.
// A second one-block launch ranks, normalises and dispatches: with
// n*k <= 2*32 pairs the counting sort is a short serial loop.
constexpr int RS_THREADS = 256;
constexpr int RS_LDS_BYTES = 64 * 1024;

static size_t rs_lds(int n, int d) { return (size_t)(1 + n) * 16 * rs_stride(d) * sizeof(float); }

bool route_small_fits(int n, int d, int E) {
    return n >= 1 && n <= ROUTE_SMALL_MAX_N && E <= MAX_E && d % 32 == 0 && rs_lds(n, d) <= RS_LDS_BYTES;
}

__global__ void __launch_bounds__(RS_THREADS)
k_route_small(RouteArgs a) {
    extern __shared__ float lds[];  // (1 + n) chain-major rows: router row r, then the n tokens
    const int r = blockIdx.x, tid = threadIdx.x;
    if (r == 0)  // the folded combine's output starts at zero (CombineOut)
        for (int i = tid; i < a.zero_count; i += RS_THREADS) a.zero_out[i] = 0.0f;
    const int d = a.d, n = a.n, E = a.E, S = rs_stride(d), RS = 16 * S;
    const float* w = r < E ? a.router + (size_t)r * d : a.shgate;
    {  // router row + token rows -> LDS: every load in flight before the first store
        constexpr int PER = (ROUTE_SMALL_MAX_N + 1) * 8192 / 4 / RS_THREADS;  // float4 slots: d <= 8192
        const int c4 = d / 4, tot = (1 + n) * c4;
        float4 v[PER];
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int i = tid + q * RS_THREADS;
            if (i >= tot) break;
            const int row = i / c4, c = i - row * c4;
            const float* src = row == 0 ? w + 4 * c : a.x + (size_t)(row - 1) * d + 4 * c;
            v[q] = *reinterpret_cast<const float4*>(src);
        }
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int i = tid + q * RS_THREADS;
            if (i >= tot) break;
            const int row = i / c4, c = i - row * c4;
            float* dst = lds + row * RS + 4 * (c & 3) * S + (c >> 2);  // elements 4c..4c+3: j = 4(c%4)+q, i = c/4
            dst[0] = v[q].x;
            dst[S] = v[q].y;
            dst[2 * S] = v[q].z;
            dst[3 * S] = v[q].w;
        }
    }
    __syncthreads();
    const int wave = tid >> 6, lane = tid & 63;
    if (wave == 0) {
        // router row r for every token: vec_dot_f32 order (src/quant.cpp:2756-2778): lane j of
        // token group t runs the FMA chain over elements 16 i + j (lanes 0-7 the reference's acc0,
        // 8-15 its acc1), then acc0 + acc1 and the sequential sum of the 8 lanes (d % 16 == 0: no
        // tails)
        const int t = lane >> 4, j = lane & 15;
        if (t < n) {
            // F16 / BF16 router rows: columns jc and jc + 8 interleaved (as k_route); the shared gate fp32
            const bool c8 = a.chain8 && r < E;
            const float s = chain_sum(chain_dot_lds(lds, lds + (1 + t) * RS, S, d, j, c8), c8);
            if (j == 0) {
                if (r < E) a.logits[(size_t)t * E + r] = a.bias ? s + a.bias[r] : s;
                else a.shscale[t] = s;  // raw shared-gate logit; the top-k step applies the sigmoid
            }
        }
    } else {
        // this block's share of the Q8_0 blocks of x, one per half-wave of waves 1..
        const int nb = d / 32, tot = n * nb;
        const int per = (tot + gridDim.x - 1) / gridDim.x;
        const int b0 = r * per, b1 = min(tot, b0 + per);
        const int half = lane >> 5, l32 = lane & 31;
        constexpr int QW = RS_THREADS / 64 - 1;
        for (int bb = b0 + (wave - 1) * 2; bb < b1; bb += QW * 2) {
            const int b = bb + half;  // token-major: b = t*nb + block
            const bool ok = b < b1;
            const int t = ok ? b / nb : 0, q = ok ? (b % nb) * 32 + l32 : 0;
            const float xv = lds[(1 + t) * RS + (q & 15) * S + (q >> 4)];
            quant_block(xv, l32, ok, a.xq, (size_t)t, ok ? b % nb : 0);
        }
    }
}

// Second launch of the few-token router: top-k and dispatch tables from the
// logits of k_route_small (raw shared-gate logits in shscale), one wave.
template <int NC>
__global__ void __launch_bounds__(64) k_topk_small(RouteArgs a, DispatchOut o) {
    topk_dispatch_wave<NC>(a, o, a.logits, a.shgate ? a.shscale : nullptr);
}

// The whole few-token routing in one block when the router fits in LDS
// (Mixtral-sized routers: 8 x 4096 fp32 = 128 KB): stage router + tokens with
// every load in flight, Q8_0 of x, the vec_dot_f32 chains (16 lanes each, as
// in k_route), then top-k, softmax and dispatch.  One launch instead of two,
// one HBM round trip.
constexpr int R1_THREADS = 1024;
constexpr int R1_PER = 10;  // float4 staging slots per thread
constexpr size_t R1_LDS_BYTES = (size_t)R1_THREADS * R1_PER * 16;

static size_t route_one_lds(int n, int d, int E, bool shgate) {
    return ((size_t)(E + (shgate ? 1 : 0) + n) * d + (size_t)std::max(n, 2) * E) * sizeof(float);
}

bool route_one_fits(int n, int d, int E, bool shgate) {
    return n >= 1 && n <= ROUTE_SMALL_MAX_N && E <= 64 && d % 16 == 0 &&
           (size_t)(E + (shgate ? 1 : 0) + n) * d * sizeof(float) <= R1_LDS_BYTES &&
           route_one_lds(n, d, E, shgate) <= 160 * 1024;
}

__global__ void __launch_bounds__(R1_THREADS) k_route_one(RouteArgs a, DispatchOut o) {
    extern __shared__ float lds[];  // [rows][d] router (+ shared gate), [n][d] tokens, [n][E] logits
    __shared__ float shl[ROUTE_SMALL_MAX_N];
    const int tid = threadIdx.x;
    const int d = a.d, n = a.n, E = a.E, rows = E + (a.shgate ? 1 : 0);
    for (int i = tid; i < a.zero_count; i += R1_THREADS) a.zero_out[i] = 0.0f;  // folded combine (CombineOut)
    float* xs = lds + (size_t)rows * d;
    float* lgs = xs + (size_t)n * d;
    {
        const int c4 = d / 4, tot = (rows + n) * c4;  // route_one_fits: tot <= R1_THREADS * R1_PER
        float4 v[R1_PER];
#pragma unroll
        for (int q = 0; q < R1_PER; ++q) {
            const int i = min(tid + q * R1_THREADS, tot - 1);
            const int row = i / c4, c = i - row * c4;
            const float* src = row < E ? a.router + (size_t)row * d : (row < rows ? a.shgate : a.x + (size_t)(row - rows) * d);
            v[q] = *reinterpret_cast<const float4*>(src + 4 * c);
        }
#pragma unroll
        for (int q = 0; q < R1_PER; ++q) {
            const int i = min(tid + q * R1_THREADS, tot - 1);
            *reinterpret_cast<float4*>(lds + 4 * i) = v[q];
        }
    }
    __syncthreads();
    // the first CW waves run the (token, router row) chains, the others quantize x
    const int chains = n * rows, CW = min(R1_THREADS / 64 - 1, (chains + 3) / 4);
    if ((tid >> 6) >= CW) {  // Q8_0 of x, one 32-block per half-wave
        const int nb = d / 32, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
        for (int b = ((tid >> 6) - CW) * 2 + half; b < n * nb; b += (R1_THREADS / 64 - CW) * 2)
            quant_block(xs[(size_t)b * 32 + l32], l32, true, a.xq, (size_t)(b / nb), b % nb);
    }
    // chains, 16 lanes each, vec_dot_f32 order (d % 16 == 0: no tails)
    for (int c = tid >> 4; c < chains && (tid >> 6) < CW; c += CW * 4) {
        const int t = c / rows, r = c % rows, j = tid & 15;
        const float* w = lds + (size_t)r * d;
        const float* xt = xs + (size_t)t * d;
        // F16 / BF16 router rows: 8 chains over 8-element steps (lanes 8-15 repeat lanes 0-7)
        const bool c8 = a.chain8 && r < E;
        float acc = 0.0f;
        if (c8) {
            const int jc = j & 7;
#pragma unroll 32
            for (int i = 0; i < d; i += 8) acc = __builtin_fmaf(w[i + jc], xt[i + jc], acc);
        } else {
#pragma unroll 32
            for (int i = 0; i < d; i += 16) acc = __builtin_fmaf(w[i + j], xt[i + j], acc);
        }
        const float s = chain_sum(acc, c8);
        if (j == 0) {
            if (r < E) {
                const float l = a.bias ? s + a.bias[r] : s;
                lgs[t * E + r] = l;
                a.logits[(size_t)t * E + r] = l;
            } else {
                shl[t] = s;
            }
        }
    }
    __syncthreads();
    if (tid < 64) topk_dispatch_wave<1>(a, o, lgs, a.shgate ? shl : nullptr);
}

void launch_route_logits(const RouteArgs& a, hipStream_t st) {
    const int rows = a.E + (a.shgate ? 1 : 0);
    hipLaunchKernelGGL(k_route_small, dim3(rows), dim3(RS_THREADS), rs_lds(a.n, a.d), st, a);
}

void launch_route_small(const RouteArgs& a, const DispatchOut& o, hipStream_t st) {
    const int rows = a.E + (a.shgate ? 1 : 0);
    if (route_one_fits(a.n, a.d, a.E, a.shgate != nullptr)) {
        const size_t lds = route_one_lds(a.n, a.d, a.E, a.shgate != nullptr);
        // dynamic LDS above 64 KB needs the kernel's opt-in; without it, the two-launch path
        const bool ok = lds <= 65536 || hipFuncSetAttribute(reinterpret_cast<const void*>(k_route_one),
                                                            hipFuncAttributeMaxDynamicSharedMemorySize,
                                                            (int)lds) == hipSuccess;
        if (ok) {
            hipLaunchKernelGGL(k_route_one, dim3(1), dim3(R1_THREADS), lds, st, a, o);
            return;
        }
        (void)hipGetLastError();  // clear the refused opt-in
    }
    hipLaunchKernelGGL(k_route_small, dim3(rows), dim3(RS_THREADS), rs_lds(a.n, a.d), st, a);
    const int nc = (a.E + 63) / 64;
    if (nc <= 1) hipLaunchKernelGGL(k_topk_small<1>, dim3(1), dim3(64), 0, st, a, o);
    else if (nc <= 2) hipLaunchKernelGGL(k_topk_small<2>, dim3(1), dim3(64), 0, st, a, o);
    else if (nc <= 4) hipLaunchKernelGGL(k_topk_small<4>, dim3(1), dim3(64), 0, st, a, o);
    else hipLaunchKernelGGL(k_topk_small<MAX_E / 64>, dim3(1), dim3(64), 0, st, a, o);
}

// One block per expert.  Every block builds the full per-expert histogram in
// LDS (no global atomics, nothing to clear between calls), derives its pair
// offset, MFMA tile offset and active-list slot, then writes the positions of
// its (token, slot) pairs in flat order -- a stable counting sort, so tokens
// keep their order inside each expert.
//  - ids: rounds of 4 x U x 256 ids, each wave a contiguous quarter; a lane's U 16-byte loads of a round are all
//    in flight at once (loaded one by one, their latencies were most of the kernel: 16384 ids over 128 experts
//    20 -> 15 us), and a batch of one round keeps them in registers for both passes;
//  - histogram: up to 16 experts by packed per-thread counters (LDS atomics on so few bins would serialize), else
//    LDS atomics;
//  - positions: the matches as a 64-bit mask per lane (4 ids x U loads),
//    one barrier exchanges the wave totals, and the writes follow the masks
//    in flat order (lane prefixes from three ballots of the per-lane count).
constexpr int DISPATCH_THREADS = 256;
constexpr int DP_U = 16;  // 16-byte id loads per lane per round, at most

template <int U>
__global__ void __launch_bounds__(DISPATCH_THREADS)
k_dispatch(const int* ids, int nk, int E, int top_k, DispatchOut o) {
    extern __shared__ int hist[];
    __shared__ int red[3][DISPATCH_THREADS / 64];
    __shared__ int wtot[2][DISPATCH_THREADS / 64];
    const int e = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    constexpr int NW = DISPATCH_THREADS / 64, ROUND = NW * 256 * U;
    for (int i = tid; i < E; i += DISPATCH_THREADS) hist[i] = 0;
    // a round's ids, -1 past the last: group f (4 ids) by one load where it is whole, the last partial one from `tail`
    const int whole = nk & ~3;
    int4 v[U];
    const int4 tail = make_int4(whole < nk ? ids[whole] : -1, whole + 1 < nk ? ids[whole + 1] : -1,
                                whole + 2 < nk ? ids[whole + 2] : -1, -1);
    auto load = [&](int r0) {
        const int f0 = r0 + wave * 256 * U + 4 * lane;
        if (whole > 0)  // block-uniform
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = *reinterpret_cast<const int4*>(ids + min(f0 + 256 * u, whole - 4));
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int f = f0 + 256 * u;
            if (f >= whole) v[u] = f == whole ? tail : make_int4(-1, -1, -1, -1);
        }
    };
    __syncthreads();
    if (E <= 16) {
        // per-thread 8-bit counters (experts 0-7 in lo, 8-15 in hi), flushed before any can reach 256
        uint64_t lo = 0, hi = 0;
        int since = 0;
        auto flush = [&]() {
            for (int x = 0; x < E; ++x) {  // wave-uniform
                int c = (int)(((x < 8 ? lo : hi) >> (8 * (x & 7))) & 255u);
#pragma unroll
                for (int m = 32; m >= 1; m >>= 1) c += __shfl_xor(c, m, 64);
                if (lane == 0) atomicAdd(&hist[x], c);
            }
            lo = hi = 0;
        };
        auto count = [&](int id) {
            const uint64_t one = 1ull << (8 * (id & 7));
            lo += id >= 0 && id < 8 ? one : 0ull;
            hi += id >= 8 ? one : 0ull;
        };
        for (int r0 = 0; r0 < nk; r0 += ROUND) {
            load(r0);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                count(v[u].x);
                count(v[u].y);
                count(v[u].z);
                count(v[u].w);
            }
            since += U;
            if (since + U > 63) {  // 63 * 4 = 252 per counter at most
                flush();
                since = 0;
            }
        }
        flush();
    } else {
        auto count = [&](int id) {
            if (id >= 0) atomicAdd(&hist[id], 1);
        };
        for (int r0 = 0; r0 < nk; r0 += ROUND) {
            load(r0);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                count(v[u].x);
                count(v[u].y);
                count(v[u].z);
                count(v[u].w);
            }
        }
    }
    __syncthreads();
    // pair offset, tile offset and active index of expert e: sums over the experts before it
    int off = 0, toff = 0, na = 0;
    for (int i = tid; i < e; i += DISPATCH_THREADS) {
        const int c = hist[i];
        off += c;
        toff += (c + MFMA_BN - 1) / MFMA_BN;
        na += c > 0;
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
        off += __shfl_xor(off, m, 64);
        toff += __shfl_xor(toff, m, 64);
        na += __shfl_xor(na, m, 64);
    }
    if (lane == 0) {
        red[0][wave] = off;
        red[1][wave] = toff;
        red[2][wave] = na;
    }
    __syncthreads();
    off = toff = na = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        off += red[0][w];
        toff += red[1][w];
        na += red[2][w];
    }
    const int cnt = hist[e];
    const int ntl = (cnt + MFMA_BN - 1) / MFMA_BN;  // this expert's tiles
    if (tid == 0) {
        o.counts[e] = cnt;
        o.offs[e] = off;
        if (cnt > 0) o.act[na] = e;
        else o.slots[E - 1 - (e - na)] = make_int4(0, 0, 0, 0);  // inactive experts fill slots n_act..E-1
        if (e == E - 1) {
            o.offs[E] = off + cnt;
            *o.n_act = na + (cnt > 0);
            *o.n_tiles = toff + ntl;
        }
    }
    for (int i = tid; i < ntl; i += DISPATCH_THREADS)
        o.tiles[toff + i] = make_int4(e, off + i * MFMA_BN, min(MFMA_BN, cnt - i * MFMA_BN), 0);
    if (cnt == 0) return;  // block-uniform
    const uint64_t lt_mask = (1ull << lane) - 1ull;
    int run = off;
    for (int r0 = 0, par = 0; r0 < nk; r0 += ROUND, par ^= 1) {
        const int wbase = r0 + wave * 256 * U;
        if (nk > ROUND) load(r0);  // (a single round's ids are still here)
        uint64_t bits = 0;  // bit 4u + c: id wbase + 256u + 4 lane + c is expert e
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t m = (v[u].x == e) | (v[u].y == e) << 1 | (v[u].z == e) << 2 | (v[u].w == e) << 3;
            bits |= (uint64_t)m << (4 * u);
        }
        int wt = __popcll(bits);
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) wt += __shfl_xor(wt, m, 64);
        if (lane == 0) wtot[par][wave] = wt;
        __syncthreads();  // wtot[par] complete; the previous round's readers of wtot[par ^ 1] are done
        int p = run, total = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            p += w < wave ? wtot[par][w] : 0;
            total += wtot[par][w];
        }
        for (int u = 0; u < U; ++u) {
            const uint32_t m = (uint32_t)(bits >> (4 * u)) & 15u;
            if (__ballot(m != 0) == 0) continue;  // wave-uniform
            const int c = __popc(m);
            const uint64_t b0 = __ballot(c & 1), b1 = __ballot(c & 2), b2 = __ballot(c & 4);
            int q = p + __popcll(b0 & lt_mask) + 2 * __popcll(b1 & lt_mask) + 4 * __popcll(b2 & lt_mask);
            const int f0 = wbase + 256 * u + 4 * lane;
            for (int x = 0; x < 4; ++x) {
                if ((m >> x) & 1u) {
                    const int f = f0 + x;
                    o.pair_tok[q] = f / top_k;
                    o.pos_of[f] = q;
                    if (q == off) o.slots[na] = make_int4(e, off, cnt, f / top_k);
                    ++q;
                }
            }
            p += __popcll(b0) + 2 * __popcll(b1) + 4 * __popcll(b2);
        }
        run += total;
    }
}

void launch_dispatch(const int* ids, int nk, int E, int top_k, const DispatchOut& o, hipStream_t st) {
    // loads per lane and round: the fewest (1, 4 or 16) that take the pairs in one
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(E), dim3(DISPATCH_THREADS), (size_t)E * sizeof(int), st, ids, nk, E, top_k, o);
    };
    if (nk <= DISPATCH_THREADS * 4) go(k_dispatch<1>);
    else if (nk <= DISPATCH_THREADS * 16) go(k_dispatch<4>);
    else go(k_dispatch<DP_U>);
}

// sum_i x[i] * x[i] over one row in vec_dot_f32's order (src/quant.cpp:2756-2778;
// d % 16 == 0): lane j < 16 of the calling wave runs the fma chain over the
// elements 16 i + j of the chain-major row xs (element 16 i + j at j * S + i),
// lanes 0-7 are the reference's acc0, 8-15 its acc1; then acc0 + acc1 and the
// sequential sum of the 8 lanes.  Every lane of the wave calls it; the result
// is valid in lanes 0-15.
__device__ __forceinline__ float row_sumsq_chain(const float* xs, int S, int m, int lane) {
    const int j = lane & 15;
    float acc = 0.0f;
    if (lane < 16)
        for (int i = 0; i < m; ++i) {
            const float v = xs[j * S + i];
            acc = __builtin_fmaf(v, v, acc);
        }
    const float hi = __shfl_down(acc, 8, 16);
    const float v = acc + hi;  // acc0[j] + acc1[j] for j < 8
    float s = 0.0f;
#pragma unroll
    for (int q = 0; q < 8; ++q) s += __shfl(v, q, 16);
    return s;
}

// MoETransformerEngine::rms_norm (src/transformer.cpp:67-73) of `rows` rows of
// d floats, one block per row: ss = vec_dot_f32(x, x) in the reference's
// order, inv = 1 / sqrt(ss / d + eps) (IEEE division and square root), then
// out[i] = x[i] * inv * w[i] (w == null: weight 1).
__global__ void __launch_bounds__(256) k_rms_norm(const float* x, const float* w, int d, float eps, float* out) {
    extern __shared__ float xs[];  // chain-major row
    __shared__ float inv_s;
    const size_t row = blockIdx.x;
    const int tid = threadIdx.x, S = d / 16 + 1;  // odd stride: the 16 chains hit distinct banks
    const float* xr = x + row * (size_t)d;
    for (int e = tid; e < d; e += 256) xs[(e & 15) * S + (e >> 4)] = xr[e];
    __syncthreads();
    if (tid < 64) {
        const float ss = row_sumsq_chain(xs, S, d / 16, tid);
        if (tid == 0) inv_s = 1.0f / sqrtf(ss / (float)d + eps);
    }
    __syncthreads();
    const float inv = inv_s;
    float* orow = out + row * (size_t)d;
    for (int e = tid; e < d; e += 256) {
        const float v = xr[e] * inv;
        orow[e] = w ? v * w[e] : v;
    }
}

void launch_rms_norm(const float* x, const float* w, int rows, int d, float eps, float* out, hipStream_t st) {
    const size_t lds = (size_t)16 * (d / 16 + 1) * sizeof(float);
    if (lds > 65536)
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k_rms_norm), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)lds);
    hipLaunchKernelGGL(k_rms_norm, dim3((unsigned)rows), dim3(256), lds, st, x, w, d, eps, out);
}

// MoE combine (transformer.cpp:2728-2730 and 2752-2754): starting from 0, for
// each selected expert in descending-logit order acc = fma(p, y, acc), then
// acc = fma(shared_scale, y_shared, acc).
// Four consecutive features of one token per thread (d % 32 == 0), 16-byte loads and stores; the
// per-feature order is k_combine's contract (fma in selection order, then the shared expert).
template <int KU>  // slots whose loads go out together (the fma order stays the selection order)
__global__ void __launch_bounds__(256)
k_combine(int n, int d, int k, const float* probs, const int* pos_of, const float* y, const float* ysh,
          const float* shscale, const float* resid, float* out, const float* y2, int shparts) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;  // float4 index
    const int d4 = d / 4;
    if (idx >= (size_t)n * d4) return;
    const int t = (int)(idx / d4), i = 4 * (int)(idx % d4);
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int s0 = 0; s0 < k; s0 += KU) {
        int p[KU];
        float w[KU];
        float4 v[KU];
#pragma unroll
        for (int u = 0; u < KU; ++u) {
            const int s = min(s0 + u, k - 1);
            p[u] = pos_of[(size_t)t * k + s];
            w[u] = probs[(size_t)t * k + s];
        }
#pragma unroll
        for (int u = 0; u < KU; ++u) v[u] = *reinterpret_cast<const float4*>(y + (size_t)p[u] * d + i);
        if (y2) {  // the K-split down GEMM's second part
#pragma unroll
            for (int u = 0; u < KU; ++u) {
                const float4 b = *reinterpret_cast<const float4*>(y2 + (size_t)p[u] * d + i);
                v[u] = make_float4(v[u].x + b.x, v[u].y + b.y, v[u].z + b.z, v[u].w + b.w);
            }
        }
#pragma unroll
        for (int u = 0; u < KU; ++u) {
            if (s0 + u < k) {
                acc.x = __builtin_fmaf(w[u], v[u].x, acc.x);
                acc.y = __builtin_fmaf(w[u], v[u].y, acc.y);
                acc.z = __builtin_fmaf(w[u], v[u].z, acc.z);
                acc.w = __builtin_fmaf(w[u], v[u].w, acc.w);
            }
        }
    }
    if (ysh) {
        const float w = shscale[t];
        float4 v = *reinterpret_cast<const float4*>(ysh + (size_t)t * d + i);
        for (int q = 1; q < shparts; ++q) {  // the K parts of a shared down, in part order
            const float4 b = *reinterpret_cast<const float4*>(ysh + ((size_t)q * n + t) * d + i);
            v = make_float4(v.x + b.x, v.y + b.y, v.z + b.z, v.w + b.w);
        }
        acc.x = __builtin_fmaf(w, v.x, acc.x);
        acc.y = __builtin_fmaf(w, v.y, acc.y);
        acc.z = __builtin_fmaf(w, v.z, acc.z);
        acc.w = __builtin_fmaf(w, v.w, acc.w);
    }
    if (resid) {  // the residual add after the block (transformer.cpp:2762-2764)
        const float4 r = *reinterpret_cast<const float4*>(resid + (size_t)t * d + i);
        acc = make_float4(r.x + acc.x, r.y + acc.y, r.z + acc.z, r.w + acc.w);
    }
    *reinterpret_cast<float4*>(out + (size_t)t * d + i) = acc;
}

// The combine of one token per block followed by post_ffw_norm
// (transformer.cpp:2758-2760: rms_norm of moe_accum in place) and the residual
// add (2762-2764): out = resid + rms_norm(acc, post_w).  acc as k_combine
// computes it, staged chain-major for the exact vec_dot_f32 order of the norm.
__global__ void __launch_bounds__(256)
k_combine_norm(int n, int d, int k, const float* probs, const int* pos_of, const float* y, const float* ysh,
               const float* shscale, const float* post_w, float eps, const float* resid, float* out, const float* y2,
               int shparts) {
    extern __shared__ float as[];  // chain-major acc row
    __shared__ float inv_s;
    const int t = blockIdx.x, tid = threadIdx.x, S = d / 16 + 1;
    for (int i = tid; i < d; i += 256) {
        float acc = 0.0f;
        for (int s = 0; s < k; ++s) {
            const float w = probs[(size_t)t * k + s];
            const size_t o = (size_t)pos_of[(size_t)t * k + s] * d + i;
            acc = __builtin_fmaf(w, y2 ? y[o] + y2[o] : y[o], acc);
        }
        if (ysh) {
            float v = ysh[(size_t)t * d + i];
            for (int q = 1; q < shparts; ++q) v += ysh[((size_t)q * n + t) * d + i];
            acc = __builtin_fmaf(shscale[t], v, acc);
        }
        as[(i & 15) * S + (i >> 4)] = acc;
    }
    __syncthreads();
    if (tid < 64) {
        const float ss = row_sumsq_chain(as, S, d / 16, tid);
        if (tid == 0) inv_s = 1.0f / sqrtf(ss / (float)d + eps);
    }
    __syncthreads();
    const float inv = inv_s;
    for (int i = tid; i < d; i += 256) {
        const float v = as[(i & 15) * S + (i >> 4)] * inv * post_w[i];
        out[(size_t)t * d + i] = resid ? resid[(size_t)t * d + i] + v : v;
    }
}

void launch_combine(int n, int d, int k, const float* probs, const int* pos_of, const float* y, const float* ysh,
                    const float* shscale, float* out, hipStream_t st, const float* resid, const float* post_w,
                    float eps, const float* y2, int shparts) {
    if (post_w) {
        const size_t lds = (size_t)16 * (d / 16 + 1) * sizeof(float);
        if (lds > 65536)
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k_combine_norm),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        hipLaunchKernelGGL(k_combine_norm, dim3((unsigned)n), dim3(256), lds, st, n, d, k, probs, pos_of, y, ysh,
                           shscale, post_w, eps, resid, out, y2, shparts);
        return;
    }
    const size_t tot = (size_t)n * (d / 4);
    const dim3 grid((unsigned)((tot + 255) / 256));
    if (k <= 2)
        hipLaunchKernelGGL(k_combine<2>, grid, dim3(256), 0, st, n, d, k, probs, pos_of, y, ysh, shscale, resid, out,
                           y2, shparts);
    else if (k <= 4)
        hipLaunchKernelGGL(k_combine<4>, grid, dim3(256), 0, st, n, d, k, probs, pos_of, y, ysh, shscale, resid, out,
                           y2, shparts);
    else
        hipLaunchKernelGGL(k_combine<8>, grid, dim3(256), 0, st, n, d, k, probs, pos_of, y, ysh, shscale, resid, out,
                           y2, shparts);
}

// Q8_0 of `rows` rows of K fp32 values (quantize_row_q8_0, src/quant.cpp:1029-1045),
// one 32-block per half-wave.
__global__ void __launch_bounds__(256) k_quant_q8(const float* x, int rows, int K, ActQ8 out) {
    const int nb = K / 32;
    const size_t gid = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int half = (threadIdx.x >> 5) & 1, l32 = threadIdx.x & 31;
    const size_t blk = gid * 2 + half;
    const bool ok = blk < (size_t)rows * nb;
    quant_block(ok ? x[blk * 32 + l32] : 0.0f, l32, ok, out, blk / nb, (int)(blk % nb));
}

// dst[0 .. kpad) = x[0 .. n) followed by zeros: the zero-padded fp32 activation row the
// fp32-activation GEMV reads (written by a kernel, so a captured graph holds no memset node).
__global__ void __launch_bounds__(256) k_copy_pad(const float* x, int n, int kpad, float* dst) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    const size_t row = blockIdx.y;
    if (i < kpad) dst[row * kpad + i] = i < n ? x[row * n + i] : 0.0f;
}

void launch_copy_pad(const float* x, int n, int kpad, float* dst, hipStream_t st, int rows) {
    hipLaunchKernelGGL(k_copy_pad, dim3((unsigned)((kpad + 255) / 256), (unsigned)rows), dim3(256), 0, st, x, n, kpad,
                       dst);
}

void launch_quantize_q8(const float* x, int rows, int K, ActQ8 out, hipStream_t st) {
    const size_t blocks = (size_t)rows * (K / 32);
    const size_t waves = (blocks + 1) / 2;
    hipLaunchKernelGGL(k_quant_q8, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st, x, rows, K, out);
}

// One thread per (matrix, row, K-unit): scatter a GGUF block into the tile
// layout described in jxmoe_kernels.h.
__global__ void __launch_bounds__(256) k_repack(const uint8_t* raw, QMat m, uint8_t* qs, uint8_t* sc, uint8_t* ex) {
    const size_t units = (size_t)m.n_mats * m.rows * m.nkb;
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= units) return;
    const int kb = (int)(idx % m.nkb);
    const size_t er = idx / m.nkb;  // e*rows + r
    const int r = (int)(er % m.rows);
    const int e = (int)(er / m.rows);
    const int rt = r / ROWS_PER_TILE, mm = r % ROWS_PER_TILE;
    const size_t tile = ((size_t)e * m.nrt + rt) * m.nkb + kb;
    if (m.type == T_Q4_0) {
        const uint8_t* src = raw + idx * 18;
        uint8_t* dq = qs + (tile * 32 + mm) * 16;
        for (int i = 0; i < 16; ++i) dq[i] = src[2 + i];
        sc[(tile * 32 + mm) * 2 + 0] = src[0];
        sc[(tile * 32 + mm) * 2 + 1] = src[1];
    } else if (m.type == T_Q8_0) {
        const uint8_t* src = raw + idx * 34;
        for (int h = 0; h < 2; ++h) {
            uint8_t* dq = qs + ((tile * 2 + h) * 32 + mm) * 16;
            for (int i = 0; i < 16; ++i) dq[i] = src[2 + 16 * h + i];
        }
        sc[(tile * 32 + mm) * 2 + 0] = src[0];
        sc[(tile * 32 + mm) * 2 + 1] = src[1];
    } else if (m.type == T_Q5_0) {  // block_q5_0: d, qh (u32), qs[16]
        const uint8_t* src = raw + idx * 22;
        uint8_t* dq = qs + (tile * 32 + mm) * 16;
        for (int i = 0; i < 16; ++i) dq[i] = src[6 + i];
        sc[(tile * 32 + mm) * 2 + 0] = src[0];
        sc[(tile * 32 + mm) * 2 + 1] = src[1];
        for (int i = 0; i < 4; ++i) ex[(tile * 32 + mm) * 4 + i] = src[2 + i];
    } else if (m.type == T_Q6_K) {  // block_q6_K: ql[128], qh[64], scales[16], d
        const uint8_t* src = raw + idx * 210;
        for (int n = 0; n < 2; ++n)
            for (int c = 0; c < 6; ++c) {
                const uint8_t* s = c < 4 ? src + 64 * n + 16 * c : src + 128 + 32 * n + 16 * (c - 4);
                uint8_t* dq = qs + (((tile * 2 + n) * 6 + c) * 32 + mm) * 16;
                for (int i = 0; i < 16; ++i) dq[i] = s[i];
            }
        for (int i = 0; i < 16; ++i) sc[(tile * 32 + mm) * 16 + i] = src[192 + i];
        ex[(tile * 32 + mm) * 2 + 0] = src[208];
        ex[(tile * 32 + mm) * 2 + 1] = src[209];
    } else {  // Q4_K (144 B: header, qs[128]) or Q5_K (176 B: header, qh[32], qs[128])
        const bool q5 = m.type == T_Q5_K;
        const uint8_t* src = raw + idx * (q5 ? 176 : 144);
        const uint8_t* sq = src + (q5 ? 48 : 16);
        uint8_t* dh = sc + (tile * 32 + mm) * 16;
        for (int i = 0; i < 16; ++i) dh[i] = src[i];
        for (int p = 0; p < 4; ++p)
            for (int h = 0; h < 2; ++h) {
                uint8_t* dq = qs + (((tile * 4 + p) * 2 + h) * 32 + mm) * 16;
                for (int i = 0; i < 16; ++i) dq[i] = sq[32 * p + 16 * h + i];
            }
        if (q5)
            for (int h = 0; h < 2; ++h)
                for (int i = 0; i < 16; ++i) ex[((tile * 2 + h) * 32 + mm) * 16 + i] = src[16 + 16 * h + i];
    }
}

void launch_repack(const uint8_t* raw, QMat m, uint8_t* qs, uint8_t* sc, uint8_t* ex, hipStream_t st) {
    const size_t units = (size_t)m.n_mats * m.rows * m.nkb;
    hipLaunchKernelGGL(k_repack, dim3((unsigned)((units + 255) / 256)), dim3(256), 0, st, raw, m, qs, sc, ex);
}

}  // namespace jx
