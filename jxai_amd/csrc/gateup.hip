// Prefill gate/up, and the down over a Q8_0 h: grouped GEMM on the matrix cores, one exact product per 32-block.
//
// The reference's dots (vec_dot_{q4_0,q8_0,q4_K,q5_K}_q8_0, src/quant.cpp:3307-3730)
// sum each 32-element block exactly in integers and scale it by (weight scale x
// activation scale).  Here, per 32-block and 32 x 32 result tile:
//   S  = the block's integer sums, one MFMA with a zero accumulator
//   P  = (weight scale of the row) x (activation scale of the pair), one MFMA of
//        inner length 2 (the outer product)
//   acc = fma(S, P, acc), 16 per lane
// so no accumulator is rescaled.  Forms of S, which give the same bits:
//   from the packed blocks  v_mfma_i32_32x32x32_i8 on the Q8_0 quants as they are and on the weights' quants as bytes,
//        unpacked in registers (a block's bytes feed both pair tiles): Q4_K q, Q5_K q - 16, Q8_0 q, Q4_0 16 (q - 8) (a nibble
//        in the upper half of its byte, the sign bit flipped; the result's 1/16 is exact).  |S| < 2^20: exact as the
//        fp32 that the fma takes (16 conversions a tile: with them 37 vector instructions, which bound the kernel).
//   from the FP6 codes  v_mfma_scale_f32_32x32x64_f8f6f4 on a second copy of Q4_0, Q4_K and Q5_K weights (QMat::g6, 0.75 to 0.88 B
//        per weight; built where device memory is plentiful).  A: the weight q (Q4_0: q - 8, Q5_K: q - 16) is one FP6 e2m3
//        digit (0..16 with a sign are the codes themselves in units of 1/8).  B: the Q8_0 quant is 16 a + b with |a|, |b| <= 8, two BF6
//        e3m2 digits (3 significant bits; 16 a is a shift of the exponent).  A lane half holds 16 elements: its a's, then
//        its b's, against its weights twice (three register copies per 32 weights instead of loading them in both halves:
//        Mixtral-shaped 2048 tokens gate/up 1336 -> 1194 us).  No conversion of the result: |S| < 2^17, exact in fp32.
//        Per step from the blocks and from the codes: Mixtral-shaped 150 / 512 / 2048 tokens 356 / 673 / 2075 and 343 /
//        656 / 1907 us (its Q5_K form 437 / 795 / 2385 and 372 / 688 / 1996), Qwen1.5-shaped 200 / 700 / 2048 tokens 211 /
//        284 / 491 and 203 / 248 / 439 us.
// P is exact up to one rounding: the fp16 scales themselves (dx; Q4_0 and Q8_0 d), d * sc_j as an exact
// fp16 hi + lo pair from the table built at upload (QMat::bt).  The Q4_K / Q5_K min term
// -dmin * sum_j m_j * (dx_j * sum q_j) (Q5_K: plus 16 d sc_j for the offset) is three bf16
// MFMAs on 2- and 3-piece splits of its factors once per super-block, straight into acc.  Only the fp32 rounding of
// the accumulation differs from the reference; it matters, because h = SiLU(g) * u is
// re-quantized to Q8_0 (a relative error of 2^-11 in g and u moves ~1.4% of h's quants by
// one step, ~2.6e-3 relative in the layer output).
//
// Work split: the dispatch tables cut each expert's pairs into tiles of MFMA_BN; a workgroup
// owns 64 of a tile's pairs and 128 gate rows with the same 128 up rows, so SwiGLU and h's
// Q8_0 blocks are settled in registers.  4 waves, each a gate and an up row tile x two
// pair tiles (32 x 32 each).  Weights are MFMA operand A: lane (n, g) = (lane % 32, lane / 32) of
// a result holds pair n and, in register r, row 8 (r / 4) + 4 g + r % 4.
//
// Data movement: activations go global -> LDS by DMA per half-unit (128 of K, double-buffered,
// 16-byte chunks XOR-swizzled by row so operand reads are conflict-free).  Each wave's
// weights stream into a register ring one half-unit ahead: a block's registers are
// reloaded for the next half-unit as soon as its products are issued, so loads are spread
// over the half-unit and the barrier waits only for the DMA (vmcnt counts in order, and the
// ring's loads are younger).
#include <stddef.h>

#include <algorithm>
#include <type_traits>

#include "jxmoe_gemm.h"

namespace jx {

namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v6i __attribute__((ext_vector_type(6)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v3i __attribute__((ext_vector_type(3)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));

constexpr int GU_BN = 64;     // pairs per workgroup
constexpr int GU_WAVES = 4;   // row-tile slots

// One staged half-unit of GU_BN activation rows.
template <bool F6, int NP>
struct GuStage {
    static constexpr int PB = F6 ? 256 : 128;  // bytes per row: codes and scales (ActH::q6), or quants
    uint8_t q[GU_BN * PB];                     // row r, chunk c at chunk c ^ (r % (PB / 16))
    float sx[F6 ? 4 : GU_BN * 8];              // [block pair][row][2 blocks](scale, sum)
    uint16_t xm[NP ? 3 * GU_BN * 8 : 8];       // [piece][row][8 sub-blocks] bf16 of dx * sum(q)
    // the waves' min-term weight pieces: gate hi, gate mid, up hi, up mid and with three gate lo, up lo, each [32 rows][16 B]
    uint8_t wm[NP ? GU_WAVES * NP * 1024 : 16];
};

template <bool F6, int NP>
struct alignas(16) GuSmem {
    GuStage<F6, NP> st[2];
    int src[GU_BN];  // token of each staged pair
};

// What a workgroup reads of x.
struct GuIn {
    const uint8_t* q;   // rows of Q8_0 quants, or of codes (ActH::q6)
    const uint8_t* s;   // quants: rows of (scale, sum)
    const uint8_t* xp;  // min-term pieces (ActH::xp)
    int K, KU;
};

// 32 x 32 integer sums of 32 weights x Q8_0 quants, into [row][pair] (WROW) or [pair][row] of the result layout.
template <bool WROW>
__device__ __forceinline__ v16i mfma_i8(v4i w, v4i x) {
    return WROW ? __builtin_amdgcn_mfma_i32_32x32x32_i8(w, x, v16i{}, 0, 0, 0)
                : __builtin_amdgcn_mfma_i32_32x32x32_i8(x, w, v16i{}, 0, 0, 0);
}
// The same from 16 FP6 weight codes a lane half and the quants' BF6 digits.  The scales take the codes' units (1/8,
// 1/16) away.
template <bool WROW>
__device__ __forceinline__ v16f mfma_fp6(v3i w, v6i x) {
    constexpr int sw = 130, sx = 131;  // 2^3, 2^4
    const v8i w8 = __builtin_shufflevector(w, w, 0, 1, 2, 0, 1, 2, -1, -1);
    const v8i x8 = __builtin_shufflevector(x, x, 0, 1, 2, 3, 4, 5, -1, -1);
    if constexpr (WROW) return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w8, x8, v16f{}, 2, 3, 0, sw, 0, sx);
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x8, w8, v16f{}, 3, 2, 0, sx, 0, sw);
}
template <bool WROW>
__device__ __forceinline__ v16f mfma_scales(h4 w, h4 x) {
    return WROW ? __builtin_amdgcn_mfma_f32_32x32x8f16(w, x, v16f{}, 0, 0, 0)
                : __builtin_amdgcn_mfma_f32_32x32x8f16(x, w, v16f{}, 0, 0, 0);
}
template <bool WROW>
__device__ __forceinline__ v16f mfma_min(b8 w, b8 x, v16f c) {
    return WROW ? mfma16b(w, x, c) : mfma16b(x, w, c);
}

// The lane offset beside it: redefined where it is used, so its widening stays in the load's own block.
__device__ __forceinline__ uint32_t here(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}
template <typename T>
__device__ __forceinline__ T gload(gbyte* p) {
    return *reinterpret_cast<const __attribute__((address_space(1))) T*>(p);
}
template <>
__device__ __forceinline__ v3i gload<v3i>(gbyte* p) {
    const __attribute__((address_space(1))) int* w = reinterpret_cast<const __attribute__((address_space(1))) int*>(p);
    return v3i{w[0], w[1], w[2]};
}
// What it writes.
struct BgOut {
    ActQ8 hq;           // gate/up: h as Q8_0 (null q: not written),
    ActH hh;            //   as its codes and min-term pieces (null q6, xp: not written),
    float* hf;          //   or in fp32, rows of hf_ld floats (null: not written)
    int hf_ld;
    float* y;           // down: y[pair][rows], part k of KS along K at y + k * ystride
    int KS;
    size_t ystride;
};

// The weight ring's loads: what a lane (n, g) reads of row n for elements 16g .. 16g+15, one 32-block (FP6 codes; Q8_0;
// Q4_0: both halves of the block) or two (K-quants: the low and the high nibbles of 16 bytes) at a time.
template <int TYPE, bool F6>
struct Ring {
    static_assert(!F6 || TYPE == T_Q4_0 || TYPE == T_Q4_K || TYPE == T_Q5_K, "types with codes");
    static constexpr bool KQ = TYPE == T_Q4_K || TYPE == T_Q5_K, PAIR = KQ && !F6;
    static constexpr bool FIFTH = TYPE == T_Q5_K && !F6;  // the fifth bits beside the nibbles
    static constexpr int NP = !KQ ? 0 : block_table_pieces(TYPE);
    static constexpr bool QUAD = KQ || F6;  // a half-unit's four scales in one load (else each block's d beside its quants)
    static constexpr int N = PAIR ? HB / 2 : HB;                          // loads of quants per half-unit
    static constexpr int BYTES = F6 ? 768 : TYPE == T_Q4_0 ? 512 : 1024;  // of a row tile per load
    static constexpr int HU = N * BYTES + (F6 && !KQ ? 512 : 0);          // and half-unit (Q4_0 codes: their scales behind)
    // all loads per half-unit of both row tiles: quants, scales, fifth bits
    static constexpr int LOADS = 2 * (N + (QUAD ? FIFTH ? 2 : 1 : HB));
    // The half-unit's DMAs go out after block 2's weights have arrived (PAIR): the compiler's counted waits for the
    // ring do not know of them, and with a ring of two loads a wait for its second one would wait for DMAs just
    // issued (Mixtral-shaped 512 tokens 752 -> 714 us).
    static constexpr bool LATE = PAIR;
    // row groups per band (work_item) of the gate/up, the down
    static constexpr int GU_RC = PAIR ? 4 : 8, DN_RC = PAIR ? 2 : 4;
};

// A block's 16 quants of this lane as bytes, from the 16 bytes that the ring holds: block j of the half-unit (odd: of the
// super-block's second half).
template <int TYPE>
__device__ __forceinline__ v4i unpack(v4i w, v4i fifth, int j, bool odd, int sh) {
    v4i r = w;  // (Q8_0)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t v = (uint32_t)w[i];
        if constexpr (TYPE == T_Q4_0) {
            r[i] = (int)(((v << sh) & 0xF0F0F0F0u) ^ 0x80808080u);
        } else if constexpr (TYPE != T_Q8_0) {
            uint32_t q = (j & 1 ? v >> 4 : v) & 0x0F0F0F0Fu;
            if constexpr (TYPE == T_Q5_K) {  // q - 16: the nibble, and 0xF0 (15 x 0x10) where the fifth bit is clear
                const uint32_t f = (uint32_t)fifth[i];  // bit J of a byte: sub-block J
                const int J = (odd ? 4 : 0) + j;
                const uint32_t c = ~(J >= 4 ? f >> (J - 4) : f << (4 - J)) & 0x10101010u;
                q |= (c << 4) - c;
            }
            r[i] = (int)q;
        }
    }
    return r;
}

template <int N>
struct Tiles {
    static constexpr int value = N;
};

// PARTS: a workgroup with at most 32 pairs (an expert's last part, or all of them at a few pairs per expert) stages and
// multiplies one pair tile.  The second loop costs the FP6 kernels register copies (Mixtral-shaped 512 tokens 684 ->
// 697 us per step), so they take it where the average expert has fewer than BG_FEW pairs (without and with it:
// Mixtral-shaped 20 / 25 / 30 / 37 pairs 322 / 326 / 334 / 343 and 305 / 312 / 345 / 352 us, DeepSeek-V2-Lite-shaped 19 /
// 24 / 30 pairs 205 / 198 / 209 and 201 / 200 / 208 us, Qwen1.5-shaped 13 / 20 / 24 / 36 pairs 204 / 205 / 209 / 238 and
// 203 / 205 / 215 / 242 us); the int8 kernels always (Qwen3-shaped 64 / 600 / 2048 tokens 125 / 246 / 404 -> 107 / 232 /
// 393 us).
// Registers at two waves per SIMD (256): acc 64, two (S, P) sets 64; int8: the weight ring 16 (Q4_0, Q8_0: 40), its
// scales 16 (Q5_K: and fifth bits 16), operands 20 and the unpacked weights 8; FP6: the ring 24 (Q4_0: 32), its scales
// 16, operands 16 and the doubled codes 12.
template <int TYPE, bool F6, bool GATEUP, bool PARTS>
__global__ void __launch_bounds__(GU_WAVES * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_bgemm(QMat W0, QMat W1, GuIn in, Groups grp, int R, int n_items, int RC, BgOut o) {
    using Rg = Ring<TYPE, F6>;
    constexpr bool KQ = Rg::KQ;
    constexpr int NP = Rg::NP, BTS = BT_MIN + NP * 512;  // the table's min pieces, bytes per super-block
    using St = GuStage<F6, NP>;
    constexpr int PB = St::PB, CPP = PB / 16, PPI = 64 / CPP;  // row bytes, chunks, rows per DMA
    constexpr int PER = GU_BN / PPI / GU_WAVES;                // 1 KB DMAs per wave and half-unit
    __shared__ GuSmem<F6, NP> sm;
    int ti, sub, rg;
    // the grid covers the tile upper bound; the items of the tiles that exist are spread over the XCDs as if
    // the grid were exact, and the rest exit
    int n_eff = n_items;
    if (!grp.identity) n_eff = min(n_items, R * *grp.n_tiles * (MFMA_BN / GU_BN));
    // down over a long K: KS adjacent workgroups per item (on different XCDs), each a range of K
    const int kp = GATEUP ? 0 : (int)(blockIdx.x % o.KS), LB = GATEUP ? (int)blockIdx.x : (int)(blockIdx.x / o.KS);
    if ((LB >> 3) >= (n_eff >> 3) + ((LB & 7) < (n_eff & 7) ? 1 : 0)) return;
    work_item(LB, n_eff, R, MFMA_BN / GU_BN, RC, ti, sub, rg);
    int e, p0, cnt;
    if (!pair_tile(grp, ti, e, p0, cnt)) return;  // whole workgroup
    e = __builtin_amdgcn_readfirstlane(e);  // uniform: the weight addresses stay scalar
    p0 = __builtin_amdgcn_readfirstlane(p0) + sub * GU_BN;  // this workgroup's part of the tile
    cnt = __builtin_amdgcn_readfirstlane(cnt) - sub * GU_BN;
    if (cnt <= 0) return;
    cnt = min(cnt, GU_BN);

    const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // a row tile past the matrix repeats the last one, its results are dropped
    const int slot = rg * GU_WAVES + wave;
    const bool active = (GATEUP ? slot : 2 * slot) < W0.nrt;
    const int rt0 = min(GATEUP ? slot : 2 * slot, W0.nrt - 1);  // gate/up: of both matrices; down: and the next one

    if (tid < GU_BN) {
        const int p = p0 + min(tid, cnt - 1);
        sm.src[tid] = !GATEUP || grp.identity ? p : grp.pair_tok[p];
    }
    __syncthreads();

    const int KB = in.K / 32, H = in.K / 128;
    // this workgroup's half-units [h0, h1): whole super-blocks, the last part the rest
    const int HP = GATEUP ? H : ((H + o.KS - 1) / o.KS + 1) & ~1, h0 = kp * HP, h1 = min(H, h0 + HP);
    // an expert's pairs are in token order, so the buffers are based at the first source row in 64 bits and
    // per-lane offsets stay below 2^32 (jx_moe_forward refuses larger batches)
    const size_t src0 = (size_t)(uint32_t)__builtin_amdgcn_readfirstlane(sm.src[0]);
    const int rowb = H * PB;  // global bytes per row
    uint32_t soff[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int r = PPI * (wave * PER + k) + lane / CPP;
        soff[k] = (uint32_t)(sm.src[r] - (int)src0) * (uint32_t)rowb + (uint32_t)(((lane % CPP) ^ (r % CPP)) << 4);
    }
    const uint32_t srow = (uint32_t)(sm.src[lane] - (int)src0);  // the row of the lane's side loads
    const uint8_t* qsrc = in.q + src0 * (size_t)rowb;
    const uint32_t xoff = srow * (uint32_t)(KB * 8), poff = srow * (uint32_t)(in.KU * 48);
    const uint8_t* xsrc = F6 ? nullptr : in.s + src0 * (size_t)(KB * 8);
    const uint8_t* psrc = KQ ? in.xp + src0 * (size_t)(in.KU * 48) : nullptr;

    const uint8_t* wb[2];   // the wave's gate and up row tiles: quants or codes,
    const uint8_t* wsb[2];  // scales (K-quants: the table)
    const uint8_t* wxb[2];  // and Q5_K's fifth bits
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const QMat& W = GATEUP && i ? W1 : W0;
        const int rt = GATEUP ? rt0 : min(rt0 + i, W.nrt - 1);
        wb[i] = (F6 ? W.g6 + (size_t)e * W.g6_es : W.qs + (size_t)e * W.qs_es) + (size_t)rt * H * Rg::HU;
        wsb[i] = KQ ? W.bt + (size_t)e * W.bt_es + (size_t)rt * in.KU * BTS
                    : W.sc + (size_t)e * W.sc_es + (size_t)rt * KB * 64;
        wxb[i] = Rg::FIFTH ? W.ex + (size_t)e * W.ex_es + (size_t)rt * in.KU * 1024 : nullptr;
    }

    const uint8_t* wlo = NP == 3 ? (g ? wsb[1] : wsb[0]) + BT_MIN + 1024 + n * 16 : nullptr;

    // LDS address of a stage's parts
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr)&sm;
    auto stage = [&](int h, int buf) {
        const uint32_t S = lds0 + buf * (uint32_t)sizeof(St);
        gbyte* base = dma_base(qsrc + (size_t)h * PB);
#pragma unroll
        for (int k = 0; k < PER; ++k)
            if (!PARTS || wave * PER * PPI < cnt)  // (the wave's rows are in use)
                dma16g(base, soff[k], S + (wave * PER + k) * 1024);
        // (the side loads over the waves: scales by 0 and 1, pieces by 1, 2 and 3)
        if (!F6 && wave < 2)
            dma16g(dma_base(xsrc + (size_t)h * (HB * 8) + wave * 16), xoff, S + offsetof(St, sx) + wave * (GU_BN * 16));
        if constexpr (KQ) {
            if (h & 1) {  // the super-block's min-term pieces, used at the end of its second half
                const uint32_t sb = (uint32_t)(h >> 1) * BTS;
                const uint32_t d = S + offsetof(St, wm) + wave * (NP * 1024);
                gbyte *m0 = dma_base(wsb[0] + sb + BT_MIN), *m1 = dma_base(wsb[1] + sb + BT_MIN);
                dma16g(m0, (uint32_t)lane * 16, d);
                dma16g(m1, (uint32_t)lane * 16, d + 1024);
                if constexpr (NP == 3) dma16v(wlo + sb, d + 2048);
                if (wave > 0)
                    dma16g(dma_base(psrc + (size_t)(h >> 1) * 48 + (wave - 1) * 16), poff,
                           S + offsetof(St, xm) + (wave - 1) * (GU_BN * 16));
            }
        }
    };

    v16f acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[i][t] = v16f{};
    std::conditional_t<F6, v16f, v16i> S[2];  // the block sums and scale products of the last two tiles
    v16f P[2];
    std::conditional_t<F6, v3i, v4i> ring[Rg::N][2];
    uint16_t rd[Rg::QUAD ? 1 : HB][2];  // row n's fp16 scales
    v4i wsc[2][2], fifth[2][2];         // or, by the half-unit's parity, as fp16 hi | lo << 16; Q5_K's fifth bits

    // operand B: byte offsets of this lane's chunks of block 0 in pair tile 0 (quants, scale; codes, their tail and scales)
    const uint32_t lb0 = (uint32_t)(n * PB + ((g ^ (n % CPP)) << 4));
    const uint32_t lb1 = F6 ? (uint32_t)(n * PB + ((8 ^ (n % CPP)) << 4) + 8 * g) : (uint32_t)n * 16;
    const int sh = 4 - 4 * g;  // Q4_0: the lane's nibble to the upper half of its byte
    // this lane's offsets in a load of quants (and fifth bits), of scales
    const uint32_t lo0 = F6 ? (uint32_t)lane * 12 : (uint32_t)(TYPE == T_Q4_0 ? n : lane) * 16;
    const uint32_t lo1 = (uint32_t)n * (Rg::QUAD ? 16 : 2);
    auto load = [&](int h, int j, uint32_t o0, uint32_t o1) {  // j: of the ring
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            ring[j][i] = gload<std::conditional_t<F6, v3i, v4i>>(
                scalar(wb[i] + (size_t)(uint32_t)h * Rg::HU + j * Rg::BYTES) + o0);
            if constexpr (!Rg::QUAD) rd[j][i] = gload<uint16_t>(scalar(wsb[i] + (size_t)(uint32_t)h * (HB * 64) + j * 64) + o1);
        }
    };
    auto load_scales = [&](int h, int odd, uint32_t o0, uint32_t o1) {
        if constexpr (Rg::QUAD)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const size_t sb = (size_t)(uint32_t)(h >> 1);
                wsc[odd][i] = gload<v4i>(scalar(KQ ? wsb[i] + sb * BTS + odd * 512
                                                   : wb[i] + (size_t)(uint32_t)h * Rg::HU + Rg::N * Rg::BYTES) + o1);
                if constexpr (Rg::FIFTH) fifth[odd][i] = gload<v4i>(scalar(wxb[i] + sb * 1024) + o0);
            }
    };
    // acc of tile (i, t) takes the sums of set c
    auto fold = [&](int i, int t, int c) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
            acc[i][t][r] = __builtin_fmaf((float)S[c][r], P[c][r], acc[i][t][r]);
        asm volatile("" : "+v"(acc[i][t]));  // here, not where acc is next read: (S, P) stay two sets
    };
    const uint32_t gmask = g ? 0u : 0xFFFFu;

    if (h0 >= h1) return;  // (workgroup-uniform; more parts than super-blocks: never launched)
    stage(h0, 0);
    asm volatile("" ::: "memory");
    load_scales(h0, 0, lo0, lo1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < Rg::N; ++j) {
        load(h0, j, lo0, lo1);
        __builtin_amdgcn_sched_barrier(0);  // in the ring's order: the loop waits by count
    }

    auto half = [&](int h, bool odd, auto tiles) __attribute__((always_inline)) {
        constexpr int NT = decltype(tiles)::value;  // pair tiles in use
        // this half-unit's DMAs are older than the ring's loads (LATE: its last two); the other waves' reads of the other
        // stage are done
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(Rg::LATE ? 2 : Rg::LOADS) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        auto stage_next = [&]() __attribute__((always_inline)) {
            asm volatile("" ::: "memory");
            if (h + 1 < h1) stage(h + 1, odd ? 0 : 1);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!Rg::LATE) stage_next();
        const St& cur = sm.st[odd ? 1 : 0];
        const int hn = min(h + 1, h1 - 1);
        const uint32_t o0 = here(lo0), o1 = here(lo1);
        load_scales(hn, odd ? 0 : 1, o0, o1);
        __builtin_amdgcn_sched_barrier(0);
        // operands A and B of the block
        v4i bi[2], wv[2];
        int bd[2];
        v6i bf[2];
        v2i bp[2];
        // chunk c of row r sits at chunk c ^ (r % CPP): the lane's offset for block j is an XOR away from block 0's
        const uint32_t b0 = here(lb0), b1 = here(lb1);
        auto read_b = [&](int t, int j) {
            const uint8_t* q = cur.q + t * 32 * PB;
            if constexpr (F6) {
                const v4i a = *reinterpret_cast<const v4i*>(q + (b0 ^ (j << 5)));
                const v2i b = *reinterpret_cast<const v2i*>(q + (b1 ^ (j << 4)));
                bf[t] = __builtin_shufflevector(a, __builtin_shufflevector(b, b, 0, 1, -1, -1), 0, 1, 2, 3, 4, 5);
                bp[t] = *reinterpret_cast<const v2i*>(q + (b1 ^ ((4 + j) << 4)));
            } else {
                bi[t] = *reinterpret_cast<const v4i*>(q + (b0 ^ (j << 5)));
                bd[t] = *reinterpret_cast<const int*>(reinterpret_cast<const uint8_t*>(cur.sx) + (j >> 1) * (GU_BN * 16) +
                                                      t * 512 + (j & 1) * 8 + b1);
            }
        };
#pragma unroll
        for (int t = 0; t < NT; ++t) read_b(t, 0);
#pragma unroll
        for (int j = 0; j < HB; ++j) {
#pragma unroll
            for (int k = 0; k < 2 * NT; ++k) {
                const int i = k & 1, t = k >> 1, c = k & 1;
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (Rg::LATE) {
                    if (j == 2 && k == 2 * NT - 1) {
                        asm volatile("" : "+v"(ring[1][0]), "+v"(ring[1][1]));
                        stage_next();
                    }
                }
                if constexpr (!F6) {
                    if (t == 0) wv[i] = unpack<TYPE>(ring[Rg::PAIR ? j >> 1 : j][i], fifth[odd ? 1 : 0][i], j, odd, sh);
                    if (i == 0) {  // (dx, dx) in the block's place of its pair, as FP6 rows hold it
                        const uint32_t d16 = __builtin_bit_cast(uint16_t, (_Float16)__int_as_float(bd[t])) & gmask;
                        const int dx = (int)(d16 * (KQ ? 0x10001u : 1u));
                        bp[t] = KQ && (j & 1) ? v2i{0, dx} : v2i{dx, 0};
                    }
                    S[c] = mfma_i8<GATEUP>(wv[i], bi[t]);
                } else {
                    S[c] = mfma_fp6<GATEUP>(ring[j][i], bf[t]);
                }
                // the weight scales (hi, lo) of blocks j & ~1 and j | 1, the other's meets a zero; or the block's d
                v2i ws;
                if constexpr (Rg::QUAD) {
                    const v4i w4 = wsc[odd ? 1 : 0][i];
                    ws = j < 2 ? v2i{w4[0], w4[1]} : v2i{w4[2], w4[3]};
                } else {
                    ws = v2i{(int)(uint32_t)rd[j][i], 0};
                }
                P[c] = mfma_scales<GATEUP>(__builtin_bit_cast(h4, ws), __builtin_bit_cast(h4, bp[t]));
                if (j > 0 || k > 0) fold(c ^ 1, ((k + 2 * NT - 1) % (2 * NT)) >> 1, c ^ 1);  // the tile before
                if (i == 1 && j + 1 < HB) read_b(t, j + 1);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
                __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);  // VALU
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (!Rg::PAIR || (j & 1)) load(hn, Rg::PAIR ? j >> 1 : j, o0, o1);
        }
        fold(1, NT - 1, 1);
        if constexpr (KQ) {
            if (odd) {
                // acc += sum_j (dx_j sum q_j)(-dmin m_j) in three MFMAs, (MFMA, lane half) -> (weight piece,
                // activation piece).  Two exact weight pieces (h, m), all products:
                //   (0,0) h.h (0,1) h.m (1,0) m.h (1,1) m.m (2,0) h.l (2,1) m.l
                // Three (Q5_K), the six of nine above 2^-24 relative:
                //   (0,0) h.h (0,1) h.m (1,0) m.h (1,1) h.l (2,0) l.h (2,1) m.m
                const uint8_t* wm = cur.wm + wave * (NP * 1024) + n * 16;
                b8 x0[2], x1[2];
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const uint16_t* xp = cur.xm + (32 * t + n) * 8;
                    x0[t] = *reinterpret_cast<const b8*>(xp + (g ? 1 : 0) * GU_BN * 8);
                    x1[t] = *reinterpret_cast<const b8*>(xp + (NP == 3 && !g ? 0 : 2) * GU_BN * 8);
                }
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const b8 w0 = *reinterpret_cast<const b8*>(wm + i * 1024);
                    const b8 w1 = *reinterpret_cast<const b8*>(wm + i * 1024 + (NP == 3 && g ? 0 : 512));
                    const b8 w2 = *reinterpret_cast<const b8*>(wm + (g ? i * 1024 + 512 : NP == 3 ? 2048 + i * 512 : i * 1024));
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        acc[i][t] = mfma_min<GATEUP>(w0, x0[t], acc[i][t]);
                        acc[i][t] = mfma_min<GATEUP>(w1, NP == 3 ? x1[t] : x0[t], acc[i][t]);
                        acc[i][t] = mfma_min<GATEUP>(w2, NP == 3 ? x0[t] : x1[t], acc[i][t]);
                    }
                }
            }
        }
    };
    auto run = [&](auto tiles) __attribute__((always_inline)) {
        for (int h = h0; h < h1; h += 2) {
            half(h, false, tiles);
            if (h + 1 < h1) half(h + 1, true, tiles);
        }
    };
    if (!PARTS || cnt > 32) run(Tiles<2>{});
    else run(Tiles<1>{});

    if constexpr (TYPE == T_Q4_0 && !F6)  // 16 (q - 8)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][t][r] *= 0.0625f;
    if constexpr (!GATEUP) {
        // lane (n, g) holds row n of a row tile and, in register r, pair 8 (r / 4) + 4 g + r % 4 of a pair tile
        float* y = o.y + (size_t)kp * o.ystride + (size_t)p0 * W0.rows;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if (2 * slot + i >= W0.nrt) return;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    if (32 * t >= cnt) break;
                    const int pr = 32 * t + 8 * (r >> 2) + 4 * g + (r & 3);
                    if (pr < cnt) y[(size_t)pr * W0.rows + (2 * slot + i) * 32 + n] = acc[i][t][r];
                }
        }
        return;
    }
    // h = act(gate) * up, and h's block of 32 rows (row tile rt0) split over lanes n and n + 32
    if (!active) return;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        if (32 * t >= cnt) return;
        float v[16];
#pragma unroll
        for (int c = 0; c < 16; ++c) v[c] = gated(acc[0][t][c], acc[1][t][c], W0.act);
        const int pr = 32 * t + n;
        const size_t p = (size_t)(p0 + pr);
        const bool valid = pr < cnt;
        if (o.hf && valid) {
            float* fd = o.hf + p * (size_t)o.hf_ld + rt0 * 32 + 4 * g;
#pragma unroll
            for (int ii = 0; ii < 4; ++ii)
                *reinterpret_cast<float4*>(fd + 8 * ii) = make_float4(v[4 * ii], v[4 * ii + 1], v[4 * ii + 2], v[4 * ii + 3]);
        }
        if (!o.hq.q && !o.hh.q6) continue;
        // Q8_0 of the block (quantize_row_q8_0): both halves' lanes hold the same scale and sum
        float amax = 0.0f;
#pragma unroll
        for (int c = 0; c < 16; ++c) amax = fmaxf(amax, __builtin_fabsf(v[c]));
        amax = fmaxf(amax, __shfl_xor(amax, 32));
        const float d = amax / 127.0f;
        const float id = (d != 0.0f) ? 1.0f / d : 0.0f;
        int s = 0;
        uint32_t w[4];
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            float r = round_away(v[c] * id);
            r = fminf(fmaxf(r, -127.0f), 127.0f);
            const int q = (int)r;
            s += q;
            if ((c & 3) == 0) w[c >> 2] = 0;
            w[c >> 2] |= ((uint32_t)q & 0xFFu) << (8 * (c & 3));
        }
        s += __shfl_xor(s, 32);
        // word ii of half g is rows 8 ii + 4 g ..: exchange so half g stores rows 16 g .. 16 g + 15
        const auto x0 = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
        const auto x1 = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
        if (!valid) continue;
        const float2 sv = make_float2(f16_to_f32(f32_to_f16_trunc(d)), (float)s);
        if (o.hq.q) {
            *reinterpret_cast<uint4*>(o.hq.q + p * (size_t)o.hq.K + rt0 * 32 + 16 * g) = make_uint4(x0[0], x0[1], x1[0], x1[1]);
            if (g == 0) o.hq.s[p * (size_t)(o.hq.K / 32) + rt0] = sv;
        }
        if (o.hh.q6) {
            const uint32_t w4[4] = {x0[0], x0[1], x1[0], x1[1]};
            write_q6_part(w4, sv, o.hh, p, rt0, g);
        }
        if (o.hh.xp && g == 0) q8_pieces(sv, o.hh, p, rt0);
    }
}

// The bf16 nearest v, as fp32 (halves away from zero: the exactness below needs no ties to even).
__device__ __forceinline__ float nearest_bf16(float v) { return __uint_as_float((__float_as_uint(v) + 0x8000u) & 0xFFFF0000u); }

// The table of a repacked Q4_K / Q5_K matrix (QMat::bt), one thread per (expert, row tile, super-block, row): the 8
// sub-blocks' d * sc_j as an exact fp16 hi + lo pair, and -dmin * m_j as an exact bf16 pair (both products have 17
// bits: past the 8 of the nearest bf16 an integer of magnitude 2^8 at most is left); Q5_K, whose quants are taken from
// q - 16, -dmin * m_j + 16 d * sc_j in three pieces.  A scale past fp16 sets *over (d above
// 1000: no model's; such a matrix then has no table).
__global__ void __launch_bounds__(256) k_block_table(QMat m, uint8_t* out, int* over) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)m.n_mats * m.nrt * m.nkb * 32) return;
    const size_t t = idx / 32;
    const int row = (int)(idx % 32);
    const uint4 hd = ld16(m.sc + (t * 32 + row) * 16);
    const float d = f16_to_f32(hd.x & 0xFFFFu), dmin = f16_to_f32(hd.x >> 16);
    uint32_t pw[3][4] = {}, sw[8];
    const int np = block_table_pieces(m.type);
    bool bad = false;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        int sc, mv;
        hdr_scale_min(hd, j, sc, mv);
        const float scale = d * (float)sc;
        const _Float16 h = (_Float16)scale;
        bad |= !(__builtin_fabsf((float)h) < __builtin_inff());
        const _Float16 l = (_Float16)(scale - (float)h);  // exact: scale is a multiple of 2^-24 of 17 bits at most
        sw[j] = (uint32_t)__builtin_bit_cast(uint16_t, h) | (uint32_t)__builtin_bit_cast(uint16_t, l) << 16;
        uint16_t pc[3] = {};
        if (np == 3) {
            split3(__builtin_fmaf(16.0f * d, (float)sc, -dmin * (float)mv), pc[0], pc[1], pc[2]);
        } else {
            const float v = -dmin * (float)mv, vh = nearest_bf16(v);
            pc[0] = (uint16_t)(__float_as_uint(vh) >> 16);
            pc[1] = (uint16_t)(__float_as_uint(v - vh) >> 16);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) pw[c][j / 2] |= (uint32_t)pc[c] << (16 * (j & 1));
    }
    if (bad) atomicOr(over, 1);
    uint8_t* o = out + t * (size_t)(BT_MIN + np * 512) + row * 16;
#pragma unroll
    for (int c = 0; c < 2; ++c)
        *reinterpret_cast<uint4*>(o + c * 512) = make_uint4(sw[4 * c], sw[4 * c + 1], sw[4 * c + 2], sw[4 * c + 3]);
    for (int c = 0; c < np; ++c)
        *reinterpret_cast<uint4*>(o + BT_MIN + c * 512) = make_uint4(pw[c][0], pw[c][1], pw[c][2], pw[c][3]);
}

// The FP6 codes of a repacked Q4_0 / Q4_K / Q5_K matrix and Q4_0's scales beside them (QMat::g6), one thread per (expert, row
// tile, 32-block, row).
__global__ void __launch_bounds__(256) k_g6_codes(QMat m, int KB, uint8_t* out) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)m.n_mats * m.nrt * KB * 32) return;
    const size_t t = idx / 32;  // (e * nrt + rt) * KB + b
    const int row = (int)(idx % 32), b = (int)(t % KB);
    const size_t er = t / KB;   // e * nrt + rt
    uint32_t lo[8];             // the 32 quants, a byte each
    int off = 0;
    if (m.type == T_Q4_0) {
        off = 8;
        const uint4 q = ld16(m.qs + (t * 32 + row) * 16);
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) lo[i] = w[i] & 0x0F0F0F0Fu, lo[4 + i] = (w[i] >> 4) & 0x0F0F0F0Fu;
    } else {
        const int j = b & 7;
        const uint8_t* qs = m.qs + ((er * m.nkb + (b >> 3)) * 8 + (j >> 1) * 2) * 512 + row * 16;
        const uint4 q0 = ld16(qs), q1 = ld16(qs + 512);
        const uint32_t w[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) lo[i] = (w[i] >> (j & 1 ? 4 : 0)) & 0x0F0F0F0Fu;
        if (m.type == T_Q5_K) {
            off = 16;
            const uint8_t* ex = m.ex + (er * m.nkb + (b >> 3)) * 1024 + row * 16;
            const uint4 h0 = ld16(ex), h1 = ld16(ex + 512);
            const uint32_t hb[8] = {h0.x, h0.y, h0.z, h0.w, h1.x, h1.y, h1.z, h1.w};
#pragma unroll
            for (int i = 0; i < 8; ++i) lo[i] |= ((hb[i] >> j) & 0x01010101u) << 4;
        }
    }
    uint32_t c[6] = {0, 0, 0, 0, 0, 0};  // two parts of 16 codes
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        const int v = (int)((lo[i >> 2] >> (8 * (i & 3))) & 0xFFu) - off;
        const uint32_t code = v < 0 ? 32u | (uint32_t)-v : (uint32_t)v;
        const int at = (6 * i) / 32, sh = (6 * i) % 32;
        c[at] |= code << sh;
        if (sh > 26) c[at + 1] |= code >> (32 - sh);
    }
    uint8_t* o = out + (t / HB) * (size_t)g6_half_unit(m.type);
    if (m.type == T_Q4_0)
        *reinterpret_cast<uint32_t*>(o + 3072 + row * 16 + (b % HB) * 4) =
            *reinterpret_cast<const uint16_t*>(m.sc + (t * 32 + row) * 2);
    uint32_t* oc = reinterpret_cast<uint32_t*>(o + (b % HB) * 768 + row * 12);
#pragma unroll
    for (int w = 0; w < 3; ++w) {
        oc[w] = c[w];
        oc[96 + w] = c[3 + w];
    }
}

// Workgroups of an item list over row groups of `slots` row-tile slots.
template <int TYPE, bool F6, bool GATEUP, bool PARTS>
void launch_t(const QMat& w0, const QMat& w1, const GuIn& in, const Groups& grp, int tiles_ub, const BgOut& o, hipStream_t st) {
    const int slots = GATEUP ? w0.nrt : (w0.nrt + 1) / 2;
    const int R = (slots + GU_WAVES - 1) / GU_WAVES;
    const int n_items = R * tiles_ub * (MFMA_BN / GU_BN);
    if (n_items <= 0) return;
    using Rg = Ring<TYPE, F6>;
    hipLaunchKernelGGL((k_bgemm<TYPE, F6, GATEUP, PARTS>), dim3(n_items * (GATEUP ? 1 : o.KS)), dim3(GU_WAVES * 64), 0, st, w0,
                       w1, in, grp, R, n_items, std::min(GATEUP ? Rg::GU_RC : Rg::DN_RC, R), o);
}

// The launch of a matrix (pair)'s format over x's forms; false: a form is missing and nothing was launched.
template <bool GATEUP>
bool launch_form(const QMat& w0, const QMat& w1, const ActQ8& xq, const ActH& xh, const Groups& grp, int tiles_ub,
                 const BgOut& o, bool few, hipStream_t st) {
    if (is_kquant(w0.type) && (!w0.bt || !w1.bt || !xh.xp)) return false;
    GuIn in{xh.q6, nullptr, reinterpret_cast<const uint8_t*>(xh.xp), w0.cols, (w0.cols + 255) / 256};
    if (w0.g6 && w1.g6) {
        if (!in.q) return false;
        auto go = [&](auto type) {
            constexpr int T = decltype(type)::value;
            if (few) launch_t<T, true, GATEUP, true>(w0, w1, in, grp, tiles_ub, o, st);
            else launch_t<T, true, GATEUP, false>(w0, w1, in, grp, tiles_ub, o, st);
            return true;
        };
        switch (w0.type) {
            case T_Q4_0: return go(std::integral_constant<int, T_Q4_0>{});
            case T_Q4_K: return go(std::integral_constant<int, T_Q4_K>{});
            case T_Q5_K: return go(std::integral_constant<int, T_Q5_K>{});
            default: return false;
        }
    }
    if (!xq.q || !xq.s) return false;
    in.q = reinterpret_cast<const uint8_t*>(xq.q);
    in.s = reinterpret_cast<const uint8_t*>(xq.s);
    switch (w0.type) {
        case T_Q4_0: launch_t<T_Q4_0, false, GATEUP, true>(w0, w1, in, grp, tiles_ub, o, st); return true;
        case T_Q8_0: launch_t<T_Q8_0, false, GATEUP, true>(w0, w1, in, grp, tiles_ub, o, st); return true;
        case T_Q4_K: launch_t<T_Q4_K, false, GATEUP, true>(w0, w1, in, grp, tiles_ub, o, st); return true;
        case T_Q5_K: launch_t<T_Q5_K, false, GATEUP, true>(w0, w1, in, grp, tiles_ub, o, st); return true;
        default: return false;
    }
}

}  // namespace

bool gemm_block_ok(const QMat& m) { return m.type == T_Q4_0 || m.type == T_Q8_0 || m.bt; }

void launch_block_table(const QMat& m, uint8_t* bt, int* over, hipStream_t st) {
    const size_t n = (size_t)m.n_mats * m.nrt * m.nkb * 32;
    hipLaunchKernelGGL(k_block_table, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, m, bt, over);
}

void launch_g6_codes(const QMat& m, uint8_t* g6, hipStream_t st) {
    const int KB = m.cols / 32;
    const size_t n = (size_t)m.n_mats * m.nrt * KB * 32;
    hipLaunchKernelGGL(k_g6_codes, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, m, KB, g6);
}

bool launch_mfma_gateup(const QMat& g, const QMat& u, const ActQ8& xq, const ActH& xh, const Groups& grp, int tiles_ub,
                        const ActQ8& hq, const ActH& hh, float* hf, hipStream_t st, bool few) {
    return launch_form<true>(g, u, xq, xh, grp, tiles_ub, BgOut{hq, hh, hf, ((g.rows + 255) / 256) * 256, nullptr, 1, 0}, few, st);
}

bool launch_mfma_down_block(const QMat& dn, const ActQ8& hq, const ActH& hh, const Groups& grp, int tiles_ub, float* y,
                            hipStream_t st, int KS, size_t ystride, bool few) {
    return launch_form<false>(dn, dn, hq, hh, grp, tiles_ub, BgOut{ActQ8{}, ActH{}, nullptr, 0, y, KS, ystride}, few, st);
}

}  // namespace jx
