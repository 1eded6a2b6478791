// Device helpers shared by the grouped matrix-core GEMMs (gateup.hip, gemm.hip).
#pragma once

#include "jxmoe_device.h"
#include "jxmoe_kernels.h"

namespace jx {

typedef __bf16 b8 __attribute__((ext_vector_type(8)));

constexpr int HB = 4;  // 32-blocks per staged half-unit

typedef __attribute__((address_space(3))) void* lds_ptr;

// 64 lanes x 16 (4) bytes from per-lane global addresses into LDS at `base`
// (wave-uniform), lane i at base + 16 i (4 i).
__device__ __forceinline__ void dma16(const void* src, void* base) {
    __builtin_amdgcn_global_load_lds(src, (lds_ptr)base, 16, 0, 0);
}
__device__ __forceinline__ void dma4(const void* src, void* base) {
    __builtin_amdgcn_global_load_lds(src, (lds_ptr)base, 4, 0, 0);
}

// Keeps a uniform address in scalar registers, so loads take it with a 32-bit lane offset (the compiler
// would otherwise add the lane offsets first and hold 64-bit vector addresses).
typedef const __attribute__((address_space(1))) uint8_t gbyte;
__device__ __forceinline__ gbyte* scalar(const uint8_t* p) {
    gbyte* g = (gbyte*)p;
    asm("" : "+s"(g));
    return g;
}
// The same as the base of dma16g: past the wait states that a vector-memory read of a scalar register needs after a
// vector instruction wrote it, which the compiler does not count into asm.
__device__ __forceinline__ gbyte* dma_base(const uint8_t* p) {
    gbyte* g = (gbyte*)p;
    asm("s_nop 4" : "+s"(g));
    return g;
}
// A wave-uniform address that the compiler computed in vector registers (a 64-bit product), in scalar ones.  (The
// asm keeps the compiler from dropping the readfirstlane of a value it knows to be uniform.)
__device__ __forceinline__ const uint8_t* uniform_ptr(const void* p) {
    uint32_t lo = (uint32_t)(uint64_t)p, hi = (uint32_t)((uint64_t)p >> 32);
    asm("s_nop 1" : "+v"(lo), "+v"(hi));
    lo = __builtin_amdgcn_readfirstlane(lo);
    hi = __builtin_amdgcn_readfirstlane(hi);
    return reinterpret_cast<const uint8_t*>((uint64_t)hi << 32 | lo);
}

// 64 lanes x 16 bytes from src (dma_base) + off (per lane) into LDS at byte `lds` (wave-uniform), lane i at lds + 16 i.  In
// asm because the compiler, which counts the builtin as a flat access, then waits for every load in flight
// before it uses any.  It has no result registers; the waits are the kernel's own (vmcnt counts in order, so the
// compiler's counted waits for the weights only get stricter).
__device__ __forceinline__ void dma16g(gbyte* src, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(src)
                 : "memory", "m0");
}
// The same from per-lane addresses.
__device__ __forceinline__ void dma16v(const uint8_t* src, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(src) : "memory", "m0");
}

__device__ __forceinline__ v16f mfma16(h8 a, h8 b, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ v16f mfma16b(b8 a, b8 b, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Exact 3-piece bf16 split of an fp32 value with at most 24 significant bits
// (truncation keeps each remainder exact).
__device__ __forceinline__ void split3(float v, uint16_t& h, uint16_t& m, uint16_t& l) {
    const uint32_t bh = __float_as_uint(v) & 0xFFFF0000u;
    const float r1 = v - __uint_as_float(bh);
    const uint32_t bm = __float_as_uint(r1) & 0xFFFF0000u;
    const float r2 = r1 - __uint_as_float(bm);
    h = (uint16_t)(bh >> 16);
    m = (uint16_t)(bm >> 16);
    l = (uint16_t)(__float_as_uint(r2) >> 16);
}

// Exact bf16 (hi, mid, lo) pieces of an fp32 value (truncation keeps each
// remainder exact) at xm[0], xm[8], xm[16].
__device__ __forceinline__ void store_pieces3(uint16_t* xm, float X) { split3(X, xm[0], xm[8], xm[16]); }

// The BF6 form (ActH::q6) of part `part` (16 quants, four signed bytes
// a word) of block b with (scale, sum) sb.
__device__ __forceinline__ void write_q6_part(const uint32_t (&w)[4], float2 sb, const ActH& o, size_t row, int b, int part) {
    uint32_t c[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int q = (int)(int8_t)(w[i >> 2] >> (8 * (i & 3)));
        const int a = (q + 8) >> 4, l = q - 16 * a;
        const uint32_t ma = (uint32_t)(a < 0 ? -a : a), ml = (uint32_t)(l < 0 ? -l : l);
        // |b| is its own code; 16 |a| = 16, 32, 48, 64 .. 128 units: 12, 16, 18, 20 .. 24
        const uint32_t ca = (a < 0 ? 32u : 0u) | (ma >= 4 ? 16 + ma : ma >= 2 ? 12 + 2 * ma : 12 * ma);
        const uint32_t cl = (l < 0 ? 32u : 0u) | ml;
        const int ba = 6 * i, bl = 96 + ba;
        c[ba / 32] |= ca << (ba % 32);
        c[bl / 32] |= cl << (bl % 32);
        if (ba % 32 > 26) {
            c[ba / 32 + 1] |= ca >> (32 - ba % 32);
            c[bl / 32 + 1] |= cl >> (32 - bl % 32);
        }
    }
    // exact: sb.x is an fp16 widened
    const uint32_t dx = part ? 0u : (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)sb.x) * 0x00010001u;
    const int j = b & 3;
    uint8_t* d = o.q6 + row * (size_t)o.K * 2 + (b >> 2) * 256;
    *reinterpret_cast<uint4*>(d + j * 32 + part * 16) = make_uint4(c[0], c[1], c[2], c[3]);
    *reinterpret_cast<uint2*>(d + 128 + j * 16 + part * 8) = make_uint2(c[4], c[5]);
    *reinterpret_cast<uint2*>(d + 192 + j * 16 + part * 8) = make_uint2(j & 1 ? 0u : dx, j & 1 ? dx : 0u);
}

// The min-term pieces (ActH::xp) of block b of a row with (scale, sum) sv.
__device__ __forceinline__ void q8_pieces(float2 sv, const ActH& o, size_t row, int b) {
    store_pieces3(o.xp + row * (size_t)o.KU * 24 + (b / 8) * 24 + b % 8, sv.x * sv.y);  // product exact
}

// (scale, min) j of a Q4_K header in registers (get_scale_min_k4,
// src/quant.cpp:1107-1115).
__device__ __forceinline__ void hdr_scale_min(const uint4& hd, int j, int& sc, int& mn) {
    const uint32_t s0 = hd.y, s1 = hd.z, s2 = hd.w;  // scales[0..3], [4..7], [8..11]
    const int sh = 8 * (j & 3);
    if (j < 4) {
        sc = (s0 >> sh) & 63;
        mn = (s1 >> sh) & 63;
    } else {
        const uint32_t b = (s2 >> sh) & 0xFF;
        sc = (b & 0x0F) | ((((s0 >> sh) >> 6) & 3) << 4);
        mn = (b >> 4) | ((((s1 >> sh) >> 6) & 3) << 4);
    }
}

// ---------------------------------------------------------------- tiles
__device__ __forceinline__ bool pair_tile(const Groups& grp, int ti, int& e, int& p0, int& cnt) {
    if (grp.identity) {
        e = 0;
        p0 = ti * MFMA_BN;
        cnt = min(MFMA_BN, grp.n_tok - p0);
        return cnt > 0;
    }
    if (ti >= *grp.n_tiles) return false;
    const int4 t = grp.tiles[ti];
    e = t.x;
    p0 = t.y;
    cnt = t.z;
    return true;
}

// Workgroup -> (pair tile, part of the tile, row group).  Numbering is
// XCD-major (hardware deals workgroups round-robin over the 8 XCDs, so XCD x
// runs a contiguous range of items), and within it bands of RC row groups
// sweep every pair tile: the ~64 workgroups resident on one XCD then cover
// about RC row groups x 64 / RC tile parts, and each weight row group and each
// staged activation tile is fetched into that XCD's L2 once for several
// workgroups.  RC = R: all row groups of a tile part before the next part.
__device__ __forceinline__ void work_item(int L, int n_items, int R, int S, int RC, int& ti, int& sub, int& rg) {
    const int x = L & 7, s = L >> 3;
    const int q = n_items >> 3, rem = n_items & 7;
    const int i = x * q + min(x, rem) + s;
    const int TS = n_items / R;             // tile parts
    const int band = i / (RC * TS);         // full bands hold RC * TS items; the last one fewer rows
    const int rows = min(RC, R - band * RC);
    const int j = i - band * RC * TS;
    const int ts = j / rows;
    rg = band * RC + (j - ts * rows);
    ti = ts / S;
    sub = ts - ti * S;
}

}  // namespace jx
