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
