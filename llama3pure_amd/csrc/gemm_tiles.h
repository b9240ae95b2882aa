// gemm_tiles.h — what the batched-product kernels share: the launch
// arguments, and one thread's slice of the weight tile as fetched.
#pragma once

#include "device_common.h"
#include "internal.h"
#include "l3p.h"

namespace l3pd {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef int int32x4 __attribute__((ext_vector_type(4)));

struct GemmArgs {
    const uint8_t* w[3];   // per segment: weight rows,
    float* y[3];           // output rows [m][ldy],
    int ldy[3];
    int n[3];              // output features,
    int noff[3];           // first column in the split workspace's rows
    int tbeg[4];           // first N tile (tbeg[nseg] = all tiles)
    int nseg;
    size_t rb;             // bytes per weight row (same K and type for every segment)
    int k, m;              // inputs, batch rows
    const float* x;
    int ldx;
    int add;               // 1: Y += W.X (residual), 0: Y = W.X
    int nsplit, ksteps;    // K splits and kBK-steps per split
    float* part;           // [nsplit][m][ntot] partials when nsplit > 1
    int ntot;
    int streamk;           // > 0: stream-K over that many workgroups (grid.x), nsplit = most slots of a tile
    int kst;               // stream-K: kBK steps of a whole tile
    int bn;                // output columns per tile
};

// One thread's slice of a step's W tile: row t / 4 of the tile, elements
// e0 .. e0 + 15 of that row with e0 = k0 + 16 (t % 4).  Sixteen consecutive
// elements lie in one Q8_0 block or one scale group of a K-quant, so the
// slice needs at most three 16-byte pieces and a few header words, which are
// fetched one step ahead like the X tile.
struct WRaw {
    uint4 a, b, c, d;       // quant bytes / header / F32 values, by type
    uint32_t h0, h1, h2;    // scale words and scale bytes, by type
};

__device__ __forceinline__ uint32_t byte_of(const uint4& u, int i) {   // byte i (0..15, not constant)
    const uint32_t w = i < 4 ? u.x : (i < 8 ? u.y : (i < 12 ? u.z : u.w));
    return (w >> (8 * (i & 3))) & 0xffu;
}
__device__ __forceinline__ uint32_t byte_c(const uint4& u, int j) {     // byte j (constant after unrolling)
    const uint32_t w = (j >> 2) == 0 ? u.x : ((j >> 2) == 1 ? u.y : ((j >> 2) == 2 ? u.z : u.w));
    return (w >> (8 * (j & 3))) & 0xffu;
}

template <int QT>
__device__ __forceinline__ void fetch_slice(WRaw& r, const uint8_t* row, int e0) {
    if constexpr (QT == L3P_Q8_0) {   // 34-byte blocks: d, 32 quants
        const uint8_t* b = row + (size_t)(e0 >> 5) * 34;
        r.h0 = *reinterpret_cast<const uint16_t*>(b);
        // 2-byte aligned: one unaligned 16-byte load, left untouched until
        // store_step so that nothing waits for it here
        __builtin_memcpy(&r.a, b + 2 + 16 * ((e0 >> 4) & 1), 16);
    } else if constexpr (QT == L3P_Q4_K) {   // 144 bytes: d, dmin, 12 scale bytes, 128 nibble pairs
        const uint8_t* b = row + (size_t)(e0 >> 8) * 144;
        const int e = e0 & 255;
        __builtin_memcpy(&r.b, b, 16);
        __builtin_memcpy(&r.a, b + 16 + 32 * (e >> 6) + (e & 31), 16);
    } else if constexpr (QT == L3P_Q5_K) {   // 176 bytes: d, dmin, 12 scale bytes, 32 high-bit bytes, 128 nibble pairs
        const uint8_t* b = row + (size_t)(e0 >> 8) * 176;
        const int e = e0 & 255;
        __builtin_memcpy(&r.c, b, 16);
        __builtin_memcpy(&r.b, b + 16 + (e & 31), 16);
        __builtin_memcpy(&r.a, b + 48 + 32 * (e >> 6) + (e & 31), 16);
    } else if constexpr (QT == L3P_Q6_K) {   // 210 bytes: ql[128], qh[64], 16 int8 scales, d
        const uint8_t* b = row + (size_t)(e0 >> 8) * 210;
        const int e = e0 & 255, half = e >> 7, g = (e & 127) >> 5, l0 = e & 31;
        __builtin_memcpy(&r.a, b + 64 * half + 32 * (g & 1) + l0, 16);
        __builtin_memcpy(&r.b, b + 128 + 32 * half + l0, 16);
        r.h0 = *reinterpret_cast<const uint16_t*>(b + 208);
        r.h1 = b[192 + 8 * half + (l0 >> 4) + 2 * g];
    } else if constexpr (QT == L3P_Q3_K) {   // 110 bytes: hmask[32], qs[64], 12 scale bytes, d
        const uint8_t* b = row + (size_t)(e0 >> 8) * 110;
        const int g = (e0 & 255) >> 4, half = g >> 3, second = g & 1;
        __builtin_memcpy(&r.a, b + 32 + 32 * half + 16 * second, 16);
        __builtin_memcpy(&r.b, b + 16 * second, 16);
        r.h0 = *reinterpret_cast<const uint16_t*>(b + 108);
        r.h1 = b[96 + (g & 7)];
        r.h2 = b[104 + (g & 3)];
    } else if constexpr (QT == L3P_Q2_K) {   // 84 bytes: 16 scale bytes, qs[64], d, dmin
        const uint8_t* b = row + (size_t)(e0 >> 8) * 84;
        const int g = (e0 & 255) >> 4, half = g >> 3, second = g & 1;
        __builtin_memcpy(&r.a, b + 16 + 32 * half + 16 * second, 16);
        __builtin_memcpy(&r.h0, b + 80, 4);
        r.h1 = b[g];
    } else if constexpr (QT == L3P_F16 || QT == L3P_BF16) {
        const uint4* p = reinterpret_cast<const uint4*>(row + 2 * (size_t)e0);
        r.a = p[0];
        r.b = p[1];
    } else {   // F32
        const uint4* p = reinterpret_cast<const uint4*>(row + 4 * (size_t)e0);
        r.a = p[0];
        r.b = p[1];
        r.c = p[2];
        r.d = p[3];
    }
}

}  // namespace l3pd

// Y (=|+=) the sum of the partials of a launch that cut K (gemm.hip)
void launch_gemm_reduce(const l3pd::GemmArgs& a, hipStream_t st);
