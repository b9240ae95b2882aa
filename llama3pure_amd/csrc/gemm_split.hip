// gemm_split.hip — the prefill GEMMs of the types the reference dequantizes
// before its batched dot (matmul_deq_batch_4row, llama3pure-c-engine.c:
// 2179-2273; F32 weights: gemm.hip), on the bf16 matrix cores with fp32's
// precision:
//   Y[m][n] (=|+=) sum_k W[n][k] * X[m][k]
//
// Operands.  An integer code of at most 8 bits is a bf16 value, and the 24
// significant bits of an fp32 x are three (truncations of 8 bits each, their
// sum is x exactly), so three bf16 products give the exact code * x, summed in
// fp32: Q8_0, Q4_K, Q5_K and Q6_K multiply their quants, Q3_K and Q2_K their
// quants times the 6- or 4-bit group scale (at most 128), BF16 its values, F16
// a high and a low part (six products).  The block's fp32 scale (d, or d times
// the group's) multiplies the sum over its 32 (Q6_K: 16) columns.  Offsets
// (Q4_K, Q5_K, Q2_K) are one more product per super-block: the groups' offset
// codes times the groups' sums of x, split alike, times dmin.  Every weight
// enters as exactly as before, and fewer fp32 additions follow it: against 64
// bits the results lie closer than those of fp32 products summed column by
// column.  x is scaled by 2^-14 and the results back, so that sums of codes
// times x stay finite for every finite x (below 2^-98 in magnitude x's last
// part is subnormal).
//
// Why.  The fp32 matrix cores do 256 FLOP a cycle and CU, the bf16 ones 4096:
// three products are 3/16 of the time.  Q8_0 14336 x 4096 x 1024 rows: 966 ->
// 388 us (125 -> 310 TFLOP/s).
//
// What bounds it.  MFMA and VALU issue add up (64 x 128 tiles: 38% and 59% of
// the SIMDs' cycles, at a clock that falls from 2.4 to 1.7-2 GHz), so what
// counts is VALU work per output: 7.5 operations an x and 1.5-4 a weight for
// each tile that expands it, and one fused multiply-add per output and block.
// A 128 x 256 tile, each of four waves 64 x 128, is the largest whose
// accumulators leave room for two workgroups a CU.  Two LDS buffers with the
// expansion between a wave's own MFMAs cost the second workgroup and were
// slower (Q8_0 458 us, Q4_K 738).
//
// A workgroup walks K in steps of 32: x and weights of a step, fetched one step
// earlier, go to LDS (80-byte rows), and each wave forms its 32 x 32 tiles with
// v_mfma_f32_32x32x16_bf16, a tile's scaling issued beside the next tile's
// products.  x fragments are held for one row of tiles and the weights' re-read:
// holding all of x's spilled (Q6_K 703 -> 477 us).  Where the tiles are too few
// for the CUs, K is cut in equal runs (multiples of a super-block where there
// are offsets), whose fp32 partials gemm_reduce_kernel adds in order.
#include <algorithm>

#include "device_common.h"
#include "gemm_tiles.h"
#include "internal.h"

namespace {

using namespace l3pd;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kK = 32;     // K step
constexpr int kLD = 40;    // LDS row stride in bf16: 80-byte rows spread eight b128 reads over all banks

template <int QT>
struct WType {
    static constexpr bool kScaled = QT != L3P_F16 && QT != L3P_BF16;   // integer codes and a scale
    static constexpr bool kHalves = QT == L3P_Q6_K;                    // a scale per 16 columns, not 32
    static constexpr int kMinGroup = QT == L3P_Q2_K ? 16 : (QT == L3P_Q4_K || QT == L3P_Q5_K) ? 32 : 0;
    static constexpr int kMins = kMinGroup ? 256 / kMinGroup : 0;      // offsets of a super-block
    static constexpr int kParts = QT == L3P_F16 ? 2 : 1;               // bf16 parts of a weight
    static constexpr int kUnit = kMinGroup ? 256 : kK;                 // K is cut at multiples of this
};

// sums of 256 columns' offset products (6-bit codes times sums of 32 x) stay finite for every finite x
constexpr float kXScale = 1.0f / 16384, kXUnscale = 16384.0f;

__device__ __forceinline__ uint32_t bits(float f) { return __float_as_uint(f); }
__device__ __forceinline__ float high_half(float f) { return __uint_as_float(bits(f) & 0xffff0000u); }
// the upper halves of two floats: their bf16 values, truncated
__device__ __forceinline__ uint32_t pack_high(float lo, float hi) {
    return __builtin_amdgcn_perm(bits(hi), bits(lo), 0x07060302u);
}

template <int kCtrl>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), kCtrl, 0xf, 0xf, true));
}

// byte-wise x - 32 for bytes 0..63, as int8
__device__ __forceinline__ uint32_t minus32(uint32_t x) { return ((x | 0x80808080u) - 0x20202020u) ^ 0x80808080u; }
template <bool kSigned>
__device__ __forceinline__ float byte_float(uint32_t w, int j) {
    return kSigned ? (float)(int8_t)(w >> (8 * j)) : (float)((w >> (8 * j)) & 0xffu);
}

// The slice's codes (or values) as bf16 pairs c (and c2, the low parts of
// F16 values), its scale, and for types with offsets the group's code mn and
// the super-block's factor dmin.
struct WSlice {
    uint32_t c[8], c2[8];
    float scale, mn, dmin;
};
template <int QT>
__device__ __forceinline__ void decode_codes(const WRaw& r, int e0, WSlice& o) {
    const uint32_t aw[4] = {r.a.x, r.a.y, r.a.z, r.a.w}, bw[4] = {r.b.x, r.b.y, r.b.z, r.b.w};
    if constexpr (QT == L3P_BF16 || QT == L3P_F16) {
        const uint32_t w[8] = {aw[0], aw[1], aw[2], aw[3], bw[0], bw[1], bw[2], bw[3]};
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if constexpr (QT == L3P_BF16) {
                o.c[j] = w[j];
            } else {   // 11 significant bits: 8 and 3; an infinity has no low part
                const float v0 = h2f_exact(w[j] & 0xffffu), v1 = h2f_exact(w[j] >> 16);
                o.c[j] = pack_high(v0, v1);
                o.c2[j] = pack_high(fabsf(v0) == INFINITY ? 0.0f : v0 - high_half(v0),
                                    fabsf(v1) == INFINITY ? 0.0f : v1 - high_half(v1));
            }
        }
        return;
    }
    float mul = 1.0f, sub = 0.0f;   // code = mul * byte - sub (Q2_K, Q3_K)
    uint32_t q[4];
    constexpr bool kSigned = QT == L3P_Q8_0 || QT == L3P_Q6_K;
    if constexpr (QT == L3P_Q8_0) {
        o.scale = h2f_exact(r.h0);
#pragma unroll
        for (int j = 0; j < 4; ++j) q[j] = aw[j];
    } else if constexpr (QT == L3P_Q4_K || QT == L3P_Q5_K) {
        const uint4& hd = QT == L3P_Q4_K ? r.b : r.c;
        const int js = (e0 & 255) >> 5;
        // sub-block js's 6-bit scale and min of the 12 bytes in hd.y, hd.z, hd.w
        const int sh = 8 * (js & 3);
        const uint32_t s0 = hd.y >> sh, s1 = hd.z >> sh, s2 = hd.w >> sh;
        const uint32_t sc = js < 4 ? s0 & 63u : (s2 & 15u) | ((s0 >> 2) & 0x30u);
        const uint32_t mn = js < 4 ? s1 & 63u : ((s2 >> 4) & 15u) | ((s1 >> 2) & 0x30u);
        o.scale = h2f_exact(hd.x & 0xffffu) * (float)sc;
        o.dmin = h2f_exact(hd.x >> 16);
        o.mn = (float)mn;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            q[j] = (aw[j] >> (4 * (js & 1))) & 0x0f0f0f0fu;
            if constexpr (QT == L3P_Q5_K) q[j] |= ((bw[j] >> js) & 0x01010101u) << 4;
        }
    } else if constexpr (QT == L3P_Q6_K) {
        const int g = (e0 & 127) >> 5;
        o.scale = h2f_exact(r.h0) * (float)(int8_t)r.h1;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            q[j] = minus32(((aw[j] >> (2 * (g & 2))) & 0x0f0f0f0fu) | (((bw[j] >> (2 * g)) & 0x03030303u) << 4));
    } else if constexpr (QT == L3P_Q3_K) {   // code = scale * (u - 4), at most 128
        const int g = (e0 & 255) >> 4, half = g >> 3, j4 = (g >> 1) & 3;
        const uint32_t lo = g < 8 ? r.h1 & 0x0fu : (r.h1 >> 4) & 0x0fu;
        mul = (float)((int)(lo | (((r.h2 >> (2 * (g >> 2))) & 3u) << 4)) - 32);
        sub = 4.0f * mul;
        o.scale = h2f_exact(r.h0);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            q[j] = ((aw[j] >> (2 * j4)) & 0x03030303u) | (((bw[j] >> (4 * half + j4)) & 0x01010101u) << 2);
    } else {   // Q2_K: code = scale * u, at most 45
        const int j4 = ((e0 & 255) >> 5) & 3;
        mul = (float)(r.h1 & 0x0fu);
        o.mn = (float)((r.h1 >> 4) & 0x0fu);
        o.scale = h2f_exact(r.h0 & 0xffffu);
        o.dmin = h2f_exact(r.h0 >> 16);
#pragma unroll
        for (int j = 0; j < 4; ++j) q[j] = (aw[j] >> (2 * j4)) & 0x03030303u;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        float v0 = byte_float<kSigned>(q[j >> 1], 2 * (j & 1)), v1 = byte_float<kSigned>(q[j >> 1], 2 * (j & 1) + 1);
        if constexpr (QT == L3P_Q3_K || QT == L3P_Q2_K) {
            v0 = __builtin_fmaf(mul, v0, -sub);
            v1 = __builtin_fmaf(mul, v1, -sub);
        }
        o.c[j] = pack_high(v0, v1);
    }
}

// x 2^-14 as three bf16 values whose sum it is: 24 significant bits in three
// truncations of 8.  The clamp lies above any finite remainder; an infinity
// (or NaN), whose remainder is NaN, gets a finite second part, so its first
// part decides.
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& p1, uint32_t& p2, uint32_t& p3) {
    constexpr float kTop = 0x1p113f;
    const float xa = a * kXScale, xb = b * kXScale;
    p1 = pack_high(xa, xb);
    const float ra = __builtin_amdgcn_fmed3f(xa - high_half(xa), -kTop, kTop);
    const float rb = __builtin_amdgcn_fmed3f(xb - high_half(xb), -kTop, kTop);
    p2 = pack_high(ra, rb);
    p3 = pack_high(ra - high_half(ra), rb - high_half(rb));
}

template <int QT, int BM, int BN, int WM>
struct Tile {
    static constexpr int kWN = 4 / WM;                            // waves along N
    static constexpr int TM = BM / WM / 32, TN = BN / kWN / 32;   // 32 x 32 tiles of a wave
    static constexpr int XU = BM / 32;                            // a thread's x quads of a step
    static constexpr int WU = BN / 128;                           // and its 16-code slices
};

template <int QT, int BM, int BN, int WM, int OCC>
__global__ void __launch_bounds__(256, OCC) gemm_split_kernel(GemmArgs a) {
    using T = Tile<QT, BM, BN, WM>;
    using W = WType<QT>;
    constexpr int TM = T::TM, TN = T::TN, XU = T::XU, WU = T::WU, NM = W::kMins, NS = W::kHalves ? 2 : 1;
    __shared__ __align__(16) uint16_t xs[3][BM * kLD];
    __shared__ __align__(16) uint16_t ws[W::kParts][BN * kLD];
    __shared__ float dsc[NS][BN];
    // the x sums (three parts) and offset codes of a super-block's groups
    __shared__ __align__(16) uint16_t xm[3][NM ? BM * NM : 8];
    __shared__ __align__(16) uint16_t wm[NM ? BN * NM : 8];
    __shared__ float dmn[NM ? BN : 1];

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int mw = (wave / T::kWN) * TM * 32, nw = (wave % T::kWN) * TN * 32;
    const int i32 = lane & 31, h = lane >> 5;

    // workgroup -> (K run, N tile, M tile), M fastest; each XCD (workgroups go
    // round the eight of them) takes one contiguous run of the items, so the
    // tiles that share weights share an L2
    const int G = gridDim.x, xcd = blockIdx.x & 7, q = G >> 3, rem = G & 7;
    const int item = xcd * q + min(xcd, rem) + (blockIdx.x >> 3);
    const int MT = (a.m + BM - 1) / BM, NT = a.tbeg[a.nseg];
    const int m0 = (item % MT) * BM, ntile = (item / MT) % NT, z = item / (MT * NT);
    const int sg = (a.nseg > 1 && ntile >= a.tbeg[1]) ? ((a.nseg > 2 && ntile >= a.tbeg[2]) ? 2 : 1) : 0;
    const uint8_t* const Wp = a.w[sg];
    const int N = a.n[sg], n0 = (ntile - a.tbeg[sg]) * BN;
    const int kbeg = z * a.ksteps * kK, kend = min(a.k, kbeg + a.ksteps * kK);

    // This thread's quads of x (rows t / 8 + 32 u: eight lanes read a row's 128
    // bytes) and its weight rows; past the matrix the last row again, whose
    // results are not stored.
    const int xr = t >> 3, xc = 4 * (t & 7);
    const float* xrow[XU];
#pragma unroll
    for (int u = 0; u < XU; ++u) xrow[u] = a.x + (size_t)min(m0 + xr + 32 * u, a.m - 1) * a.ldx + xc;
    const uint8_t* wrow[WU];
#pragma unroll
    for (int u = 0; u < WU; ++u) wrow[u] = Wp + (size_t)min(n0 + ((t + 256 * u) >> 1), N - 1) * a.rb;
    float4 xv[XU];
    WRaw wr[WU];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int u = 0; u < XU; ++u) xv[u] = *reinterpret_cast<const float4*>(xrow[u] + k0);
#pragma unroll
        for (int u = 0; u < WU; ++u) fetch_slice<QT>(wr[u], wrow[u], k0 + 16 * (t & 1));
    };
    auto store = [&](int k0) {
#pragma unroll
        for (int u = 0; u < XU; ++u) {
            uint2 p[3];
            split_pair(xv[u].x, xv[u].y, p[0].x, p[1].x, p[2].x);
            split_pair(xv[u].z, xv[u].w, p[0].y, p[1].y, p[2].y);
#pragma unroll
            for (int c = 0; c < 3; ++c) *reinterpret_cast<uint2*>(&xs[c][(xr + 32 * u) * kLD + xc]) = p[c];
        }
        if constexpr (NM > 0) {   // the group's sum of x: four or eight lanes
#pragma unroll
            for (int u = 0; u < XU; ++u) {
                float s = (xv[u].x + xv[u].y) + (xv[u].z + xv[u].w);
                s += dpp<0xB1>(s);                                  // lane ^ 1
                s += dpp<0x4E>(s);                                  // lane ^ 2
                if (W::kMinGroup == 32) s += dpp<0x141>(s);         // the other four of eight
                if ((t & (W::kMinGroup / 4 - 1)) == 0) {
                    uint32_t p1, p2, p3;
                    split_pair(s, 0.0f, p1, p2, p3);
                    const int i = (xr + 32 * u) * NM + ((k0 + xc) & 255) / W::kMinGroup;
                    xm[0][i] = (uint16_t)p1;
                    xm[1][i] = (uint16_t)p2;
                    xm[2][i] = (uint16_t)p3;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < WU; ++u) {
            const int i = t + 256 * u, n = i >> 1, half = i & 1, e0 = k0 + 16 * half;
            WSlice o;
            decode_codes<QT>(wr[u], e0, o);
            uint4* dst = reinterpret_cast<uint4*>(&ws[0][n * kLD + 16 * half]);
            dst[0] = make_uint4(o.c[0], o.c[1], o.c[2], o.c[3]);
            dst[1] = make_uint4(o.c[4], o.c[5], o.c[6], o.c[7]);
            if constexpr (W::kParts == 2) {
                uint4* dst2 = reinterpret_cast<uint4*>(&ws[W::kParts - 1][n * kLD + 16 * half]);
                dst2[0] = make_uint4(o.c2[0], o.c2[1], o.c2[2], o.c2[3]);
                dst2[1] = make_uint4(o.c2[4], o.c2[5], o.c2[6], o.c2[7]);
            }
            if constexpr (W::kScaled) {
                if (NS == 2 || half == 0) dsc[NS == 2 ? half : 0][n] = o.scale * kXUnscale;
            }
            if constexpr (NM > 0) {
                if (W::kMinGroup == 16 || half == 0) {
                    wm[n * NM + (e0 & 255) / W::kMinGroup] = (uint16_t)(bits(o.mn) >> 16);
                    dmn[n] = -o.dmin * kXUnscale;
                }
            }
        }
    };

    floatx16 acc[TM][TN];
#pragma unroll
    for (int im = 0; im < TM; ++im)
#pragma unroll
        for (int in = 0; in < TN; ++in)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[im][in][r] = 0.0f;

    auto frag = [&](const uint16_t* p) { return *reinterpret_cast<const bf16x8*>(p); };
    fetch(kbeg);
    for (int k0 = kbeg; k0 < kend; k0 += kK) {
        store(k0);
        __syncthreads();
        if (k0 + kK < kend) fetch(k0 + kK);   // in flight during this step's matrix work
        // The wave's 32 x 32 tiles one after the other: a tile's products go to
        // b, and its scaling into acc runs in the shadow of the next tile's.
        floatx16 b[2];
        float sc[2];
#pragma unroll
        for (int im = 0; im < TM; ++im) {
            bf16x8 xf[2][3];
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int c = 0; c < 3; ++c) xf[s][c] = frag(&xs[c][(mw + 32 * im + i32) * kLD + 16 * s + 8 * h]);
#pragma unroll
            for (int in = 0; in < TN; ++in) {
                const int n = nw + 32 * in + i32;
                bf16x8 wf[2][W::kParts];
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int c = 0; c < W::kParts; ++c) wf[s][c] = frag(&ws[c][n * kLD + 16 * s + 8 * h]);
                if constexpr (!W::kScaled) {
#pragma unroll
                    for (int s = 0; s < 2; ++s)
#pragma unroll
                        for (int c = 2; c >= 0; --c)
#pragma unroll
                            for (int wc = W::kParts - 1; wc >= 0; --wc)
                                acc[im][in] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[s][c], wf[s][wc],
                                                                                     acc[im][in], 0, 0, 0);
                } else {
#pragma unroll
                    for (int g = 0; g < NS; ++g) {
                        constexpr int kChain = 2 / NS;               // slabs of 16 columns under one scale
                        const int p = (im * TN + in) * NS + g;       // chain p; chain p - 1 is scaled beside it
                        b[p & 1] = floatx16{};
                        sc[p & 1] = dsc[g][n];
#pragma unroll
                        for (int s = g * kChain; s < (g + 1) * kChain; ++s)
#pragma unroll
                            for (int c = 2; c >= 0; --c)
                                b[p & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[s][c], wf[s][0], b[p & 1], 0, 0, 0);
                        if (p > 0) {
                            const int o = (p - 1) / NS;
#pragma unroll
                            for (int r = 0; r < 16; ++r)
                                acc[o / TN][o % TN][r] =
                                    __builtin_fmaf(sc[(p - 1) & 1], b[(p - 1) & 1][r], acc[o / TN][o % TN][r]);
                        }
#pragma unroll
                        for (int i = 0; i < 3 * kChain; ++i) {
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                       // one MFMA,
                            __builtin_amdgcn_sched_group_barrier(0x002, 16 / (3 * kChain) + 1, 0);   // then VALU
                        }
                    }
                }
            }
        }
        if constexpr (W::kScaled) {
            constexpr int p = TM * TN * NS - 1;
#pragma unroll
            for (int r = 0; r < 16; ++r)
                acc[TM - 1][TN - 1][r] = __builtin_fmaf(sc[p & 1], b[p & 1][r], acc[TM - 1][TN - 1][r]);
        }
        if constexpr (NM > 0) {
            if ((k0 & 255) == 256 - kK) {   // the super-block's offsets: one more slab of 16 (or 8 and 8 zeros)
#pragma unroll
                for (int in = 0; in < TN; ++in) {
                    const int n = nw + 32 * in + i32;
                    bf16x8 wf = {};
                    if (NM == 16 || h == 0) wf = frag(&wm[n * NM + (NM == 16 ? 8 * h : 0)]);
                    const float dm = dmn[n];
#pragma unroll
                    for (int im = 0; im < TM; ++im) {
                        floatx16 b = {};
#pragma unroll
                        for (int c = 2; c >= 0; --c) {
                            bf16x8 xg = {};
                            if (NM == 16 || h == 0)
                                xg = frag(&xm[c][(mw + 32 * im + i32) * NM + (NM == 16 ? 8 * h : 0)]);
                            b = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xg, wf, b, 0, 0, 0);
                        }
#pragma unroll
                        for (int r = 0; r < 16; ++r) acc[im][in][r] = __builtin_fmaf(dm, b[r], acc[im][in][r]);
                    }
                }
            }
        }
        __syncthreads();
    }

    // D layout: lane (h, i32) holds rows 8 (r / 4) + 4 h + r % 4 of column i32
    float* const Y = a.y[sg];
    const size_t ldy = a.ldy[sg];
    float* const P = a.nsplit > 1 ? a.part + (size_t)z * a.m * a.ntot + a.noff[sg] : nullptr;
#pragma unroll
    for (int im = 0; im < TM; ++im)
#pragma unroll
        for (int in = 0; in < TN; ++in) {
            const int n = n0 + nw + 32 * in + i32;
            if (n >= N) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + mw + 32 * im + 8 * (r >> 2) + 4 * h + (r & 3);
                if (m >= a.m) continue;
                const float v = W::kScaled ? acc[im][in][r] : acc[im][in][r] * kXUnscale;
                if (P) {
                    P[(size_t)m * a.ntot + n] = v;
                } else {
                    float* p = Y + (size_t)m * ldy + n;
                    *p = a.add ? *p + v : v;
                }
            }
        }
}

// The tile shapes.  128 x 256 expands fewest values per output and wins full
// grids (14336 x 4096 x 1024: Q8_0 388 us against 449 and 461 of 64 x 128 and
// 64 x 256, Q6_K 477 / 570 / 619), but with super-block offsets its 256
// registers a lane do not hold the slices (Q4_K 922 / 550 / 543), so those types
// have the first three; 32 x 128 is for few rows (1000 x 2304 x 37: 15.0 against
// 16.5) and 64 x 128 for what leaves CUs idle otherwise.
struct Shape {
    int bm, bn;
    float alone, step;   // us of a K step of one workgroup: a CU to itself; its share of a full CU (Q8_0, measured)
};
constexpr Shape kShapes[4] = {{32, 128, 0.66f, 0.35f}, {64, 128, 0.82f, 0.47f}, {64, 256, 1.25f, 0.92f},
                              {128, 256, 1.85f, 1.45f}};
constexpr bool has_offsets(int type) { return type == L3P_Q2_K || type == L3P_Q4_K || type == L3P_Q5_K; }

template <int QT>
void launch_type(const GemmArgs& a, int shape, int grid, hipStream_t st) {
    switch (shape) {
    case 0: launch_kernel(gemm_split_kernel<QT, 32, 128, 1, 4>, dim3(grid), dim3(256), 0u, st, a); break;
    case 1: launch_kernel(gemm_split_kernel<QT, 64, 128, 2, 3>, dim3(grid), dim3(256), 0u, st, a); break;
    case 2: launch_kernel(gemm_split_kernel<QT, 64, 256, 2, 2>, dim3(grid), dim3(256), 0u, st, a); break;
    default:
        if constexpr (!has_offsets(QT))
            launch_kernel(gemm_split_kernel<QT, 128, 256, 2, 2>, dim3(grid), dim3(256), 0u, st, a);
    }
}

int unit_of(int type) { return has_offsets(type) ? 256 : kK; }

}  // namespace

bool gemm_split_supported(int type) { return gemm_mfma_supported(type) && type != L3P_F32; }

GemmPlan gemm_split_plan(const GemmJob& j, size_t ws_floats) {
    GemmPlan best;
    float best_us = 1e30f;
    const int unit = unit_of(j.type), units = (j.k + unit - 1) / unit, cus = device_cus();
    size_t ntot = 0;
    for (int i = 0; i < j.nseg; ++i) ntot += j.seg[i].n;
    // l3p_gemm_static takes the shapes whose fp32 plan fits its array, with
    // l3p_gemm's values: for them the partials of this plan fit it too
    if (ws_floats > kGemmStaticScratchFloats && gemm_plan(j, ws_floats).partial_floats <= kGemmStaticScratchFloats)
        ws_floats = kGemmStaticScratchFloats;
    for (int s = 0; s < (has_offsets(j.type) ? 3 : 4); ++s) {
        const Shape& sh = kShapes[s];
        long tiles = 0;
        for (int i = 0; i < j.nseg; ++i) tiles += (j.seg[i].n + sh.bn - 1) / sh.bn;
        tiles *= (j.m + sh.bm - 1) / sh.bm;
        for (int z = 1; z <= 32 && z <= units; ++z) {
            const int run = (units + z - 1) / z, runs = (units + run - 1) / run;   // no empty run
            if (runs != z) continue;
            const size_t partial = z > 1 ? (size_t)z * j.m * ntot : 0;
            if (partial > ws_floats) break;
            // Runs of types with offsets have two super-blocks or more: one is
            // faster still (Q5_K 512 x 512 x 11: 12.1 us, two 16.5, fp32 20.5), but
            // its rounding turns a near-tie of the small Q5_K model's greedy decode
            // the other way than the reference.
            if (z > 1 && has_offsets(j.type) && run < 2) break;
            const float n = (float)((tiles * z + cus - 1) / cus);   // workgroups a CU runs
            float us = std::max(sh.alone, n * sh.step) * (float)(run * (unit / kK));
            if (z > 1) us += 3.0f + 0.1f * z + (float)partial * 8.0f / 6e6f;   // write, read and one more launch
            if (us < best_us) {
                best_us = us;
                best.shape = s;
                best.nsplit = z;
                best.ksteps = run * (unit / kK);
                best.partial_floats = partial;
            }
        }
    }
    return best;
}

void launch_gemm_split(const GemmJob& j, const GemmPlan& plan, float* ws, hipStream_t st) {
    L3P_REQUIRE(gemm_split_supported(j.type), L3P_E_UNSUPPORTED, "gemm: type %d has no split path", j.type);
    L3P_REQUIRE(plan.nsplit == 1 || ws, L3P_E_INVALID, "gemm: split-K plan without a workspace");
    L3P_REQUIRE(j.k % kK == 0 && j.ldx % 4 == 0 && ((uintptr_t)j.x & 15) == 0, L3P_E_INVALID,
                "gemm: x rows must be 16-byte aligned");
    L3P_REQUIRE(j.m <= 65535 * 64, L3P_E_INVALID, "gemm: batch %d too large", j.m);
    L3P_REQUIRE(j.nseg >= 1 && j.nseg <= 3, L3P_E_INVALID, "gemm: %d segments", j.nseg);
    const Shape& sh = kShapes[plan.shape];
    GemmArgs a{};
    int tiles = 0, ntot = 0;
    for (int i = 0; i < j.nseg; ++i) {
        if (j.seg[i].n == 0) continue;
        a.w[a.nseg] = j.seg[i].w;
        a.y[a.nseg] = j.seg[i].y;
        a.ldy[a.nseg] = j.seg[i].ldy;
        a.n[a.nseg] = j.seg[i].n;
        a.noff[a.nseg] = ntot;
        a.tbeg[a.nseg] = tiles;
        tiles += (j.seg[i].n + sh.bn - 1) / sh.bn;
        ntot += j.seg[i].n;
        ++a.nseg;
    }
    if (j.m == 0 || a.nseg == 0) return;
    a.tbeg[a.nseg] = tiles;
    a.rb = type_row_bytes(j.type, j.k);
    a.k = j.k;
    a.m = j.m;
    a.x = j.x;
    a.ldx = j.ldx;
    a.add = j.add ? 1 : 0;
    a.ntot = ntot;
    a.ksteps = plan.ksteps;
    a.nsplit = plan.nsplit;
    a.bn = sh.bn;
    a.part = a.nsplit > 1 ? ws : nullptr;
    // every K run must hold at least one step: the kernel's loads start before its loop
    L3P_REQUIRE(plan.ksteps > 0 && (long)(plan.nsplit - 1) * plan.ksteps * kK < j.k, L3P_E_INVALID,
                "gemm: plan of %d runs of %d steps for %d columns", plan.nsplit, plan.ksteps, j.k);
    const long grid = (long)tiles * ((j.m + sh.bm - 1) / sh.bm) * plan.nsplit;
    L3P_REQUIRE(grid < (1L << 31), L3P_E_INVALID, "gemm: %ld workgroups", grid);
    switch (j.type) {
    case L3P_Q8_0: launch_type<L3P_Q8_0>(a, plan.shape, (int)grid, st); break;
    case L3P_Q2_K: launch_type<L3P_Q2_K>(a, plan.shape, (int)grid, st); break;
    case L3P_Q3_K: launch_type<L3P_Q3_K>(a, plan.shape, (int)grid, st); break;
    case L3P_Q4_K: launch_type<L3P_Q4_K>(a, plan.shape, (int)grid, st); break;
    case L3P_Q5_K: launch_type<L3P_Q5_K>(a, plan.shape, (int)grid, st); break;
    case L3P_Q6_K: launch_type<L3P_Q6_K>(a, plan.shape, (int)grid, st); break;
    case L3P_F16: launch_type<L3P_F16>(a, plan.shape, (int)grid, st); break;
    default: launch_type<L3P_BF16>(a, plan.shape, (int)grid, st); break;
    }
    if (a.nsplit > 1) launch_gemm_reduce(a, st);
}
