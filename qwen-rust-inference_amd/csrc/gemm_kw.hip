// Projections of few to a few hundred tokens on gfx950: Y[M, N] = X[M, K]
// W[N, K]^T to fp32 accuracy, with K split over the 4 waves of a block.
//
// X comes as the three BF16 planes of its values in MFMA fragment order (P3,
// common.h); W as its planes (prepared matrices) or in its own format (fp32,
// packed BF16, int8 with row scales), split or widened in registers. The part
// products are those of the prefill GEMM: six per fp32 weight, three per BF16
// or int8 weight (x2 w, x1 w, x0 w), int8 rows scaled after the sum.
//
// A 128 x 128 or 128 x 256 tile leaves most CUs idle at these sizes (a down
// projection of 128 tokens has 8 such tiles), and cutting K into chunks over
// blocks costs partials in memory and a second launch. Here a block owns a
// small output tile over the whole K: wave w takes the 16-deep k tiles w, w +
// 4, ..., its operands straight from L2 / HBM into registers (a fragment is
// one 16-byte load per lane, 1 KiB contiguous per wave; the next k tile's in
// flight while one is multiplied), and the four partial tiles are added in
// wave order through LDS: no staging, no barrier in the loop, one launch,
// results independent of timing.
//
// What bounds it: the CU's 64 bytes per clock from L2 beside the MFMAs. Per k
// tile a 64 x 64 tile moves 12 KiB for 24 MFMAs of fp32 weights (192 clocks
// either way), a 32 x 32 tile 6 KiB for 6 MFMAs; weights read from HBM or
// resident in the caches, in any k order, take the same time. A block's time
// hardly depends on how many run beside it, so the tile is the smallest of at
// most 256 blocks (pick_tile); of a launch of more, two blocks run on a CU.
//
// Measured (one call, weights cold, launch included; before: the prefill GEMM
// of gemm_p3.hip over planes, or gemm_bf3_kernel under 64 tokens and for
// matrices without planes):
//   GLU 2 x 3584 x 1024, fp32 planes: 23 tokens 70.1 -> 13.7 us, 128 tokens 25.3 -> 16.9
//   GLU, BF16 plane: 23 tokens 54.1 -> 7.1 us, 128 tokens 22.7 -> 10.3, 512 tokens 38.0 -> 28.5
//   GLU, int8 without a plane, 128 tokens: 59.5 -> 12.3 us
//   down 1024 x 3584, fp32 planes: 23 tokens 24.7 -> 12.0 us, 128 tokens 22.0 -> 12.8
//   q|k|v 5120 x 1024, 128 tokens: fp32 planes 17.1 -> 12.0 us, BF16 19.4 -> 8.6
#include <type_traits>

#include "common.h"

namespace qr {
namespace {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Waves per block. Two blocks of four share a CU (their registers and LDS allow
// it), so a launch of a few more tiles than CUs runs on: against one block of
// eight waves, 130 column tiles at 128 tokens 28.1 -> 23.8 us (fp32) and 16.5 ->
// 13.4 (BF16), the BF16 GLU of 512 tokens 34.9 -> 29.6, one round the same.
constexpr int NW = 4;

// One launch: up to kKwItems matrices of one X (their column tiles in order).
struct KwArgs {
    const __bf16* xp;
    const float* x;  // X itself (read for the few-row matrices only)
    int M, kt, tiles_m, tiles_n, count;  // kt: K / 16
    struct Item {
        float* y;
        const void* w;
        const float* scale;  // int8 row scales
        int rows, first;     // first column tile
        int raw;             // w in its own format (else planes)
    } it[kKwItems];
    // GLU: it[0] gate, it[1] up (rows of one), y the product
    __bf16* planes;  // the product's planes, or null
};

__device__ __forceinline__ void split3(float v, bf16x8 (&h)[3], int e) {
    const __bf16 h0 = __bf16(v);
    const float r1 = v - float(h0);
    const __bf16 h1 = __bf16(r1);
    h[0][e] = h0;
    h[1][e] = h1;
    h[2][e] = __bf16(r1 - float(h1));
}

template <WeightType T>
constexpr int kPlanes = T == WeightType::F32 ? 3 : 1;

// A lane's 8 consecutive k of one weight row, as loaded.
template <WeightType T, bool RAW>
struct WReg {
    bf16x8 h[kPlanes<T>];
};
template <>
struct WReg<WeightType::F32, true> {
    f4v lo, hi;
};
template <>
struct WReg<WeightType::I8, true> {
    uint2 v;
};

// The lane's operand from address `p` (planes: its 16 bytes of plane 0, the
// planes one KiB apart; raw: the 8 values).
template <WeightType T, bool RAW>
__device__ __forceinline__ void wload(WReg<T, RAW>& r, const char* p) {
    if constexpr (RAW && T == WeightType::F32) {
        r.lo = *reinterpret_cast<const f4v*>(p);
        r.hi = *reinterpret_cast<const f4v*>(p + 16);
    } else if constexpr (RAW && T == WeightType::I8) {
        r.v = *reinterpret_cast<const uint2*>(p);
    } else {
#pragma unroll
        for (int q = 0; q < kPlanes<T>; ++q) r.h[q] = *reinterpret_cast<const bf16x8*>(p + 1024 * q);
    }
}
// Plane q alone (planes only).
template <WeightType T>
__device__ __forceinline__ void wload_plane(WReg<T, false>& r, const char* p, int q) {
    r.h[q] = *reinterpret_cast<const bf16x8*>(p + 1024 * q);
}
template <WeightType T, bool RAW>
__device__ __forceinline__ void wplanes(const WReg<T, RAW>& r, bf16x8 (&h)[kPlanes<T>]) {
    if constexpr (RAW && T == WeightType::F32) {
#pragma unroll
        for (int e = 0; e < 8; ++e) split3(e < 4 ? r.lo[e] : r.hi[e - 4], h, e);
    } else if constexpr (RAW && T == WeightType::I8) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const unsigned w = e < 4 ? r.v.x : r.v.y;
            h[0][e] = __bf16(float(int(w << (24 - 8 * (e & 3))) >> 24));
        }
    } else {
#pragma unroll
        for (int q = 0; q < kPlanes<T>; ++q) h[q] = r.h[q];
    }
}
// Bytes of one raw weight.
template <WeightType T>
constexpr int kRawBytes = T == WeightType::F32 ? 4 : T == WeightType::BF16 ? 2 : 1;

// The part products of an X operand (three planes) and a W operand, from the
// smallest: product q is x_P(q) w_Q(q), after which plane xdead(q) of X and
// wdead(q) of W (-1: none) are not used again in the step.
template <WeightType T>
struct Products {
    static constexpr int N = 3;
    static constexpr int P(int q) { return 2 - q; }
    static constexpr int Q(int) { return 0; }
    static constexpr int xdead(int q) { return 2 - q; }
    static constexpr int wdead(int q) { return q == 2 ? 0 : -1; }
};
template <>
struct Products<WeightType::F32> {
    static constexpr int N = 6;
    static constexpr int P(int q) { return q == 0 ? 2 : q < 3 ? 1 : 0; }
    static constexpr int Q(int q) { return q == 1 || q == 4 ? 1 : q == 3 ? 2 : 0; }
    static constexpr int xdead(int q) { return q == 0 ? 2 : q == 2 ? 1 : q == 5 ? 0 : -1; }
    static constexpr int wdead(int q) { return q < 3 ? -1 : 5 - q; }
};

// n steps through a ring of NS (even) register buffers. step(buffer, step % 2,
// next) multiplies a buffer and, for next >= 0, loads step `next` into it plane
// by plane as the products are done with it: loads issued in a burst after the
// products stall the wave (the CU's vector memory path takes 16 clocks per KiB
// and a wave issues in order), among them they do not: q|k|v of 128 fp32 tokens
// 14.5 -> 12.0 us, of 300 25.8 -> 20.7, the BF16 GLU of 128 tokens 11.4 -> 10.3.
// The main loop's loads are unconditional (a join between a path with loads and
// one without would make the compiler wait for more than the buffer it needs).
template <int NS, class Buf, class L, class S>
__device__ __forceinline__ void ring(int n, L&& load, S&& step) {
    Buf b[NS];
#pragma unroll
    for (int i = 0; i < NS; ++i) load(b[i], min(i, n - 1));
    int s = 0;
    for (; s + 2 * NS <= n; s += NS)
#pragma unroll
        for (int i = 0; i < NS; ++i) step(b[i], i % 2, s + i + NS);
#pragma unroll
    for (int i = 0; i < NS; ++i)
        if (s + i < n) {
            step(b[i], i % 2, -1);
            if (s + i + NS < n) load(b[i], s + i + NS);
        }
    s += NS;
#pragma unroll
    for (int i = 0; i < NS - 1; ++i)
        if (s + i < n) step(b[i], i % 2, -1);
}

// Wave w's k tiles (w, w + NW, ...) of a (32 TMT) x (32 TNT) tile into acc. xb
// / wb: this lane's address of each 32-row tile's k tile 0. The leading products
// x0 w0 sum in accumulators of their own, the others, 2^-8 of them and less, in
// `rest`: a sum rounds once per k tile where it counts, not once per product.
// Error against 64 bits, all products of even and all of odd steps in one
// accumulator each -> now: k of 8 fp32 tokens 1.9e-7 -> 1.3e-7 (1.55e-7 with K
// split over the blocks of gemm_bf3_kernel), MLP of 20 fp32 tokens 4.3e-7 ->
// 2.7e-7, of 150 int8 tokens 3.0e-7 -> 2.1e-7; the same time.
template <WeightType T, bool RAW, int TMT, int TNT>
__device__ __forceinline__ void k_wave(f16v (&acc)[TMT][TNT], const char* const (&xb)[TMT], const char* const (&wb)[TNT],
                                       int kt, int w) {
    constexpr int XSTEP = 3 * 1024, WSTEP = RAW ? 16 * kRawBytes<T> : kPlanes<T> * 1024;
    const int n = (kt - w + NW - 1) / NW;
    // buffers that fit 256 VGPRs
    constexpr int NS = TMT * TNT == 4 || (T == WeightType::F32 && TMT == 1 && TNT == 2) ? 2 : 4;
    struct Buf {
        bf16x8 x[TMT][3];
        WReg<T, RAW> w[TNT];
    };
    auto load = [&](Buf& b, int step) {
        const size_t k = size_t(w + NW * step);
#pragma unroll
        for (int j = 0; j < TNT; ++j) wload<T, RAW>(b.w[j], wb[j] + k * WSTEP);
#pragma unroll
        for (int i = 0; i < TMT; ++i)
#pragma unroll
            for (int q = 0; q < 3; ++q) b.x[i][q] = *reinterpret_cast<const bf16x8*>(xb[i] + k * XSTEP + 1024 * q);
    };
    f16v rest[TMT][TNT];
#pragma unroll
    for (int i = 0; i < TMT; ++i)
#pragma unroll
        for (int j = 0; j < TNT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = rest[i][j][r] = 0.f;
    auto step = [&](Buf& b, int, int next) {
        using Pr = Products<T>;
        const size_t k = size_t(w + NW * next);
        bf16x8 h[TNT][kPlanes<T>];
#pragma unroll
        for (int j = 0; j < TNT; ++j) wplanes<T, RAW>(b.w[j], h[j]);
        if (RAW && next >= 0) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < TNT; ++j) wload<T, RAW>(b.w[j], wb[j] + k * WSTEP);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int q = 0; q < Pr::N; ++q) {
#pragma unroll
            for (int i = 0; i < TMT; ++i)
#pragma unroll
                for (int j = 0; j < TNT; ++j) {
                    f16v& a = q + 1 < Pr::N ? rest[i][j] : acc[i][j];
                    a = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b.x[i][Pr::P(q)], h[j][Pr::Q(q)], a, 0, 0, 0);
                }
            if (next < 0) continue;
            __builtin_amdgcn_sched_barrier(0);
            if (Pr::xdead(q) >= 0)
#pragma unroll
                for (int i = 0; i < TMT; ++i)
                    b.x[i][Pr::xdead(q)] =
                        *reinterpret_cast<const bf16x8*>(xb[i] + k * XSTEP + 1024 * Pr::xdead(q));
            if constexpr (!RAW)
                if (Pr::wdead(q) >= 0)
#pragma unroll
                    for (int j = 0; j < TNT; ++j) wload_plane<T>(b.w[j], wb[j] + k * WSTEP, Pr::wdead(q));
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (w < kt) ring<NS, Buf>(n, load, step);
#pragma unroll
    for (int i = 0; i < TMT; ++i)
#pragma unroll
        for (int j = 0; j < TNT; ++j) acc[i][j] += rest[i][j];
}

// Block b's tile: the 8 XCDs take blocks in turn; XCD x takes column tiles x,
// x + 8, ..., the row tiles of one column tile in a row, so a weight tile is
// read from HBM by one XCD. False for the spare blocks.
__device__ __forceinline__ bool kw_block(const KwArgs& p, int& mt, int& nt) {
    const int b = int(blockIdx.x), i = b >> 3;
    mt = i % p.tiles_m;
    nt = i / p.tiles_m * 8 + (b & 7);
    return nt < p.tiles_n;
}
__device__ __forceinline__ int kw_item(const KwArgs& p, int nt) {
    int item = 0;
    while (item + 1 < p.count && nt >= p.it[item + 1].first) ++item;
    return item;
}

// The sum of the waves' partials of 4 consecutive columns.
template <int SLOT>
__device__ __forceinline__ f4v wave_parts(const float* at) {
    f4v s = *reinterpret_cast<const f4v*>(at);
#pragma unroll
    for (int w = 1; w < NW; ++w) s += *reinterpret_cast<const f4v*>(at + w * SLOT);
    return s;
}
// 4 consecutive columns of an output row.
__device__ __forceinline__ void store4(const KwArgs::Item& it, int m, int n, f4v s) {
    if (n >= it.rows) return;
    float* y = it.y + size_t(m) * it.rows + n;
    if (it.rows % 4 == 0 && reinterpret_cast<uintptr_t>(it.y) % 16 == 0) {
        if (it.scale) s *= *reinterpret_cast<const f4v*>(it.scale + n);
        *reinterpret_cast<f4v*>(y) = s;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < it.rows) y[e] = it.scale ? it.scale[n + e] * s[e] : s[e];
    }
}

// 16 tokens of a matrix of at most 16 rows in its own format (the DeltaNet a
// and b, whose outputs set the decay and beta of every token) as whole fp32
// products on v_mfma_f32_16x16x4_f32, X from its fp32 values: the arithmetic of
// gemm_ab_mfma_kernel (gemm.hip) to the bit, so that such a matrix gives the
// same result alone and in a group, and an infinite or very large value stays
// what it is (split into BF16 parts it becomes NaN). Step m is 16 columns, MFMA
// e of it takes k = 16 m + 4 (lane / 16) + e; the even steps of wave w are those
// of wave w there, the odd ones those of wave w + 4, and the eight partial tiles
// are added in that order. A block takes 16 tokens whatever the launch's tile
// (kFewTokens; up to four blocks stand in the place of one tile): with all of a
// 64-token tile in one block these blocks ended last (DeltaNet layer, 77 BF16
// tokens: 65.8 us, now 59.3 as with split products; 128 fp32 tokens: 75.6, now
// 70.4, with split products 72.3).
constexpr int kFewTokens = 16;
template <WeightType T>
__device__ __forceinline__ void few_rows(const KwArgs& p, const KwArgs::Item& it, int m0, float* part) {
    constexpr int B = 16;  // steps in flight (K = 1024: all of a wave's)
    const int lane = int(threadIdx.x) & 63, w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const int lr = lane & 15, g = lane >> 4, K = 16 * p.kt;
    const size_t wr = size_t(min(lr, it.rows - 1)) * K;  // (rows past the matrix or the tokens: not stored)
    const float* const xr = p.x + size_t(min(m0 + lr, p.M - 1)) * K;
    f4v acc[2] = {f4v{0.f, 0.f, 0.f, 0.f}, f4v{0.f, 0.f, 0.f, 0.f}};
    for (int mb = w; mb < p.kt; mb += NW * B) {
        f4v wv[B], xv[B];
#pragma unroll
        for (int j = 0; j < B; ++j) {
            const int k = 16 * min(mb + NW * j, p.kt - 1) + 4 * g;
            xv[j] = *reinterpret_cast<const f4v*>(xr + k);
            if constexpr (T == WeightType::F32) {
                wv[j] = *reinterpret_cast<const f4v*>(static_cast<const float*>(it.w) + wr + k);
            } else if constexpr (T == WeightType::BF16) {
                const uint2 v = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(it.w) + wr + k);
                wv[j] = f4v{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                            __uint_as_float(v.y & 0xffff0000u)};
            } else {
                const unsigned v = *reinterpret_cast<const unsigned*>(static_cast<const int8_t*>(it.w) + wr + k);
                wv[j] = f4v{float(int(v << 24) >> 24), float(int(v << 16) >> 24), float(int(v << 8) >> 24),
                            float(int(v) >> 24)};
            }
        }
#pragma unroll
        for (int j = 0; j < B; ++j)
            if (mb + NW * j < p.kt)  // (a scalar)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    acc[j & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[j][e], wv[j][e], acc[j & 1], 0, 0, 0);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) part[((w + NW * h) * kFewTokens + 4 * g + r) * 16 + lr] = acc[h][r];
    __syncthreads();
    const int m = int(threadIdx.x) / 16, n = int(threadIdx.x) % 16;
    if (m0 + m >= p.M || n >= it.rows) return;
    float s = part[threadIdx.x];
#pragma unroll
    for (int v = 1; v < 2 * NW; ++v) s += part[v * kFewTokens * 16 + threadIdx.x];
    it.y[size_t(m0 + m) * it.rows + n] = it.scale ? it.scale[n] * s : s;
}

// Two waves per SIMD (256 registers each, here and in kw_narrow_kernel) also keep
// the accumulators out of the AGPRs: with 512 registers to a wave the compiler
// moved them there and back at every branch of the ring's end, and one build of
// this kernel gave wrong last sums, as if read before their MFMA had written them.
// GLU = false: a (32 TMT) x (32 TNT) tile of one item. GLU = true (TNT = 2):
// 32 gate rows and the same 32 up rows, product = silu(g) * u and its planes.
template <WeightType T, int TMT, int TNT, bool GLU>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2))) void kw_kernel(KwArgs p) {
    constexpr int TM = 32 * TMT, TN = 32 * TNT, PITCH = TN + 4, SLOT = TM * PITCH;
    __shared__ __attribute__((aligned(16))) float part[NW * SLOT];
    int mt, nt;
    if (!kw_block(p, mt, nt)) return;
    const int tid = int(threadIdx.x), lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int item = GLU ? 0 : kw_item(p, nt);
    const KwArgs::Item& it = p.it[item];
    const int m0 = mt * TM, n0 = GLU ? 32 * nt : TN * (nt - it.first);
    const int kt = p.kt;
    if constexpr (!GLU)
        if (it.raw && it.rows <= kKwFewRows) {
            const int t0 = m0 + kFewTokens * (nt - it.first);
            if (t0 < p.M) few_rows<T>(p, it, t0, part);
            return;
        }
    const char* xb[TMT];
#pragma unroll
    for (int i = 0; i < TMT; ++i)
        xb[i] = reinterpret_cast<const char*>(p.xp) + size_t(mt * TMT + i) * kt * 3072 + 16 * lane;
    f16v acc[TMT][TNT];
    const char* wb[TNT];
    if (!GLU && TNT == 2 && it.raw && it.rows <= 32) {  // half the tile
        const char* wb1[1] = {reinterpret_cast<const char*>(it.w) +
                              (size_t(min(lane & 31, it.rows - 1)) * kt * 16 + 8 * (lane >> 5)) * kRawBytes<T>};
        f16v half[TMT][1];
        k_wave<T, true, TMT, 1>(half, xb, wb1, kt, w);
#pragma unroll
        for (int i = 0; i < TMT; ++i) acc[i][0] = acc[i][TNT - 1] = half[i][0];  // (columns past the matrix: not stored)
    } else if (it.raw) {
#pragma unroll
        for (int j = 0; j < TNT; ++j) {  // rows past the matrix read its last row (not stored)
            const int row = min(n0 + (GLU ? 0 : 32 * j) + (lane & 31), it.rows - 1);
            wb[j] = reinterpret_cast<const char*>(p.it[GLU ? j : item].w) +
                    (size_t(row) * kt * 16 + 8 * (lane >> 5)) * kRawBytes<T>;
        }
        k_wave<T, true, TMT, TNT>(acc, xb, wb, kt, w);
    } else {
#pragma unroll
        for (int j = 0; j < TNT; ++j)
            wb[j] = reinterpret_cast<const char*>(p.it[GLU ? j : item].w) +
                    size_t(n0 / 32 + (GLU ? 0 : j)) * kt * (kPlanes<T> * 1024) + 16 * lane;
        k_wave<T, false, TMT, TNT>(acc, xb, wb, kt, w);
    }
    // register r of lane l in tile (i, j): row 32 i + 8 (r / 4) + 4 (l / 32) + r % 4, column 32 j + l % 32
#pragma unroll
    for (int i = 0; i < TMT; ++i)
#pragma unroll
        for (int j = 0; j < TNT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                part[w * SLOT + (32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * PITCH + 32 * j + (lane & 31)] =
                    acc[i][j][r];
    __syncthreads();
    if constexpr (!GLU) {
#pragma unroll
        for (int o = tid; o < TM * TN / 4; o += 64 * NW) {
            const int m = o / (TN / 4), c = o % (TN / 4) * 4;
            if (m0 + m < p.M) store4(it, m0 + m, n0 + c, wave_parts<SLOT>(part + m * PITCH + c));
        }
    } else {
        for (int o = tid; o < TM * 4; o += 64 * NW) {
            const int m = o / 4, c = o % 4 * 8, n = n0 + c;
            if (m0 + m >= p.M) continue;
            float v[8];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                f4v g = wave_parts<SLOT>(part + m * PITCH + c + 4 * h);
                f4v u = wave_parts<SLOT>(part + m * PITCH + 32 + c + 4 * h);
                if (it.scale) {
                    g *= *reinterpret_cast<const f4v*>(it.scale + n + 4 * h);
                    u *= *reinterpret_cast<const f4v*>(p.it[1].scale + n + 4 * h);
                }
                f4v s;
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e] = v[4 * h + e] = siluf_(g[e]) * u[e];
                *reinterpret_cast<f4v*>(it.y + size_t(m0 + m) * it.rows + n + 4 * h) = s;
            }
            if (p.planes) {
                bf16x8 h[3];
#pragma unroll
                for (int e = 0; e < 8; ++e) split3(v[e], h, e);
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    *reinterpret_cast<bf16x8*>(p.planes + p3_index(m0 + m, n, q, it.rows / 16)) = h[q];
            }
        }
    }
}

// A 32 x 16 tile on v_mfma_f32_16x16x32_bf16 (32-deep k steps): twice the
// blocks of a 32 x 32 tile for the narrow matrices. Lane l holds 8 k values
// (32 s + 8 (l / 16)) of row l % 16 of each operand; register r of its
// accumulator is row 4 (l / 16) + r, column l % 16.
template <WeightType T>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2))) void kw_narrow_kernel(KwArgs p) {
    constexpr int TM = 32, TN = 16, PITCH = TN + 4, SLOT = TM * PITCH;
    constexpr int WP = kPlanes<T>;
    __shared__ __attribute__((aligned(16))) float part[NW * SLOT];
    int mt, nt;
    if (!kw_block(p, mt, nt)) return;
    const int tid = int(threadIdx.x), lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const KwArgs::Item& it = p.it[kw_item(p, nt)];
    const int m0 = mt * TM, n0 = TN * (nt - it.first), kt = p.kt, steps = kt / 2;
    // fragment lane of row r16 (of 16) and this lane's k: r16 + 32 ((l / 16) % 2), k tile l / 32 of the step
    const int fl = (lane & 15) + 32 * ((lane >> 4) & 1), fk = lane >> 5;
    const char* xb = reinterpret_cast<const char*>(p.xp) + (size_t(mt) * kt + fk) * 3072 + 16 * fl;
    // [row half][the leading product of even and of odd steps, the other products]: as in k_wave, and
    // the leading chain half as long (this tile takes the matrices of the longest K)
    f4v acc[2][3];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][0][r] = acc[i][1][r] = acc[i][2][r] = 0.f;
    auto run = [&](auto raw, const char* wb) {
        constexpr bool RAW = decltype(raw)::value;
        constexpr int WSTEP = RAW ? 32 * kRawBytes<T> : 2 * WP * 1024;
        struct Buf {
            bf16x8 x[2][3];
            WReg<T, RAW> w;
        };
        auto load = [&](Buf& b, int step) {
            const size_t s = size_t(w + NW * step);
            wload<T, RAW>(b.w, wb + s * WSTEP);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    b.x[i][q] = *reinterpret_cast<const bf16x8*>(xb + s * 6144 + 1024 * q + 256 * i);
        };
        auto step = [&](Buf& b, int parity, int next) {
            using Pr = Products<T>;
            const size_t s = size_t(w + NW * next);
            bf16x8 h[WP];
            wplanes<T, RAW>(b.w, h);
            if (RAW && next >= 0) {
                __builtin_amdgcn_sched_barrier(0);
                wload<T, RAW>(b.w, wb + s * WSTEP);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int q = 0; q < Pr::N; ++q) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    f4v& a = acc[i][q + 1 < Pr::N ? 2 : parity];
                    a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b.x[i][Pr::P(q)], h[Pr::Q(q)], a, 0, 0, 0);
                }
                if (next < 0) continue;
                __builtin_amdgcn_sched_barrier(0);
                if (Pr::xdead(q) >= 0)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        b.x[i][Pr::xdead(q)] =
                            *reinterpret_cast<const bf16x8*>(xb + s * 6144 + 1024 * Pr::xdead(q) + 256 * i);
                if constexpr (!RAW)
                    if (Pr::wdead(q) >= 0) wload_plane<T>(b.w, wb + s * WSTEP, Pr::wdead(q));
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        if (w < steps) ring<4, Buf>((steps - w + NW - 1) / NW, load, step);
    };
    if (it.raw) {
        const int row = min(n0 + (lane & 15), it.rows - 1);
        run(std::true_type{}, reinterpret_cast<const char*>(it.w) + (size_t(row) * kt * 16 + 8 * (lane >> 4)) * kRawBytes<T>);
    } else {
        run(std::false_type{}, reinterpret_cast<const char*>(it.w) + (size_t(n0 / 32) * kt + fk) * (WP * 1024) +
                         16 * (fl + (n0 & 16)));
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            part[w * SLOT + (16 * i + 4 * (lane >> 4) + r) * PITCH + (lane & 15)] =
                acc[i][0][r] + (acc[i][1][r] + acc[i][2][r]);
    __syncthreads();
    if (tid < TM * TN / 4) {
        const int m = tid / (TN / 4), c = tid % (TN / 4) * 4;
        if (m0 + m < p.M) store4(it, m0 + m, n0 + c, wave_parts<SLOT>(part + m * PITCH + c));
    }
}

// Output tile of a block, tokens x weight rows (the GLU: 32 gate and the same
// 32 up rows, k64x64 or k32x64).
enum Tile { k64x64, k64x32, k32x64, k32x32, k32x16 };
constexpr int tile_m(Tile t) { return t == k64x64 || t == k64x32 ? 64 : 32; }
constexpr int tile_n(Tile t) { return t == k64x64 || t == k32x64 ? 64 : t == k32x16 ? 16 : 32; }

template <WeightType T>
int launch(hipStream_t s, Tile tile, bool glu, const KwArgs& a) {
    const dim3 grid{unsigned(ceil_div(a.tiles_n, 8)) * 8u * unsigned(a.tiles_m)}, block{64u * NW};
    if (glu) {
        if (tile == k64x64)
            hipLaunchKernelGGL((kw_kernel<T, 2, 2, true>), grid, block, 0, s, a);
        else
            hipLaunchKernelGGL((kw_kernel<T, 1, 2, true>), grid, block, 0, s, a);
    } else {
        switch (tile) {
        case k64x64: hipLaunchKernelGGL((kw_kernel<T, 2, 2, false>), grid, block, 0, s, a); break;
        case k64x32: hipLaunchKernelGGL((kw_kernel<T, 2, 1, false>), grid, block, 0, s, a); break;
        case k32x64: hipLaunchKernelGGL((kw_kernel<T, 1, 2, false>), grid, block, 0, s, a); break;
        case k32x32: hipLaunchKernelGGL((kw_kernel<T, 1, 1, false>), grid, block, 0, s, a); break;
        case k32x16: hipLaunchKernelGGL((kw_narrow_kernel<T>), grid, block, 0, s, a); break;
        }
    }
    return int(hipGetLastError());
}
int launch_t(hipStream_t s, WeightType t, Tile tile, bool glu, const KwArgs& a) {
    switch (t) {
    case WeightType::F32: return launch<WeightType::F32>(s, tile, glu, a);
    case WeightType::BF16: return launch<WeightType::BF16>(s, tile, glu, a);
    case WeightType::I8: return launch<WeightType::I8>(s, tile, glu, a);
    }
    return int(hipErrorInvalidValue);
}

long blocks_of(const KwItem* items, int n, int M, Tile t) {
    long cols = 0;
    for (int i = 0; i < n; ++i) cols += ceil_div(items[i].rows, tile_n(t));
    return cols * ceil_div(M, tile_m(t));
}
// The smallest tile of at most 256 blocks (one per CU), else 64 x 64. fp32
// weights in their own format are split in the kernel, once per 32 x 16
// operand: 64 x 32 splits half as many as 32 x 64 (down, 300 tokens: 28.8
// against 34.5 us). The 32 x 16 tile is for matrices of a width worth
// spreading (few_rows runs in the wider ones). Every other tile forms the same
// sums to the bit; in this one a K step is twice as deep and they round
// differently, so a matrix of 128 rows or more may differ in its last bits
// between a call of its own and a group that makes more than 256 such tiles.
Tile pick_tile(WeightType t, const KwItem* items, int n, int M) {
    bool narrow = true;
    for (int i = 0; i < n; ++i) narrow = narrow && items[i].rows >= 128;
    const Tile middle = t == WeightType::F32 && items[0].raw ? k64x32 : k32x64;
    for (Tile c : {k32x16, k32x32, middle})
        if ((c != k32x16 || narrow) && blocks_of(items, n, M, c) <= 256) return c;
    return k64x64;
}

}  // namespace

// Up to kKwMaxTokens tokens, and while the 64 x 64 tiles number at most 640
// (three planes; against the prefill GEMM's 128 x 256 tiles: 560 of the GLU at
// 300 tokens 35.1 against 41.9 us, 640 of q|k|v at 512 tokens 31.1 against
// 39.7, 1024 of 8192 rows at 512 tokens 54 against 48) or 1152 (one plane, or
// no planes at all: 896 of the GLU at 512 tokens 28.5 against 38.0 us; with
// one accumulator chain and burst loads 1792 of them took 82 against 57).
bool kw_wanted(WeightType t, bool raw, int M, int rows) {
    const long tiles = long(ceil_div(M, 64)) * long(ceil_div(rows, 64));
    return M <= kKwMaxTokens && (M <= 64 || tiles <= (t == WeightType::F32 && !raw ? 640 : 1152));
}

bool kw_raw_ok(WeightType t, const void* a, int rows, int cols) {
    return p3_cols_ok(cols) && reinterpret_cast<uintptr_t>(a) % 16 == 0 && (t != WeightType::I8 || rows % 2 == 0);
}

int kw_gemm(hipStream_t s, WeightType t, const KwItem* items, int n, const __bf16* xp, const float* x, int M, int K) {
    if (M < 1 || n < 1 || n > kKwItems || !p3_cols_ok(K) || reinterpret_cast<uintptr_t>(x) % 16)
        return int(hipErrorInvalidValue);
    for (int i = 0; i < n; ++i)
        if (items[i].rows < 1 || reinterpret_cast<uintptr_t>(items[i].scale) % 16 ||
            (kw_few_rows(items[i]) ? x == nullptr : xp == nullptr))
            return int(hipErrorInvalidValue);
    const Tile tile = pick_tile(t, items, n, M);
    KwArgs a{};
    a.xp = xp;
    a.x = x;
    a.M = M;
    a.kt = K / 16;
    a.tiles_m = int(ceil_div(M, tile_m(tile)));
    a.count = n;
    for (int i = 0; i < n; ++i) {
        a.it[i] = KwArgs::Item{items[i].y, items[i].w, items[i].scale, items[i].rows, a.tiles_n, items[i].raw ? 1 : 0};
        a.tiles_n += kw_few_rows(items[i]) ? tile_m(tile) / kFewTokens : int(ceil_div(items[i].rows, tile_n(tile)));
    }
    return launch_t(s, t, tile, false, a);
}

int kw_glu(hipStream_t s, WeightType t, float* product, __bf16* planes, const KwItem& gate, const KwItem& up,
           const __bf16* xp, int M, int K) {
    if (M < 1 || gate.rows < 32 || gate.rows % 32 != 0 || gate.rows != up.rows || gate.raw != up.raw ||
        !p3_cols_ok(K) || !gate.scale != !up.scale ||
        (reinterpret_cast<uintptr_t>(product) | reinterpret_cast<uintptr_t>(gate.scale) |
         reinterpret_cast<uintptr_t>(up.scale)) % 16)
        return int(hipErrorInvalidValue);
    // one plane: 32-token tiles also past one round of 64-token ones (300 tokens 25 against 29 us with burst loads)
    const long cols = gate.rows / 32, small = cols * ceil_div(M, 32), large = cols * ceil_div(M, 64);
    const Tile tile = small <= 256 || (large > 256 && t != WeightType::F32 && !gate.raw) ? k32x64 : k64x64;
    KwArgs a{};
    a.xp = xp;
    a.M = M;
    a.kt = K / 16;
    a.tiles_m = int(ceil_div(M, tile_m(tile)));
    a.tiles_n = int(cols);
    a.count = 1;
    a.it[0] = KwArgs::Item{product, gate.w, gate.scale, gate.rows, 0, gate.raw ? 1 : 0};
    a.it[1] = KwArgs::Item{product, up.w, up.scale, up.rows, 0, up.raw ? 1 : 0};
    a.planes = planes;
    return launch_t(s, t, tile, true, a);
}

}  // namespace qr
