// gfx950 (CDNA4) kernels of the weight-only quantized GEMV path, plus their
// launch-shape selection.
//
// Semantics follow the reference operator contracts
// (kernels/int4gemv/int4gemv_common.h:1-79 for INT4,
//  kernels/qgemv/qgemv_common.h:1-55 for INT8): FP32 accumulation, one
// round-to-nearest-even cast to fp16 per output row, fp16 subnormals kept
// (the library is never built with fast-math or flush-to-zero).
//
// Two kernel families per operator:
//
// * scalar (`*_scalar_kernel`): 16-byte loads of any alignment, any k,
//   per-element dequant `fma(q*s, x, acc)`, DPP wave reduction, LDS across
//   the waves that share a row.  It is the single source for the *_baseline
//   variants and for every fallback (bit-identity of fallback and baseline
//   follows from that and from a plan that depends on the sizes alone).
//
// * wave (`*_wave_kernel<CW, J, R>`): the CDNA4 design.
//   - Lanes of a wave64 are split into 64/CW row slots of CW lanes; lane
//     (slot, col) owns the 16-byte weight chunks col, col+CW, ...,
//     col+CW*(J-1) of every row it handles, so one wave load instruction
//     reads CW*16 contiguous bytes of each of 64/CW rows (fully coalesced).
//   - Each lane handles R rows; all R*J weight loads are issued before any
//     arithmetic, so a whole row tile is in flight at once (HBM latency is
//     the limiter for these short kernels).
//   - The lane's x values for its J chunks are loaded once and kept in
//     registers as fp16 pairs, reused across its R rows.
//   - Nibbles become fp16 with one v_bitop3 per pair:
//       ((w & 0x000F000F) ^ 0x64086408) is the fp16 pair (1032+q0, 1032+q4)
//     (4-bit two's complement q, xor 8 maps it to q+8, 0x6400 is 1024), and
//     one packed fp16 add of -1032 gives (q0, q4) exactly.  The nibbles at
//     bits 4-7 are taken in place as 16*q ((w & 0x00F000F0) ^ 0x64806480,
//     bias -1152) and their partial sum is scaled by 1/16 (exact).
//   - Products and sums use v_dot2_f32_f16 (fp16 x fp16 products are exact
//     in FP32, accumulation in FP32); the group scale is applied once per
//     16-byte chunk (one chunk lies inside one 128-element group).
//   - Cross-lane reduction uses DPP (quad_perm, row mirrors, row_bcast15/31)
//     with no LDS and no barrier; the last lane of each row segment writes.
//   INT8 uses the same structure with 16 int8 per chunk:
//       ((w & 0x00FF00FF) ^ 0x64806480) - 1152 = (q0, q2) as fp16,
//   and the per-row scale applied once after the reduction.
//
// Every wave-kernel summation order is a legal FP32 order under the
// reference's accumulation-error bound (at most three FP32 roundings per
// term: the dot2 rounding, the scale product, the accumulate).

#include "cq_internal.h"

#include <hip/hip_ext.h>

#include <algorithm>
#include <climits>
#include <cstring>
#include <type_traits>

namespace cq {
namespace {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr int kBlock = 256;  // threads per workgroup for every kernel

__device__ __forceinline__ float h2f(uint16_t bits) {
    return static_cast<float>(__builtin_bit_cast(_Float16, bits));
}

__device__ __forceinline__ uint16_t f2h(float v) {
    // v_cvt_f16_f32: round to nearest even, fp16 subnormals kept.
    return __builtin_bit_cast(uint16_t, static_cast<_Float16>(v));
}

__device__ __forceinline__ f16x2 as_f16x2(uint32_t bits) {
    return __builtin_bit_cast(f16x2, bits);
}

// v + (v moved by a DPP pattern).  Lanes of rows outside ROW_MASK receive
// +0, which leaves their value unchanged.
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ float dpp_plus(float v) {
    const int moved = __builtin_amdgcn_update_dpp(
        0, __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xF, false);
    return v + __builtin_bit_cast(float, moved);
}

// Sum over aligned segments of SEG lanes (16, 32 or 64).  The total is
// exact in the last lane of every segment (lane % SEG == SEG - 1).
template <int SEG>
__device__ __forceinline__ float segment_sum(float v) {
    v = dpp_plus<0xB1>(v);   // quad_perm [1,0,3,2]: pairs
    v = dpp_plus<0x4E>(v);   // quad_perm [2,3,0,1]: quads
    v = dpp_plus<0x141>(v);  // row_half_mirror: 8 lanes
    v = dpp_plus<0x140>(v);  // row_mirror: 16 lanes
    if constexpr (SEG >= 32) v = dpp_plus<0x142, 0xA>(v);  // row_bcast15
    if constexpr (SEG >= 64) v = dpp_plus<0x143, 0xC>(v);  // row_bcast31
    return v;
}

// Workgroups of a launch are dealt round-robin to the 8 XCDs (workgroup i
// runs on XCD i % 8), and each XCD has its own L2.  This returns a logical
// block index under which every XCD takes runs of RUN consecutive logical
// blocks, the eight XCDs one run each side by side, so that neighbouring rows
// (their scale and y lines) stay in one L2 while all XCDs together walk
// through one region of the weights.  What is left past the last whole set of
// runs is split into one run per XCD.  It is a bijection on [0, gridDim.x)
// for any grid size, so it changes which workgroup computes a row, never
// how the row is computed (outputs are bit-identical to the identity
// mapping).  Against one contiguous range of rows per XCD, where the eight
// XCDs read eight far-apart regions at once (us per call, HBM-cold, runs of
// 32): INT8 8192^2 13.5 -> 12.0, INT4 8192^2 8.1 -> 7.5, INT8 11008x4096 9.05
// -> 8.4, INT4 32000x4096 13.3 -> 12.4; launches under 10 MB level.  Runs of
// 8 and 64 are up to 3% slower than 32 in places.  Where waves hold at most
// two chunks per lane, runs of 64: such a launch of 512 workgroups is over in
// 3.4 us and 1-3% slower with runs of 32 (INT4 4096^2).  The INT8 K-tiled
// kernel keeps one run per XCD (4096x28672 20.7 us against 20.9).
// So do the FP16/FP32 kernels, for the first pass over weights not read
// before: FP16 32000x4096 57.5 us against 66.2 with runs of 32, FP32
// 4096x11008 43.0 against 50.6 (why was not established).  Later passes pay
// for it at most sizes, one run against runs of 32 (us per call from a graph):
// FP16 4096^2 7.20, 6.90; 11008x4096 16.4, 16.1; 32000x4096 43.9, 42.9;
// 4096x11008 17.2, 17.4; FP32 4096^2 13.1, 12.9; 5120x1600 6.90, 6.63;
// 4096x11008 33.3, 33.7; rows of 14000 elements and more level.
constexpr uint32_t kXcdRun = 32;
constexpr uint32_t kXcdAll = 1u << 24;   // one run per XCD
// Run for waves that load `chunks` 16-byte chunks per lane in all.
constexpr uint32_t xcd_run(int chunks) { return chunks <= 2 ? 64 : kXcdRun; }
template <uint32_t RUN = kXcdRun>
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t g) {
    constexpr uint32_t kXcds = 8, kSpan = kXcds * RUN;
    const uint32_t base = b / kSpan * kSpan, xcd = b % kXcds;
    const uint32_t span = min(g - base, kSpan);   // or what is left
    return base + xcd * (span / kXcds) + min(xcd, span % kXcds) + (b - base) / kXcds;
}
template <uint32_t RUN = kXcdRun>
__device__ __forceinline__ uint32_t xcd_block() { return xcd_block<RUN>(blockIdx.x, gridDim.x); }

// ---------------------------------------------------------------- scalar
//
// The kernels of the *_baseline variants and of every call that misses the
// vector contract (any alignment, any k): per-element arithmetic, as the
// reference's scalar kernels define it (INT4/INT8 fma(float(q) * s, x, acc),
// FP16/FP32 fma(w, x, acc)), on 16-byte loads that need no alignment.
//
// SP waves share R rows.  Lane `lane` of the i-th of them owns the 16-byte
// weight chunks lane + 64 (i + SP j) of a row (E elements each) and loads x
// for them straight from memory (every wave reads x, so it sits in the
// caches), once for its R rows.  Batches of U chunks run through two register
// sets: batch b + 1 is in flight while batch b is summed (its loads are
// unconditional, see gemv_lds_kernel).  The k % E elements past the last whole
// chunk go one per lane.  Four accumulators per lane keep the FMA chains as
// short as one element per thread of a 256-thread workgroup would; the shares
// of a row meet in LDS and are added in wave order.  Chunks past the row end
// are re-read in bounds and not summed (no zero operand stands in for them, so
// an infinite scale or x meets no extra product).
//
// With one element per load and one workgroup per row (the form before) the
// memory system was idle: INT8 4096^2 with W and x off alignment 18.2 us, now
// 7.45; FP16 18.3, now 10.8.  What bounds it now, by us per call (HBM-cold)
// on aligned data; W 1 to 3 bytes off (FP16: 2); x 2 bytes off; both; and the
// LDS kernels on the aligned data:
//   INT4 4096^2      4.7   4.9   6.4   7.15    3.4
//   INT4 11008x4096  9.1   9.2  13.1  15.2     5.8
//   INT8 4096^2      5.1   5.9   5.9   7.45    4.3
//   INT8 11008x4096 10.7  12.3  12.1  16.3     8.5
//   FP16 4096^2      7.1   9.2   7.5  10.8     6.9
//   FP16 11008x4096 15.0  20.8  16.3  25.1    15.6
// On aligned data FP16 is bound by memory (6.0 TB/s at 11008x4096), INT4 by
// its per-element arithmetic (2.6 TB/s), INT8 (4.2 TB/s) lies between.  Off
// alignment the unaligned loads themselves cost the difference; W or x off by
// 4 or 8 bytes costs nothing.

__device__ __forceinline__ uint4 load16_any(const char* p) {
    uint4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}

// float(q) * s for a value held exactly in fp16: one v_fma_mix_f32.  Adding
// -0 changes no product, signed zeros included.
__device__ __forceinline__ float times_scale(_Float16 q, float s) {
    return __builtin_fmaf(static_cast<float>(q), s, -0.0f);
}

// Per operator: E elements per 16-byte chunk, XP 16-byte pieces of x per
// chunk, `sum` one chunk into the four accumulators, `one` a single element.
struct AnyInt4 {
    using Y = uint16_t;
    static constexpr int E = 32, XP = 4, kXBytes = 2;
    static constexpr bool kGroupScale = true;
    static constexpr bool kTailFirst = false;
    static __device__ __forceinline__ float scale_of(const void* s, int64_t, int64_t i) {
        return h2f(static_cast<const uint16_t*>(s)[i]);
    }
    static __device__ __forceinline__ void sum(const uint4& w, const uint4 (&x)[XP],
                                               float s, float (&acc)[4]) {
        const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
        const f16x2 bias_lo = {static_cast<_Float16>(-1032.0f), static_cast<_Float16>(-1032.0f)};
        const f16x2 bias_hi = {static_cast<_Float16>(-72.0f), static_cast<_Float16>(-72.0f)};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t u = ws[i], u8 = u >> 8;
            const f16x2 x01 = as_f16x2(x[i].x), x23 = as_f16x2(x[i].y);
            const f16x2 x45 = as_f16x2(x[i].z), x67 = as_f16x2(x[i].w);
            // pairs (q0, q4), (q1, q5), (q2, q6), (q3, q7)
            const f16x2 qa = as_f16x2((u & 0x000F000Fu) ^ 0x64086408u) + bias_lo;
            const f16x2 qb = as_f16x2((u & 0x00F000F0u) ^ 0x54805480u) + bias_hi;
            const f16x2 qc = as_f16x2((u8 & 0x000F000Fu) ^ 0x64086408u) + bias_lo;
            const f16x2 qd = as_f16x2((u8 & 0x00F000F0u) ^ 0x54805480u) + bias_hi;
            acc[0] = __builtin_fmaf(times_scale(qa[0], s), static_cast<float>(x01[0]), acc[0]);
            acc[1] = __builtin_fmaf(times_scale(qb[0], s), static_cast<float>(x01[1]), acc[1]);
            acc[2] = __builtin_fmaf(times_scale(qc[0], s), static_cast<float>(x23[0]), acc[2]);
            acc[3] = __builtin_fmaf(times_scale(qd[0], s), static_cast<float>(x23[1]), acc[3]);
            acc[0] = __builtin_fmaf(times_scale(qa[1], s), static_cast<float>(x45[0]), acc[0]);
            acc[1] = __builtin_fmaf(times_scale(qb[1], s), static_cast<float>(x45[1]), acc[1]);
            acc[2] = __builtin_fmaf(times_scale(qc[1], s), static_cast<float>(x67[0]), acc[2]);
            acc[3] = __builtin_fmaf(times_scale(qd[1], s), static_cast<float>(x67[1]), acc[3]);
        }
    }
    // k % 128 == 0: no element past the last whole chunk
    static __device__ __forceinline__ float elem_w(const char*, int64_t) { return 0.f; }
    static __device__ __forceinline__ float elem_x(const char*, int64_t) { return 0.f; }
    static __device__ __forceinline__ float one(float, float, float, float acc) { return acc; }
    static __device__ __forceinline__ void store(Y* y, float v) { *y = f2h(v); }
};

struct AnyInt8 {
    using Y = uint16_t;
    static constexpr int E = 16, XP = 2, kXBytes = 2;
    static constexpr bool kGroupScale = false;
    static constexpr bool kTailFirst = false;
    static __device__ __forceinline__ float scale_of(const void* s, int64_t row, int64_t) {
        return static_cast<const float*>(s)[row];
    }
    static __device__ __forceinline__ void sum(const uint4& w, const uint4 (&x)[XP],
                                               float s, float (&acc)[4]) {
        const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
        const uint32_t xw[8] = {x[0].x, x[0].y, x[0].z, x[0].w, x[1].x, x[1].y, x[1].z, x[1].w};
        const f16x2 bias = {static_cast<_Float16>(-1152.0f), static_cast<_Float16>(-1152.0f)};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t u = ws[i];
            // pairs (q0, q2), (q1, q3)
            const f16x2 qa = as_f16x2((u & 0x00FF00FFu) ^ 0x64806480u) + bias;
            const f16x2 qb = as_f16x2(((u >> 8) & 0x00FF00FFu) ^ 0x64806480u) + bias;
            const f16x2 x01 = as_f16x2(xw[2 * i]), x23 = as_f16x2(xw[2 * i + 1]);
            acc[0] = __builtin_fmaf(times_scale(qa[0], s), static_cast<float>(x01[0]), acc[0]);
            acc[1] = __builtin_fmaf(times_scale(qb[0], s), static_cast<float>(x01[1]), acc[1]);
            acc[2] = __builtin_fmaf(times_scale(qa[1], s), static_cast<float>(x23[0]), acc[2]);
            acc[3] = __builtin_fmaf(times_scale(qb[1], s), static_cast<float>(x23[1]), acc[3]);
        }
    }
    static __device__ __forceinline__ float elem_w(const char* w, int64_t i) {
        return static_cast<float>(reinterpret_cast<const int8_t*>(w)[i]);
    }
    static __device__ __forceinline__ float elem_x(const char* x, int64_t i) {
        return h2f(reinterpret_cast<const uint16_t*>(x)[i]);
    }
    static __device__ __forceinline__ float one(float w, float x, float s, float acc) {
        return __builtin_fmaf(w * s, x, acc);
    }
    static __device__ __forceinline__ void store(Y* y, float v) { *y = f2h(v); }
};

struct AnyF16 {
    using Y = uint16_t;
    static constexpr int E = 8, XP = 1, kXBytes = 2;
    static constexpr bool kGroupScale = false;
    static constexpr bool kTailFirst = true;
    static __device__ __forceinline__ float scale_of(const void*, int64_t, int64_t) { return 0.f; }
    static __device__ __forceinline__ void sum(const uint4& w, const uint4 (&x)[XP], float,
                                               float (&acc)[4]) {
        const uint32_t ws[4] = {w.x, w.y, w.z, w.w}, xw[4] = {x[0].x, x[0].y, x[0].z, x[0].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const f16x2 a = as_f16x2(ws[i]), b = as_f16x2(xw[i]);
            acc[i] = __builtin_fmaf(static_cast<float>(a[0]), static_cast<float>(b[0]), acc[i]);
            acc[i] = __builtin_fmaf(static_cast<float>(a[1]), static_cast<float>(b[1]), acc[i]);
        }
    }
    static __device__ __forceinline__ float elem_w(const char* w, int64_t i) {
        return h2f(reinterpret_cast<const uint16_t*>(w)[i]);
    }
    static __device__ __forceinline__ float elem_x(const char* x, int64_t i) { return elem_w(x, i); }
    static __device__ __forceinline__ float one(float w, float x, float, float acc) {
        return __builtin_fmaf(w, x, acc);
    }
    static __device__ __forceinline__ void store(Y* y, float v) { *y = f2h(v); }
};

struct AnyF32 {
    using Y = float;
    static constexpr int E = 4, XP = 1, kXBytes = 4;
    static constexpr bool kGroupScale = false;
    static constexpr bool kTailFirst = true;
    static __device__ __forceinline__ float scale_of(const void*, int64_t, int64_t) { return 0.f; }
    static __device__ __forceinline__ void sum(const uint4& w, const uint4 (&x)[XP], float,
                                               float (&acc)[4]) {
        const uint32_t ws[4] = {w.x, w.y, w.z, w.w}, xw[4] = {x[0].x, x[0].y, x[0].z, x[0].w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
            acc[i] = __builtin_fmaf(__builtin_bit_cast(float, ws[i]),
                                    __builtin_bit_cast(float, xw[i]), acc[i]);
    }
    static __device__ __forceinline__ float elem_w(const char* w, int64_t i) {
        return reinterpret_cast<const float*>(w)[i];
    }
    static __device__ __forceinline__ float elem_x(const char* x, int64_t i) { return elem_w(x, i); }
    static __device__ __forceinline__ float one(float w, float x, float, float acc) {
        return __builtin_fmaf(w, x, acc);
    }
    static __device__ __forceinline__ void store(Y* y, float v) { *y = v; }
};

template <class Op, int R, int U, int SP>
__device__ __forceinline__ void scalar_rows(
        const char* __restrict__ w,      // [n][k] elements, any alignment
        const void* __restrict__ scale,  // INT4 [n][k/128], INT8 [n], else unused
        const char* __restrict__ x,      // [k]
        typename Op::Y* __restrict__ y, int n, int64_t k) {
    constexpr int E = Op::E, XP = Op::XP;
    constexpr int64_t kXStep = 64 * E * Op::kXBytes;    // x bytes of 64 chunks
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int part = wave % SP;                // this wave's share of its rows' chunks
    const int64_t row0 = (static_cast<int64_t>(xcd_block()) * (kBlock / 64 / SP) +
                          wave / SP) * R;
    const int64_t nfull = k / E;               // whole chunks of a row
    const int64_t niter = (nfull + 63) / 64;   // 64 chunks each; this wave takes part + SP i
    const int64_t wrow_bytes = nfull * 16 + (k - nfull * E) * (16 / E);
    const int64_t groups = k / 128;
    const char* wr[R];
    float srow[R];
    int64_t rows[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        rows[r] = std::min<int64_t>(row0 + r, n - 1);
        wr[r] = w + rows[r] * wrow_bytes;
        srow[r] = Op::kGroupScale ? 0.f : Op::scale_of(scale, rows[r], 0);
    }
    struct Batch {
        uint4 w[R][U];
        uint4 x[U][XP];
        float s[R][U];
    };
    auto load = [&](Batch& b, int64_t it0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // wave-uniform bases; iterations past the last re-read it, lanes
            // past the row end re-read its last chunk
            const int64_t it = std::min<int64_t>(it0 + SP * u, niter - 1);
            const int last = static_cast<int>(std::min<int64_t>(63, nfull - 1 - 64 * it));
            const uint32_t l = static_cast<uint32_t>(std::min(lane, last));
#pragma unroll
            for (int r = 0; r < R; ++r) {
                b.w[r][u] = load16_any(wr[r] + it * 1024 + l * 16u);
                b.s[r][u] = Op::kGroupScale
                    ? Op::scale_of(scale, 0, rows[r] * groups + it * 16 + (l >> 2)) : srow[r];
            }
            const char* xp = x + it * kXStep + l * static_cast<uint32_t>(16 * XP);
#pragma unroll
            for (int p = 0; p < XP; ++p) b.x[u][p] = load16_any(xp + 16 * p);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // The elements past the last whole chunk, one per lane, in the last wave;
    // loaded ahead of the chunks where those are few elements each (FP16
    // 32000x2050 20.8 us against 22.6, FP32 20000x1001 13.4 against 15.2), at
    // the end for INT8 (4001x4099 6.1 against 6.2, 16001x4099 16.8 against 17.5).
    const int64_t tail = nfull * E + lane;
    const int64_t tail_in = std::min<int64_t>(tail, k - 1);
    float tail_w[R] = {}, tail_x = 0.f;
    auto load_tail = [&] {
        tail_x = Op::elem_x(x, tail_in);
#pragma unroll
        for (int r = 0; r < R; ++r) tail_w[r] = Op::elem_w(wr[r], tail_in);
    };
    if constexpr (Op::kTailFirst) load_tail();
    float acc[R][4] = {};
    auto sum = [&](const Batch& b, int64_t it0) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if ((it0 + SP * u) * 64 + lane < nfull)
#pragma unroll
                for (int r = 0; r < R; ++r) Op::sum(b.w[r][u], b.x[u], b.s[r][u], acc[r]);
    };
    if (part < niter) {
        constexpr int64_t kStep = SP * U;
        Batch b0, b1;
        load(b0, part);
        int64_t it = part;
        for (; it + 2 * kStep < niter; it += 2 * kStep) {
            load(b1, it + kStep);
            sum(b0, it);
            load(b0, it + 2 * kStep);
            sum(b1, it + kStep);
        }
        if (it + kStep < niter) {
            load(b1, it + kStep);
            sum(b0, it);
            sum(b1, it + kStep);
        } else {
            sum(b0, it);
        }
    }
    if (part == SP - 1 && tail < k) {
        if constexpr (!Op::kTailFirst) load_tail();
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r][0] = Op::one(tail_w[r], tail_x, srow[r], acc[r][0]);
    }
    float a[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
        a[r] = segment_sum<64>((acc[r][0] + acc[r][1]) + (acc[r][2] + acc[r][3]));
    if constexpr (SP > 1) {
        __shared__ float shares[kBlock / 64][R];
        if (lane == 63)
#pragma unroll
            for (int r = 0; r < R; ++r) shares[wave][r] = a[r];
        __syncthreads();
        if (part != 0) return;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            a[r] = shares[wave][r];
#pragma unroll
            for (int i = 1; i < SP; ++i) a[r] += shares[wave + i][r];
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (lane == 63 && row0 + r < n) Op::store(y + row0 + r, a[r]);
}

template <int R, int U, int SP>
__global__ __launch_bounds__(kBlock) void int4gemv_scalar_kernel(
        const char* __restrict__ w, const void* __restrict__ scale,
        const char* __restrict__ x, uint16_t* __restrict__ y, int n, int64_t k) {
    scalar_rows<AnyInt4, R, U, SP>(w, scale, x, y, n, k);
}
template <int R, int U, int SP>
__global__ __launch_bounds__(kBlock) void qgemv_scalar_kernel(
        const char* __restrict__ w, const void* __restrict__ scale,
        const char* __restrict__ x, uint16_t* __restrict__ y, int n, int64_t k) {
    scalar_rows<AnyInt8, R, U, SP>(w, scale, x, y, n, k);
}
template <typename S, int R, int U, int SP>
__global__ __launch_bounds__(kBlock) void gemv_scalar_kernel(
        const char* __restrict__ w, const void* __restrict__ scale,
        const char* __restrict__ x, S* __restrict__ y, int n, int64_t k) {
    scalar_rows<std::conditional_t<sizeof(S) == 4, AnyF32, AnyF16>, R, U, SP>(
        w, scale, x, y, n, k);
}

// ------------------------------------------------------------------ wave

// Rows per lane that the register budget of a J-chunk instance allows.
constexpr int int4_rmax(int j) { return j <= 2 ? 4 : (j <= 4 ? 2 : 1); }
constexpr int q8_rmax(int j) { return j <= 4 ? 4 : (j <= 8 ? 2 : 1); }
constexpr int kInt4MaxJ = 8;   // 8 * 64 chunks * 32 = 16384 elements
constexpr int kQ8MaxJ = 16;    // 16 * 64 chunks * 16 = 16384 elements

template <int CW, int J, int R>
__global__ __launch_bounds__(kBlock) void int4gemv_wave_kernel(
        const uint4* __restrict__ w,         // [n][nchunks] 16-byte chunks
        const uint16_t* __restrict__ scale,  // [n][nchunks/4]
        const uint4* __restrict__ x,         // [nchunks][4] 16-byte pieces
        uint16_t* __restrict__ y, int n, int nchunks) {
    constexpr int SLOTS = 64 / CW;
    const int lane = threadIdx.x & 63;
    const int col = lane % CW;
    const int slot = lane / CW;
    const int ngroups = nchunks >> 2;
    const int64_t wave_id =
        static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int64_t row0 = wave_id * (SLOTS * R) + slot;

    // Every load is unconditional on a clamped, in-bounds index (lanes past
    // the row end or past n re-read a valid chunk) so that no load sits
    // behind a branch and all of them are in flight together; inactive
    // lanes are zeroed afterwards with a select.  Weight chunks of all R
    // rows go first: the HBM requests leave at once.
    int cidx[J];
    bool act[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int c = col + CW * j;
        act[j] = c < nchunks;
        cidx[j] = act[j] ? c : nchunks - 1;
    }
    uint4 wv[R][J];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int64_t row = std::min<int64_t>(row0 + SLOTS * r, n - 1);
#pragma unroll
        for (int j = 0; j < J; ++j) wv[r][j] = w[row * nchunks + cidx[j]];
    }
    uint16_t sv[R][J];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int64_t row = std::min<int64_t>(row0 + SLOTS * r, n - 1);
#pragma unroll
        for (int j = 0; j < J; ++j) sv[r][j] = scale[row * ngroups + (cidx[j] >> 2)];
    }
    uint4 xv[J][4];
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int p = 0; p < 4; ++p) xv[j][p] = x[4 * cidx[j] + p];

    // x of the lane's chunks, re-paired for the nibble order of a weight
    // word: xa = (x0,x4), xb = (x1,x5), xc = (x2,x6), xd = (x3,x7).  An
    // inactive chunk gets x = 0, so its (valid, re-read) weights add +-0.
    uint32_t xa[J][4], xb[J][4], xc[J][4], xd[J][4];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        uint32_t d[16];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            d[4 * p + 0] = act[j] ? xv[j][p].x : 0u;
            d[4 * p + 1] = act[j] ? xv[j][p].y : 0u;
            d[4 * p + 2] = act[j] ? xv[j][p].z : 0u;
            d[4 * p + 3] = act[j] ? xv[j][p].w : 0u;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t d0 = d[4 * q], d1 = d[4 * q + 1];
            const uint32_t d2 = d[4 * q + 2], d3 = d[4 * q + 3];
            xa[j][q] = (d0 & 0xFFFFu) | (d2 << 16);
            xb[j][q] = (d0 >> 16) | (d2 & 0xFFFF0000u);
            xc[j][q] = (d1 & 0xFFFFu) | (d3 << 16);
            xd[j][q] = (d1 >> 16) | (d3 & 0xFFFF0000u);
        }
    }

    const f16x2 bias1 = {static_cast<_Float16>(-1032.0f),
                         static_cast<_Float16>(-1032.0f)};
    const f16x2 bias16 = {static_cast<_Float16>(-1152.0f),
                          static_cast<_Float16>(-1152.0f)};
#pragma unroll
    for (int r = 0; r < R; ++r) {
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const uint32_t words[4] = {wv[r][j].x, wv[r][j].y, wv[r][j].z,
                                       wv[r][j].w};
            float d1 = 0.f, d16 = 0.f;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t u = words[q];
                const uint32_t u8 = u >> 8;
                const f16x2 qa = as_f16x2((u & 0x000F000Fu) ^ 0x64086408u) + bias1;
                const f16x2 qb = as_f16x2((u & 0x00F000F0u) ^ 0x64806480u) + bias16;
                const f16x2 qc = as_f16x2((u8 & 0x000F000Fu) ^ 0x64086408u) + bias1;
                const f16x2 qd = as_f16x2((u8 & 0x00F000F0u) ^ 0x64806480u) + bias16;
                d1 = __builtin_amdgcn_fdot2(qa, as_f16x2(xa[j][q]), d1, false);
                d16 = __builtin_amdgcn_fdot2(qb, as_f16x2(xb[j][q]), d16, false);
                d1 = __builtin_amdgcn_fdot2(qc, as_f16x2(xc[j][q]), d1, false);
                d16 = __builtin_amdgcn_fdot2(qd, as_f16x2(xd[j][q]), d16, false);
            }
            const float s = h2f(sv[r][j]);
            acc = __builtin_fmaf(s, d1, acc);
            acc = __builtin_fmaf(s * 0.0625f, d16, acc);
        }
        acc = segment_sum<CW>(acc);
        const int64_t row = row0 + SLOTS * r;
        if (col == CW - 1 && row < n) y[row] = f2h(acc);
    }
}

template <int CW, int J, int R>
__global__ __launch_bounds__(kBlock) void qgemv_wave_kernel(
        const uint4* __restrict__ w,       // [n][nchunks] 16 int8 per chunk
        const float* __restrict__ scale,   // [n]
        const uint4* __restrict__ x,       // [nchunks][2] 16-byte pieces
        uint16_t* __restrict__ y, int n, int nchunks) {
    constexpr int SLOTS = 64 / CW;
    const int lane = threadIdx.x & 63;
    const int col = lane % CW;
    const int slot = lane / CW;
    const int64_t wave_id =
        static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int64_t row0 = wave_id * (SLOTS * R) + slot;

    // Unconditional loads on clamped indices, as in the INT4 kernel.
    int cidx[J];
    bool act[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int c = col + CW * j;
        act[j] = c < nchunks;
        cidx[j] = act[j] ? c : nchunks - 1;
    }
    uint4 wv[R][J];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int64_t row = std::min<int64_t>(row0 + SLOTS * r, n - 1);
#pragma unroll
        for (int j = 0; j < J; ++j) wv[r][j] = w[row * nchunks + cidx[j]];
    }
    uint4 xv[J][2];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        xv[j][0] = x[2 * cidx[j]];
        xv[j][1] = x[2 * cidx[j] + 1];
    }
    // x re-paired for a weight word's byte order: xp = (x0,x2), xq = (x1,x3);
    // an inactive chunk gets x = 0.
    uint32_t xp[J][4], xq[J][4];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const uint4 v0 = xv[j][0], v1 = xv[j][1];
        uint32_t d[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) d[i] = act[j] ? d[i] : 0u;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t d0 = d[2 * q], d1 = d[2 * q + 1];
            xp[j][q] = (d0 & 0xFFFFu) | (d1 << 16);
            xq[j][q] = (d0 >> 16) | (d1 & 0xFFFF0000u);
        }
    }

    const f16x2 bias = {static_cast<_Float16>(-1152.0f),
                        static_cast<_Float16>(-1152.0f)};
#pragma unroll
    for (int r = 0; r < R; ++r) {
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const uint32_t words[4] = {wv[r][j].x, wv[r][j].y, wv[r][j].z,
                                       wv[r][j].w};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t u = words[q];
                const f16x2 qp = as_f16x2((u & 0x00FF00FFu) ^ 0x64806480u) + bias;
                const f16x2 qq = as_f16x2(((u >> 8) & 0x00FF00FFu) ^ 0x64806480u) + bias;
                acc = __builtin_amdgcn_fdot2(qp, as_f16x2(xp[j][q]), acc, false);
                acc = __builtin_amdgcn_fdot2(qq, as_f16x2(xq[j][q]), acc, false);
            }
        }
        acc = segment_sum<CW>(acc);
        const int64_t row = row0 + SLOTS * r;
        if (col == CW - 1 && row < n) y[row] = f2h(scale[row] * acc);
    }
}

// ------------------------------------------------------------- wave+LDS
//
// Second CDNA4 design: x is staged once per workgroup in LDS, already
// re-paired for the weight words, instead of every wave loading and
// re-pairing its own copy.  Per lane the x pairs of its J chunks then come
// from 4*J ds_read_b128.  Both nibbles of a byte feed one accumulator: the
// high nibble is taken in place (bits 4-7) under the fp16 exponent of 64,
// where the mantissa step is 1/16, so ((w & 0x00F000F0) ^ 0x54805480) is
// the fp16 pair (72+q1, 72+q5) and a packed add of -72 gives (q1, q5)
// exactly.  Workgroups take their rows through xcd_block(); NT
// (256 or 512 threads) is chosen by the host plan.
//
// Address work is kept off the VALU, which these kernels are short of (the
// INT4 dequant and dot take 13 VALU instructions per 8 weights):
// - The host plans J = ceil(nchunks / CW), so a lane's chunks col + CW*j for
//   j < J - 1 always lie inside the row; only the last one is clamped.
//   The others sit at compile-time offsets from one per-lane address.
// - The LDS planes have the compile-time stride CW*J + 1; column CW*J is
//   zero and is what lanes past the row end read.  Every x read but the
//   last chunk's is then an immediate offset from one address.
// - The row base is wave-uniform when a row spans the wave (CW = 64), so it
//   lives in scalar registers.
// Issue order, pinned with scheduling barriers: the workgroup's x pieces,
// then per row, chunk by chunk, the weight chunk and the group scale (the
// grouped kernels know the weights' address before the scales'; INT8: the
// chunks, then the row scale), so that the wait before chunk j covers chunks
// 0..j only and each chunk is summed as it lands.  A scheduling barrier after
// the workgroup barrier keeps weight arithmetic (and its waits) from being
// hoisted above it.

// The timeline stamps pin their clock reads by data dependence, not by
// scheduling fences (the compiler places pure arithmetic before the machine
// scheduler sees a fence, and a full fence also held every LDS read of x
// live at once, doubling the VGPRs at J = 6).  wall_clock_through(v) reads
// the wall clock with `v` passed through as an operand it may modify: the
// read waits for the arithmetic that produces v, and whatever uses v after
// it waits for the read.  The read is a scalar memory instruction the
// compiler does not track, so it waits for its own result before anything
// else counts on the LGKM counter.
__device__ __forceinline__ uint64_t wall_clock_through(float& v) {
    uint64_t t;
    asm volatile("s_memrealtime %0\n\ts_waitcnt lgkmcnt(0)" : "=s"(t), "+v"(v));
    return t;
}
__device__ __forceinline__ uint64_t wall_clock_through(uint32_t& a, uint32_t& b,
                                                       uint32_t& c) {
    uint64_t t;
    asm volatile("s_memrealtime %0\n\ts_waitcnt lgkmcnt(0)"
                 : "=s"(t), "+v"(a), "+v"(b), "+v"(c));
    return t;
}

// The rows a workgroup computes: logical workgroup `blk` of a problem of n
// rows, problem `p` of its group.
struct RowSlot {
    int p;
    uint32_t blk;
    int n;
};

// Operands of a launch of one problem; the grouped kernels have their own.
// `slot()` is evaluated behind the x loads, `scale` behind the first weight
// load, `store` at the end: none holds back a load that does not need it.
template <typename S, uint32_t RUN>
struct OneProblem {
    const uint4* w_;
    const S* scale_;
    uint16_t* y_;
    int n_;
    __device__ __forceinline__ RowSlot slot() const { return {0, xcd_block<RUN>(), n_}; }
    __device__ __forceinline__ const uint4* w(const RowSlot&) const { return w_; }
    __device__ __forceinline__ const S* scale(const RowSlot&) const { return scale_; }
    __device__ __forceinline__ void store(const RowSlot&, int64_t row, uint16_t v) const {
        y_[row] = v;
    }
};

// One workgroup's rows of one INT4 problem.  `xs` is the workgroup's LDS:
// [4][CW*J + 1] re-paired x pieces, q-major.  `ops` names the workgroup's
// operands (OneProblem).
//
// STAMP (the timeline diagnostic only; every GEMV instance has it false, and
// then none of its code exists): lane 0 of each wave writes 8 words to
// stamps[wave * 8 ..]: the 100 MHz wall clock at the wave's start, after the
// x barrier, after its first chunk is summed, after its last chunk is
// summed and after its y stores are issued; then the hardware CU id.
template <int CW, int J, int R, int NT, bool STAMP = false, class Ops>
__device__ __forceinline__ void int4_lds_rows(
        const uint4* __restrict__ x,         // [4*nchunks] 16-byte pieces
        int nchunks, uint4* __restrict__ xs, const Ops ops,
        uint64_t* __restrict__ stamps = nullptr) {
    [[maybe_unused]] uint64_t ts[5] = {};
    if constexpr (STAMP) ts[0] = wall_clock64();
    constexpr int SLOTS = 64 / CW;
    constexpr int S = CW * J + 1;                     // LDS plane stride
    constexpr int XPER = (4 * CW * J + NT - 1) / NT;  // x pieces per thread
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int col = lane % CW;
    const int slot = lane / CW;
    const int npieces = 4 * nchunks;

    // (1) this thread's share of x first
    uint4 xv[XPER];
#pragma unroll
    for (int i = 0; i < XPER; ++i) xv[i] = x[std::min(tid + i * NT, npieces - 1)];
    __builtin_amdgcn_sched_barrier(0);
    const RowSlot g = ops.slot();
    const int n = g.n;
    const uint32_t blk = g.blk;
    const int64_t wave_id = static_cast<int64_t>(blk) * (NT >> 6) +
                            __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t row0 = wave_id * (SLOTS * R) + slot;
    // Byte offsets fit in 32 bits (the host checks n * k / 2 < 2^32).
    const char* wb = reinterpret_cast<const char*>(ops.w(g));
    const char* sb = nullptr;
    const uint32_t wrow_bytes = static_cast<uint32_t>(nchunks) * 16u;
    const uint32_t srow_bytes = static_cast<uint32_t>(nchunks >> 2) * 2u;
    // (2) per row, each chunk and then its group scale, all in flight
    //     together; a last chunk past the row end re-reads chunk
    //     nchunks - 1 (x is zero there)
    const int clast = col + CW * (J - 1);
    const int cl = clast < nchunks ? clast : nchunks - 1;
    const uint32_t wcol = static_cast<uint32_t>(col) * 16u;
    const uint32_t scol = static_cast<uint32_t>(col >> 2) * 2u;
    uint4 wv[R][J];
    uint16_t sv[R][J];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t row = static_cast<uint32_t>(std::min<int64_t>(row0 + SLOTS * r, n - 1));
        const char* wr = wb + row * wrow_bytes;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const bool in_row = j < J - 1;
            wv[r][j] = *reinterpret_cast<const uint4*>(
                wr + (in_row ? wcol + CW * 16 * j : static_cast<uint32_t>(cl) * 16u));
            __builtin_amdgcn_sched_barrier(0);
            if (r == 0 && j == 0) sb = reinterpret_cast<const char*>(ops.scale(g));
            const char* sr = sb + row * srow_bytes;
            sv[r][j] = *reinterpret_cast<const uint16_t*>(
                sr + (in_row ? scol + (CW / 2) * j : static_cast<uint32_t>(cl >> 2) * 2u));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // (3) re-pair x: piece = x0..x7 -> [(x0,x4), (x1,x5), (x2,x6), (x3,x7)]
#pragma unroll
    for (int i = 0; i < XPER; ++i) {
        // unconditional store on the clamped index (threads past the end
        // rewrite the last piece with the same value), so that no load is
        // sunk behind a branch
        const int p = std::min(tid + i * NT, npieces - 1);
        const uint4 v = xv[i];
        uint4 o;
        o.x = (v.x & 0xFFFFu) | (v.z << 16);
        o.y = (v.x >> 16) | (v.z & 0xFFFF0000u);
        o.z = (v.y & 0xFFFFu) | (v.w << 16);
        o.w = (v.y >> 16) | (v.w & 0xFFFF0000u);
        xs[(p & 3) * S + (p >> 2)] = o;
    }
    if (tid < 4) xs[tid * S + CW * J] = uint4{0, 0, 0, 0};
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    // nibble masks and byte shift of the dequant; the stamped copy passes
    // them through the barrier stamp's clock read, so no dequant (nor its
    // wait for the weights) is placed above that read
    uint32_t m_lo = 0x000F000Fu, m_hi = 0x00F000F0u, sh8 = 8;
    if constexpr (STAMP) ts[1] = wall_clock_through(m_lo, m_hi, sh8);
    uint4 xp[J][4];
    const int xlast = clast < nchunks ? clast : CW * J;
    // the stamped copy reads each chunk's x next to its use (below): its
    // clock reads keep loads from crossing them, and reads issued all up
    // front would hold J x 16 VGPRs at once
    if constexpr (!STAMP) {
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                xp[j][q] = xs[q * S + (j < J - 1 ? col + CW * j : xlast)];
    }

    const f16x2 bias_lo = {static_cast<_Float16>(-1032.0f),
                           static_cast<_Float16>(-1032.0f)};
    const f16x2 bias_hi = {static_cast<_Float16>(-72.0f),
                           static_cast<_Float16>(-72.0f)};
#pragma unroll
    for (int r = 0; r < R; ++r) {
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            if constexpr (STAMP) {
                if (r == 0) {
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        xp[j][q] = xs[q * S + (j < J - 1 ? col + CW * j : xlast)];
                }
            }
            float d = 0.f;
            if constexpr (STAMP) {
                // the second chunk's dequant and sum start after the first stamp
                if (r * J + j == 1)
                    asm volatile("" : "+v"(d), "+v"(wv[r][j].x), "+v"(wv[r][j].y),
                                 "+v"(wv[r][j].z), "+v"(wv[r][j].w) : "v"(acc));
            }
            const uint32_t words[4] = {wv[r][j].x, wv[r][j].y, wv[r][j].z,
                                       wv[r][j].w};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t u = words[q];
                const uint32_t u8 = u >> sh8;
                const f16x2 qa = as_f16x2((u & m_lo) ^ 0x64086408u) + bias_lo;
                const f16x2 qb = as_f16x2((u & m_hi) ^ 0x54805480u) + bias_hi;
                const f16x2 qc = as_f16x2((u8 & m_lo) ^ 0x64086408u) + bias_lo;
                const f16x2 qd = as_f16x2((u8 & m_hi) ^ 0x54805480u) + bias_hi;
                d = __builtin_amdgcn_fdot2(qa, as_f16x2(xp[j][q].x), d, false);
                d = __builtin_amdgcn_fdot2(qb, as_f16x2(xp[j][q].y), d, false);
                d = __builtin_amdgcn_fdot2(qc, as_f16x2(xp[j][q].z), d, false);
                d = __builtin_amdgcn_fdot2(qd, as_f16x2(xp[j][q].w), d, false);
            }
            acc = __builtin_fmaf(h2f(sv[r][j]), d, acc);
            if constexpr (STAMP) {
                if (r == 0 && j == 0) ts[2] = wall_clock_through(acc);
                if (r == R - 1 && j == J - 1) ts[3] = wall_clock_through(acc);
            }
        }
        acc = segment_sum<CW>(acc);
        const int64_t row = row0 + SLOTS * r;
        if (col == CW - 1 && row < n) ops.store(g, row, f2h(acc));
    }
    if constexpr (STAMP) {
        __builtin_amdgcn_sched_barrier(0);
        ts[4] = wall_clock64();
        if (lane == 0) {
            const uint64_t wave = static_cast<uint64_t>(blk) * (NT >> 6) +
                                  static_cast<uint64_t>(tid >> 6);
            uint64_t* o = stamps + wave * 8;
#pragma unroll
            for (int i = 0; i < 5; ++i) o[i] = ts[i];
            o[5] = __smid();
            o[6] = 0;
            o[7] = 0;
        }
    }
}

// One workgroup's rows of one INT8 problem; `xs` holds [2][CW*J + 1]
// re-paired x pieces, q-major, column CW*J zero.  Same layout and issue order
// as the INT4 rows; the row's scale is loaded right after its weights, so the
// final scaling waits on no load of its own.
template <int CW, int J, int R, int NT, class Ops>
__device__ __forceinline__ void q8_lds_rows(
        const uint4* __restrict__ x,       // [2*nchunks] 16-byte pieces
        int nchunks, uint4* __restrict__ xs, const Ops ops) {
    constexpr int SLOTS = 64 / CW;
    constexpr int S = CW * J + 1;
    constexpr int XPER = (2 * CW * J + NT - 1) / NT;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int col = lane % CW;
    const int slot = lane / CW;
    const int npieces = 2 * nchunks;

    uint4 xv[XPER];
#pragma unroll
    for (int i = 0; i < XPER; ++i) xv[i] = x[std::min(tid + i * NT, npieces - 1)];
    __builtin_amdgcn_sched_barrier(0);
    const RowSlot g = ops.slot();
    const int n = g.n;
    const int64_t wave_id = static_cast<int64_t>(g.blk) * (NT >> 6) +
                            __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t row0 = wave_id * (SLOTS * R) + slot;
    const char* wb = reinterpret_cast<const char*>(ops.w(g));
    const uint32_t wrow_bytes = static_cast<uint32_t>(nchunks) * 16u;
    const int clast = col + CW * (J - 1);
    const int cl = clast < nchunks ? clast : nchunks - 1;
    const uint32_t wcol = static_cast<uint32_t>(col) * 16u;
    uint4 wv[R][J];
    float sc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t row = static_cast<uint32_t>(std::min<int64_t>(row0 + SLOTS * r, n - 1));
        const char* wr = wb + row * wrow_bytes;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const uint32_t off = j < J - 1 ? wcol + CW * 16 * j
                                           : static_cast<uint32_t>(cl) * 16u;
            wv[r][j] = *reinterpret_cast<const uint4*>(wr + off);
            __builtin_amdgcn_sched_barrier(0);
        }
        sc[r] = ops.scale(g)[row];
        __builtin_amdgcn_sched_barrier(0);
    }
    // re-pair x: piece = x0..x7 -> [(x0,x2), (x1,x3), (x4,x6), (x5,x7)]
#pragma unroll
    for (int i = 0; i < XPER; ++i) {
        const int p = std::min(tid + i * NT, npieces - 1);
        const uint4 v = xv[i];
        uint4 o;
        o.x = (v.x & 0xFFFFu) | (v.y << 16);
        o.y = (v.x >> 16) | (v.y & 0xFFFF0000u);
        o.z = (v.z & 0xFFFFu) | (v.w << 16);
        o.w = (v.z >> 16) | (v.w & 0xFFFF0000u);
        xs[(p & 1) * S + (p >> 1)] = o;
    }
    if (tid < 2) xs[tid * S + CW * J] = uint4{0, 0, 0, 0};
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    uint4 xp[J][2];
    const int xlast = clast < nchunks ? clast : CW * J;
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int q = 0; q < 2; ++q)
            xp[j][q] = xs[q * S + (j < J - 1 ? col + CW * j : xlast)];

    const f16x2 bias = {static_cast<_Float16>(-1152.0f),
                        static_cast<_Float16>(-1152.0f)};
#pragma unroll
    for (int r = 0; r < R; ++r) {
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const uint32_t words[4] = {wv[r][j].x, wv[r][j].y, wv[r][j].z,
                                       wv[r][j].w};
            const uint32_t xpair[8] = {xp[j][0].x, xp[j][0].y, xp[j][0].z,
                                       xp[j][0].w, xp[j][1].x, xp[j][1].y,
                                       xp[j][1].z, xp[j][1].w};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t u = words[q];
                const f16x2 qp = as_f16x2((u & 0x00FF00FFu) ^ 0x64806480u) + bias;
                const f16x2 qq = as_f16x2(((u >> 8) & 0x00FF00FFu) ^ 0x64806480u) + bias;
                acc = __builtin_amdgcn_fdot2(qp, as_f16x2(xpair[2 * q]), acc, false);
                acc = __builtin_amdgcn_fdot2(qq, as_f16x2(xpair[2 * q + 1]), acc, false);
            }
        }
        acc = segment_sum<CW>(acc);
        const int64_t row = row0 + SLOTS * r;
        if (col == CW - 1 && row < n) ops.store(g, row, f2h(sc[r] * acc));
    }
}

// LDS bytes of the untiled INT4 / INT8 LDS kernels for plan (cw, j).
constexpr uint32_t int4_lds_bytes(int cw, int j) {
    return 4u * 16u * static_cast<uint32_t>(cw * j + 1);
}
constexpr uint32_t q8_lds_bytes(int cw, int j) {
    return 2u * 16u * static_cast<uint32_t>(cw * j + 1);
}
// The LDS kernels read chunks col + cw*j for j < J - 1 unclamped, which
// stays inside a row only when J = ceil(nchunks / cw); every plan has that
// form, and launches check it.
inline bool lds_chunks_ok(const Plan& p, int64_t nchunks) {
    return p.cw > 0 && p.j == (nchunks + p.cw - 1) / p.cw;
}

// One problem per launch.
template <int CW, int J, int R, int NT>
__global__ __launch_bounds__(NT) void int4gemv_lds_kernel(
        const uint4* __restrict__ w, const uint16_t* __restrict__ scale,
        const uint4* __restrict__ x, uint16_t* __restrict__ y, int n,
        int nchunks) {
    extern __shared__ uint4 xs[];
    int4_lds_rows<CW, J, R, NT>(x, nchunks, xs, OneProblem<uint16_t, xcd_run(J * R)>{w, scale, y, n});
}

// The INT4 LDS kernel with the timeline stamps (diagnostic, cq_int4_timeline):
// the same arithmetic and launch shape; `stamps` holds 8 words per wave.
template <int CW, int J, int R, int NT>
__global__ __launch_bounds__(NT) void int4gemv_lds_stamp_kernel(
        const uint4* __restrict__ w, const uint16_t* __restrict__ scale,
        const uint4* __restrict__ x, uint16_t* __restrict__ y, int n,
        int nchunks, uint64_t* __restrict__ stamps) {
    extern __shared__ uint4 xs[];
    int4_lds_rows<CW, J, R, NT, true>(x, nchunks, xs,
                                      OneProblem<uint16_t, xcd_run(J * R)>{w, scale, y, n}, stamps);
}

template <int CW, int J, int R, int NT>
__global__ __launch_bounds__(NT) void qgemv_lds_kernel(
        const uint4* __restrict__ w, const float* __restrict__ scale,
        const uint4* __restrict__ x, uint16_t* __restrict__ y, int n,
        int nchunks) {
    extern __shared__ uint4 xs[];
    q8_lds_rows<CW, J, R, NT>(x, nchunks, xs, OneProblem<float, xcd_run(J * R)>{w, scale, y, n});
}

// K-tiled LDS kernels, for rows longer than one batch of chunks held per
// lane (k > 16384; the *_lds_tiled variants force them at any k).  R rows
// per wave (CW = 64), both read against one copy of x.  x is staged tile by
// tile: TJ * 64 chunks of the row per tile (TJ = 2..8: TJ * 2048 INT4 or
// TJ * 1024 INT8 elements), re-paired in LDS, with a barrier before the
// tile is read and one before the next tile overwrites it.  Every thread of
// the workgroup runs the same tiles (they depend on nchunks only; rows past n
// are clamped, never skipped), so every barrier is reached by all.  In the last,
// partial tile only the first ceil(tc / 64) chunks of each lane are loaded
// and summed (a wave-uniform bound).  Lane `col` takes chunks col + 64 j of
// its rows in j order, as the untiled kernels do, so each row's sum
// accumulates in the same order as an untiled kernel with J =
// ceil(nchunks / 64): at k <= 16384 the result is bit-identical to the LDS
// kernel with CW = 64 (for any R).
template <int NT, int TJ, int R>
__global__ __launch_bounds__(NT) void int4gemv_tiled_kernel(
        const uint4* __restrict__ w, const uint16_t* __restrict__ scale,
        const uint4* __restrict__ x, uint16_t* __restrict__ y, int n,
        int nchunks) {
    extern __shared__ uint4 xs[];                  // [4][TC + 1]
    constexpr int TC = TJ * 64;                    // chunks per tile
    constexpr int XPER = 4 * TC / NT;              // x pieces per thread per tile
    static_assert(4 * TC % NT == 0, "a tile's pieces divide over the workgroup");
    constexpr int ldsw = TC + 1;
    const int tid = threadIdx.x;
    const int col = tid & 63;
    const int64_t row0 = (static_cast<int64_t>(xcd_block()) * (NT >> 6) + (tid >> 6)) * R;
    // Byte offsets within a row fit in 32 bits (the host checks
    // n * k / 2 < 2^32); row bases are 64-bit.
    const char* wrow[R];
    const char* srow[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint64_t rc = static_cast<uint64_t>(std::min<int64_t>(row0 + r, n - 1));
        wrow[r] = reinterpret_cast<const char*>(w) + rc * (static_cast<uint32_t>(nchunks) * 16u);
        srow[r] = reinterpret_cast<const char*>(scale) + rc * ((static_cast<uint32_t>(nchunks) >> 2) * 2u);
    }
    const f16x2 bias_lo = {static_cast<_Float16>(-1032.0f),
                           static_cast<_Float16>(-1032.0f)};
    const f16x2 bias_hi = {static_cast<_Float16>(-72.0f),
                           static_cast<_Float16>(-72.0f)};
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.f;
    auto tile = [&]<bool PARTIAL>(int c0, int tc) {
        const int jn = PARTIAL ? (tc + 63) >> 6 : TJ;   // chunks per lane, wave-uniform
        const int np = 4 * tc;                          // x pieces in this tile
        const uint4* xt = x + 4 * static_cast<int64_t>(c0);
        uint4 xv[XPER];
#pragma unroll
        for (int i = 0; i < XPER; ++i) xv[i] = xt[std::min(tid + i * NT, np - 1)];
        __builtin_amdgcn_sched_barrier(0);
        // this lane's chunks of the tile; lanes past the row end re-read the
        // tile's last chunk against the zero column of x
        uint4 wv[R][TJ];
        uint16_t sv[R][TJ];
        int xcol[TJ];
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            if (PARTIAL && j >= jn) break;
            const int c = col + 64 * j;
            const uint32_t cl = static_cast<uint32_t>(c0 + (c < tc ? c : tc - 1));
            xcol[j] = c < tc ? c : TC;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                wv[r][j] = *reinterpret_cast<const uint4*>(wrow[r] + cl * 16u);
                sv[r][j] = *reinterpret_cast<const uint16_t*>(srow[r] + (cl >> 2) * 2u);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < XPER; ++i) {
            const int p = std::min(tid + i * NT, np - 1);
            const uint4 v = xv[i];
            uint4 o;
            o.x = (v.x & 0xFFFFu) | (v.z << 16);
            o.y = (v.x >> 16) | (v.z & 0xFFFF0000u);
            o.z = (v.y & 0xFFFFu) | (v.w << 16);
            o.w = (v.y >> 16) | (v.w & 0xFFFF0000u);
            xs[(p & 3) * ldsw + (p >> 2)] = o;
        }
        if (tid < 4) xs[tid * ldsw + TC] = uint4{0, 0, 0, 0};
        __syncthreads();
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            if (PARTIAL && j >= jn) break;
            float d[R];
#pragma unroll
            for (int r = 0; r < R; ++r) d[r] = 0.f;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint4 xq = xs[q * ldsw + xcol[j]];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const uint32_t u = q == 0 ? wv[r][j].x : q == 1 ? wv[r][j].y
                                     : q == 2 ? wv[r][j].z : wv[r][j].w;
                    const uint32_t u8 = u >> 8;
                    const f16x2 qa = as_f16x2((u & 0x000F000Fu) ^ 0x64086408u) + bias_lo;
                    const f16x2 qb = as_f16x2((u & 0x00F000F0u) ^ 0x54805480u) + bias_hi;
                    const f16x2 qc = as_f16x2((u8 & 0x000F000Fu) ^ 0x64086408u) + bias_lo;
                    const f16x2 qd = as_f16x2((u8 & 0x00F000F0u) ^ 0x54805480u) + bias_hi;
                    d[r] = __builtin_amdgcn_fdot2(qa, as_f16x2(xq.x), d[r], false);
                    d[r] = __builtin_amdgcn_fdot2(qb, as_f16x2(xq.y), d[r], false);
                    d[r] = __builtin_amdgcn_fdot2(qc, as_f16x2(xq.z), d[r], false);
                    d[r] = __builtin_amdgcn_fdot2(qd, as_f16x2(xq.w), d[r], false);
                }
            }
#pragma unroll
            for (int r = 0; r < R; ++r) acc[r] = __builtin_fmaf(h2f(sv[r][j]), d[r], acc[r]);
        }
        __syncthreads();
    };
    int c0 = 0;
    for (; c0 + TC <= nchunks; c0 += TC) tile.template operator()<false>(c0, TC);
    if (c0 < nchunks) tile.template operator()<true>(c0, nchunks - c0);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float a = segment_sum<64>(acc[r]);
        if (col == 63 && row0 + r < n) y[row0 + r] = f2h(a);
    }
}

template <int NT, int TJ, int R>
__global__ __launch_bounds__(NT) void qgemv_tiled_kernel(
        const uint4* __restrict__ w, const float* __restrict__ scale,
        const uint4* __restrict__ x, uint16_t* __restrict__ y, int n,
        int nchunks) {
    extern __shared__ uint4 xs[];                  // [2][TC + 1]
    constexpr int TC = TJ * 64;
    constexpr int XPER = 2 * TC / NT;
    static_assert(2 * TC % NT == 0, "a tile's pieces divide over the workgroup");
    constexpr int ldsw = TC + 1;
    const int tid = threadIdx.x;
    const int col = tid & 63;
    const int64_t row0 = (static_cast<int64_t>(xcd_block<kXcdAll>()) * (NT >> 6) + (tid >> 6)) * R;
    const char* wrow[R];
    float sc[R];   // row scales, loaded first so the final scaling waits on nothing
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint64_t rc = static_cast<uint64_t>(std::min<int64_t>(row0 + r, n - 1));
        wrow[r] = reinterpret_cast<const char*>(w) + rc * (static_cast<uint32_t>(nchunks) * 16u);
        sc[r] = scale[rc];
    }
    const f16x2 bias = {static_cast<_Float16>(-1152.0f),
                        static_cast<_Float16>(-1152.0f)};
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.f;
    auto tile = [&]<bool PARTIAL>(int c0, int tc) {
        const int jn = PARTIAL ? (tc + 63) >> 6 : TJ;
        const int np = 2 * tc;
        const uint4* xt = x + 2 * static_cast<int64_t>(c0);
        uint4 xv[XPER];
#pragma unroll
        for (int i = 0; i < XPER; ++i) xv[i] = xt[std::min(tid + i * NT, np - 1)];
        __builtin_amdgcn_sched_barrier(0);
        uint4 wv[R][TJ];
        int xcol[TJ];
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            if (PARTIAL && j >= jn) break;
            const int c = col + 64 * j;
            const uint32_t cl = static_cast<uint32_t>(c0 + (c < tc ? c : tc - 1));
            xcol[j] = c < tc ? c : TC;
#pragma unroll
            for (int r = 0; r < R; ++r)
                wv[r][j] = *reinterpret_cast<const uint4*>(wrow[r] + cl * 16u);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < XPER; ++i) {
            const int p = std::min(tid + i * NT, np - 1);
            const uint4 v = xv[i];
            uint4 o;
            o.x = (v.x & 0xFFFFu) | (v.y << 16);
            o.y = (v.x >> 16) | (v.y & 0xFFFF0000u);
            o.z = (v.z & 0xFFFFu) | (v.w << 16);
            o.w = (v.z >> 16) | (v.w & 0xFFFF0000u);
            xs[(p & 1) * ldsw + (p >> 1)] = o;
        }
        if (tid < 2) xs[tid * ldsw + TC] = uint4{0, 0, 0, 0};
        __syncthreads();
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            if (PARTIAL && j >= jn) break;
            const uint4 x0 = xs[xcol[j]];
            const uint4 x1 = xs[ldsw + xcol[j]];
            const uint32_t xpair[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t words[4] = {wv[r][j].x, wv[r][j].y, wv[r][j].z, wv[r][j].w};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t u = words[q];
                    const f16x2 qp = as_f16x2((u & 0x00FF00FFu) ^ 0x64806480u) + bias;
                    const f16x2 qq = as_f16x2(((u >> 8) & 0x00FF00FFu) ^ 0x64806480u) + bias;
                    acc[r] = __builtin_amdgcn_fdot2(qp, as_f16x2(xpair[2 * q]), acc[r], false);
                    acc[r] = __builtin_amdgcn_fdot2(qq, as_f16x2(xpair[2 * q + 1]), acc[r], false);
                }
            }
        }
        __syncthreads();
    };
    int c0 = 0;
    for (; c0 + TC <= nchunks; c0 += TC) tile.template operator()<false>(c0, TC);
    if (c0 < nchunks) tile.template operator()<true>(c0, nchunks - c0);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float a = segment_sum<64>(acc[r]);
        const int64_t row = row0 + r;
        if (col == 63 && row < n) y[row] = f2h(sc[r] * a);
    }
}

// Tile size of the K-tiled kernels (chunks per lane per tile); 256-thread
// workgroups throughout.  Measured on MI355X over HBM-cold pools, every
// instance bit-identical:
// - INT4, one row per wave: 7 chunks per lane per tile.  Against 8 it avoids
//   a small last tile (k = 28672 splits into two full tiles of 7): 1-13%
//   faster at 512..3072 x 20480..53248, level at 65536.
// - INT4, two rows per wave: 2 chunks per lane per tile while the row has at
//   most 16 chunks per lane (k <= 32768, at most 8 tiles): 2-8% faster than 4
//   at 4096..16384 x 20480..28672; with more tiles the barriers cost more
//   than the smaller tile saves (4096x65536: 5% slower), so 4 there.
// - INT8 (tiles of an even number of chunks, so that a tile's x pieces
//   divide over the workgroup): two rows per wave with 4 chunks per lane
//   per tile, one row with 8.  2, 6 and 14 were no faster (14 spills).
constexpr int int4_tile_j(int r, int j) { return r == 1 ? 7 : (j <= 16 ? 2 : 4); }
constexpr int q8_tile_j(int r) { return r == 2 ? 4 : 8; }
// LDS bytes of one tile of `tj` chunks per lane: `pieces` 16-byte x pieces
// per chunk (INT4 4, INT8 2), plus the zero column.
constexpr uint32_t tile_lds(int pieces, int tj) {
    return static_cast<uint32_t>(pieces) * (tj * 64 + 1) * 16u;
}

// Several independent problems of one k per launch (grouped GEMV).  Logical
// workgroups [start[p], start[p+1]) belong to problem p, and each computes
// exactly the rows it would compute in a launch of that problem alone, so
// the outputs are bit-identical to separate launches.
//
// What a workgroup needs before its first load travels in the kernel
// arguments that the hardware preloads into scalar registers (the first 14
// words), and the prefix sums of the workgroup counts are computed from the
// row counts: a workgroup that first has to read a table from the argument
// memory stands still for each dependent read (a table cost 0.7-1.2 us a
// launch: four dependent reads):
// - Group3 (up to three problems with one x: q/k/v, gate/up): x, the weights
//   and the row counts are preloaded; scale and y are read behind the first
//   weight loads.
// - Group8 (any other group): the row counts are preloaded; one 32-byte read
//   brings the problem's pointers.
// INT4 us per call, with the table and now (problems with one x): 3 x
// 4096x4096 7.6 -> 6.4 (one matrix of the same rows 6.3), 2 x 11008x4096
// 10.9 -> 9.7, 1024 + 256 + 256 x 1024 3.17 -> 2.22; with an x each: 3 x
// 4096x4096 6.7, 1024 + 256 + 256 x 1024 2.54.
constexpr int log2_of(int v) { return v <= 1 ? 0 : 1 + log2_of(v / 2); }

// Selects of values: written on the arguments themselves, they would select
// among the arguments' addresses and put the arguments into scratch memory
// (a grouped launch then takes twice as long).
template <typename T>
__device__ __forceinline__ T pick2(bool second, T a, T b) { return second ? b : a; }
template <typename T>
__device__ __forceinline__ T pick3(int p, T a, T b, T c) {
    return pick2(p == 2, pick2(p == 1, a, b), c);
}

template <int ROWS, uint32_t RUN, int COUNT>   // rows per workgroup, run of xcd_block
__device__ __forceinline__ RowSlot group_slot(const int (&n)[COUNT]) {
    constexpr int kShift = log2_of(ROWS);
    static_assert(ROWS == 1 << kShift, "rows per workgroup are a power of two");
    uint32_t start[COUNT + 1] = {0};
#pragma unroll
    for (int i = 0; i < COUNT; ++i)
        start[i + 1] = start[i] + ((static_cast<uint32_t>(n[i]) + ROWS - 1) >> kShift);
    const uint32_t lb = xcd_block<RUN>(blockIdx.x, start[COUNT]);
    RowSlot s{0, lb, n[0]};
#pragma unroll
    for (int i = 1; i < COUNT; ++i) {
        const bool past = lb >= start[i];       // absent problems have no workgroups
        s.p = pick2(past, s.p, i);
        s.blk = pick2(past, s.blk, lb - start[i]);
        s.n = pick2(past, s.n, n[i]);
    }
    return s;
}

// A second copy of problem p's output with every run of 2^shift rows (a head)
// written `times` times in a row.  It is written with the rows themselves: a
// decode step that repeats v for its query heads paid a copy launch of its own
// for it (two 70B layers as a graph 165.9 us with the copy, 159.4 without).
struct RepeatRows {
    uint16_t* y;
    int p, shift, times;
};

// Up to three problems with one x.  Rep is RepeatRows, or NoRepeat in the
// kernels without a second copy (its test and arguments cost the other groups
// 0.02-0.05 us a launch).
struct NoRepeat {};
template <typename S, int ROWS, uint32_t RUN, class Rep>
struct Group3 {
    const uint4* w_[3];
    const S* scale_[3];
    uint16_t* y_[3];
    int n_[3];
    Rep rep_;
    __device__ __forceinline__ RowSlot slot() const { return group_slot<ROWS, RUN>(n_); }
    __device__ __forceinline__ const uint4* w(const RowSlot& s) const {
        return pick3(s.p, w_[0], w_[1], w_[2]);
    }
    __device__ __forceinline__ const S* scale(const RowSlot& s) const {
        return pick3(s.p, scale_[0], scale_[1], scale_[2]);
    }
    __device__ __forceinline__ void store(const RowSlot& s, int64_t row, uint16_t v) const {
        pick3(s.p, y_[0], y_[1], y_[2])[row] = v;
        if constexpr (std::is_same_v<Rep, RepeatRows>) {
            if (s.p != rep_.p) return;
            const int64_t head = row >> rep_.shift;
            uint16_t* y = rep_.y + ((head * rep_.times) << rep_.shift) +
                          (row - (head << rep_.shift));
            for (int t = 0; t < rep_.times; ++t) y[static_cast<int64_t>(t) << rep_.shift] = v;
        }
    }
};

// A problem of a larger group, its slot known before x.
template <typename S>
struct OneSlot {
    const uint4* w_;
    const S* scale_;
    uint16_t* y_;
    RowSlot s_;
    __device__ __forceinline__ RowSlot slot() const { return s_; }
    __device__ __forceinline__ const uint4* w(const RowSlot&) const { return w_; }
    __device__ __forceinline__ const S* scale(const RowSlot&) const { return scale_; }
    __device__ __forceinline__ void store(const RowSlot&, int64_t row, uint16_t v) const {
        y_[row] = v;
    }
};

struct GroupRecord {
    const void* w;
    const void* scale;
    const void* x;
    void* y;
};
struct Group8Records {
    GroupRecord r[kMaxGroup];
};

template <int CW, int J, int R, int NT, class Rep>
__global__ __launch_bounds__(NT) void int4gemv_lds_group3_kernel(
        const uint4* x, const uint4* w0, const uint4* w1, const uint4* w2, int n0,
        int n1, int n2, int nchunks, const uint16_t* s0, const uint16_t* s1, const uint16_t* s2,
        uint16_t* y0, uint16_t* y1, uint16_t* y2, Rep rep) {
    extern __shared__ uint4 xs[];
    constexpr int kRows = 64 / CW * R * (NT / 64);
    int4_lds_rows<CW, J, R, NT>(x, nchunks, xs,
        Group3<uint16_t, kRows, xcd_run(J * R), Rep>{{w0, w1, w2}, {s0, s1, s2}, {y0, y1, y2},
                                               {n0, n1, n2}, rep});
}

template <int CW, int J, int R, int NT>
__global__ __launch_bounds__(NT) void int4gemv_lds_group8_kernel(
        int n0, int n1, int n2, int n3, int n4, int n5, int n6, int n7, int nchunks,
        Group8Records g) {
    extern __shared__ uint4 xs[];
    const int n[kMaxGroup] = {n0, n1, n2, n3, n4, n5, n6, n7};
    const RowSlot s = group_slot<64 / CW * R * (NT / 64), xcd_run(J * R)>(n);
    const GroupRecord r = g.r[s.p];
    int4_lds_rows<CW, J, R, NT>(static_cast<const uint4*>(r.x), nchunks, xs,
        OneSlot<uint16_t>{static_cast<const uint4*>(r.w), static_cast<const uint16_t*>(r.scale),
                    static_cast<uint16_t*>(r.y), s});
}

template <int CW, int J, int R, int NT, class Rep>
__global__ __launch_bounds__(NT) void qgemv_lds_group3_kernel(
        const uint4* x, const uint4* w0, const uint4* w1, const uint4* w2, int n0,
        int n1, int n2, int nchunks, const float* s0, const float* s1, const float* s2,
        uint16_t* y0, uint16_t* y1, uint16_t* y2, Rep rep) {
    extern __shared__ uint4 xs[];
    constexpr int kRows = 64 / CW * R * (NT / 64);
    q8_lds_rows<CW, J, R, NT>(x, nchunks, xs,
        Group3<float, kRows, xcd_run(J * R), Rep>{{w0, w1, w2}, {s0, s1, s2}, {y0, y1, y2},
                                               {n0, n1, n2}, rep});
}

template <int CW, int J, int R, int NT>
__global__ __launch_bounds__(NT) void qgemv_lds_group8_kernel(
        int n0, int n1, int n2, int n3, int n4, int n5, int n6, int n7, int nchunks,
        Group8Records g) {
    extern __shared__ uint4 xs[];
    const int n[kMaxGroup] = {n0, n1, n2, n3, n4, n5, n6, n7};
    const RowSlot s = group_slot<64 / CW * R * (NT / 64), xcd_run(J * R)>(n);
    const GroupRecord r = g.r[s.p];
    q8_lds_rows<CW, J, R, NT>(static_cast<const uint4*>(r.x), nchunks, xs,
        OneSlot<float>{static_cast<const uint4*>(r.w), static_cast<const float*>(r.scale),
                    static_cast<uint16_t*>(r.y), s});
}

// ------------------------------------------------------------- FP16/FP32
//
// The reference's FP16/FP32 GEMV (kernels/gemv/gemv_common.h:1-79):
// y[n] = sum_k W[n,k] * x[k] accumulated in FP32 and cast once to the
// dtype of W (RNE for fp16).  W and x are fp16 or fp32, same dtype.

__device__ __forceinline__ void fp_store(uint16_t* p, float v) { *p = f2h(v); }
__device__ __forceinline__ void fp_store(float* p, float v) { *p = v; }

// One 16-byte chunk of W against the matching chunk of x, into acc, one
// FMA per element: fp16 operands go straight into v_fma_mix_f32 (the
// fp16 x fp16 product is exact in FP32, the add is one round-to-nearest-
// even), fp32 as plain FMAs.  v_dot2_f32_f16 would halve the instructions
// but measured on gfx950 it is not a single RNE rounding (about 1% of
// random operands differ from one, in a sign-asymmetric way), and this
// path is memory-bound at 2 or 4 bytes per element, so the FMA costs
// nothing.
__device__ __forceinline__ float fma_pair(uint32_t w, uint32_t x, float acc) {
    const f16x2 a = as_f16x2(w), b = as_f16x2(x);
    acc = __builtin_fmaf(static_cast<float>(a[0]), static_cast<float>(b[0]), acc);
    return __builtin_fmaf(static_cast<float>(a[1]), static_cast<float>(b[1]), acc);
}
// Four independent accumulators per lane (one per 32-bit word of a chunk)
// keep consecutive FMAs free of dependencies; they are summed at the end.
__device__ __forceinline__ void dot_chunk(uint16_t, const uint4& w,
                                          const uint4& x, float (&acc)[4]) {
    acc[0] = fma_pair(w.x, x.x, acc[0]);
    acc[1] = fma_pair(w.y, x.y, acc[1]);
    acc[2] = fma_pair(w.z, x.z, acc[2]);
    acc[3] = fma_pair(w.w, x.w, acc[3]);
}
__device__ __forceinline__ void dot_chunk(float, const uint4& w,
                                          const uint4& x, float (&acc)[4]) {
    acc[0] = __builtin_fmaf(__builtin_bit_cast(float, w.x), __builtin_bit_cast(float, x.x), acc[0]);
    acc[1] = __builtin_fmaf(__builtin_bit_cast(float, w.y), __builtin_bit_cast(float, x.y), acc[1]);
    acc[2] = __builtin_fmaf(__builtin_bit_cast(float, w.z), __builtin_bit_cast(float, x.z), acc[2]);
    acc[3] = __builtin_fmaf(__builtin_bit_cast(float, w.w), __builtin_bit_cast(float, x.w), acc[3]);
}

// Vector: CW lanes per row (64/CW rows per wave), lane `col` owns the
// 16-byte chunks col + CW*j.  x is staged once per workgroup in LDS
// ([nchunks + 1] chunks, the last one zero: what lanes past the row end
// read).  The lane's W chunks stream through two register batches of JB
// chunks: batch b+1 is in flight while batch b is multiplied, so any K
// runs with a bounded register budget.  The loop's loads are unconditional (the
// last batch is peeled): after a load under a condition the compiler no longer
// knows how many are in flight and waits for all of them before it multiplies.
// FP16 4096x11008 17.4 -> 17.2 us (a graph's calls), 1000x30000 13.8 -> 13.6,
// FP32 2000x14000 26.9 -> 26.7, others level.  (The K-tiled kernel below keeps
// its conditional loads: four batches a tile between two barriers gained
// nothing.)
constexpr int kGemvBatch = 8;

// A chunk of x on its way to LDS is held as a vector: a uint4 that is only
// copied is forwarded from x to LDS as one memory copy, which moves the load
// behind the weight loads, and the barrier then waits for all of them (us per
// call of a graph that way and with x first: FP16 1024x4096 3.57, 3.23;
// 1024x16384 8.17, 7.89; FP32 1024x4096 5.16, 4.55; 4096^2 level; on the K-tiled
// kernel FP16 3000x65536 121, 70.7, FP32 1000x30000 37.6, 24.0).
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x4 load_chunk(const uint4* p) {
    return *reinterpret_cast<const u32x4*>(p);
}
__device__ __forceinline__ void store_chunk(uint4* p, u32x4 v) {
    *reinterpret_cast<u32x4*>(p) = v;
}

// Chunk w of a row, or zero where the lane re-read it past the row end.  x is
// zero there too, but 0 * w is NaN where w is infinite.  Only LDS reads may be
// scheduled across: moved ahead of the earlier chunks' products, the selects
// wait for every load of the batch (us per call of a graph: FP16 1024x4096
// 3.34, in place 3.23, without the selects 3.22; in place and without them
// 4096^2 7.22, 7.16, 4096x11008 17.2, 17.1).
__device__ __forceinline__ uint4 if_in_row(bool in, const uint4& w) {
    __builtin_amdgcn_sched_barrier(0x100);
    return {in ? w.x : 0u, in ? w.y : 0u, in ? w.z : 0u, in ? w.w : 0u};
}

// JB: chunks per lane per register batch.  ONE: the row is one batch of
// exactly the lane's chunk count (only its last chunk can pass the row end);
// the kernel is then a third of the size, and all of x is staged in one pass.
// Longer rows go in batches of kGemvBatch.
template <typename S, int CW, int NT, int JB, bool ONE>
__global__ __launch_bounds__(NT) void gemv_lds_kernel(
        const uint4* __restrict__ w,   // [n][nchunks] 16-byte chunks
        const uint4* __restrict__ x,   // [nchunks] 16-byte chunks
        S* __restrict__ y, int n, int nchunks) {
    extern __shared__ uint4 xs[];
    constexpr int SLOTS = 64 / CW;
    // x chunks per thread per staging pass (all of x where the row is one batch)
    constexpr int XB = ONE ? (CW * JB + NT - 1) / NT : 4;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int col = lane % CW;
    const int slot = lane / CW;
    // x first (the barrier waits for it), in passes of XB chunks per thread
    u32x4 xv[XB];
#pragma unroll
    for (int i = 0; i < XB; ++i) xv[i] = load_chunk(x + std::min(tid + i * NT, nchunks - 1));
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t blk = xcd_block<kXcdAll>();
    const int64_t row =
        (static_cast<int64_t>(blk) * (NT >> 6) + (tid >> 6)) * SLOTS + slot;
    const uint32_t rowc = static_cast<uint32_t>(std::min<int64_t>(row, n - 1));
    const char* wb = reinterpret_cast<const char*>(w);
    const uint32_t wrow_bytes = static_cast<uint32_t>(nchunks) * 16u;
    const int nbatch = ((nchunks + CW - 1) / CW + JB - 1) / JB;

    uint4 wa[JB];
    constexpr int kOneFull = ONE ? JB - 1 : 0;   // chunks that are inside the row
    auto load = [&](uint4 (&dst)[JB], int b) {
#pragma unroll
        for (int jj = 0; jj < JB; ++jj) {
            const int c = col + CW * (b * JB + jj);
            const uint32_t cl =
                static_cast<uint32_t>(jj < kOneFull || c < nchunks ? c : nchunks - 1);
            dst[jj] = *reinterpret_cast<const uint4*>(wb + (rowc * wrow_bytes + cl * 16u));
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    load(wa, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < XB; ++i) store_chunk(xs + std::min(tid + i * NT, nchunks - 1), xv[i]);
#pragma unroll 1
    for (int base = XB * NT; !ONE && base < nchunks; base += XB * NT) {   // K beyond one pass
#pragma unroll
        for (int i = 0; i < XB; ++i)
            xv[i] = load_chunk(x + std::min(base + tid + i * NT, nchunks - 1));
#pragma unroll
        for (int i = 0; i < XB; ++i)
            store_chunk(xs + std::min(base + tid + i * NT, nchunks - 1), xv[i]);
    }
    if (tid == 0) xs[nchunks] = uint4{0, 0, 0, 0};
    __syncthreads();

    float accs[4] = {0.f, 0.f, 0.f, 0.f};
    // The first FULL chunks of the batch are inside the row in every lane.
    // CLAMP: their x is read as if they might not be (in the loop below the
    // compiler then keeps two LDS reads in flight: FP16 1024x16384 7.90 us
    // against 8.05).  The last whole chunk stays behind the others for the
    // reason given at if_in_row.
    auto comp = [&]<int FULL, bool CLAMP = false>(const uint4 (&src)[JB], int b) {
#pragma unroll
        for (int jj = 0; jj < JB; ++jj) {
            const int c = col + CW * (b * JB + jj);
            if (!CLAMP && jj == FULL - 1) __builtin_amdgcn_sched_barrier(0x100);
            if (jj < FULL) dot_chunk(S{}, src[jj], xs[CLAMP ? std::min(c, nchunks) : c], accs);
            else dot_chunk(S{}, if_in_row(c < nchunks, src[jj]), xs[std::min(c, nchunks)], accs);
        }
    };
    if constexpr (ONE) {
        comp.template operator()<kOneFull>(wa, 0);
    } else {
        uint4 wn[JB];
        // a last batch that the row fills needs no selects (FP32 1024x4096
        // 4.54 us against 4.65; a row of one batch is no faster for it)
        auto last = [&](const uint4 (&src)[JB], int b) {
            if (nchunks % (CW * JB) == 0) comp.template operator()<JB>(src, b);
            else comp.template operator()<0>(src, b);
        };
        int b = 0;
        for (; b + 2 < nbatch; b += 2) {
            load(wn, b + 1);
            comp.template operator()<JB, true>(wa, b);
            load(wa, b + 2);
            comp.template operator()<JB, true>(wn, b + 1);
        }
        if (b + 1 < nbatch) {
            load(wn, b + 1);
            comp.template operator()<JB, true>(wa, b);
            last(wn, b + 1);
        } else {
            last(wa, b);
        }
    }
    float acc = (accs[0] + accs[1]) + (accs[2] + accs[3]);
    acc = segment_sum<CW>(acc);
    if (col == CW - 1 && row < n) fp_store(y + row, acc);
}

// K-tiled FP16/FP32 GEMV, for rows whose x does not fit the 64 KiB stage
// (k > 32768 fp16, > 16384 fp32; gemv_lds_tiled forces it at any k).  64
// lanes per row, one row per wave.  x is staged tile by tile (kGemvTileJ
// chunks per lane per tile, 32 KB), with a barrier before the tile is read
// and one before the next tile overwrites it; every thread runs the same
// tiles (they depend on nchunks only; rows past n are clamped), so every
// barrier is reached by all.  Within a tile the lane's W chunks stream
// through two register batches of kGemvBatch chunks as in gemv_lds_kernel.
// Lane `col` takes chunks col + 64 j in j order, so where x fits one stage
// the sums are bit-identical to gemv_lds_kernel with CW = 64.
constexpr int kGemvTileJ = 4 * kGemvBatch;    // 32 chunks per lane per tile
constexpr uint32_t kGemvTileLds = (kGemvTileJ * 64 + 1) * 16u;   // 32,784 B

// ONE: the row is shorter than a tile (gemv_lds_tiled at such k, or weights of
// 4 GiB and more).  A kernel of its own, as the loop over whole tiles takes 168
// VGPRs with fp16 and halves the workgroups per CU: FP16 4096^2 7.6 us against
// 8.8.
template <typename S, int NT, bool ONE>
__global__ __launch_bounds__(NT) void gemv_tiled_kernel(
        const uint4* __restrict__ w,   // [n][nchunks] 16-byte chunks
        const uint4* __restrict__ x,   // [nchunks] 16-byte chunks
        S* __restrict__ y, int n, int nchunks) {
    extern __shared__ uint4 xs[];                 // [TC + 1], the last zero
    constexpr int JB = kGemvBatch;
    constexpr int TC = kGemvTileJ * 64;           // chunks per tile
    constexpr int XPER = TC / NT;                 // x chunks per thread per tile
    static_assert(TC % NT == 0, "a tile's chunks divide over the workgroup");
    const int tid = threadIdx.x;
    const int col = tid & 63;
    const int64_t row = static_cast<int64_t>(xcd_block<kXcdAll>()) * (NT >> 6) + (tid >> 6);
    const uint64_t rowc = static_cast<uint64_t>(std::min<int64_t>(row, n - 1));
    const char* wrow = reinterpret_cast<const char*>(w) +
                       rowc * (static_cast<uint32_t>(nchunks) * 16u);
    float accs[4] = {0.f, 0.f, 0.f, 0.f};
    auto tile = [&]<bool PARTIAL>(int c0, int tc) {           // chunks [c0, c0 + tc)
        const int nbatch = ((tc + 63) / 64 + JB - 1) / JB;    // wave-uniform
        const uint4* xt = x + c0;
        u32x4 xv[XPER];
#pragma unroll
        for (int i = 0; i < XPER; ++i) xv[i] = load_chunk(xt + std::min(tid + i * NT, tc - 1));
        __builtin_amdgcn_sched_barrier(0);
        uint4 wa[JB], wn[JB];
        auto load = [&](uint4 (&dst)[JB], int b) {
#pragma unroll
            for (int jj = 0; jj < JB; ++jj) {
                const int c = col + 64 * (b * JB + jj);
                const uint32_t cl = static_cast<uint32_t>(c0 + (c < tc ? c : tc - 1));
                dst[jj] = *reinterpret_cast<const uint4*>(wrow + cl * 16u);
            }
        };
        load(wa, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < XPER; ++i) store_chunk(xs + std::min(tid + i * NT, tc - 1), xv[i]);
        if (tid == 0) xs[TC] = uint4{0, 0, 0, 0};
        __syncthreads();
        auto comp = [&](const uint4 (&src)[JB], int b) {
#pragma unroll
            for (int jj = 0; jj < JB; ++jj) {
                const int c = col + 64 * (b * JB + jj);
                if (PARTIAL) dot_chunk(S{}, if_in_row(c < tc, src[jj]), xs[c < tc ? c : TC], accs);
                else dot_chunk(S{}, src[jj], xs[c], accs);
            }
        };
        for (int b = 0; b < nbatch; b += 2) {
            if (b + 1 < nbatch) load(wn, b + 1);
            comp(wa, b);
            if (b + 1 < nbatch) {
                if (b + 2 < nbatch) load(wa, b + 2);
                comp(wn, b + 1);
            }
        }
        __syncthreads();
    };
    if constexpr (ONE) {
        tile.template operator()<true>(0, nchunks);
    } else {
        int c0 = 0;
        for (; c0 + TC <= nchunks; c0 += TC) tile.template operator()<false>(c0, TC);
        if (c0 < nchunks) tile.template operator()<true>(c0, nchunks - c0);
    }
    float acc = (accs[0] + accs[1]) + (accs[2] + accs[3]);
    acc = segment_sum<64>(acc);
    if (col == 63 && row < n) fp_store(y + row, acc);
}

// The copy RepeatRows describes, for outputs the grouped kernels did not
// write it with.
__global__ __launch_bounds__(kBlock) void repeat_rows_kernel(
        const uint16_t* __restrict__ src, uint16_t* __restrict__ dst, int n, int head,
        int times) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= n) return;
    const int64_t h = i / head;
    const uint16_t v = src[i];
    for (int t = 0; t < times; ++t) dst[(h * times + t) * head + (i - h * head)] = v;
}

// ------------------------------------------------- read-only ceiling
//
// A plain streaming read of `bytes`, one 16-byte load per thread.  Of the
// read patterns measured for one 8.67 MB launch over an HBM-cold pool (1, 2,
// 4, 8 or 16 loads per thread at 256, 512 or 1024 threads, strided or
// contiguous, with and without the nontemporal hint), one load per thread
// in 256-thread workgroups was fastest (2.89 us; 4 loads per thread 3.18 us,
// 16 loads 3.49 us): the most waves, each with the shortest dependency.  The
// loaded words are folded and compared with `key`, a launch argument the
// compiler cannot see, so the loads cannot be removed; the store to `sink`
// runs only if a thread's fold equals the key (harmless either way: sink is
// the caller's scratch word).  It is the measured bandwidth ceiling of one
// launch that reads the same number of bytes as a GEMV call.
__global__ __launch_bounds__(kBlock) void stream_read_kernel(
        const uint4* __restrict__ p, uint32_t* __restrict__ sink, int64_t n16,
        uint32_t key) {
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    const uint4 v = p[idx < n16 ? idx : n16 - 1];
    const uint32_t a = v.x ^ v.y ^ v.z ^ v.w;
    if (a == key) sink[0] = a;
}

// A workgroup that does no memory work: launched back to back on one stream
// it measures what one dispatch of a given grid and workgroup size costs
// before any kernel body runs (command processing, workgroup launch, the
// end-of-kernel release).  The store is never taken: the host passes a key
// no thread index reaches.
__global__ __launch_bounds__(1024) void empty_launch_kernel(
        uint32_t* __restrict__ sink, uint32_t key) {
    if (threadIdx.x == key) sink[0] = blockIdx.x;
}

// A bounded on-device wait for the timing loops: one wave sleeps until the
// constant-rate wall clock has advanced `ticks`, or until it has gone round
// its loop `max_iters` times, whichever comes first (so it ends even if the
// clock were not running).  Queued ahead of a timed window it keeps the GPU
// busy while the host enqueues the window's launches, so the window times
// the GPU and not the host's submission rate (about 2.5-3.5 us per launch
// on MI355X, close to a short GEMV's own time).  It touches no memory.
__global__ __launch_bounds__(64) void delay_kernel(uint64_t ticks,
                                                   uint64_t max_iters) {
    const uint64_t t0 = wall_clock64();
    for (uint64_t i = 0; i < max_iters; ++i) {
        if (wall_clock64() - t0 >= ticks) break;
        __builtin_amdgcn_s_sleep(8);
    }
}

// --------------------------------------------------------- instance tables

using Int4Fn = void (*)(const uint4*, const uint16_t*, const uint4*,
                        uint16_t*, int, int);
using Q8Fn = void (*)(const uint4*, const float*, const uint4*, uint16_t*,
                      int, int);

// One traits type per kernel family: the instance for (CW, J, R), or null
// where the register budget does not allow R rows per lane at J chunks.
struct Int4Wave {
    using Fn = Int4Fn;
    static constexpr int kMaxJ = kInt4MaxJ;
    template <int CW, int J, int R>
    static constexpr Fn get() {
        if constexpr (R <= int4_rmax(J)) return &int4gemv_wave_kernel<CW, J, R>;
        else return nullptr;
    }
};
// The INT4 plans take 512-thread workgroups only with one row per lane
// (lds_threads), so only those instances exist at 512 threads.
template <int NT, int R>
constexpr bool int4_lds_shape(int j) {
    return R <= int4_rmax(j) && (NT != 512 || R == 1);
}
template <int NT>
struct Int4Lds {
    using Fn = Int4Fn;
    static constexpr int kMaxJ = kInt4MaxJ;
    template <int CW, int J, int R>
    static constexpr Fn get() {
        if constexpr (int4_lds_shape<NT, R>(J)) return &int4gemv_lds_kernel<CW, J, R, NT>;
        else return nullptr;
    }
};
struct Q8Wave {
    using Fn = Q8Fn;
    static constexpr int kMaxJ = kQ8MaxJ;
    template <int CW, int J, int R>
    static constexpr Fn get() {
        if constexpr (R <= q8_rmax(J)) return &qgemv_wave_kernel<CW, J, R>;
        else return nullptr;
    }
};
template <int NT>
struct Q8Lds {
    using Fn = Q8Fn;
    static constexpr int kMaxJ = kQ8MaxJ;
    template <int CW, int J, int R>
    static constexpr Fn get() {
        if constexpr (R <= q8_rmax(J)) return &qgemv_lds_kernel<CW, J, R, NT>;
        else return nullptr;
    }
};

using Int4StampFn = void (*)(const uint4*, const uint16_t*, const uint4*,
                             uint16_t*, int, int, uint64_t*);
template <int NT>
struct Int4LdsStamp {
    using Fn = Int4StampFn;
    static constexpr int kMaxJ = kInt4MaxJ;
    template <int CW, int J, int R>
    static constexpr Fn get() {
        if constexpr (int4_lds_shape<NT, R>(J)) return &int4gemv_lds_stamp_kernel<CW, J, R, NT>;
        else return nullptr;
    }
};

template <typename S, class Rep>
using Group3Fn = void (*)(const uint4*, const uint4*, const uint4*, const uint4*, int,
                          int, int, int, const S*, const S*, const S*, uint16_t*,
                          uint16_t*, uint16_t*, Rep);
using Group8Fn = void (*)(int, int, int, int, int, int, int, int, int, Group8Records);

template <int NT, class Rep>
struct Int4LdsGroup3 {
    using Fn = Group3Fn<uint16_t, Rep>;
    static constexpr int kMaxJ = kInt4MaxJ;
    template <int CW, int J, int R>
    static constexpr Fn get() {
        if constexpr (R <= int4_rmax(J)) return &int4gemv_lds_group3_kernel<CW, J, R, NT, Rep>;
        else return nullptr;
    }
};
template <int NT>
struct Int4LdsGroup8 {
    using Fn = Group8Fn;
    static constexpr int kMaxJ = kInt4MaxJ;
    template <int CW, int J, int R>
    static constexpr Fn get() {
        if constexpr (R <= int4_rmax(J)) return &int4gemv_lds_group8_kernel<CW, J, R, NT>;
        else return nullptr;
    }
};
template <int NT, class Rep>
struct Q8LdsGroup3 {
    using Fn = Group3Fn<float, Rep>;
    static constexpr int kMaxJ = kQ8MaxJ;
    template <int CW, int J, int R>
    static constexpr Fn get() {
        if constexpr (R <= q8_rmax(J)) return &qgemv_lds_group3_kernel<CW, J, R, NT, Rep>;
        else return nullptr;
    }
};
template <int NT>
struct Q8LdsGroup8 {
    using Fn = Group8Fn;
    static constexpr int kMaxJ = kQ8MaxJ;
    template <int CW, int J, int R>
    static constexpr Fn get() {
        if constexpr (R <= q8_rmax(J)) return &qgemv_lds_group8_kernel<CW, J, R, NT>;
        else return nullptr;
    }
};

constexpr int r_index(int r) { return r == 1 ? 0 : (r == 2 ? 1 : 2); }

template <class F, int CW, int J>
typename F::Fn pick_r(int r) {
    static constexpr typename F::Fn t[3] = {F::template get<CW, J, 1>(),
                                            F::template get<CW, J, 2>(),
                                            F::template get<CW, J, 4>()};
    return t[r_index(r)];
}

template <class F, int... Js>
typename F::Fn pick_j64(int j, int r, std::integer_sequence<int, Js...>) {
    typename F::Fn f = nullptr;
    ((j == Js + 1 ? (f = pick_r<F, 64, Js + 1>(r), 0) : 0), ...);
    return f;
}

template <class F>
typename F::Fn instance(int cw, int j, int r) {
    if (cw == 16 && j == 1) return pick_r<F, 16, 1>(r);
    if (cw == 32 && j == 1) return pick_r<F, 32, 1>(r);
    if (cw == 64 && j >= 1 && j <= F::kMaxJ)
        return pick_j64<F>(j, r, std::make_integer_sequence<int, F::kMaxJ>{});
    return nullptr;
}

// Launch with the argument types taken from the kernel's own signature.
template <typename... Params>
hipError_t launch(void (*kernel)(Params...), int64_t grid, int block,
                  uint32_t shmem, hipStream_t stream, hipEvent_t ev0,
                  hipEvent_t ev1, std::type_identity_t<Params>... args) {
    void* argv[] = {static_cast<void*>(&args)...};
    const dim3 g(static_cast<uint32_t>(grid)), b(static_cast<uint32_t>(block));
    if (ev0 == nullptr && ev1 == nullptr)
        return hipLaunchKernel(reinterpret_cast<const void*>(kernel), g, b,
                               argv, shmem, stream);
    return hipExtLaunchKernel(reinterpret_cast<const void*>(kernel), g, b,
                              argv, shmem, stream, ev0, ev1, 0);
}

// The same launch resolved into a Launch record instead of enqueued: the
// kernel, its shape and its arguments, each argument copied into an 8-byte
// slot (the runtime reads each argument's own size from the slot's start).
template <typename... Params>
hipError_t bind(Launch* out, void (*kernel)(Params...), int64_t grid,
                int block, uint32_t shmem, std::type_identity_t<Params>... args) {
    static_assert(sizeof...(Params) <= kMaxLaunchArgs, "too many kernel arguments");
    static_assert(((sizeof(Params) <= 8 && std::is_trivially_copyable_v<Params>) && ...),
                  "kernel arguments must fit an 8-byte slot");
    if (grid < 1 || grid > UINT32_MAX) return hipErrorInvalidConfiguration;
    Launch L;
    L.fn = reinterpret_cast<const void*>(kernel);
    L.grid = static_cast<uint32_t>(grid);
    L.block = static_cast<uint32_t>(block);
    L.shmem = shmem;
    L.nargs = sizeof...(Params);
    int i = 0;
    ((std::memcpy(&L.args[i++], &args, sizeof(args))), ...);
    *out = L;
    return hipSuccess;
}

// Instances of the scalar kernels that scalar_plan can ask for.
struct Int4Scalar {
    template <int R, int U, int SP>
    static constexpr auto get() { return &int4gemv_scalar_kernel<R, U, SP>; }
};
struct Q8Scalar {
    template <int R, int U, int SP>
    static constexpr auto get() { return &qgemv_scalar_kernel<R, U, SP>; }
};
template <typename S>
struct GemvScalar {
    template <int R, int U, int SP>
    static constexpr auto get() { return &gemv_scalar_kernel<S, R, U, SP>; }
};
template <class F>
auto scalar_instance(const Plan& p) {
    if (p.split == 1) return p.r == 1 ? F::template get<1, 1, 1>() : F::template get<2, 1, 1>();
    if (p.split == 2) return p.r == 1 ? F::template get<1, 1, 2>() : F::template get<2, 1, 2>();
    if (p.batch == 1) return p.r == 1 ? F::template get<1, 1, 4>() : F::template get<2, 1, 4>();
    return p.r == 1 ? F::template get<1, 2, 4>() : F::template get<2, 2, 4>();
}

int pow2_at_least(int64_t v, int lo) {
    int p = lo;
    while (p < v && p < 64) p <<= 1;
    return p;
}

// Default rows per lane (measured on MI355X with kernel arguments
// preloaded, HBM-cold pools, back-to-back launches on a pre-filled queue;
// every candidate bit-identical).  INT4 with at most 3 chunks per lane:
// - rows of at most 32 chunks (64 // CW >= 2 row slots per wave): two rows
//   (4096x1024: 2.39 us against 2.55);
// - otherwise one row while one row per wave keeps the whole grid resident
//   (at most 32 waves per CU on kCus CUs), two above, where one row per wave
//   would run a second round of waves: 4096^2 one row 3.38 us against two
//   3.56-3.63; 6144x4096 4.18 against 4.34; 11008x4096 two rows 6.05 against
//   6.36; 14336x4096 7.41 against 7.65; 13824x5120 9.32 against 10.14.
// With 4 or more chunks per lane one row throughout (8192^2 8.19 us against
// 9.01, 28672x8192 24.3 against 25.0).  INT8 does best with one row per lane
// at every shape measured.
constexpr int64_t kCus = 256;
constexpr int64_t kResidentWaves = 32 * kCus;
int default_rows_int4(int64_t n, int slots, int j, int rmax) {
    if (j > 3 || rmax < 2) return 1;
    if (slots >= 2) return 2;
    return n > kResidentWaves ? 2 : 1;
}

// Workgroup size of the LDS kernels.  512 threads halve the number of
// workgroups that stage x.  Measured on MI355X (same launch path, HBM-cold
// pools) this pays when x is large next to each workgroup's weights (INT4
// with one row per lane, INT8 with 8+ chunks per lane: 4096x11008 INT4
// 7.44 -> 6.93 us, INT8 10.48 -> 9.88 us) and the 512-thread grid fills the
// CUs in whole rounds (a multiple of kCus workgroups) or runs many (8+) of
// them.  A partial round among few costs
// more than the staging saves: 5120x13824 (640 workgroups of 512, 2.5
// rounds; 1280 of 256) INT4 10.2 us with 512 threads, 9.8 with 256, INT8
// 15.4 and 14.6; 5120^2 INT4 5.15 and 4.8.  Among many rounds the partial
// one matters less: 27648x5120 (13.5 rounds) 15.8-16.0 us with 512, 16.0-16.3
// with 256.  INT8 at K = 4096 was 1-3% slower with 512.
// True when `waves` in 512-thread workgroups fill the CUs in whole rounds
// or in 8+ rounds (the condition for 512-thread plans, all operators).
bool rounds_ok_512(int64_t waves) {
    const int64_t grid = (waves + 7) / 8;
    return grid >= kCus && (grid % kCus == 0 || grid >= 8 * kCus);
}

int lds_threads(bool int4, int r, int j, int64_t waves) {
    const bool rounds_ok = rounds_ok_512(waves);
    // INT4: 512 threads with one row per lane (4096^2 3.38 us against 3.43,
    // 4096x11008 6.82 against 7.14, 8192^2 8.19 against 8.48); with two
    // rows 256 threads (11008x4096 6.05 against 6.14, 13824x5120 9.32
    // against 10.30)
    if (int4 && r == 1 && rounds_ok) return 512;
    if (!int4 && j >= 8 && rounds_ok) return 512;
    return kBlock;
}

void finish_wave_plan(Plan& p, int64_t n, bool int4) {
    const int slots = 64 / p.cw;
    const int64_t rows_per_wave = static_cast<int64_t>(slots) * p.r;
    const int64_t waves = (n + rows_per_wave - 1) / rows_per_wave;
    // the LDS kernels stage x with every thread of a full block
    const int64_t block_waves =
        p.kind == kLds ? lds_threads(int4, p.r, p.j, waves) / 64
                       : std::min<int64_t>(kBlock / 64, waves);
    p.block = static_cast<int>(block_waves * 64);
    p.grid = (waves + block_waves - 1) / block_waves;
}

// Plan of the scalar kernels, from the sizes alone (so that a call off the
// vector contract and the same call of a *_baseline variant sum in the same
// order).  `per` is the elements of a 16-byte chunk.  A row is `steps` rounds
// of 64 chunks; measured over HBM-cold pools (us per call):
// - waves per row: 1 for one step (INT8 32000x333: 8.7; 2 waves 10.2, 4 14.8),
//   2 for two or three (INT4 4096^2 5.0; 1 wave 6.2, 4 5.6), 4 from there
//   (INT8 1000x30001 11.0; 1 wave 27, 2 15.7);
// - rows per wave: 2 (INT8 4001x4099 6.3; 1 row 6.9), but 1 up to 512 rows,
//   where two would leave CUs idle (FP32 500x5001 4.4 against 4.6, INT8
//   256x4099 2.4 against 2.9);
// - chunks per batch: 2 from 16 steps (INT8 300x131071 18.9, one chunk 25.4),
//   else 1 (INT8 4001x4099 with two: 8.6).
Plan scalar_plan(int64_t n, int64_t k, int per, bool fallback, const char* why) {
    Plan p;
    p.kind = kScalar;
    p.block = kBlock;
    const int64_t steps = (k / per + 63) / 64;
    p.split = steps <= 1 ? 1 : steps <= 3 ? 2 : 4;
    p.batch = steps >= 16 ? 2 : 1;
    p.r = n <= 512 ? 1 : 2;
    const int64_t rows = p.r * (kBlock / 64 / p.split);    // per workgroup
    p.grid = (n + rows - 1) / rows;
    p.fallback = fallback;
    p.why = why;
    return p;
}

// The K-tiled kernel: `rows` rows per wave if requested (1 or 2), else one
// up to n = 3072 and two above.  Up to 3072 rows one row per wave (n / 4
// workgroups, at most 3 per CU) with the longer tile keeps more bytes in
// flight: INT4 2048 and 3072 x 28672 10-11% faster than two rows, INT8
// 2048x28672 15%, 2048x65536 13%, 3072x28672 level.  From 3328 rows two rows
// per wave are faster for both (INT4 3328x28672 7%, INT8 3328x28672 11%,
// 3584x65536 6%): one row would leave a fourth, partial workgroup on some CUs.
Plan tiled_plan(int rows, int64_t n, int64_t nchunks, bool int4) {
    Plan p;
    p.kind = kTiled;
    p.cw = 64;
    p.j = static_cast<int>((nchunks + 63) / 64);
    p.r = rows > 0 ? std::min(rows, 2) : (n > 3072 ? 2 : 1);
    p.tile = int4 ? int4_tile_j(p.r, p.j) : q8_tile_j(p.r);
    p.block = kBlock;
    const int64_t waves = (n + p.r - 1) / p.r;
    p.grid = (waves + kBlock / 64 - 1) / (kBlock / 64);
    return p;
}

}  // namespace

bool int4_contract_ok(const void* w, const void* x, int64_t k) {
    if (k % 32 != 0) return false;
    return (reinterpret_cast<uintptr_t>(w) & 15u) == 0 &&
           (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
}

bool q8_contract_ok(const void* w, const void* x, int64_t k) {
    if (k % 16 != 0) return false;
    return (reinterpret_cast<uintptr_t>(w) & 15u) == 0 &&
           (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
}


Plan plan_int4(int kind, int rows, int64_t n, int64_t k, const void* w,
               const void* x) {
    if (kind == kScalar) return scalar_plan(n, k, AnyInt4::E, false, "");
    if (!int4_contract_ok(w, x, k))
        return scalar_plan(n, k, AnyInt4::E, true, "vector contract unmet (w/x 16B alignment, k%32)");
    const int64_t nchunks = k / 32;
    // the untiled LDS kernels address W with 32-bit byte offsets; the tiled
    // kernel keeps 64-bit row bases, so it also takes weights of 4 GiB or more
    const bool big = n * (k / 2) >= (int64_t{1} << 32);
    if (kind == kTiled || (kind == kLds && (k > kMaxWaveK || big)))
        return tiled_plan(rows, n, nchunks, true);
    if (k > kMaxWaveK) return scalar_plan(n, k, AnyInt4::E, true, "k above the wave kernels' register-resident x");
    Plan p;
    p.kind = kind;
    p.cw = pow2_at_least(nchunks, 16);
    p.j = static_cast<int>((nchunks + p.cw - 1) / p.cw);
    const int rmax = int4_rmax(p.j);
    p.r = rows > 0 ? std::min(rows, rmax) : default_rows_int4(n, 64 / p.cw, p.j, rmax);
    if (p.r == 3) p.r = 2;
    finish_wave_plan(p, n, true);
    return p;
}

Plan plan_q8(int kind, int rows, int64_t n, int64_t k, const void* w,
             const void* x) {
    if (kind == kScalar) return scalar_plan(n, k, AnyInt8::E, false, "");
    if (!q8_contract_ok(w, x, k))
        return scalar_plan(n, k, AnyInt8::E, true, "vector contract unmet (w/x 16B alignment, k%16)");
    const int64_t nchunks = k / 16;
    const bool big = n * k >= (int64_t{1} << 32);    // as in plan_int4
    if (kind == kTiled || (kind == kLds && (k > kMaxWaveK || big)))
        return tiled_plan(rows, n, nchunks, false);
    if (k > kMaxWaveK) return scalar_plan(n, k, AnyInt8::E, true, "k above the wave kernels' register-resident x");
    Plan p;
    p.kind = kind;
    p.cw = pow2_at_least(nchunks, 16);
    p.j = static_cast<int>((nchunks + p.cw - 1) / p.cw);
    const int rmax = q8_rmax(p.j);
    p.r = rows > 0 ? std::min(rows, rmax) : 1;
    if (p.r == 3) p.r = 2;
    finish_wave_plan(p, n, false);
    return p;
}

hipError_t prepare_int4(const Plan& p, const void* w, const void* scale,
                        const void* x, void* y, int64_t n, int64_t k, Launch* L) {
    if (p.kind == kScalar)
        return bind(L, scalar_instance<Int4Scalar>(p),
                    p.grid, p.block, 0, static_cast<const char*>(w), scale,
                    static_cast<const char*>(x), static_cast<uint16_t*>(y),
                    static_cast<int>(n), k);
    if (p.kind == kTiled) {
        const Int4Fn tfn =
            p.r == 1 && p.tile == 7   ? &int4gemv_tiled_kernel<kBlock, 7, 1>
            : p.r == 2 && p.tile == 2 ? &int4gemv_tiled_kernel<kBlock, 2, 2>
            : p.r == 2 && p.tile == 4 ? &int4gemv_tiled_kernel<kBlock, 4, 2>
                                      : nullptr;
        if (tfn == nullptr) return hipErrorInvalidConfiguration;
        return bind(L, tfn, p.grid, kBlock, tile_lds(4, p.tile),
                    static_cast<const uint4*>(w), static_cast<const uint16_t*>(scale),
                    static_cast<const uint4*>(x), static_cast<uint16_t*>(y),
                    static_cast<int>(n), static_cast<int>(k / 32));
    }
    const Int4Fn fn =
        p.kind == kWave ? instance<Int4Wave>(p.cw, p.j, p.r)
        : p.block == 512 ? instance<Int4Lds<512>>(p.cw, p.j, p.r)
                         : instance<Int4Lds<kBlock>>(p.cw, p.j, p.r);
    if (fn == nullptr) return hipErrorInvalidConfiguration;
    if (p.kind == kLds && !lds_chunks_ok(p, k / 32)) return hipErrorInvalidConfiguration;
    const uint32_t shmem = p.kind == kLds ? int4_lds_bytes(p.cw, p.j) : 0;
    return bind(L, fn, p.grid, p.block, shmem, static_cast<const uint4*>(w),
                static_cast<const uint16_t*>(scale), static_cast<const uint4*>(x),
                static_cast<uint16_t*>(y), static_cast<int>(n),
                static_cast<int>(k / 32));
}

hipError_t prepare_q8(const Plan& p, const void* w, const void* scale,
                      const void* x, void* y, int64_t n, int64_t k, Launch* L) {
    if (p.kind == kScalar)
        return bind(L, scalar_instance<Q8Scalar>(p),
                    p.grid, p.block, 0, static_cast<const char*>(w), scale,
                    static_cast<const char*>(x), static_cast<uint16_t*>(y),
                    static_cast<int>(n), k);
    if (p.kind == kTiled) {
        const Q8Fn tfn = p.r == 2 && p.tile == q8_tile_j(2) ? &qgemv_tiled_kernel<kBlock, q8_tile_j(2), 2>
                         : p.r == 1 && p.tile == q8_tile_j(1) ? &qgemv_tiled_kernel<kBlock, q8_tile_j(1), 1>
                                                               : nullptr;
        if (tfn == nullptr) return hipErrorInvalidConfiguration;
        return bind(L, tfn, p.grid, kBlock, tile_lds(2, p.tile),
                    static_cast<const uint4*>(w), static_cast<const float*>(scale),
                    static_cast<const uint4*>(x), static_cast<uint16_t*>(y),
                    static_cast<int>(n), static_cast<int>(k / 16));
    }
    const Q8Fn fn = p.kind == kWave ? instance<Q8Wave>(p.cw, p.j, p.r)
                    : p.block == 512 ? instance<Q8Lds<512>>(p.cw, p.j, p.r)
                                     : instance<Q8Lds<kBlock>>(p.cw, p.j, p.r);
    if (fn == nullptr) return hipErrorInvalidConfiguration;
    if (p.kind == kLds && !lds_chunks_ok(p, k / 16)) return hipErrorInvalidConfiguration;
    const uint32_t shmem = p.kind == kLds ? q8_lds_bytes(p.cw, p.j) : 0;
    return bind(L, fn, p.grid, p.block, shmem, static_cast<const uint4*>(w),
                static_cast<const float*>(scale), static_cast<const uint4*>(x),
                static_cast<uint16_t*>(y), static_cast<int>(n),
                static_cast<int>(k / 16));
}

hipError_t enqueue(const Launch& L, hipStream_t stream, hipEvent_t ev0,
                   hipEvent_t ev1) {
    if (L.fn == nullptr || L.nargs > kMaxLaunchArgs) return hipErrorInvalidConfiguration;
    void* argv[kMaxLaunchArgs];
    for (uint32_t i = 0; i < L.nargs; ++i)
        argv[i] = const_cast<uint64_t*>(&L.args[i]);
    const dim3 g(L.grid), b(L.block);
    if (ev0 == nullptr && ev1 == nullptr)
        return hipLaunchKernel(L.fn, g, b, argv, L.shmem, stream);
    return hipExtLaunchKernel(L.fn, g, b, argv, L.shmem, stream, ev0, ev1, 0);
}

hipError_t launch_int4(const Plan& p, const void* w, const void* scale,
                       const void* x, void* y, int64_t n, int64_t k,
                       hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1) {
    Launch L;
    const hipError_t e = prepare_int4(p, w, scale, x, y, n, k, &L);
    return e != hipSuccess ? e : enqueue(L, stream, ev0, ev1);
}

hipError_t launch_int4_stamped(const Plan& p, const void* w, const void* scale,
                               const void* x, void* y, int64_t n, int64_t k,
                               uint64_t* stamps, hipStream_t stream) {
    if (p.kind != kLds || !lds_chunks_ok(p, k / 32)) return hipErrorInvalidConfiguration;
    if (p.block != 512 && p.block != kBlock) return hipErrorInvalidConfiguration;
    const Int4StampFn fn = p.block == 512 ? instance<Int4LdsStamp<512>>(p.cw, p.j, p.r)
                                          : instance<Int4LdsStamp<kBlock>>(p.cw, p.j, p.r);
    if (fn == nullptr) return hipErrorInvalidConfiguration;
    return launch(fn, p.grid, p.block, int4_lds_bytes(p.cw, p.j), stream, nullptr,
                  nullptr, static_cast<const uint4*>(w),
                  static_cast<const uint16_t*>(scale), static_cast<const uint4*>(x),
                  static_cast<uint16_t*>(y), static_cast<int>(n),
                  static_cast<int>(k / 32), stamps);
}

hipError_t launch_q8(const Plan& p, const void* w, const void* scale,
                     const void* x, void* y, int64_t n, int64_t k,
                     hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1) {
    Launch L;
    const hipError_t e = prepare_q8(p, w, scale, x, y, n, k, &L);
    return e != hipSuccess ? e : enqueue(L, stream, ev0, ev1);
}

namespace {

// Shared part of the grouped plans: the plan of the whole group's rows for
// the LDS kernel (cw, j from k; r and block from the total row count), or a
// "launch one by one" plan when any problem cannot take the LDS kernel.
template <typename PlanFn, typename OkFn>
Plan group_plan(PlanFn plan_one, OkFn lds_ok, int rows,
                const GroupProblem* probs, int count, int64_t k) {
    Plan p;
    int64_t total = 0;
    for (int i = 0; i < count; ++i) {
        if (!lds_ok(probs[i])) {
            p.fallback = true;
            p.why = "a problem misses the vector contract or the LDS limits";
            return p;
        }
        total += probs[i].n;
    }
    p = plan_one(kLds, rows, total, k, probs[0].w, probs[0].x);
    if (p.kind != kLds) {
        p.kind = kScalar;
        p.fallback = true;
    }
    return p;
}

// One grouped launch of plan `p`: the kernel for up to three problems that
// share x, or the general one.  An absent problem has no rows.
template <typename S, template <int, class> class F3, template <int> class F8>
hipError_t launch_group(const Plan& p, const GroupProblem* probs, int count,
                        uint32_t shmem, int nchunks, const Repeat* rep, bool* repeated,
                        hipStream_t stream) {
    const bool wide = p.block == 512;
    const int64_t rows = static_cast<int64_t>(64 / p.cw) * p.r * (p.block / 64);
    int64_t grid = 0;
    int n[kMaxGroup] = {};
    bool one_x = true;
    for (int i = 0; i < count; ++i) {
        n[i] = static_cast<int>(probs[i].n);
        grid += (probs[i].n + rows - 1) / rows;
        one_x = one_x && probs[i].x == probs[0].x;
    }
    if (grid > INT32_MAX) return hipErrorInvalidConfiguration;
    if (count <= 3 && one_x) {
        const uint4* w[3] = {};
        const S* sc[3] = {};
        uint16_t* y[3] = {};
        for (int i = 0; i < count; ++i) {
            w[i] = static_cast<const uint4*>(probs[i].w);
            sc[i] = static_cast<const S*>(probs[i].scale);
            y[i] = static_cast<uint16_t*>(probs[i].y);
        }
        auto go = [&](auto fn, auto r) {
            if (fn == nullptr) return hipErrorInvalidConfiguration;
            return launch(fn, grid, p.block, shmem, stream, nullptr, nullptr,
                          static_cast<const uint4*>(probs[0].x), w[0], w[1], w[2], n[0],
                          n[1], n[2], nchunks, sc[0], sc[1], sc[2], y[0], y[1], y[2], r);
        };
        if (rep != nullptr && (rep->head & (rep->head - 1)) == 0) {
            RepeatRows r{static_cast<uint16_t*>(rep->y), rep->problem, 0, rep->times};
            while ((1 << r.shift) < rep->head) ++r.shift;
            *repeated = true;
            return go(wide ? instance<F3<512, RepeatRows>>(p.cw, p.j, p.r)
                           : instance<F3<kBlock, RepeatRows>>(p.cw, p.j, p.r), r);
        }
        return go(wide ? instance<F3<512, NoRepeat>>(p.cw, p.j, p.r)
                       : instance<F3<kBlock, NoRepeat>>(p.cw, p.j, p.r), NoRepeat{});
    }
    const Group8Fn fn = wide ? instance<F8<512>>(p.cw, p.j, p.r)
                             : instance<F8<kBlock>>(p.cw, p.j, p.r);
    if (fn == nullptr) return hipErrorInvalidConfiguration;
    Group8Records g = {};
    for (int i = 0; i < count; ++i)
        g.r[i] = {probs[i].w, probs[i].scale, probs[i].x, probs[i].y};
    return launch(fn, grid, p.block, shmem, stream, nullptr, nullptr, n[0], n[1], n[2],
                  n[3], n[4], n[5], n[6], n[7], nchunks, g);
}

}  // namespace

Plan plan_int4_group(int rows, const GroupProblem* probs, int count, int64_t k) {
    return group_plan(
        plan_int4,
        [k](const GroupProblem& q) {
            return int4_contract_ok(q.w, q.x, k) && k <= kMaxWaveK &&
                   q.n * (k / 2) < (int64_t{1} << 32);
        },
        rows, probs, count, k);
}

Plan plan_q8_group(int rows, const GroupProblem* probs, int count, int64_t k) {
    return group_plan(
        plan_q8,
        [k](const GroupProblem& q) {
            return q8_contract_ok(q.w, q.x, k) && k <= kMaxWaveK &&
                   q.n * k < (int64_t{1} << 32);
        },
        rows, probs, count, k);
}

hipError_t launch_int4_group(const Plan& p, const GroupProblem* probs,
                             int count, int64_t k, const Repeat* rep,
                             bool* repeated, hipStream_t stream) {
    if (p.kind != kLds || count < 1 || count > kMaxGroup || !lds_chunks_ok(p, k / 32))
        return hipErrorInvalidConfiguration;
    return launch_group<uint16_t, Int4LdsGroup3, Int4LdsGroup8>(
        p, probs, count, int4_lds_bytes(p.cw, p.j), static_cast<int>(k / 32), rep, repeated,
        stream);
}

hipError_t launch_q8_group(const Plan& p, const GroupProblem* probs,
                             int count, int64_t k, const Repeat* rep,
                             bool* repeated, hipStream_t stream) {
    if (p.kind != kLds || count < 1 || count > kMaxGroup || !lds_chunks_ok(p, k / 16))
        return hipErrorInvalidConfiguration;
    return launch_group<float, Q8LdsGroup3, Q8LdsGroup8>(
        p, probs, count, q8_lds_bytes(p.cw, p.j), static_cast<int>(k / 16), rep, repeated,
        stream);
}

// ---- FP16/FP32 GEMV
constexpr int64_t kGemvMaxLdsBytes = 64 * 1024;   // x staged per workgroup

bool gemv_contract_ok(int dtype, const void* w, const void* x, int64_t k) {
    const int64_t per = dtype == kF32 ? 4 : 8;     // elements per 16 bytes
    if (k % per != 0) return false;
    return (reinterpret_cast<uintptr_t>(w) & 15u) == 0 &&
           (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
}

Plan plan_gemv(int kind, int dtype, int64_t n, int64_t k, const void* w,
               const void* x) {
    const int per = dtype == kF32 ? AnyF32::E : AnyF16::E;
    if (kind == kScalar) return scalar_plan(n, k, per, false, "");
    if (!gemv_contract_ok(dtype, w, x, k))
        return scalar_plan(n, k, per, true, "vector contract unmet (w/x 16B alignment, k % elements per 16 B)");
    const int64_t es = dtype == kF32 ? 4 : 2;
    const int64_t nchunks = k * es / 16;
    // in-row byte offsets are 32-bit in every vector kernel; row bases are
    // 64-bit only in the tiled kernel, which therefore also takes weights
    // of 4 GiB or more
    if (k * es >= (int64_t{1} << 32))
        return scalar_plan(n, k, per, true, "rows of 4 GiB or more (32-bit offsets)");
    const bool big = n * k * es >= (int64_t{1} << 32);
    Plan p;
    if (kind == kTiled || big || (nchunks + 1) * 16 > kGemvMaxLdsBytes) {
        // x staged tile by tile: 64 lanes per row, one row per wave
        p.kind = kTiled;
        p.cw = 64;
        p.j = static_cast<int>((nchunks + 63) / 64);
        p.r = 1;
        p.tile = kGemvTileJ;
        p.block = rounds_ok_512(n) ? 512 : kBlock;
        p.grid = (n + p.block / 64 - 1) / (p.block / 64);
        return p;
    }
    p.kind = kLds;
    p.cw = pow2_at_least(nchunks, 16);
    p.j = static_cast<int>((nchunks + p.cw - 1) / p.cw);
    p.r = 1;
    const int64_t waves = (n + (64 / p.cw) - 1) / (64 / p.cw);
    // 512-thread workgroups halve the x stagings: 16-20% faster at fp16
    // 4096^2 and 15% at 6144x4096 (whole rounds of CUs); with a partial
    // round among few (5120^2, 5120x13824: 2.5 rounds) 256 threads are 6-7%
    // faster; among 5+ rounds the two are level
    p.block = rounds_ok_512(waves) ? 512 : kBlock;
    p.grid = (waves + p.block / 64 - 1) / (p.block / 64);
    return p;
}

namespace {
template <typename S>
using GemvFn = void (*)(const uint4*, const uint4*, S*, int, int);

template <typename S, int NT>
GemvFn<S> gemv_instance_nt(int cw, int j) {
    if (cw == 16 && j == 1) return &gemv_lds_kernel<S, 16, NT, 1, true>;
    if (cw == 32 && j == 1) return &gemv_lds_kernel<S, 32, NT, 1, true>;
    if (cw != 64 || j < 1) return nullptr;
    switch (j) {
    case 1: return &gemv_lds_kernel<S, 64, NT, 1, true>;
    case 2: return &gemv_lds_kernel<S, 64, NT, 2, true>;
    case 3: return &gemv_lds_kernel<S, 64, NT, 3, true>;
    case 4: return &gemv_lds_kernel<S, 64, NT, 4, true>;
    case 5: return &gemv_lds_kernel<S, 64, NT, 5, true>;
    case 6: return &gemv_lds_kernel<S, 64, NT, 6, true>;
    case 7: return &gemv_lds_kernel<S, 64, NT, 7, true>;
    case kGemvBatch: return &gemv_lds_kernel<S, 64, NT, kGemvBatch, true>;
    default: return &gemv_lds_kernel<S, 64, NT, kGemvBatch, false>;
    }
}

template <typename S>
GemvFn<S> gemv_tiled_instance(int block, bool one) {
    if (block == 512) return one ? &gemv_tiled_kernel<S, 512, true> : &gemv_tiled_kernel<S, 512, false>;
    return one ? &gemv_tiled_kernel<S, kBlock, true> : &gemv_tiled_kernel<S, kBlock, false>;
}

template <typename S>
GemvFn<S> gemv_instance(int cw, int j, int block) {
    if (block == 512) return gemv_instance_nt<S, 512>(cw, j);
    if (block == kBlock) return gemv_instance_nt<S, kBlock>(cw, j);
    return nullptr;
}

template <typename S>
hipError_t prepare_gemv_t(const Plan& p, const void* w, const void* x, void* y,
                          int64_t n, int64_t k, Launch* L) {
    if (p.kind == kScalar)
        return bind(L, scalar_instance<GemvScalar<S>>(p), p.grid, p.block, 0,
                    static_cast<const char*>(w), nullptr, static_cast<const char*>(x),
                    static_cast<S*>(y), static_cast<int>(n), k);
    const int nchunks = static_cast<int>(k * static_cast<int64_t>(sizeof(S)) / 16);
    if (p.kind == kTiled)
        return bind(L, gemv_tiled_instance<S>(p.block, nchunks < kGemvTileJ * 64), p.grid, p.block, kGemvTileLds, static_cast<const uint4*>(w),
                    static_cast<const uint4*>(x), static_cast<S*>(y),
                    static_cast<int>(n), nchunks);
    const GemvFn<S> fn = gemv_instance<S>(p.cw, p.j, p.block);
    if (fn == nullptr || !lds_chunks_ok(p, nchunks)) return hipErrorInvalidConfiguration;
    return bind(L, fn, p.grid, p.block, static_cast<uint32_t>((nchunks + 1) * 16),
                static_cast<const uint4*>(w), static_cast<const uint4*>(x),
                static_cast<S*>(y), static_cast<int>(n), nchunks);
}
}  // namespace

hipError_t prepare_gemv(const Plan& p, int dtype, const void* w, const void* x,
                        void* y, int64_t n, int64_t k, Launch* L) {
    return dtype == kF32 ? prepare_gemv_t<float>(p, w, x, y, n, k, L)
                         : prepare_gemv_t<uint16_t>(p, w, x, y, n, k, L);
}

hipError_t launch_gemv(const Plan& p, int dtype, const void* w, const void* x,
                       void* y, int64_t n, int64_t k, hipStream_t stream,
                       hipEvent_t ev0, hipEvent_t ev1) {
    Launch L;
    const hipError_t e = prepare_gemv(p, dtype, w, x, y, n, k, &L);
    return e != hipSuccess ? e : enqueue(L, stream, ev0, ev1);
}

hipError_t launch_repeat(const void* src, int64_t n, const Repeat& rep, hipStream_t stream) {
    return launch(repeat_rows_kernel, (n + kBlock - 1) / kBlock, kBlock, 0, stream, nullptr,
                  nullptr, static_cast<const uint16_t*>(src), static_cast<uint16_t*>(rep.y),
                  static_cast<int>(n), rep.head, rep.times);
}

hipError_t launch_stream_read(const void* buf, int64_t bytes, void* sink,
                              hipStream_t stream) {
    const int64_t n16 = bytes / 16;
    const int64_t grid = (n16 + kBlock - 1) / kBlock;
    return launch(stream_read_kernel, grid, kBlock, 0, stream, nullptr,
                  nullptr, static_cast<const uint4*>(buf),
                  static_cast<uint32_t*>(sink), n16, 0x9E3779B9u);
}

hipError_t launch_delay(double us, hipStream_t stream) {
    if (!(us > 0.0)) return hipSuccess;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    int khz = 0;   // wall clock rate in kHz (100 MHz on MI355X)
    e = hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev);
    if (e != hipSuccess) return e;
    if (khz <= 0) return hipErrorInvalidValue;
    const double t = us * static_cast<double>(khz) / 1000.0;
    if (t > 1e12) return hipErrorInvalidValue;
    const uint64_t ticks = static_cast<uint64_t>(t) + 1;
    // each pass sleeps 8 x 64 cycles, several ticks: ticks + 1024 passes
    // always outlast the wait and bound it if the clock were stuck
    return launch(delay_kernel, 1, 64, 0, stream, nullptr, nullptr, ticks,
                  ticks + 1024);
}

hipError_t launch_empty(int64_t grid, int block, void* sink,
                        hipStream_t stream) {
    return launch(empty_launch_kernel, grid, block, 0, stream, nullptr,
                  nullptr, static_cast<uint32_t*>(sink), 0xFFFFFFFFu);
}

}  // namespace cq
