// noncausal_mfma.hip -- bucket reductions and token maps of the non-causal
// forward and backward on the fp32 matrix cores, for widths that are multiples
// of 4 (analysis/hot-path.md:157-162 and its VJP):
//   reduction  R[a][b] = sum_t x[t][a] y[t][b],  colsum[a] = sum_t x[t][a]
//              (B = K^T V and A in the forward, dE = Q^T dOut in the backward)
//   map        out[t][c] = sum_a x[t][a] M[a][c] (+ bias[c])
//              (out = Q E, dQ = dOut E^T, dK = V dB^T + dA, dV = K dB)
// fp32 tokens: every product is v_mfma_f32_16x16x4_f32 -- fp32 operands,
// products and sums, the arithmetic of a chain of fp32 fused multiply-adds at
// twice the rate of the vector ALU (this build has no packed fp32).
// bf16 tokens: v_mfma_f32_16x16x32_bf16, sixteen times that rate.  A reduction's
// products of two bf16 values are exact in its fp32 sums; a map's fp32 matrix
// is split into three bf16 terms that add up to it exactly (8 bits each,
// truncated; below 2^-110 to within 2^-133, the least a bf16 term holds), so
// its products are the fp32 ones too (for finite tokens; those with an infinity
// or NaN take fp32 products, whole_products).
// The token rows never go through workgroup-wide LDS staging: a wave loads
// whole rows into registers and, where the products want the other layout,
// turns 16 or 32 rows through a piece of LDS of its own, without barriers.
//
// A lane is (g, lr) = (lane / 16, lane % 16).  An MFMA takes A[row lr][k of g]
// and B[k of g][column lr] from each lane and returns D[4 g + r][lr].
//   reduction  the contraction runs over tokens: lane (g, lr) loads x and y of
//              tokens 4 i + g, columns EA lr .. and EB lr .. (a load
//              instruction covers four whole rows); block (ea, eb) of R holds
//              rows EA m + ea and columns EB n + eb.
//   map        the contraction runs over columns: lane (g, lr) holds x of
//              token lr, four (fp32) or eight (bf16) columns per step.  M comes
//              from LDS in that order, one 16-byte read per block and step (and
//              term), and the result is transposed (D = M^T X^T) so that a lane
//              holds four consecutive columns of one token.
// Sums over waves and tiles have a fixed order: results are bitwise
// reproducible.
//
// Measured against the vector-ALU kernels (noncausal_v4.hip), S = d = 64,
// kernel times in us, reduction / map / query side / key side:
//   fp32, N = 384, T = 1024: 50 / 62 / 101 / 107 -> 36 / 44 / 61 / 81, at 5.6,
//     4.6, 5.0 and 5.0 TB/s of tokens: bound by memory (the query side's two
//     products alone are 41 us of fp32 matrix instructions); 44 for the
//     reduction where no token is left in a cache by the call before;
//   bf16, N = 192, T = 577: 20 + 10 (reduce) / 41 / 41 + 7 (finalize) / 41
//     -> 9 / 11 / 13 / 15: launches of one workgroup per stream, bound by the
//     latency of staging, the loop's few steps and the launch itself.
// Other widths (S 12 .. 256, d 20 .. 128) ran 1.2x (100 x 36, fp32) to 9x.
#include <algorithm>

#include "mfma_common.h"

namespace race {
namespace {

using mfma::bf16x8;
using mfma::f32x4;
using mfma::kOutside;
using mfma::mfma16;
using mfma::mfma4;
using mfma::u32x2;
using mfma::u32x4;

constexpr int kWaves = kThreads / 64;  // waves of a reduction workgroup
constexpr int kMapWaves = 8;            // waves of a map workgroup: they share one staged matrix
constexpr int64_t kMapMaxTokens = 1024;
// Tokens a wave takes at a time: one fp32 MFMA tile, or the 32-token
// contraction of a bf16 one.
template <typename TIn>
constexpr int kStep = sizeof(TIn) == 4 ? 16 : 32;
constexpr int kNcStorePolicy = 2;  // nontemporal: the results are not read again here

// E consecutive elements of a token row.
template <typename TIn, int E>
struct Vec {
    static constexpr int kBytes = E * int(sizeof(TIn));
    using Raw = std::conditional_t<kBytes == 16, uint4, std::conditional_t<kBytes == 8, uint2, uint32_t>>;
    static_assert(kBytes >= 4, "whole words");
    Raw v;
    template <int P = mfma::kPolicyDefault>
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, int off) {
        if constexpr (kBytes == 16)
            v = mfma::buf_load16<P>(r, off);
        else if constexpr (kBytes == 8)
            v = mfma::buf_load8<P>(r, off);
        else
            v = __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, P);
    }
    __device__ __forceinline__ uint32_t word(int i) const {
        if constexpr (kBytes == 16)
            return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
        else if constexpr (kBytes == 8)
            return i == 0 ? v.x : v.y;
        else
            return v;
    }
    __device__ __forceinline__ float get(int e) const {
        if constexpr (sizeof(TIn) == 4) return __uint_as_float(word(e));
        const uint32_t w = word(e >> 1);
        return (e & 1) ? mfma::hi_half(w) : mfma::lo_half(w);
    }
    __device__ __forceinline__ f32x4 f32() const {
        static_assert(E == 4, "four values");
        return f32x4{get(0), get(1), get(2), get(3)};
    }
};

// ---------------------------------------------------------------------------
// Reduction.

// A step's rows by column: c[e] holds column E lr + e of the lane's tokens
// 4 i + g, as four fp32 operands or one bf16 operand of eight.
template <typename TIn, int E>
struct Columns;
template <int E>
struct Columns<float, E> {
    float c[E][4];
    __device__ __forceinline__ explicit Columns(const Vec<float, E> (&x)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < E; ++e) c[e][i] = x[i].get(e);
    }
};
template <int E>
struct Columns<bf16_t, E> {
    bf16x8 c[E];
    __device__ __forceinline__ explicit Columns(const Vec<bf16_t, E> (&x)[8]) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            u32x4 r;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                r[i] = __builtin_amdgcn_perm(x[2 * i + 1].word(e >> 1), x[2 * i].word(e >> 1),
                                             (e & 1) ? 0x07060302u : 0x05040100u);
            c[e] = __builtin_bit_cast(bf16x8, r);
        }
    }
};

// One wave's accumulators of a 16 EA x 16 EB block of R, and the column sums
// of x it has seen.
template <int EA, int EB>
struct Outer {
    f32x4 acc[EA][EB];
    float csum[EA];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int a = 0; a < EA; ++a) {
            csum[a] = 0.f;
#pragma unroll
            for (int b = 0; b < EB; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    // The products of one step's operands, and with kSums x's column sums.
    template <bool kSums>
    __device__ __forceinline__ void add(const Columns<float, EA>& x, const Columns<float, EB>& y) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int a = 0; a < EA; ++a) {
                if constexpr (kSums) csum[a] += x.c[a][i];
#pragma unroll
                for (int b = 0; b < EB; ++b) acc[a][b] = mfma4(x.c[a][i], y.c[b][i], acc[a][b]);
            }
    }
    template <bool kSums>
    __device__ __forceinline__ void add(const Columns<bf16_t, EA>& x, const Columns<bf16_t, EB>& y) {
#pragma unroll
        for (int a = 0; a < EA; ++a) {
            if constexpr (kSums) {
                const u32x4 xc = __builtin_bit_cast(u32x4, x.c[a]);
#pragma unroll
                for (int i = 0; i < 4; ++i) csum[a] += mfma::lo_half(xc[i]) + mfma::hi_half(xc[i]);
            }
#pragma unroll
            for (int b = 0; b < EB; ++b) acc[a][b] = mfma16(x.c[a], y.c[b], acc[a][b]);
        }
    }
    static constexpr int kBlockFloats = 16 * EA * 16 * EB;
    // The partial block in `part` [16 EA][16 EB]: written, or replaced by
    // itself plus this wave's.
    template <bool kAdd>
    __device__ __forceinline__ void spill(float* __restrict__ part, int g, int lr) const {
#pragma unroll
        for (int a = 0; a < EA; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float* p = part + (EA * (4 * g + r) + a) * 16 * EB + EB * lr;
#pragma unroll
                for (int b = 0; b < EB; ++b) p[b] = kAdd ? acc[a][b][r] + p[b] : acc[a][b][r];
            }
    }
    // The workgroup's block: waves 0 .. 3 added as (0 + 2) + (1 + 3) through
    // two LDS buffers of kBlockFloats, and the column sums over lane groups
    // and waves in order; rows a0 .., columns b0 .. of the record `r`
    // ([Wa][Wb], then the column sums when `sums` asks for them).
    __device__ __forceinline__ void combine(float* __restrict__ lds, float* __restrict__ r, int Wa, int Wb,
                                            int a0, int b0, bool sums, int w, int g, int lr) {
        float* cs = lds + 2 * kBlockFloats;  // [4 waves][4 groups][16 EA]
        __syncthreads();
        if (w >= 2) spill<false>(lds + (w - 2) * kBlockFloats, g, lr);
#pragma unroll
        for (int a = 0; a < EA; ++a) cs[(w * 4 + g) * 16 * EA + EA * lr + a] = csum[a];
        __syncthreads();
        if (w < 2) spill<true>(lds + w * kBlockFloats, g, lr);
        __syncthreads();
        // Whole rows out, 16 bytes a thread.
        const int rows = min(16 * EA, Wa - a0), cols = min(16 * EB, Wb - b0);
        for (int e = threadIdx.x; e < 16 * EA * 4 * EB; e += kThreads) {
            const int a = e / (4 * EB), c = 4 * (e % (4 * EB));
            if (a < rows && c < cols)
                *reinterpret_cast<f32x4*>(r + int64_t(a0 + a) * Wb + b0 + c) =
                    *reinterpret_cast<const f32x4*>(lds + a * 16 * EB + c) +
                    *reinterpret_cast<const f32x4*>(lds + kBlockFloats + a * 16 * EB + c);
        }
        if (sums && int(threadIdx.x) < rows) {
            float s = 0.f;
#pragma unroll
            for (int i = 0; i < 16; ++i) s += cs[i * 16 * EA + threadIdx.x];
            r[int64_t(Wa) * Wb + a0 + threadIdx.x] = s;
        }
    }
    static constexpr int kLdsFloats = 2 * kBlockFloats + 16 * 16 * EA;
};

// One workgroup per (chunk of tokens, stream, block of R).  Wave w takes the
// steps w, w + 4, .. of the chunk.  The operand vectors of the next step are
// loaded before the current step's products.
// kEndFirst (the causal tile sums, whose tiles the output pass then walks from
// their start): the steps go from the chunk's end to its start, past the
// caches except for the first `kept` rows (cache_kept_rows), which come last.
template <typename TIn, int EA, int EB, bool kEndFirst>
__global__ __launch_bounds__(kThreads, 3) void nc_sums_kernel(
    const TIn* __restrict__ x, const TIn* __restrict__ y, float* __restrict__ records, int64_t T, int chunk,
    int64_t chunks, int64_t rec, int Wa, int Wb, int bblocks, int kept) {
    extern __shared__ __align__(16) float smem[];
    constexpr int es = int(sizeof(TIn)), kTok = kStep<TIn>, kLoads = kTok / 4;
    const int lane = threadIdx.x & 63, g = lane >> 4, lr = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t n = blockIdx.y, ci = blockIdx.x;
    const int a0 = 16 * EA * int(blockIdx.z / bblocks), b0 = 16 * EB * int(blockIdx.z % bblocks);
    const int64_t t0 = ci * chunk;
    const int rows = int(min(T, t0 + chunk) - t0);
    const auto xr = mfma::make_rsrc(x + (n * T + t0) * Wa, int64_t(rows) * Wa * es);
    const auto yr = mfma::make_rsrc(y + (n * T + t0) * Wb, int64_t(rows) * Wb * es);
    const int ca = a0 + EA * lr, cb = b0 + EB * lr;
    Vec<TIn, EA> xv[kLoads];
    Vec<TIn, EB> yv[kLoads];
    auto load = [&](auto pol, int r0) {
        constexpr int P = decltype(pol)::value;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int row = r0 + 4 * i + g;
            xv[i].template load<P>(xr, ca < Wa ? (row * Wa + ca) * es : kOutside);
            yv[i].template load<P>(yr, cb < Wb ? (row * Wb + cb) * es : kOutside);
        }
    };
    using Alloc = std::integral_constant<int, mfma::kPolicyDefault>;
    using Stream = std::integral_constant<int, mfma::kPolicyStream>;
    Outer<EA, EB> o;
    o.clear();
    // The products of the rows held, the next step's rows loaded meanwhile
    // (past either end of the chunk: zeros, never used).
    auto step = [&](auto pol, int next) {
        const Columns<TIn, EA> xc(xv);
        const Columns<TIn, EB> yc(yv);
        load(pol, next);
        o.template add<true>(xc, yc);
    };
    constexpr int kAll = kTok * kWaves;
    if constexpr (kEndFirst) {
        const int cut = (kept + kAll - 1) / kAll * kAll;
        int r0 = (rows - 1) / kAll * kAll + kTok * w;
        if (r0 < cut)
            load(Alloc{}, r0);
        else
            load(Stream{}, r0);
        for (; r0 - kAll >= cut; r0 -= kAll) step(Stream{}, r0 - kAll);
#pragma unroll 2
        for (; r0 >= 0; r0 -= kAll) step(Alloc{}, r0 >= kAll ? r0 - kAll : rows);
    } else {
        load(Alloc{}, kTok * w);
#pragma unroll 2
        for (int r0 = kTok * w; r0 < rows; r0 += kAll) step(Alloc{}, r0 + kAll);
    }
    o.combine(smem, records + (n * chunks + ci) * rec, Wa, Wb, a0, b0, b0 == 0, w, g, lr);
}

// ---------------------------------------------------------------------------
// Map.

// The operands of 16 tokens' rows of (at most) 16 NJ values and their product
// with a staged matrix, acc[cb] += M^T X^T.
//   kB16 = false: operand j of lane (g, lr) is x[lr][16 j + 4 g .. + 3], and
//     entry (j NCB + cb) 64 + lane of `m` holds M[16 j + 4 g .. + 3][16 cb + lr].
//   kB16 = true: operand j is x[lr][32 j + 8 g .. + 7], and entry
//     ((j NCB + cb) 3 + term) 64 + lane holds that term of M[32 j + 8 g .. + 7][16 cb + lr].
template <typename TIn, int NJ, bool kB16>
struct MapRows {
    static constexpr int kPer = kB16 ? 8 : 4;                   // values per operand
    static constexpr int kOps = kB16 ? (NJ + 1) / 2 : NJ;       // operands
    static constexpr int kUnit = kPer * int(sizeof(TIn));       // bytes
    using V = Vec<TIn, kPer>;
    using Raw = typename V::Raw;
    // A row is 4 kOps units; a wave's 16 rows are kOps units per lane.
    static constexpr int kUnits = 4 * kOps;
    static constexpr int kBytes = 16 * kUnits * kUnit;
    V x[kOps];

    // Unit i 64 + lane of the 16 rows (row-major): a load covers whole rows.
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, int row0, int W, int lane) {
#pragma unroll
        for (int i = 0; i < kOps; ++i) {
            const int u = i * 64 + lane, row = u / kUnits, c = (u % kUnits) * kPer;
            x[i].load(r, c < W ? ((row0 + row) * W + c) * int(sizeof(TIn)) : kOutside);
        }
    }
    // From the loads' layout to the operands', through kBytes of LDS that only
    // this wave uses (LDS serves a wave in order: only the compiler's order has
    // to be held).  Unit u of row r sits at u ^ r, so both sides spread over
    // the banks.
    __device__ __forceinline__ static int at(int row, int u) { return row * kUnits + (u ^ (row & (kUnits - 1))); }
    __device__ __forceinline__ void turn(Raw* __restrict__ t, int lane, int g, int lr) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int i = 0; i < kOps; ++i) {
            const int u = i * 64 + lane;
            t[at(u / kUnits, u % kUnits)] = x[i].v;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int j = 0; j < kOps; ++j) x[j].v = t[at(lr, 4 * j + g)];
    }
    // The lanes that hold an infinity or NaN, where the products are of terms:
    // a zero term times an infinity is NaN, so those tokens need whole_products.
    __device__ __forceinline__ uint64_t nonfinite() const {
        if constexpr (kB16) {
            typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
            u16x2 top = {0, 0};
#pragma unroll
            for (int j = 0; j < kOps; ++j)
#pragma unroll
                for (int i = 0; i < kUnit / 4; ++i)
                    top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, x[j].word(i) & 0x7fff7fffu));
            return __ballot(top[0] >= 0x7f80 || top[1] >= 0x7f80);
        } else {
            return 0;
        }
    }
    template <int NCB>
    __device__ __forceinline__ void times(const float* __restrict__ m, int lane, f32x4 (&acc)[NCB]) const {
        if constexpr (kB16) {
            const bf16x8* mb = reinterpret_cast<const bf16x8*>(m);
#pragma unroll
            for (int j = 0; j < kOps; ++j) {
                const bf16x8 xv = __builtin_bit_cast(bf16x8, x[j].v);
                // Smallest terms first.
#pragma unroll
                for (int t = 2; t >= 0; --t)
#pragma unroll
                    for (int cb = 0; cb < NCB; ++cb)
                        acc[cb] = mfma16(mb[((j * NCB + cb) * 3 + t) * 64 + lane], xv, acc[cb]);
            }
        } else {
            const f32x4* mf = reinterpret_cast<const f32x4*>(m);
#pragma unroll
            for (int j = 0; j < kOps; ++j) {
                f32x4 mv[NCB];
#pragma unroll
                for (int cb = 0; cb < NCB; ++cb) mv[cb] = mf[(j * NCB + cb) * 64 + lane];
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int cb = 0; cb < NCB; ++cb) acc[cb] = mfma4(mv[cb][e], x[j].get(e), acc[cb]);
            }
        }
    }
};

// LDS floats of a staged matrix.
template <int NJ, int NCB, bool kB16>
constexpr int kMatrixFloats = kB16 ? 32 * ((NJ + 1) / 2) * 16 * NCB * 3 / 2 : 16 * NJ * 16 * NCB;

// The three bf16 terms of x: 8 bits each by truncation, so hi + mid + lo is x
// exactly (from 2^-110 up); infinities and NaN stay in hi alone.
__device__ __forceinline__ void split3(float x, uint16_t (&t)[3]) {
    const uint32_t u = __float_as_uint(x);
    const float r1 = x - __uint_as_float(u & 0xffff0000u);
    const uint32_t u1 = __float_as_uint(r1);
    const float r2 = r1 - __uint_as_float(u1 & 0xffff0000u);
    const bool finite = (u & 0x7f800000u) != 0x7f800000u;
    t[0] = uint16_t(u >> 16) | uint16_t(!finite && (u & 0x007fffffu) ? 0x40u : 0u);  // NaN stays NaN
    t[1] = finite ? uint16_t(u1 >> 16) : uint16_t(0);
    t[2] = finite ? uint16_t(__float_as_uint(r2) >> 16) : uint16_t(0);
}

// M[k][c .. c + 3] (kAcross) or M[k .. k + 3][c] = x into the operand order of
// MapRows::times.
template <int NCB, bool kB16, bool kAcross>
__device__ __forceinline__ void put_matrix(float* __restrict__ dst, int k, int c, const f32x4& x) {
    const int cb = c >> 4, lr = c & 15;
    if constexpr (kB16) {
        uint16_t* d = reinterpret_cast<uint16_t*>(dst);
        const int j = k >> 5, g = (k >> 3) & 3, e = k & 7;
        uint16_t t[4][3];
#pragma unroll
        for (int i = 0; i < 4; ++i) split3(x[i], t[i]);
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            const int at = (((j * NCB + cb) * 3 + s) * 64 + 16 * g + lr) * 8 + e;
            if constexpr (kAcross) {
#pragma unroll
                for (int i = 0; i < 4; ++i) d[at + 8 * i] = t[i][s];
            } else {
                *reinterpret_cast<uint2*>(d + at) = make_uint2(t[0][s] | uint32_t(t[1][s]) << 16,
                                                               t[2][s] | uint32_t(t[3][s]) << 16);
            }
        }
    } else {
        const int j = k >> 4, g = (k >> 2) & 3, e = k & 3;
        if constexpr (kAcross) {
#pragma unroll
            for (int i = 0; i < 4; ++i) dst[((j * NCB + cb) * 64 + 16 * g + lr + i) * 4 + e] = x[i];
        } else {
            reinterpret_cast<f32x4*>(dst)[(j * NCB + cb) * 64 + 16 * g + lr] = x;
        }
    }
}

// A wave's 16 result rows of 16 NCB columns, from the accumulators to memory
// as whole rows (row pieces of 64 bytes straight from the accumulators left
// lines half written: the map of 393216 fp32 rows of 64 took 68 us with
// nontemporal stores), through 16 rows of 4 NCB four-value units of this
// wave's LDS, swizzled as MapRows::turn.
template <typename TIn, int NCB>
struct OutRows {
    static constexpr int kUnits = 4 * NCB;
    static constexpr int kBytes = 16 * kUnits * 4 * int(sizeof(TIn));
    using Raw = std::conditional_t<sizeof(TIn) == 4, u32x4, u32x2>;
    __device__ __forceinline__ static int at(int row, int u) { return row * kUnits + (u ^ (row & (kUnits - 1))); }
    __device__ __forceinline__ static void put(Raw* __restrict__ t, int cb, const f32x4& y, int g, int lr) {
        if constexpr (sizeof(TIn) == 4)
            t[at(lr, 4 * cb + g)] = __builtin_bit_cast(u32x4, y);
        else
            t[at(lr, 4 * cb + g)] = u32x2{mfma::pack2(y[0], y[1]), mfma::pack2(y[2], y[3])};
    }
    // Rows row0 .. of the view `o`, row length W; columns c0 .. of it, ncols of
    // them.  `replace` runs with the results in `t`.
    template <typename Replace>
    __device__ __forceinline__ static void store(Raw* __restrict__ t, const f32x4 (&acc)[NCB], __amdgpu_buffer_rsrc_t o,
                                                 int row0, int W, int c0, int ncols, int lane, int g, int lr,
                                                 Replace replace) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) put(t, cb, acc[cb], g, lr);
        replace();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int i = 0; i < NCB; ++i) {
            const int u = i * 64 + lane, row = u / kUnits, c = 4 * (u % kUnits);
            const int off = c < ncols ? ((row0 + row) * W + c0 + c) * int(sizeof(TIn)) : kOutside;
            const Raw v = t[at(row, u % kUnits)];
            if constexpr (sizeof(TIn) == 4)
                __builtin_amdgcn_raw_buffer_store_b128(v, o, off, 0, kNcStorePolicy);
            else
                __builtin_amdgcn_raw_buffer_store_b64(v, o, off, 0, kNcStorePolicy);
        }
    }
};

// The results in `t` of the tokens whose lanes are set in `bad` (bf16 rows row0
// .. of `xr`, row length W; MapRows::nonfinite), replaced by the products with
// the staged matrix put together again from its terms: fp32 products, as the
// other tokens' terms add up to.  init(cb, g) gives the values a lane's sums
// start from.  Operands are read again and nothing is unrolled: rows like these are
// the exception, and the registers the loop around it holds are not.
template <typename TIn, int NJ, int NCB, typename Init>
__device__ __forceinline__ void whole_products(typename OutRows<TIn, NCB>::Raw* __restrict__ t, uint64_t bad,
                                               __amdgpu_buffer_rsrc_t xr, int row0, int W,
                                               const float* __restrict__ m, int lane, Init init) {
    using X = MapRows<TIn, NJ, true>;
    asm volatile("" : "+v"(lane));  // the addresses below are not kept for the loop either
    const int g = lane >> 4, lr = lane & 15;
    const bool mine = ((bad | bad >> 16 | bad >> 32 | bad >> 48) >> lr) & 1;
    const uint2* mt = reinterpret_cast<const uint2*>(m);
#pragma unroll 1
    for (int cb = 0; cb < NCB; ++cb) {
        f32x4 acc = init(cb, g);
#pragma unroll 1
        for (int h = 0; h < 2 * X::kOps; ++h) {  // half operands
            const int j = h >> 1, c = 32 * j + 8 * g + 4 * (h & 1);
            Vec<bf16_t, 4> x, t0, t1, t2;
            x.load(xr, c < W ? ((row0 + lr) * W + c) * int(sizeof(TIn)) : kOutside);
            const uint2* at = mt + ((j * NCB + cb) * 3 * 64 + lane) * 2 + (h & 1);
            t0.v = at[0];
            t1.v = at[128];
            t2.v = at[256];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = mfma4(t0.get(e) + (t1.get(e) + t2.get(e)), x.get(e), acc);
        }
        if (mine) OutRows<TIn, NCB>::put(t, cb, acc, g, lr);
    }
}

// Columns c0 .. c0 + 16 NCB - 1 of the map operand's matrix in operand order,
// zero past Wa rows and `ncols` columns; the workgroups of a stream's first
// token block also save the undivided values when the operand asks for it.
// The operand is a row-major matrix m[s][c] (rows of `ld` values, the divisor
// by s), taken plain (M[s][c]) or transposed (M[c][s]); a thread takes four
// consecutive c of a row, the loads of four such groups and two parts in
// flight together.
template <int NT, int NJ, int NCB, bool kB16>
__device__ __forceinline__ void stage_operand(float* __restrict__ dst, const MapOperand& op, int64_t n, int Wa,
                                              int c0, int ncols, bool first_block, bool first_slice) {
    constexpr int kCols = 16 * NCB, kRows = kB16 ? 32 * ((NJ + 1) / 2) : 16 * NJ, kQuads = kRows * kCols / 4;
    const bool plain = op.col == 1;
    const int64_t ld = plain ? op.row : op.col;
    const float* mn = op.m + n * op.stream;
    const float* dv = op.div ? op.div + n * op.div_stream : nullptr;
    float* sv = op.save && first_block ? op.save + n * op.save_stream : nullptr;
    constexpr int kPer = kQuads >= 4 * NT ? 4 : kQuads >= 2 * NT ? 2 : 1;
    for (int e0 = 0; e0 < kQuads; e0 += kPer * NT) {
        f32x4 v[kPer];
        float q[kPer];
        int row[kPer], col[kPer];  // of M: plain, columns col .. + 3; transposed, rows row .. + 3
        int64_t at[kPer];
        int div[kPer];
        bool ok[kPer];
#pragma unroll
        for (int m = 0; m < kPer; ++m) {
            const int e = e0 + int(threadIdx.x) + m * NT;
            row[m] = plain ? e / (kCols / 4) : 4 * (e % (kRows / 4));
            col[m] = plain ? 4 * (e % (kCols / 4)) : e / (kRows / 4);
            ok[m] = e < kQuads && row[m] < Wa && col[m] < ncols;
            at[m] = ok[m] ? (plain ? row[m] * ld + c0 + col[m] : (c0 + col[m]) * ld + row[m]) : 0;
            div[m] = ok[m] ? (plain ? row[m] : c0 + col[m]) : 0;
            v[m] = f32x4{0.f, 0.f, 0.f, 0.f};
            q[m] = 0.f;
        }
        for (int p0 = 0; p0 < op.parts; p0 += 2) {
            const int64_t o0 = p0 * op.part_stride, o1 = min(p0 + 1, op.parts - 1) * op.part_stride;
            f32x4 v0[kPer], v1[kPer];
            float q0[kPer], q1[kPer];
#pragma unroll
            for (int m = 0; m < kPer; ++m) {
                v0[m] = *reinterpret_cast<const f32x4*>(mn + at[m] + o0);
                v1[m] = *reinterpret_cast<const f32x4*>(mn + at[m] + o1);
                q0[m] = dv ? dv[div[m] + o0] : 0.f;
                q1[m] = dv ? dv[div[m] + o1] : 0.f;
            }
#pragma unroll
            for (int m = 0; m < kPer; ++m) {
                v[m] += v0[m];
                q[m] += q0[m];
                if (p0 + 1 < op.parts) {
                    v[m] += v1[m];
                    q[m] += q1[m];
                }
            }
        }
#pragma unroll
        for (int m = 0; m < kPer; ++m) {
            if (e0 + int(threadIdx.x) + m * NT >= kQuads) continue;
            if (sv && ok[m]) {
                *reinterpret_cast<f32x4*>(sv + at[m]) = v[m];
                // Each divisor once: by the first values of its row of m.
                if (dv && (plain ? col[m] == 0 && first_slice : row[m] == 0)) sv[op.save_div_off + div[m]] = q[m];
            }
            f32x4 x = ok[m] ? v[m] : f32x4{0.f, 0.f, 0.f, 0.f};
            if (dv && ok[m]) {
                const float den = q[m] + kEps;
                x = f32x4{x[0] / den, x[1] / den, x[2] / den, x[3] / den};
            }
            if (plain)
                put_matrix<NCB, kB16, true>(dst, row[m], col[m], x);
            else
                put_matrix<NCB, kB16, false>(dst, row[m], col[m], x);
        }
    }
}

// Stream and block of a workgroup: gfx950 hands consecutive workgroups to its 8
// XCDs in turn, so the `per` blocks of one stream are 8 apart in launch order
// and share an XCD's L2 (the matrix records a stream's workgroups all read).
__device__ __forceinline__ void stream_block(int64_t id, int64_t N, int per, int64_t& n, int& blk) {
    const int64_t group = id / (8 * per);
    const int in = int(id - group * 8 * per);
    const int streams = int(min<int64_t>(8, N - 8 * group));
    n = 8 * group + in % streams;
    blk = in / streams;
}

// One workgroup per (block of `wg_tokens` tokens, stream, slice of 16 NCB
// output columns); wave w takes the 16-token tiles w, w + NW, ..  Rows of up to
// 128 values are loaded as whole rows a tile ahead; longer ones straight in
// the operands' layout (their turn would take 64 KB of LDS).
template <typename TIn, int NJ, int NCB, bool kB16, int NW>
__global__ __launch_bounds__(64 * NW) void nc_map_kernel(const TIn* __restrict__ x, TIn* __restrict__ out,
                                                          const MapOperand op, int64_t N, int64_t T, int Wa,
                                                          int Wb, int wg_tokens, int per) {
    extern __shared__ __align__(16) float smem[];
    using X = MapRows<TIn, NJ, kB16>;
    using O = OutRows<TIn, NCB>;
    constexpr int es = int(sizeof(TIn));
    constexpr bool kTurn = NJ <= 8;
    constexpr int kWaveBytes = kTurn && X::kBytes > O::kBytes ? X::kBytes : O::kBytes;
    const int lane = threadIdx.x & 63, g = lane >> 4, lr = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    unsigned char* mine = reinterpret_cast<unsigned char*>(smem + kMatrixFloats<NJ, NCB, kB16>) + w * kWaveBytes;
    int64_t n;
    int blk;
    stream_block(blockIdx.x, N, per, n, blk);
    const int64_t t0 = int64_t(blk) * wg_tokens;
    const int rows = int(min<int64_t>(T - t0, wg_tokens));
    const int c0 = 16 * NCB * int(blockIdx.y), ncols = min(16 * NCB, Wb - c0);
    const auto xr = mfma::make_rsrc(x + (n * T + t0) * Wa, int64_t(rows) * Wa * es);
    const auto orr = mfma::make_rsrc(out + (n * T + t0) * Wb, int64_t(rows) * Wb * es);
    auto load = [&](X& v, int row0) {
        if constexpr (kTurn) {
            v.load(xr, row0, Wa, lane);
        } else {
#pragma unroll
            for (int j = 0; j < X::kOps; ++j) {
                const int c = X::kPer * (4 * j + g);
                v.x[j].load(xr, c < Wa ? ((row0 + lr) * Wa + c) * es : kOutside);
            }
        }
    };
    X next;
    load(next, 16 * w);
    stage_operand<64 * NW, NJ, NCB, kB16>(smem, op, n, Wa, c0, ncols, blk == 0, blockIdx.y == 0);
    auto bias_of = [&](int cb, int g) {
        f32x4 b;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int c = 16 * cb + 4 * g + r;
            b[r] = op.bias && c < ncols ? op.bias[n * op.bias_stream + c0 + c] : 0.f;
        }
        return b;
    };
    f32x4 bias[NCB];
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) bias[cb] = bias_of(cb, g);
    __syncthreads();
    for (int r0 = 16 * w; r0 < rows; r0 += 16 * NW) {
        X cur = next;
        if constexpr (kTurn) cur.turn(reinterpret_cast<typename X::Raw*>(mine), lane, g, lr);
        load(next, r0 + 16 * NW);  // past the block: zeros
        f32x4 acc[NCB];
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) acc[cb] = bias[cb];
        const uint64_t bad = cur.nonfinite();
        cur.template times<NCB>(smem, lane, acc);
        typename O::Raw* to = reinterpret_cast<typename O::Raw*>(mine);
        O::store(to, acc, orr, r0, Wb, c0, ncols, lane, g, lr, [&] {
            if constexpr (kB16) {
                if (bad) whole_products<TIn, NJ, NCB>(to, bad, xr, r0, Wa, smem, lane, bias_of);
            }
        });
    }
}

// ---------------------------------------------------------------------------
// The backward at S = d = 64 in two passes, as the vector-ALU kernels split it
// (noncausal_v4.hip): the query side reads Q and dOut once (dQ, and the dE
// records), the key side K and V once (dK, dV), forming dB and dA from the dE
// records as it stages them.

// Query side: one workgroup per (tile, stream), wave w on the steps w, w + 4,
// .. of the tile; the dE records have nc_sums_kernel's order of sums, bit for
// bit.  dOut's rows, loaded for the reduction, are turned for the map through
// the wave's LDS.
template <typename TIn>
__global__ __launch_bounds__(kThreads, 2) void nc_query64_kernel(
    const TIn* __restrict__ q, const TIn* __restrict__ gout, TIn* __restrict__ dq, const float* __restrict__ state,
    float* __restrict__ records, int64_t N, int64_t T, int chunk, int64_t chunks, int64_t rec) {
    constexpr int W = 64, es = int(sizeof(TIn)), kTok = kStep<TIn>, kLoads = kTok / 4;
    constexpr bool kB16 = sizeof(TIn) == 2;
    using V4 = Vec<TIn, 4>;
    using X = MapRows<TIn, 4, kB16>;
    using O = OutRows<TIn, 4>;
    extern __shared__ __align__(16) float smem[];
    float* Em = smem;  // E^T in operand order
    const int lane = threadIdx.x & 63, g = lane >> 4, lr = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    unsigned char* mine = reinterpret_cast<unsigned char*>(smem + kMatrixFloats<4, 4, kB16>) + w * kTok * W * es;
    int64_t n;
    int ci;
    stream_block(blockIdx.x, N, int(chunks), n, ci);
    const int64_t t0 = int64_t(ci) * chunk;
    const int rows = int(min(T, t0 + chunk) - t0);
    const auto qr = mfma::make_rsrc(q + (n * T + t0) * W, int64_t(rows) * W * es);
    const auto gr = mfma::make_rsrc(gout + (n * T + t0) * W, int64_t(rows) * W * es);
    const auto dr = mfma::make_rsrc(dq + (n * T + t0) * W, int64_t(rows) * W * es);
    V4 qv[kLoads], gv[kLoads];
    auto load = [&](int r0) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            qv[i].load(qr, ((r0 + 4 * i + g) * W + 4 * lr) * es);
            gv[i].load(gr, ((r0 + 4 * i + g) * W + 4 * lr) * es);
        }
    };
    load(kTok * w);
    {
        // Thread (row, quad) = (tid / 16, tid % 16) stages E[s][4 quad ..] of
        // rows s = row + 16 m: M[a = c][b = s] = E[s][c].
        const float* sn = state + n * (W * W + W);
        const int row = threadIdx.x >> 4, quad = threadIdx.x & 15;
        f32x4 b[4];
        float a[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            b[m] = *reinterpret_cast<const f32x4*>(sn + (row + 16 * m) * W + 4 * quad);
            a[m] = sn[W * W + row + 16 * m];
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const float den = a[m] + kEps;
            put_matrix<4, kB16, false>(Em, 4 * quad, row + 16 * m,
                                       f32x4{b[m][0] / den, b[m][1] / den, b[m][2] / den, b[m][3] / den});
        }
    }
    __syncthreads();
    Outer<4, 4> o;
    o.clear();
    typename V4::Raw* t = reinterpret_cast<typename V4::Raw*>(mine);
    // dOut's rows as MapRows::turn leaves them, 16 rows at a time: four-value
    // units, two of which make a bf16 operand.
    constexpr int kPerOp = X::kPer / 4;
    auto at = [](int row, int u) { return row * 16 + kPerOp * ((u / kPerOp) ^ (row & (X::kUnits - 1))) + u % kPerOp; };
    for (int r0 = kTok * w; r0 < rows; r0 += kTok * kWaves) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int i = 0; i < kLoads; ++i) t[at(4 * i + g, lr)] = gv[i].v;
        const Columns<TIn, 4> qc(qv), gc(gv);
        load(r0 + kTok * kWaves);  // past the tile: zeros
        o.template add<false>(qc, gc);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        X gm[kTok / 16];
#pragma unroll
        for (int h = 0; h < kTok / 16; ++h)
#pragma unroll
            for (int j = 0; j < X::kOps; ++j)
                gm[h].x[j].v = *reinterpret_cast<const typename X::Raw*>(t + at(16 * h + lr, kPerOp * (4 * j + g)));
#pragma unroll
        for (int h = 0; h < kTok / 16; ++h) {
            f32x4 acc[4];
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) acc[cb] = f32x4{0.f, 0.f, 0.f, 0.f};
            const uint64_t bad = gm[h].nonfinite();
            gm[h].template times<4>(Em, lane, acc);
            typename O::Raw* to = reinterpret_cast<typename O::Raw*>(mine);
            O::store(to, acc, dr, r0 + 16 * h, W, 0, W, lane, g, lr, [&] {
                if constexpr (kB16) {
                    if (bad)
                        whole_products<TIn, 4, 4>(to, bad, gr, r0 + 16 * h, W, Em, lane,
                                                  [](int, int) { return f32x4{0.f, 0.f, 0.f, 0.f}; });
                }
            });
        }
    }
    o.combine(smem, records + (n * chunks + ci) * rec, W, W, 0, 0, false, w, g, lr);
}

// Key side: one workgroup per (block of wg_tokens tokens, stream).  dB and dA
// come from `parts` dE records (summed in order) and the state, or with
// dB_ready from bwd_finalize_kernel's dB and dA.  dk or dv may be null.
template <typename TIn, int NW>
__global__ __launch_bounds__(64 * NW) void nc_key64_kernel(
    const TIn* __restrict__ k, const TIn* __restrict__ v, TIn* __restrict__ dk, TIn* __restrict__ dv,
    const float* __restrict__ dE_records, int parts, int64_t rec, const float* __restrict__ state,
    const float* __restrict__ dB_ready, const float* __restrict__ dA_ready, int64_t N, int64_t T, int wg_tokens,
    int per) {
    constexpr int W = 64, es = int(sizeof(TIn));
    constexpr bool kB16 = sizeof(TIn) == 2;
    using X = MapRows<TIn, 4, kB16>;
    using O = OutRows<TIn, 4>;
    static_assert(X::kBytes == O::kBytes, "one turn buffer");
    extern __shared__ __align__(16) float smem[];
    float* Mv = smem;                                    // dV's operand: M[a = s][b = c] = dB[s][c]
    float* Mk = Mv + kMatrixFloats<4, 4, kB16>;          // dK's operand: M[a = c][b = s] = dB[s][c]
    float* dAs = Mk + kMatrixFloats<4, 4, kB16>;         // [64]
    const int lane = threadIdx.x & 63, g = lane >> 4, lr = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    unsigned char* mine = reinterpret_cast<unsigned char*>(dAs + W) + w * X::kBytes;
    int64_t n;
    int blk;
    stream_block(blockIdx.x, N, per, n, blk);
    const int64_t t0 = int64_t(blk) * wg_tokens;
    const int rows = int(min<int64_t>(T - t0, wg_tokens));
    // A gradient that is not asked for: its rows are neither read nor written.
    const int64_t kb = dv ? int64_t(rows) * W * es : 0, vb = dk ? int64_t(rows) * W * es : 0;
    const auto kr = mfma::make_rsrc(dv ? k + (n * T + t0) * W : nullptr, kb);
    const auto vr = mfma::make_rsrc(dk ? v + (n * T + t0) * W : nullptr, vb);
    const auto dkr = mfma::make_rsrc(dk ? dk + (n * T + t0) * W : nullptr, vb);
    const auto dvr = mfma::make_rsrc(dv ? dv + (n * T + t0) * W : nullptr, kb);
    X kn, vn;
    kn.load(kr, 16 * w, W, lane);
    vn.load(vr, 16 * w, W, lane);
    {
        // Thread (row, quad) forms dB[s][4 quad ..] of rows s = row + kRows m
        // (the 16 threads of a row are 16 lanes of one wave).
        constexpr int kRows = 4 * NW, kPer = W / kRows;
        const int row = threadIdx.x >> 4, quad = threadIdx.x & 15;
        f32x4 db[kPer];
        float da[kPer];
        if (dB_ready) {
#pragma unroll
            for (int m = 0; m < kPer; ++m) {
                db[m] = *reinterpret_cast<const f32x4*>(dB_ready + n * W * W + (row + kRows * m) * W + 4 * quad);
                da[m] = dA_ready[n * W + row + kRows * m];
            }
        } else {
            const float* sn = state + n * (W * W + W);
            const float* rn = dE_records + n * int64_t(parts) * rec;
            f32x4 b[kPer], gs[kPer];
            float a[kPer];
#pragma unroll
            for (int m = 0; m < kPer; ++m) {
                b[m] = *reinterpret_cast<const f32x4*>(sn + (row + kRows * m) * W + 4 * quad);
                a[m] = sn[W * W + row + kRows * m];
                gs[m] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
            // Two parts' loads in flight at a time.
            for (int t = 0; t < parts; t += 2) {
                const float* r0 = rn + int64_t(t) * rec;
                const float* r1 = rn + int64_t(min(t + 1, parts - 1)) * rec;
                f32x4 p0[kPer], p1[kPer];
#pragma unroll
                for (int m = 0; m < kPer; ++m) {
                    p0[m] = *reinterpret_cast<const f32x4*>(r0 + (row + kRows * m) * W + 4 * quad);
                    p1[m] = *reinterpret_cast<const f32x4*>(r1 + (row + kRows * m) * W + 4 * quad);
                }
#pragma unroll
                for (int m = 0; m < kPer; ++m) {
                    gs[m] += p0[m];
                    if (t + 1 < parts) gs[m] += p1[m];
                }
            }
#pragma unroll
            for (int m = 0; m < kPer; ++m) {
                const float den = a[m] + kEps;
                float sum = 0.f;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    db[m][i] = gs[m][i] / den;
                    sum = fmaf(gs[m][i], b[m][i] / den, sum);
                }
#pragma unroll
                for (int off = 8; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
                da[m] = -sum / den;
            }
        }
#pragma unroll
        for (int m = 0; m < kPer; ++m) {
            put_matrix<4, kB16, false>(Mk, 4 * quad, row + kRows * m, db[m]);
            put_matrix<4, kB16, true>(Mv, row + kRows * m, 4 * quad, db[m]);
            if (quad == 0) dAs[row + kRows * m] = da[m];
        }
    }
    __syncthreads();
    f32x4 bias[4];
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) bias[cb] = *reinterpret_cast<const f32x4*>(dAs + 16 * cb + 4 * g);
    typename X::Raw* tx = reinterpret_cast<typename X::Raw*>(mine);
    typename O::Raw* to = reinterpret_cast<typename O::Raw*>(mine);
    for (int r0 = 16 * w; r0 < rows; r0 += 16 * NW) {
        const int rn = r0 + 16 * NW;  // past the block: zeros
        X vc = vn;
        vc.turn(tx, lane, g, lr);
        vn.load(vr, rn, W, lane);
        if (dk) {
            f32x4 acc[4];
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) acc[cb] = bias[cb];
            const uint64_t bad = vc.nonfinite();
            vc.template times<4>(Mk, lane, acc);
            O::store(to, acc, dkr, r0, W, 0, W, lane, g, lr, [&] {
                if constexpr (kB16) {
                    if (bad)
                        whole_products<TIn, 4, 4>(to, bad, vr, r0, W, Mk, lane, [&](int cb, int g) {
                            return *reinterpret_cast<const f32x4*>(dAs + 16 * cb + 4 * g);
                        });
                }
            });
        }
        X kc = kn;
        kc.turn(tx, lane, g, lr);
        kn.load(kr, rn, W, lane);
        if (dv) {
            f32x4 acc[4];
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) acc[cb] = f32x4{0.f, 0.f, 0.f, 0.f};
            const uint64_t bad = kc.nonfinite();
            kc.template times<4>(Mv, lane, acc);
            O::store(to, acc, dvr, r0, W, 0, W, lane, g, lr, [&] {
                if constexpr (kB16) {
                    if (bad)
                        whole_products<TIn, 4, 4>(to, bad, kr, r0, W, Mv, lane,
                                                  [](int, int) { return f32x4{0.f, 0.f, 0.f, 0.f}; });
                }
            });
        }
    }
}

// Values per lane for a width: 16 lanes cover it, or a block of 64.
int lane_values(int W) { return W <= 16 ? 1 : W <= 32 ? 2 : 4; }

// Tokens per workgroup of a map, whole 16-token tiles.  The blocks of all
// streams are one grid dimension, and a launch of 2^32 threads or more wraps
// around without an error.
int map_wg_tokens(const Problem& p, int slices) {
    const int64_t most = ((int64_t(1) << 32) - 1) / (64 * kMapWaves) / p.N;
    const int64_t per = std::min(most, nc_blocks_per_stream(p.N * slices, p.T, p.dtype, kMapMaxTokens));
    return int(((p.T + per - 1) / per + 15) / 16 * 16);
}

template <typename TIn, int EA, int EB, bool kEndFirst = false>
hipError_t launch_sums_e(const void* x, const void* y, float* records, const Problem& p, int Wa, int Wb,
                         hipStream_t stream) {
    const int ab = (Wa + 16 * EA - 1) / (16 * EA), bb = (Wb + 16 * EB - 1) / (16 * EB);
    const dim3 grid(unsigned(p.tiles), unsigned(p.N), unsigned(ab * bb));
    nc_sums_kernel<TIn, EA, EB, kEndFirst><<<grid, kThreads, Outer<EA, EB>::kLdsFloats * sizeof(float), stream>>>(
        static_cast<const TIn*>(x), static_cast<const TIn*>(y), records, p.T, p.tile, p.tiles, p.rec, Wa, Wb, bb,
        kEndFirst ? cache_kept_rows(p) : 0);
    return hipGetLastError();
}

template <typename TIn>
hipError_t launch_sums_t(const void* x, const void* y, float* records, const Problem& p, int Wa, int Wb,
                         hipStream_t stream) {
    // bf16 vectors are at least one word.
    const int ea = lane_values(Wa) < 2 ? 2 : lane_values(Wa), eb = lane_values(Wb) < 2 ? 2 : lane_values(Wb);
    if (ea == 2 && eb == 2) return launch_sums_e<TIn, 2, 2>(x, y, records, p, Wa, Wb, stream);
    if (ea == 2) return launch_sums_e<TIn, 2, 4>(x, y, records, p, Wa, Wb, stream);
    if (eb == 2) return launch_sums_e<TIn, 4, 2>(x, y, records, p, Wa, Wb, stream);
    return launch_sums_e<TIn, 4, 4>(x, y, records, p, Wa, Wb, stream);
}

template <typename TIn, int NJ, int NCB, bool kB16>
hipError_t launch_map_b(const void* x, void* out, const MapOperand& op, const Problem& p, int Wa, int Wb,
                        hipStream_t stream) {
    const int slices = (Wb + 16 * NCB - 1) / (16 * NCB);
    const int wt = map_wg_tokens(p, slices);
    const int per = int((p.T + wt - 1) / wt);
    const dim3 grid(unsigned(per * p.N), unsigned(slices));
    constexpr int NW = kMapWaves;
    constexpr size_t kTurn = NJ <= 8 ? MapRows<TIn, NJ, kB16>::kBytes : 0, kOut = OutRows<TIn, NCB>::kBytes;
    const size_t lds = kMatrixFloats<NJ, NCB, kB16> * sizeof(float) + NW * (kTurn > kOut ? kTurn : kOut);
    nc_map_kernel<TIn, NJ, NCB, kB16, NW><<<grid, 64 * NW, lds, stream>>>(static_cast<const TIn*>(x), static_cast<TIn*>(out),
                                                                 op, p.N, p.T, Wa, Wb, wt, per);
    return hipGetLastError();
}

// bf16 rows of whole 8-value operands take the bf16 matrix instructions; rows
// that end in half an operand are widened to fp32.
template <typename TIn, int NJ, int NCB>
hipError_t launch_map_e(const void* x, void* out, const MapOperand& op, const Problem& p, int Wa, int Wb,
                        hipStream_t stream) {
    if constexpr (sizeof(TIn) == 2) {
        if (Wa % 8 == 0) return launch_map_b<TIn, NJ, NCB, true>(x, out, op, p, Wa, Wb, stream);
    }
    return launch_map_b<TIn, NJ, NCB, false>(x, out, op, p, Wa, Wb, stream);
}

template <typename TIn, int NJ>
hipError_t launch_map_j(const void* x, void* out, const MapOperand& op, const Problem& p, int Wa, int Wb,
                        hipStream_t stream) {
    if (Wb <= 16) return launch_map_e<TIn, NJ, 1>(x, out, op, p, Wa, Wb, stream);
    if (Wb <= 32) return launch_map_e<TIn, NJ, 2>(x, out, op, p, Wa, Wb, stream);
    return launch_map_e<TIn, NJ, 4>(x, out, op, p, Wa, Wb, stream);
}

template <typename TIn>
hipError_t launch_map_t(const void* x, void* out, const MapOperand& op, const Problem& p, int Wa, int Wb,
                        hipStream_t stream) {
    if (Wa <= 16) return launch_map_j<TIn, 1>(x, out, op, p, Wa, Wb, stream);
    if (Wa <= 32) return launch_map_j<TIn, 2>(x, out, op, p, Wa, Wb, stream);
    if (Wa <= 64) return launch_map_j<TIn, 4>(x, out, op, p, Wa, Wb, stream);
    if (Wa <= 128) return launch_map_j<TIn, 8>(x, out, op, p, Wa, Wb, stream);
    return launch_map_j<TIn, 16>(x, out, op, p, Wa, Wb, stream);
}

template <typename TIn>
size_t query64_lds_bytes() {
    const size_t loop = kMatrixFloats<4, 4, sizeof(TIn) == 2> * sizeof(float) +
                        size_t(kWaves) * kStep<TIn> * 64 * sizeof(TIn);
    const size_t combine = Outer<4, 4>::kLdsFloats * sizeof(float);
    return loop > combine ? loop : combine;
}

template <typename TIn>
size_t key64_lds_bytes() {
    return size_t(2 * kMatrixFloats<4, 4, sizeof(TIn) == 2> + 64) * sizeof(float) +
           kMapWaves * MapRows<TIn, 4, sizeof(TIn) == 2>::kBytes;
}

}  // namespace

// Every workgroup has a fixed cost (staging its matrix or adding its waves'
// partial sums) next to its tokens, and a launch takes as long as the CU with
// the most workgroups: the split with the least (workgroups per CU) (tokens +
// fixed) wins.  The fixed cost in tokens' worth of the loop is about 96 (fp32)
// or 256 (bf16, whose loop is faster).  Measured forward + backward, bf16, S =
// d = 64: N = 192, T = 577: 47 us with 1 block per stream, 50 with 2, 65 with 3;
// N = 96, T = 1024: 58, 43 (2), 50 (3), 47 (4), 65 (6); fp32, N = 384, T = 1024:
// 263, 234 (2), 247 (3), 239 (4).
int64_t nc_blocks_per_stream(int64_t streams, int64_t T, int dtype, int64_t max_tokens) {
    constexpr int64_t kCus = 256;
    const int64_t fixed = dtype == RACE_BF16 ? 256 : 96;
    const int64_t least = (T + max_tokens - 1) / max_tokens, most = (T + 63) / 64;
    int64_t best = least, best_cost = INT64_MAX;
    for (int64_t per = least; per <= most && (per == least || streams * (per - 1) < 4 * kCus); ++per) {
        const int64_t cost = (streams * per + kCus - 1) / kCus * ((T + per - 1) / per + fixed);
        if (cost < best_cost) {
            best_cost = cost;
            best = per;
        }
    }
    return best;
}

hipError_t launch_nc_sums(const void* x, const void* y, float* records, const Problem& p, int Wa, int Wb,
                          hipStream_t stream) {
    if (p.dtype == RACE_BF16) return launch_sums_t<bf16_t>(x, y, records, p, Wa, Wb, stream);
    return launch_sums_t<float>(x, y, records, p, Wa, Wb, stream);
}

hipError_t launch_tile_sums_b16(const void* k, const void* v, float* records, const Problem& p, hipStream_t stream) {
    if (p.S != 64 || p.d != 64 || p.dtype != RACE_BF16) return hipErrorInvalidValue;
    return launch_sums_e<bf16_t, 4, 4, true>(k, v, records, p, 64, 64, stream);
}

hipError_t launch_nc_map(const void* x, void* out, const MapOperand& op, const Problem& p, int Wa, int Wb,
                         hipStream_t stream) {
    if (p.dtype == RACE_BF16) return launch_map_t<bf16_t>(x, out, op, p, Wa, Wb, stream);
    return launch_map_t<float>(x, out, op, p, Wa, Wb, stream);
}

hipError_t launch_nc_query64(const void* q, const void* g, void* dq, const float* state, float* records,
                             const Problem& p, hipStream_t stream) {
    if (p.S != 64 || p.d != 64) return hipErrorInvalidValue;
    const dim3 grid(unsigned(p.tiles * p.N));
    const size_t lds = p.dtype == RACE_BF16 ? query64_lds_bytes<bf16_t>() : query64_lds_bytes<float>();
    if (p.dtype == RACE_BF16)
        nc_query64_kernel<bf16_t><<<grid, kThreads, lds, stream>>>(
            static_cast<const bf16_t*>(q), static_cast<const bf16_t*>(g), static_cast<bf16_t*>(dq), state, records,
            p.N, p.T, p.tile, p.tiles, p.rec);
    else
        nc_query64_kernel<float><<<grid, kThreads, lds, stream>>>(
            static_cast<const float*>(q), static_cast<const float*>(g), static_cast<float*>(dq), state, records,
            p.N, p.T, p.tile, p.tiles, p.rec);
    return hipGetLastError();
}

hipError_t launch_nc_key64(const void* k, const void* v, void* dk, void* dv, const float* dE_records,
                           const float* state, const float* dB_ready, const float* dA_ready, const Problem& p,
                           hipStream_t stream) {
    if (p.S != 64 || p.d != 64) return hipErrorInvalidValue;
    if (!dB_ready && (p.tiles > kNcFoldParts || !dE_records || !state)) return hipErrorInvalidValue;
    const int wt = map_wg_tokens(p, 1);
    const int per = int((p.T + wt - 1) / wt);
    const dim3 grid(unsigned(per * p.N));
    const size_t lds = p.dtype == RACE_BF16 ? key64_lds_bytes<bf16_t>() : key64_lds_bytes<float>();
    const int parts = int(p.tiles);
    if (p.dtype == RACE_BF16)
        nc_key64_kernel<bf16_t, kMapWaves><<<grid, 64 * kMapWaves, lds, stream>>>(
            static_cast<const bf16_t*>(k), static_cast<const bf16_t*>(v), static_cast<bf16_t*>(dk),
            static_cast<bf16_t*>(dv), dE_records, parts, p.rec, state, dB_ready, dA_ready, p.N, p.T, wt, per);
    else
        nc_key64_kernel<float, kMapWaves><<<grid, 64 * kMapWaves, lds, stream>>>(
            static_cast<const float*>(k), static_cast<const float*>(v), static_cast<float*>(dk),
            static_cast<float*>(dv), dE_records, parts, p.rec, state, dB_ready, dA_ready, p.N, p.T, wt, per);
    return hipGetLastError();
}

}  // namespace race
