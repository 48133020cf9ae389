// hash_rows.hip -- the hashing of BatchedACE (src/race_baseline.py:41-44) and
// its gradient on the fp32 matrix cores, for rows of whole 4-value groups
// (d_k a multiple of 4), 2 to 6 planes per table and 16-byte probability rows.
// hashing.hip holds the functions' definitions and takes every other call.
//
// A wave takes 16 rows at a time and keeps everything of them in registers:
//   projection  U^T [slots][rows] = P X^T on v_mfma_f32_16x16x4_f32 (fp32
//               products and sums, as a scalar dot product has them).  Lane
//               (g, lr) = (lane / 16, lane % 16) loads x[row lr][16 j + 4 g ..
//               + 3]: one 16-byte load per 16 columns, and the four lanes of a
//               row read 64 contiguous bytes.
//   slots       The rows of P are laid out so that the four accumulator values
//               of a lane are whole tables: 4 planes (K = 3, 4; the fourth
//               slot of K = 3 is zero), two tables of 2 (K = 2), or half a
//               table whose other half is the next block's (K = 5, 6).  Lane
//               (g, lr) then holds every plane value of its tables of row lr,
//               and the 2^K corners need no exchange between lanes.
//   corners     A lane's probabilities (or upstream gradients) are one
//               contiguous run of the row; its 16-byte chunks are exchanged
//               with the other three lanes of the row (v_permlane16_swap,
//               v_permlane32_swap: registers against lane groups), so that a
//               load or store instruction covers 64 contiguous bytes per row.
//   gradient    dX^T [columns][rows] = P^T dU^T, the contraction over slots in
//               the order the lanes hold them (step e of lane group g is slot
//               4 g + e): the plane gradients are the operand as they stand.
// The planes sit in LDS in operand order (one 16-byte read per 16 columns or
// slots), staged once per workgroup.
//
// The kernels are bound by memory and, for the gradient, by the latency of one
// group's chain of loads, tanh and products, which the waves of a SIMD cover.
// Measured against one row per thread (hashing.hip), fp32, L = K = 4, d_k = 64:
// 131072 rows forward 29 -> 17 us (67 MB), gradient 110 -> 24.5 us (101 MB);
// 400000 rows 61 -> 35 and 407 -> 64 us; 500 rows 20 -> 5.5 and 39 -> 7 us.
#include "mfma_common.h"

namespace race {
namespace {

using mfma::f32x4;
using mfma::kOutside;
using mfma::mfma4;
using mfma::u32x2;
using mfma::u32x4;

constexpr int kGroups = 2;                          // 16-row groups per wave
constexpr int kWaves = kThreads / 64;
constexpr int kWgRows = 16 * kGroups * kWaves;      // rows per workgroup

// Which table and plane the slot `row` (0..15) of slot block `b` carries.
template <int K>
struct Slots {
    static constexpr int kBlk = K <= 4 ? 1 : 2;     // slot blocks per set of tables
    static constexpr int kTpq = K == 2 ? 2 : 1;     // tables per lane and set
    static constexpr int kTables = 4 * kTpq;        // tables per set
    static constexpr int kVals = kTpq << K;         // probabilities per lane and set
    __device__ static int table(int b, int row) {
        return K == 2 ? 8 * b + (row >> 1) : 4 * (b / kBlk) + (row >> 2);
    }
    __device__ static int plane(int b, int row) {
        return K == 2 ? (row & 1) : 4 * (b % kBlk) + (row & 3);
    }
    static int blocks(int L) { return ((L + kTables - 1) / kTables) * kBlk; }
};

template <typename TIn>
struct Row4;  // four consecutive row values
template <>
struct Row4<float> {
    uint4 v;
    __device__ void load(__amdgpu_buffer_rsrc_t r, int off) { v = mfma::buf_load16<0>(r, off); }
    __device__ f32x4 f32() const { return __builtin_bit_cast(f32x4, v); }
};
template <>
struct Row4<bf16_t> {
    uint2 v;
    __device__ void load(__amdgpu_buffer_rsrc_t r, int off) { v = mfma::buf_load8<0>(r, off); }
    __device__ f32x4 f32() const {
        return f32x4{mfma::lo_half(v.x), mfma::hi_half(v.x), mfma::lo_half(v.y), mfma::hi_half(v.y)};
    }
};

// Lane group g's register i against lane group i's register g, for the four
// 16-byte chunks of a lane (its own inverse).
__device__ __forceinline__ void swap_pair32(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ void swap_pair16(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
template <int NC>
__device__ __forceinline__ void exchange(u32x4 (&q)[NC]) {
    if constexpr (NC == 2) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            uint32_t a = q[0][w], b = q[1][w];
            swap_pair16(a, b);
            q[0][w] = a;
            q[1][w] = b;
        }
    } else if constexpr (NC >= 4) {
#pragma unroll
        for (int c = 0; c < NC; c += 4)
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                uint32_t x0 = q[c][w], x1 = q[c + 1][w], x2 = q[c + 2][w], x3 = q[c + 3][w];
                swap_pair32(x0, x2);
                swap_pair32(x1, x3);
                swap_pair16(x0, x1);
                swap_pair16(x2, x3);
                q[c][w] = x0;
                q[c + 1][w] = x1;
                q[c + 2][w] = x2;
                q[c + 3][w] = x3;
            }
    }
}
// Byte offset in its row of the chunk that register i of lane group g carries
// once exchanged (the lane whose run it belongs to, then the chunk of it).
template <int NC>
__device__ __forceinline__ int chunk_byte(int i, int g) {
    const int owner = NC == 1 ? g : NC == 2 ? ((g & 2) | i) : (i & 3);
    const int chunk = NC == 1 ? 0 : NC == 2 ? (g & 1) : ((i & ~3) | g);
    return 16 * (owner * NC + chunk);
}

// Planes as operands in LDS.  Projection: entry (b NJ + j) 64 + lane holds
// P[slot 16 b + lr][16 j + 4 g .. + 3].  Gradient: P[slot 16 b + 4 g .. + 3][16 j + lr].
template <int K, int NJ, bool kGrad>
__device__ __forceinline__ void stage_planes(f32x4* __restrict__ dst, const float* __restrict__ planes_T,
                                             int blocks, int dk, int L) {
    const int LK = L * K;
    for (int e = threadIdx.x; e < blocks * NJ * 64; e += kThreads) {
        const int lane = e & 63, j = (e >> 6) % NJ, b = (e >> 6) / NJ;
        const int g = lane >> 4, lr = lane & 15;
        f32x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = kGrad ? 4 * g + i : lr, col = kGrad ? 16 * j + lr : 16 * j + 4 * g + i;
            const int t = Slots<K>::table(b, row), k = Slots<K>::plane(b, row);
            const bool ok = t < L && k < K && col < dk;
            const float p = planes_T[ok ? col * LK + t * K + k : 0];
            v[i] = ok ? p : 0.f;
        }
        dst[e] = v;
    }
}

template <typename TIn, int NJ>
__device__ __forceinline__ void load_rows(Row4<TIn> (&x)[NJ], __amdgpu_buffer_rsrc_t xr, int r0, int dk,
                                          int g, int lr) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int c = 16 * j + 4 * g;
        x[j].load(xr, c < dk ? ((r0 + lr) * dk + c) * int(sizeof(TIn)) : kOutside);
    }
}

// Plane values of slot block b, rows of `x`: lane (g, lr) gets slots 4 g .. + 3 of row lr.
template <typename TIn, int NJ>
__device__ __forceinline__ f32x4 project(const f32x4* __restrict__ pa, const Row4<TIn> (&x)[NJ], int b, int lane) {
    f32x4 a[4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const f32x4 p = pa[(b * NJ + j) * 64 + lane], xv = x[j].f32();
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = mfma4(p[e], xv[e], a[e]);
    }
    return (a[0] + a[1]) + (a[2] + a[3]);
}

// The product over the planes above the last two of corner quad `quad` (its
// four corners share them), sg the table's K values of sigma(2 u).
template <int K>
__device__ __forceinline__ float upper_product(const float* sg, int quad) {
    float p = 1.f;
#pragma unroll
    for (int k = 0; k + 2 < K; ++k) p *= ((quad >> (K - 3 - k)) & 1) ? sg[k] : 1.0f - sg[k];
    return p;
}

template <typename TIn, int K, int NJ>
__global__ __launch_bounds__(kThreads) void hash_rows_kernel(const TIn* __restrict__ x,
                                                             const float* __restrict__ planes_T,
                                                             TIn* __restrict__ probs, int64_t rows, int dk,
                                                             int L, int blocks) {
    using SL = Slots<K>;
    constexpr int es = int(sizeof(TIn)), NC = SL::kVals * es / 16;
    extern __shared__ __align__(16) unsigned char lds[];
    f32x4* pa = reinterpret_cast<f32x4*>(lds);
    const int lane = threadIdx.x & 63, g = lane >> 4, lr = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t row0 = int64_t(blockIdx.x) * kWgRows;
    const int cnt = int(min<int64_t>(kWgRows, rows - row0));
    const int row_bytes = (L << K) * es;
    const auto xr = mfma::make_rsrc(x + row0 * dk, int64_t(cnt) * dk * es);
    const auto pr = mfma::make_rsrc(probs + (row0 * L << K), int64_t(cnt) * row_bytes);
    Row4<TIn> xs[kGroups][NJ];
#pragma unroll
    for (int gi = 0; gi < kGroups; ++gi) load_rows<TIn, NJ>(xs[gi], xr, 16 * (w + kWaves * gi), dk, g, lr);
    stage_planes<K, NJ, false>(pa, planes_T, blocks, dk, L);
    __syncthreads();
    const float two_over_scale = 2.0f / sqrtf(float(dk));
#pragma unroll
    for (int gi = 0; gi < kGroups; ++gi) {
        const int r0 = 16 * (w + kWaves * gi);
        if (r0 >= cnt) break;
        for (int b = 0, set_byte = 0; b < blocks; b += SL::kBlk, set_byte += 64 * NC) {
            float sg[4 * SL::kBlk];
#pragma unroll
            for (int h = 0; h < SL::kBlk; ++h) {
                const f32x4 u = project<TIn, NJ>(pa, xs[gi], b + h, lane);
#pragma unroll
                for (int i = 0; i < 4; ++i) sg[4 * h + i] = 1.0f / (1.0f + expf(-two_over_scale * tanhf(u[i])));
            }
            u32x4 q[NC];
#pragma unroll
            for (int t = 0; t < SL::kTpq; ++t) {
                const float* s = sg + 2 * t;  // two tables only for K = 2
                const float s1 = s[K - 2], s0 = s[K - 1];
                const float n1 = 1.0f - s1, n0 = 1.0f - s0;
#pragma unroll
                for (int u = 0; u < (1 << K) / 4; ++u) {
                    const float p = upper_product<K>(s, u);
                    const float p0 = (p * n1) * n0, p1 = (p * n1) * s0, p2 = (p * s1) * n0, p3 = (p * s1) * s0;
                    const int quad = t * ((1 << K) / 4) + u;
                    if constexpr (es == 4) {
                        q[quad] = __builtin_bit_cast(u32x4, f32x4{p0, p1, p2, p3});
                    } else {
                        q[quad / 2][2 * (quad & 1)] = mfma::pack2(p0, p1);
                        q[quad / 2][2 * (quad & 1) + 1] = mfma::pack2(p2, p3);
                    }
                }
            }
            exchange<NC>(q);
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                const int byte = set_byte + chunk_byte<NC>(i, g);
                __builtin_amdgcn_raw_buffer_store_b128(
                    q[i], pr, byte < row_bytes ? (r0 + lr) * row_bytes + byte : kOutside, 0, 0);
            }
        }
    }
}

template <typename TIn, int K, int NJ>
__global__ __launch_bounds__(kThreads) void hash_rows_bwd_kernel(
    const TIn* __restrict__ x, const float* __restrict__ planes_T, const TIn* __restrict__ dprobs,
    TIn* __restrict__ dx, int64_t rows, int dk, int L, int blocks) {
    using SL = Slots<K>;
    constexpr int es = int(sizeof(TIn)), NC = SL::kVals * es / 16, R = 1 << K;
    extern __shared__ __align__(16) unsigned char lds[];
    f32x4* pa = reinterpret_cast<f32x4*>(lds);
    f32x4* pt = pa + blocks * NJ * 64;
    const int lane = threadIdx.x & 63, g = lane >> 4, lr = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t row0 = int64_t(blockIdx.x) * kWgRows;
    const int cnt = int(min<int64_t>(kWgRows, rows - row0));
    const int row_bytes = (L << K) * es;
    const auto xr = mfma::make_rsrc(x + row0 * dk, int64_t(cnt) * dk * es);
    const auto gr = mfma::make_rsrc(dprobs + (row0 * L << K), int64_t(cnt) * row_bytes);
    const auto dr = mfma::make_rsrc(dx + row0 * dk, int64_t(cnt) * dk * es);
    // A set of tables' upstream gradients, chunks as exchanged.
    auto load_grads = [&](u32x4 (&q)[NC], int r0, int set_byte) {
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int byte = set_byte + chunk_byte<NC>(i, g);
            q[i] = __builtin_bit_cast(
                u32x4, mfma::buf_load16<0>(gr, byte < row_bytes ? (r0 + lr) * row_bytes + byte : kOutside));
        }
    };
    Row4<TIn> xs[NJ];
    u32x4 q[NC];
    load_rows<TIn, NJ>(xs, xr, 16 * w, dk, g, lr);
    load_grads(q, 16 * w, 0);
    stage_planes<K, NJ, false>(pa, planes_T, blocks, dk, L);
    stage_planes<K, NJ, true>(pt, planes_T, blocks, dk, L);
    __syncthreads();
    const float inv_scale = 1.0f / sqrtf(float(dk));
    for (int r0 = 16 * w; r0 < cnt; r0 += 16 * kWaves) {
        f32x4 acc[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int b = 0, set_byte = 0; b < blocks; b += SL::kBlk, set_byte += 64 * NC) {
            float th[4 * SL::kBlk], sg[4 * SL::kBlk], dp[4 * SL::kBlk];
#pragma unroll
            for (int h = 0; h < SL::kBlk; ++h) {
                const f32x4 u = project<TIn, NJ>(pa, xs, b + h, lane);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    th[4 * h + i] = tanhf(u[i]);
                    sg[4 * h + i] = 1.0f / (1.0f + expf(-2.0f * inv_scale * th[4 * h + i]));
                    dp[4 * h + i] = 0.f;
                }
            }
            u32x4 c[NC];
#pragma unroll
            for (int i = 0; i < NC; ++i) c[i] = q[i];
            // The next set's (or rows') loads go out before this set's arithmetic.
            const bool last = b + SL::kBlk >= blocks;
            if (last) {
                const int rn = r0 + 16 * kWaves;  // past the rows: zeros, never used
                load_rows<TIn, NJ>(xs, xr, rn, dk, g, lr);
                load_grads(q, rn, 0);
            } else {
                load_grads(q, r0, set_byte + 64 * NC);
            }
            exchange<NC>(c);
#pragma unroll
            for (int t = 0; t < SL::kTpq; ++t) {
                const float* s = sg + 2 * t;
                const float s1 = s[K - 2], s0 = s[K - 1];
                const float n1 = 1.0f - s1, n0 = 1.0f - s0;
                float tot = 0.f, pos[K];
#pragma unroll
                for (int k = 0; k < K; ++k) pos[k] = 0.f;
#pragma unroll
                for (int u = 0; u < R / 4; ++u) {
                    const int quad = t * (R / 4) + u;
                    float v[4];
                    if constexpr (es == 4) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(c[quad][i]);
                    } else {
                        const uint32_t w0 = c[quad / 2][2 * (quad & 1)], w1 = c[quad / 2][2 * (quad & 1) + 1];
                        v[0] = mfma::lo_half(w0);
                        v[1] = mfma::hi_half(w0);
                        v[2] = mfma::lo_half(w1);
                        v[3] = mfma::hi_half(w1);
                    }
                    const float p = upper_product<K>(s, u);
                    v[0] *= (p * n1) * n0;
                    v[1] *= (p * n1) * s0;
                    v[2] *= (p * s1) * n0;
                    v[3] *= (p * s1) * s0;
                    const float q4 = (v[0] + v[1]) + (v[2] + v[3]);
                    tot += q4;
                    pos[K - 1] += v[1] + v[3];
                    pos[K - 2] += v[2] + v[3];
#pragma unroll
                    for (int k = 0; k + 2 < K; ++k)
                        if ((u >> (K - 3 - k)) & 1) pos[k] += q4;
                }
                // The slots of a table past L take part in the products below: a
                // row with an infinity left NaN in them (0 * inf).
                const bool there = SL::table(b, 4 * g + 2 * t) < L;
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const float tk = th[2 * t + k];
                    const float du = 2.0f * (pos[k] - s[k] * tot) * (1.0f - tk * tk) * inv_scale;
                    dp[2 * t + k] = there ? du : 0.f;
                }
            }
#pragma unroll
            for (int h = 0; h < SL::kBlk; ++h)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const f32x4 p = pt[((b + h) * NJ + j) * 64 + lane];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        acc[j] = mfma4(p[e], dp[4 * h + e], acc[j]);
                }
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int col = 16 * j + 4 * g;
            mfma::store4<TIn, 0>(dr, col < dk ? ((r0 + lr) * dk + col) * es : kOutside, acc[j]);
        }
    }
}

bool aligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

template <int K>
size_t operand_bytes(int dk, int L) {
    return size_t(Slots<K>::blocks(L)) * (dk <= 64 ? 4 : 8) * 64 * sizeof(f32x4);
}

template <typename TIn, int K>
hipError_t launch_k(const void* x, const float* planes_T, const void* dprobs, void* out, int64_t rows, int dk,
                    int L, hipStream_t stream) {
    const dim3 grid(unsigned((rows + kWgRows - 1) / kWgRows));
    const int blocks = Slots<K>::blocks(L);
    const size_t lds = operand_bytes<K>(dk, L) * (dprobs ? 2 : 1);
    const TIn* xi = static_cast<const TIn*>(x);
    const TIn* gi = static_cast<const TIn*>(dprobs);
    TIn* o = static_cast<TIn*>(out);
    if (dprobs) {
        if (dk <= 64)
            hash_rows_bwd_kernel<TIn, K, 4><<<grid, kThreads, lds, stream>>>(xi, planes_T, gi, o, rows, dk, L, blocks);
        else
            hash_rows_bwd_kernel<TIn, K, 8><<<grid, kThreads, lds, stream>>>(xi, planes_T, gi, o, rows, dk, L, blocks);
    } else {
        if (dk <= 64)
            hash_rows_kernel<TIn, K, 4><<<grid, kThreads, lds, stream>>>(xi, planes_T, o, rows, dk, L, blocks);
        else
            hash_rows_kernel<TIn, K, 8><<<grid, kThreads, lds, stream>>>(xi, planes_T, o, rows, dk, L, blocks);
    }
    return hipGetLastError();
}

template <typename TIn>
hipError_t launch_t(const void* x, const float* planes_T, const void* dprobs, void* out, int64_t rows, int dk,
                    int L, int K, hipStream_t stream) {
    switch (K) {
        case 2: return launch_k<TIn, 2>(x, planes_T, dprobs, out, rows, dk, L, stream);
        case 3: return launch_k<TIn, 3>(x, planes_T, dprobs, out, rows, dk, L, stream);
        case 4: return launch_k<TIn, 4>(x, planes_T, dprobs, out, rows, dk, L, stream);
        case 5: return launch_k<TIn, 5>(x, planes_T, dprobs, out, rows, dk, L, stream);
        case 6: return launch_k<TIn, 6>(x, planes_T, dprobs, out, rows, dk, L, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

// Rows are loaded as 16- or 8-byte groups of four values (d_k a multiple of 4)
// and probability rows as whole 16-byte chunks, from 16-byte aligned arrays;
// K = 1 (no quads of corners), K = 7, 8 (32 and 64 quads of corners unrolled
// per lane) and every other row layout take the row-per-thread kernels.
//
// So do few tables of narrow rows: a set (8 tables of 2 planes, 4 of more) costs
// the same however many of its tables there are, and 16 or fewer columns as much
// as 64, while a thread of the row-per-thread kernels does only what a row
// needs.  Measured against those, fp32, 200000 / 800000 rows, forward: L = 1,
// K = 4, d_k = 32 1.06 / 1.04 of their time, 40 0.86 / 0.90; L = 2 16 0.96 / 1.04,
// 20 0.92 / 1.02; L = 4, K = 2 20 1.04 / 1.11, 24 0.99 / 1.06.  Gradient: L = 1, K = 3
// 12 0.98 / 1.27, 16 0.83 / 1.07; L = 2, K = 3 4 0.80 / 0.97.  bf16 rows cost these
// kernels less (L = 1, K = 4, d_k = 24 1.06 / 1.09, 32 0.98 / 0.99).  Up to 20000
// rows these kernels took 0.6 to 0.95 of the time there too, but a row's result
// does not depend on how many there are.  Within the rest they were faster: at
// d_k = 64, K = 2 .. 6, forward 0.2 to 0.95 of the time, gradient 0.04 to 0.4 (past
// 800000 rows of one table of 64 or three of 32 corners, fp32, bound by the
// writes, forward up to 1.16).
bool hash_rows_supported(const void* x, const void* probs, const void* dx, int dk, int L, int K, int dtype,
                         bool gradient) {
    const int es = dtype == RACE_BF16 ? 2 : 4;
    if (K < 2 || K > 6 || dk % 4 != 0 || ((L << K) * es) % 16 != 0 || !aligned(x) || !aligned(probs) || !aligned(dx))
        return false;
    const int set = K == 2 ? 8 : 4;
    if (gradient) return !(K <= 4 && 4 * L <= set && dk <= 12);
    const int columns = (dtype == RACE_BF16 ? 6 : 8) + (K == 2 ? 2 : 0);
    return !(2 * L <= set && dk <= 32 && L * dk <= columns * set);
}

hipError_t launch_hash_rows(const void* x, const float* planes_T, const void* dprobs, void* out, int64_t rows,
                            int dk, int L, int K, int dtype, hipStream_t stream) {
    if (dtype == RACE_BF16) return launch_t<bf16_t>(x, planes_T, dprobs, out, rows, dk, L, K, stream);
    return launch_t<float>(x, planes_T, dprobs, out, rows, dk, L, K, stream);
}

}  // namespace race
