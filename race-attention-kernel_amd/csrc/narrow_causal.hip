// narrow_causal.hip -- causal output pass on the fp32 matrix cores for the
// shapes the tiled MFMA kernels have no specialization for: up to 64 buckets,
// any number of value columns (in slices of up to 64), both multiples of 4.
//
// The chunk identity of mfma_causal.hip in steps of 16 tokens, a wave keeping
// its whole state and step in registers (no LDS and no barrier in the walk).
// Every product is v_mfma_f32_16x16x4_f32, so operands, products and sums are
// fp32 as in the vector-ALU pass (causal_output_valu_kernel, which walks a
// tile with one workgroup and serial dot products).
//
// Lane (g, lr) = (lane / 16, lane % 16).  NE = values per lane of a bucket row
// (16 lanes cover S <= 16 NE), ND the same for the value columns of a slice.
//   row layout      token 4 g + i, buckets NE lr .. (K) and columns ND lr ..
//                   (V): operands of K^T V (A and B) and of P V (V)
//   quarter layout  token lr, buckets 4 NE g .. + 4 NE - 1 (Q, K, W): operands
//                   of K W^T and W B0.  A running sum over tokens is a scan over
//                   the 16 lanes of a row (DPP).
//   B0              the accumulators of K^T V: row 4 g + r of block e is bucket
//                   4 NE g + NE r + e, column lr of block f is column ND lr + f:
//                   the A operand of (W B0)^T as they stand, step (r, e) taking
//                   value NE r + e of W's quarter
//   P^T             the accumulator of K W^T: row 4 g + r is token j = 4 g + r of
//                   query lr, the B operand of (P V)^T as it stands.
// Per step: Abar = A0 + scan(K), W = Q / (Abar + eps), P = tril(W K^T),
// O = W B0 + P V, A0 += 1^T K, B0 += K^T V.
//
// A workgroup of four waves owns a tile and slice; each wave walks a quarter
// of the tile, from the tile's prefix record plus the sums of the earlier
// quarters, which the waves form first (K and V again, mostly from cache):
// four times the waves of one walk per tile, which is what a launch of a few
// hundred tiles lacks.
//
// Bound by the chain of one step (scan, division, products) at the few waves
// such launches have.  Measured against the vector-ALU pass, fp32: N = 32, T =
// 5001, S = 16, d = 32 228 -> 17 us (the whole op 261 -> 28 us with the sums on
// the matrix cores too); whole ops over S 4 .. 64, d 4 .. 128, N T 128 to 524288
// tokens, both dtypes, 2.3x to 23x.
#include "mfma_common.h"

namespace race {
namespace {

using mfma::f32x4;
using mfma::kOutside;
using mfma::mfma4;
using mfma::u32x4;

constexpr int kWaves = kThreads / 64;

// E consecutive values at byte offset `off`, as floats.
template <typename TIn, int E>
__device__ __forceinline__ void load_vals(__amdgpu_buffer_rsrc_t r, int off, float (&x)[E]) {
    if constexpr (sizeof(TIn) == 4) {
        if constexpr (E == 4) {
            const f32x4 v = __builtin_bit_cast(f32x4, mfma::buf_load16<0>(r, off));
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = v[e];
        } else if constexpr (E == 2) {
            const uint2 v = mfma::buf_load8<0>(r, off);
            x[0] = __uint_as_float(v.x);
            x[1] = __uint_as_float(v.y);
        } else {
            x[0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
        }
    } else {
        if constexpr (E == 4) {
            const uint2 v = mfma::buf_load8<0>(r, off);
            x[0] = mfma::lo_half(v.x);
            x[1] = mfma::hi_half(v.x);
            x[2] = mfma::lo_half(v.y);
            x[3] = mfma::hi_half(v.y);
        } else if constexpr (E == 2) {
            const uint32_t v = __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
            x[0] = mfma::lo_half(v);
            x[1] = mfma::hi_half(v);
        } else {
            x[0] = __uint_as_float(uint32_t(__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0)) << 16);
        }
    }
}

// x plus the value `n` lanes back in the 16-lane row (zero past its start).
template <int kShift>
__device__ __forceinline__ float add_back(float x) {
    const int y = __builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x110 + kShift, 0xf, 0xf, true);
    return x + __int_as_float(y);
}
// Inclusive sum over the lanes of a 16-lane row.
__device__ __forceinline__ float scan16(float x) {
    x = add_back<1>(x);
    x = add_back<2>(x);
    x = add_back<4>(x);
    return add_back<8>(x);
}

// The value of the 16-lane row's last lane, in every lane of it.
__device__ __forceinline__ float last16(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x15f, 0xf, 0xf, true));
}

template <typename TIn, int NE, int ND>
__global__ __launch_bounds__(kThreads, 2) void causal_output_narrow_kernel(
    const TIn* __restrict__ q, const TIn* __restrict__ k, const TIn* __restrict__ v, TIn* __restrict__ out,
    const float* __restrict__ records, int64_t T, int S, int d, int tile, int64_t tiles, int64_t rec) {
    constexpr int es = int(sizeof(TIn));
    constexpr int kState = NE * ND * 64 * 4;  // floats of one wave's B accumulators
    extern __shared__ __align__(16) float smem[];
    f32x4* Bs = reinterpret_cast<f32x4*>(smem);         // [3 waves][NE ND][64 lanes]
    float* As = smem + (kWaves - 1) * kState;           // [3 waves][16 NE]
    const int lane = threadIdx.x & 63, g = lane >> 4, lr = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t n = blockIdx.y, ti = blockIdx.x, t0 = ti * tile;
    const int rows = int(min(T, t0 + tile) - t0);
    const int c0 = 16 * ND * int(blockIdx.z);
    const int seg = tile / kWaves, first = w * seg, end = min(rows, first + seg);
    const auto qr = mfma::make_rsrc(q + (n * T + t0) * S, int64_t(rows) * S * es);
    const auto kr = mfma::make_rsrc(k + (n * T + t0) * S, int64_t(rows) * S * es);
    const auto vr = mfma::make_rsrc(v + (n * T + t0) * d, int64_t(rows) * d * es);
    const auto orr = mfma::make_rsrc(out + (n * T + t0) * d, int64_t(rows) * d * es);

    struct Rows {
        float k[4][NE], v[4][ND];
    };
    auto load_rows = [&](Rows& x, int r0) {
        const int s = NE * lr, c = c0 + ND * lr;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = r0 + 4 * g + i;
            load_vals<TIn, NE>(kr, s < S ? (row * S + s) * es : kOutside, x.k[i]);
            load_vals<TIn, ND>(vr, c < d ? (row * d + c) * es : kOutside, x.v[i]);
        }
    };
    struct Quarter {
        float x[4 * NE];
    };
    auto load_quarter = [&](Quarter& x, __amdgpu_buffer_rsrc_t r, int r0) {
#pragma unroll
        for (int m = 0; m < NE; ++m) {
            const int s = 4 * NE * g + 4 * m;
            float y[4];
            load_vals<TIn, 4>(r, s < S ? ((r0 + lr) * S + s) * es : kOutside, y);
#pragma unroll
            for (int e = 0; e < 4; ++e) x.x[4 * m + e] = y[e];
        }
    };
    f32x4 B[NE][ND];
    auto add_state = [&](const Rows& x) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < NE; ++e)
#pragma unroll
                for (int f = 0; f < ND; ++f) B[e][f] = mfma4(x.k[i][e], x.v[i][f], B[e][f]);
    };
    auto bucket = [&](int e, int r) { return 4 * NE * g + NE * r + e; };

    // The sums of the quarters a later wave starts after.
    Rows x;
    load_rows(x, first);
    if (w < kWaves - 1 && first + seg < rows) {
        float sum[NE];
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            sum[e] = 0.f;
#pragma unroll
            for (int f = 0; f < ND; ++f) B[e][f] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        for (int r0 = first; r0 < end; r0 += 16) {
            const Rows cur = x;
            load_rows(x, r0 + 16);
            add_state(cur);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int e = 0; e < NE; ++e) sum[e] += cur.k[i][e];
        }
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            sum[e] += __shfl_xor(sum[e], 16);
            sum[e] += __shfl_xor(sum[e], 32);
            if (g == 0) As[w * 16 * NE + NE * lr + e] = sum[e];
#pragma unroll
            for (int f = 0; f < ND; ++f) Bs[(w * NE * ND + e * ND + f) * 64 + lane] = B[e][f];
        }
        load_rows(x, first);
    }
    // State at the wave's first token: the tile's record, then the earlier
    // quarters in order.
    Quarter qn, kn;
    load_quarter(qn, qr, first);
    load_quarter(kn, kr, first);
    const float* rp = records + (n * tiles + ti) * rec;
    float A[4 * NE];
#pragma unroll
    for (int e = 0; e < NE; ++e)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int s = bucket(e, r);
            A[NE * r + e] = s < S ? rp[int64_t(S) * d + s] : 0.f;
#pragma unroll
            for (int f = 0; f < ND; ++f) {
                const int c = c0 + ND * lr + f;
                B[e][f][r] = s < S && c < d ? rp[int64_t(s) * d + c] : 0.f;
            }
        }
    __syncthreads();
    if (first >= rows) return;
    for (int u = 0; u < w; ++u) {
#pragma unroll
        for (int e = 0; e < NE; ++e) {
#pragma unroll
            for (int f = 0; f < ND; ++f) {
                const f32x4 p = Bs[(u * NE * ND + e * ND + f) * 64 + lane];
                // Buckets past S hold nothing but products with zero keys (NaN
                // next to an infinite value).
#pragma unroll
                for (int r = 0; r < 4; ++r) B[e][f][r] += bucket(e, r) < S ? p[r] : 0.f;
            }
        }
#pragma unroll
        for (int i = 0; i < 4 * NE; ++i) A[i] += As[u * 16 * NE + 4 * NE * g + i];
    }

    for (int r0 = first; r0 < end; r0 += 16) {
        const Rows cur = x;
        Quarter W = qn;
        const Quarter kq = kn;
        load_rows(x, r0 + 16);  // past the quarter: never used
        load_quarter(qn, qr, r0 + 16);
        load_quarter(kn, kr, r0 + 16);
        // Running mass and W; the mass after the step's last token.
#pragma unroll
        for (int i = 0; i < 4 * NE; ++i) {
            const float mass = A[i] + scan16(kq.x[i]);
            W.x[i] = W.x[i] / (mass + kEps);
            A[i] = last16(mass);
        }
        // P^T, masked to j <= i.
        f32x4 p0 = {0.f, 0.f, 0.f, 0.f}, p1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4 * NE; i += 2) {
            p0 = mfma4(kq.x[i], W.x[i], p0);
            p1 = mfma4(kq.x[i + 1], W.x[i + 1], p1);
        }
        f32x4 P = p0 + p1;
#pragma unroll
        for (int r = 0; r < 4; ++r) P[r] = 4 * g + r <= lr ? P[r] : 0.f;
        f32x4 o[ND];
#pragma unroll
        for (int f = 0; f < ND; ++f) o[f] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int e = 0; e < NE; ++e)
#pragma unroll
                for (int f = 0; f < ND; ++f) o[f] = mfma4(B[e][f][r], W.x[NE * r + e], o[f]);
        // P V as a product takes the zeros above the diagonal times later
        // tokens' values: with an infinity or NaN among the step's values the
        // sum over j <= i is taken one token at a time instead.
        bool finite = true;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int f = 0; f < ND; ++f) finite = finite && fabsf(cur.v[i][f]) < __builtin_inff();
        if (__all(finite)) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int f = 0; f < ND; ++f) o[f] = mfma4(cur.v[r][f], P[r], o[f]);
            add_state(cur);
        } else {
            for (int jg = 0; jg < 4; ++jg)
#pragma unroll
                for (int jr = 0; jr < 4; ++jr) {
                    const float p = __shfl(P[jr], 16 * jg + lr);
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int f = 0; f < ND; ++f) {
                            const float val = __shfl(cur.v[jr][f], 16 * jg + 4 * g + r);
                            if (4 * jg + jr <= lr) o[f][r] = fmaf(p, val, o[f][r]);
                        }
                }
            add_state(cur);
#pragma unroll
            for (int e = 0; e < NE; ++e)
#pragma unroll
                for (int f = 0; f < ND; ++f)
#pragma unroll
                    for (int r = 0; r < 4; ++r) B[e][f][r] = bucket(e, r) < S ? B[e][f][r] : 0.f;
        }
        // Token lr, columns 4 ND g + ND r + f.
#pragma unroll
        for (int m = 0; m < ND; ++m) {
            f32x4 y;
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = o[(4 * m + i) % ND][(4 * m + i) / ND];
            const int c = c0 + 4 * ND * g + 4 * m;
            mfma::store4<TIn, 0>(orr, c < d ? ((r0 + lr) * d + c) * es : kOutside, y);
        }
    }
}

template <typename TIn, int NE, int ND>
hipError_t launch_e(const void* q, const void* k, const void* v, void* out, const float* records, const Problem& p,
                    hipStream_t stream) {
    const dim3 grid(unsigned(p.tiles), unsigned(p.N), unsigned((p.d + 16 * ND - 1) / (16 * ND)));
    const size_t lds = size_t(kWaves - 1) * (NE * ND * 64 * 4 + 16 * NE) * sizeof(float);
    causal_output_narrow_kernel<TIn, NE, ND><<<grid, kThreads, lds, stream>>>(
        static_cast<const TIn*>(q), static_cast<const TIn*>(k), static_cast<const TIn*>(v), static_cast<TIn*>(out),
        records, p.T, p.S, p.d, p.tile, p.tiles, p.rec);
    return hipGetLastError();
}

template <typename TIn, int NE>
hipError_t launch_d(const void* q, const void* k, const void* v, void* out, const float* records, const Problem& p,
                    hipStream_t stream) {
    if (p.d <= 16) return launch_e<TIn, NE, 1>(q, k, v, out, records, p, stream);
    // With 33 to 64 buckets a slice of 64 columns takes every register of a SIMD
    // (or spills); slices of 32 measured 20 to 25% faster (S = 48, 64, d = 80, 96).
    if constexpr (NE <= 2) {
        if (p.d > 32) return launch_e<TIn, NE, 4>(q, k, v, out, records, p, stream);
    }
    return launch_e<TIn, NE, 2>(q, k, v, out, records, p, stream);
}

template <typename TIn>
hipError_t launch_t(const void* q, const void* k, const void* v, void* out, const float* records, const Problem& p,
                    hipStream_t stream) {
    if (p.S <= 16) return launch_d<TIn, 1>(q, k, v, out, records, p, stream);
    if (p.S <= 32) return launch_d<TIn, 2>(q, k, v, out, records, p, stream);
    return launch_d<TIn, 4>(q, k, v, out, records, p, stream);
}

}  // namespace

bool narrow_causal_supported(int S, int d) { return S <= 64 && S % 4 == 0 && d % 4 == 0; }

hipError_t launch_causal_output_narrow(const void* q, const void* k, const void* v, void* out, const float* records,
                                       const Problem& p, hipStream_t stream) {
    if (!narrow_causal_supported(p.S, p.d) || p.tile % (16 * kWaves) != 0) return hipErrorInvalidValue;
    if (p.dtype == RACE_BF16) return launch_t<bf16_t>(q, k, v, out, records, p, stream);
    return launch_t<float>(q, k, v, out, records, p, stream);
}

}  // namespace race
