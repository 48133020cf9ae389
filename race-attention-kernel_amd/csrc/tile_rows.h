// tile_rows.h -- token rows loaded straight into MFMA operand registers, and the
// sums K^T V and 1^T K of a run of tokens by one workgroup of four waves (S = d
// = 64): the tile sums of mfma_direct.hip, and the prefixes of short sequences
// in mfma_causal.hip.  Not part of the ABI.
#pragma once

#include "mfma_common.h"

namespace race {
namespace mfma {

constexpr int kDirC = 32;  // tokens per sub-chunk
// Eight floats (permuted-k order) to bf16 hi/lo fragments.
template <bool kSplit>
__device__ __forceinline__ void split8(const float (&v)[8], bf16x8& hi, bf16x8& lo) {
    uint2 h0, l0, h1, l1;
    split4<kSplit>(v[0], v[1], v[2], v[3], h0, l0);
    split4<kSplit>(v[4], v[5], v[6], v[7], h1, l1);
    hi = __builtin_bit_cast(bf16x8, make_uint4(h0.x, h0.y, h1.x, h1.y));
    if constexpr (kSplit) lo = __builtin_bit_cast(bf16x8, make_uint4(l0.x, l0.y, l1.x, l1.y));
}

// One sub-chunk of a [tokens][W] tensor in the lane layout above.
template <typename TIn, int W, int P>
struct DRows {
    static constexpr int NG = W / 64;
    f32x4 x[NG][2][4];  // [column group][h][r]: columns 64 gg + 4 lr .. + 3 of row 16 h + 4 g + r

    template <int PP = P>
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, int r0, int g, int lr) {
#pragma unroll
        for (int gg = 0; gg < NG; ++gg)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    x[gg][h][r] = load_q4<TIn, PP>(
                        rs, ((r0 + 16 * h + 4 * g + r) * W + 64 * gg + 4 * lr) * int(sizeof(TIn)));
    }
    // The 8 rows of column 64 gg + 4 lr + c, in permuted-k order.
    __device__ __forceinline__ void col(int gg, int c, float (&v)[8]) const {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int r = 0; r < 4; ++r) v[4 * h + r] = x[gg][h][r][c];
    }
};

// Floats of LDS quad_sums takes.
constexpr int kQuadLdsFloats = 4 * (64 * 64 + 64);

// The sums over rows 0 .. rows - 1 of k and v (rows of 64) into the record rp
// (B [64][64], then A [64]), plus `init`'s when it is given.  The sub-chunk pairs
// (64 tokens) are dealt to the four waves round-robin from the last pair down:
// at each step the workgroup reads the 256 tokens below the previous step's, so
// it walks from the end to the start, the first `kept` rows with
// cache-allocating loads, the rest past the caches.  The four partial sums meet
// in LDS (`part`) and are added in wave order, so the record is the same bit for
// bit on every run.
template <typename TIn>
__device__ __forceinline__ void quad_sums(const TIn* __restrict__ k, const TIn* __restrict__ v, int rows, int kept,
                                          float* __restrict__ part, float* rp, const float* init) {
    constexpr int S = 64, D = 64, C = kDirC, LP = kPolicyDefault, es = int(sizeof(TIn));
    constexpr bool kSplit = std::is_same<TIn, float>::value;
    constexpr int kPart = S * D + S;  // floats of one wave's partial record in LDS
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l = threadIdx.x & 63, g = l >> 4, lr = l & 15;
    const __amdgpu_buffer_rsrc_t kr = make_rsrc(k, int64_t(rows) * S * es);
    const __amdgpu_buffer_rsrc_t vr = make_rsrc(v, int64_t(rows) * D * es);

    f32x4 acc[4][4];  // [sb][cb]: B[4 (4 g + r) + sb][4 lr + cb] at element r
#pragma unroll
    for (int sb = 0; sb < 4; ++sb)
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) acc[sb][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
    float asum[4] = {0.f, 0.f, 0.f, 0.f};

    // Consume the sub-chunk held in (kx, vx), then refill them from row
    // `next` (past the tile the loads read zeros, which are never consumed).
    auto chunk = [&](auto pol, DRows<TIn, S, LP>& kx, DRows<TIn, D, LP>& vx, int next) {
        constexpr int PP = decltype(pol)::value;
        bf16x8 vh[4], vl[4];
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            float e[8];
            vx.col(0, cb, e);
            split8<kSplit>(e, vh[cb], vl[cb]);
        }
        vx.template load<PP>(vr, next, g, lr);
#pragma unroll
        for (int sb = 0; sb < 4; ++sb) {
            float e[8];
            kx.col(0, sb, e);
            asum[sb] += (((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7])));
            bf16x8 kh, kl;
            split8<kSplit>(e, kh, kl);
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) acc[sb][cb] = mfma3<kSplit>(kh, kl, vh[cb], vl[cb], acc[sb][cb]);
        }
        kx.template load<PP>(kr, next, g, lr);
    };

    // Pair p covers rows 2 C p .. 2 C p + 2 C - 1 (the second half may lie
    // past the tile and read zeros).  Wave w takes pairs P-1-w, P-5-w, ...
    const int pairs = (rows + 2 * C - 1) / (2 * C);
    int p = pairs - 1 - w;
    const int first = p >= 0 ? 2 * C * p : rows;
    // Pairs from `pcut` up are read `nt`, the rest with the allocating policy.
    const int pcut = min(pairs, (kept + 2 * C - 1) / (2 * C));
    const int cut = 2 * C * pcut;
    DRows<TIn, S, LP> k0, k1;
    DRows<TIn, D, LP> v0, v1;
    if (first < cut) {
        k0.load(kr, first, g, lr);
        v0.load(vr, first, g, lr);
        k1.load(kr, first + C, g, lr);
        v1.load(vr, first + C, g, lr);
    } else {
        k0.template load<kPolicyStream>(kr, first, g, lr);
        v0.template load<kPolicyStream>(vr, first, g, lr);
        k1.template load<kPolicyStream>(kr, first + C, g, lr);
        v1.template load<kPolicyStream>(vr, first + C, g, lr);
    }
    using Alloc = std::integral_constant<int, LP>;
    using Stream = std::integral_constant<int, kPolicyStream>;
    for (; p - 4 >= pcut; p -= 4) {
        const int nx = 2 * C * (p - 4);
        chunk(Stream{}, k0, v0, nx);
        chunk(Stream{}, k1, v1, nx + C);
    }
    for (; p >= 0; p -= 4) {
        const int nx = 2 * C * (p - 4);  // below row 0 (last round): outside the range, zeros
        chunk(Alloc{}, k0, v0, nx);
        chunk(Alloc{}, k1, v1, nx + C);
    }

    // Partial record of wave w: B row 16 g + 4 r + sb, columns 4 lr .. + 3,
    // then A (the token groups g added in a fixed order).
    float* mine = part + w * kPart;
#pragma unroll
    for (int sb = 0; sb < 4; ++sb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            *reinterpret_cast<f32x4*>(mine + (16 * g + 4 * r + sb) * D + 4 * lr) =
                f32x4{acc[sb][0][r], acc[sb][1][r], acc[sb][2][r], acc[sb][3][r]};
    {
        f32x4 a;
#pragma unroll
        for (int sb = 0; sb < 4; ++sb) {
            float x = asum[sb];
            x = x + __shfl_xor(x, 16);
            x = x + __shfl_xor(x, 32);
            a[sb] = x;
        }
        if (g == 0) *reinterpret_cast<f32x4*>(mine + S * D + 4 * lr) = a;
    }
    __syncthreads();
    // record = ((part0 + part1) + part2) + part3, 16-byte pieces.
    for (int i = threadIdx.x; i < kPart / 4; i += kThreads) {
        f32x4 x = *reinterpret_cast<const f32x4*>(part + 4 * i);
#pragma unroll
        for (int j = 1; j < 4; ++j) x += *reinterpret_cast<const f32x4*>(part + j * kPart + 4 * i);
        if (init) x += *reinterpret_cast<const f32x4*>(init + 4 * i);
        *reinterpret_cast<f32x4*>(rp + 4 * i) = x;
    }
}

}  // namespace mfma
}  // namespace race
