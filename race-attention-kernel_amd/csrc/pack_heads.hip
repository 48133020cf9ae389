// pack_heads.hip -- token rows of several heads, [B][T][H][d] as a projection
// leaves them, to one stream of rows per head, [B * H][T][d], as the op's
// kernels take them (the permutes of src/race_baseline.py:35-40), for up to
// three tensors in one launch.
//
// A copy, bound by memory.  A workgroup writes one contiguous run of rows of
// one stream and reads them H rows apart; the H workgroups that read one run
// of the source are next to each other in launch order.  (Reading in source
// order, a workgroup's writes are H streams apart, a power of two in the usual
// shapes, and meet on the same memory channels.)  The source is read past the
// caches (nontemporal: it is not read again) and the destination stays in them
// for the kernels that follow: three tensors of 131072 fp32 rows of 64 (201 MB
// moved) 47 -> 33 us with the nontemporal reads, 37 with nontemporal writes
// too; torch's permuted copies took 50.
#include <algorithm>

#include "race_internal.h"

namespace race {
namespace {

constexpr int kPackChunks = 1024;  // 16-byte chunks per workgroup: 4 per thread
constexpr int kPackUnroll = kPackChunks / kThreads;
// Workgroups of a batch in one launch: one of 2^32 threads or more wraps around
// without an error.
constexpr int64_t kPackLaunch = int64_t(1) << 23;

typedef uint32_t Chunk __attribute__((ext_vector_type(4)));

struct PackArgs {
    const Chunk* src[3];
    Chunk* dst[3];
};

// vec: 16-byte chunks per row (1 << shift where that is a power of two, else
// shift < 0); tokens: rows per workgroup, at most kPackChunks chunks; first: the
// launch's first workgroup of a batch.
__global__ __launch_bounds__(kThreads) void pack_heads_kernel(PackArgs a, int64_t T, int H, int vec, int shift,
                                                              int tokens, unsigned first) {
    const Chunk* src = a.src[blockIdx.z];
    Chunk* dst = a.dst[blockIdx.z];
    const int64_t b = blockIdx.y;
    const unsigned wg = first + blockIdx.x;
    const int h = int(wg % unsigned(H));
    const int64_t t0 = int64_t(wg / unsigned(H)) * tokens;
    const int chunks = int(min<int64_t>(tokens, T - t0)) * vec;
    const int64_t from = ((b * T + t0) * H + h) * vec, to = ((b * H + h) * T + t0) * vec;
    Chunk v[kPackUnroll];
#pragma unroll
    for (int m = 0; m < kPackUnroll; ++m) {
        const int c = min(int(threadIdx.x) + m * kThreads, chunks - 1);
        const int t = shift >= 0 ? c >> shift : c / vec;
        v[m] = __builtin_nontemporal_load(src + from + int64_t(t) * H * vec + (c - t * vec));
    }
#pragma unroll
    for (int m = 0; m < kPackUnroll; ++m) {
        const int c = int(threadIdx.x) + m * kThreads;
        if (c < chunks) dst[to + c] = v[m];
    }
}

}  // namespace

hipError_t launch_pack_heads(const void* const* src, void* const* dst, int count, int64_t batch, int64_t T, int H,
                             int row_bytes, hipStream_t stream) {
    PackArgs a = {};
    for (int i = 0; i < count; ++i) {
        a.src[i] = static_cast<const Chunk*>(src[i]);
        a.dst[i] = static_cast<Chunk*>(dst[i]);
    }
    const int vec = row_bytes / 16;
    const int shift = (vec & (vec - 1)) == 0 ? __builtin_ctz(vec) : -1;
    const int tokens = kPackChunks / vec;
    const int64_t wgs = (T + tokens - 1) / tokens * H;
    for (int64_t w = 0; w < wgs; w += kPackLaunch) {
        const dim3 grid(unsigned(std::min(wgs - w, kPackLaunch)), unsigned(batch), unsigned(count));
        pack_heads_kernel<<<grid, kThreads, 0, stream>>>(a, T, H, vec, shift, tokens, unsigned(w));
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) return err;
    }
    return hipSuccess;
}

}  // namespace race
