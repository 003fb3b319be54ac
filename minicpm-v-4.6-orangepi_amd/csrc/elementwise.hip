// elementwise.hip -- silu*mul and the greedy argmax for gfx950.
#include "common.h"
#include "row_norm.h"

namespace mcv {
namespace {

// out = silu_mul_f16(g, u) elementwise (common.h), 8 elements a thread and trip in
// 16-byte accesses; VEC = false (an operand not 16-byte aligned) and the last n
// % 8 elements one at a time.  MI355X, 3000 x 3584: 16.1 us element by element,
// 13.6 in chunks; ~35 VALU per element (the correctly rounded division and
// expf) keep it from the 13 us of its 64 MB.
template <bool VEC>
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* __restrict__ g, const uint16_t* __restrict__ u,
                                                       uint16_t* __restrict__ out, int64_t n) {
    const int64_t tid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int64_t threads = static_cast<int64_t>(gridDim.x) * blockDim.x;
    const int64_t chunks = VEC ? n / 8 : 0;
    for (int64_t i = tid; i < chunks; i += threads) {
        const uint4 a = reinterpret_cast<const uint4*>(g)[i], b = reinterpret_cast<const uint4*>(u)[i];
        auto two = [](uint32_t p, uint32_t q) {
            return uint32_t(silu_mul_f16(static_cast<uint16_t>(p), static_cast<uint16_t>(q))) |
                   (uint32_t(silu_mul_f16(static_cast<uint16_t>(p >> 16), static_cast<uint16_t>(q >> 16))) << 16);
        };
        reinterpret_cast<uint4*>(out)[i] = make_uint4(two(a.x, b.x), two(a.y, b.y), two(a.z, b.z), two(a.w, b.w));
    }
    for (int64_t i = chunks * 8 + tid; i < n; i += threads) out[i] = silu_mul_f16(g[i], u[i]);
}

// Greedy argmax of fp16 rows, first maximum, with argmax_key16's order: NaN and
// -inf never win, subnormals and -0 count as +0.
//
// One workgroup of 1024 threads per row, read in 16-byte chunks of eight values, U
// = 4 in flight per lane (eight: rows of 31012 4.9 us against 4.1, longer ones the
// same).  U = 1: rows that leave a lane one chunk, which stays in registers for the
// lookup below (one row of 8192: per value 3.7 us, U = 4 4.1, U = 1 3.4).
// What bounds it is the VALU work per value, so a chunk is compared as a whole:
// packed 16-bit integer steps map a value to a signed order (rank16) in which
// every value that cannot win sits below kRankNone, a packed maximum folds the
// eight, and one comparison keeps the lane's best rank and the first chunk that
// holds it; the index inside the chunk is looked up once, at the end (a lane
// visits its chunks in increasing order, so only a strictly larger rank
// replaces).  At most seven values up to the first 16-byte boundary and after
// the last chunk go one by one.  The lanes' 64-bit keys (value, then lowest
// index) meet through wave shuffles and LDS.  MI355X, rows of 248094: building
// argmax_key16 per value took 31 us; chunks 10.3, 6
// rows 10.5, 32 rows 11.0, 6 rows of 31012 6.4 -> 4.1.  Cutting a row over
// workgroups whose keys meet by atomic maximum takes two more launches: 7.1 us
// for one row, 8.7 for 6, 12.1 for 32, and ~6 us more of the host.

// The order-preserving rank of two packed fp16 values: sign-magnitude to two's
// complement, then + 0x3ff, which wraps positive NaN (above +inf) around to the
// bottom, next to negative NaN and -inf.
typedef short short2_t __attribute__((ext_vector_type(2)));
constexpr int kRankShift = 0x3ff;
constexpr int kRankNone = static_cast<int16_t>(0x87fe);      // -inf; NaN is below
__device__ __forceinline__ short2_t rank16(uint32_t w) {
    const short2_t v = __builtin_bit_cast(short2_t, w);
    const uint32_t neg = __builtin_bit_cast(uint32_t, static_cast<short2_t>(v >> 15)) & 0x7fff7fffu;
    return __builtin_bit_cast(short2_t, w ^ neg) + short2_t{kRankShift, kRankShift};
}
// Subnormals and zeros of either sign (two's complement -1024 .. 1023) are one value.
__device__ __forceinline__ int rank_flush(int r) {
    const int v = r - kRankShift;
    return static_cast<uint32_t>(v + 1024) < 2048u ? kRankShift : r;
}
__device__ __forceinline__ int rank_max8(const uint4& q) {
    const short2_t m = __builtin_elementwise_max(__builtin_elementwise_max(rank16(q.x), rank16(q.y)),
                                                 __builtin_elementwise_max(rank16(q.z), rank16(q.w)));
    return rank_flush(m[0] > m[1] ? m[0] : m[1]);
}

constexpr int kArgThreads = 1024;
template <int U>
__global__ __launch_bounds__(kArgThreads) void argmax_kernel(const uint16_t* __restrict__ x, int64_t N,
                                                             int64_t* __restrict__ idx) {
    const uint16_t* xr = x + static_cast<size_t>(blockIdx.x) * N;
    const int tid = threadIdx.x;
    const int64_t head64 = static_cast<int64_t>((16u - (reinterpret_cast<uintptr_t>(xr) & 15u)) & 15u) / 2;
    const int64_t head = head64 < N ? head64 : N;
    const uint4* __restrict__ v = reinterpret_cast<const uint4*>(xr + head);
    const int64_t nv = (N - head) / 8;
    int br = kRankNone;                          // best rank so far and its first chunk
    int64_t bc = 0;
    uint4 bq = make_uint4(0, 0, 0, 0);           // U = 1: the lane's only chunk
    for (int64_t j0 = tid; j0 < nv; j0 += int64_t(kArgThreads) * U) {
        uint4 q[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {            // past the end: -inf, never a candidate
            const int64_t j = j0 + int64_t(u) * kArgThreads;
            q[u] = j < nv ? v[j] : make_uint4(0xfc00fc00u, 0xfc00fc00u, 0xfc00fc00u, 0xfc00fc00u);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int r = rank_max8(q[u]);
            const bool take = r > br;
            br = take ? r : br;
            bc = take ? j0 + int64_t(u) * kArgThreads : bc;
        }
        if constexpr (U == 1) {
            bq = q[0];
            break;
        }
    }
    unsigned long long best = 0ull;
    auto visit = [&](int64_t i) {
        const unsigned long long k = argmax_key64(argmax_key16(xr[i]), static_cast<uint32_t>(i));
        best = k > best ? k : best;
    };
    if (br > kRankNone) {
        if constexpr (U != 1) bq = v[bc];
        const uint32_t w[4] = {bq.x, bq.y, bq.z, bq.w};
        int first = 7;
#pragma unroll
        for (int e = 7; e >= 0; --e) first = rank_flush(rank16(w[e / 2])[e & 1]) == br ? e : first;
        visit(head + 8 * bc + first);
    }
    if (tid < head) visit(tid);
    if (head + 8 * nv + tid < N) visit(head + 8 * nv + tid);
    best = wave_max_u64(best);
    __shared__ unsigned long long wbest[kArgThreads / 64];
    if ((tid & 63) == 0) wbest[tid >> 6] = best;
    __syncthreads();
    if (tid < 64) {
        best = wave_max_u64(tid < kArgThreads / 64 ? wbest[tid] : 0ull);
        if (tid == 0) idx[blockIdx.x] = argmax_index(best);
    }
}

}  // namespace
}  // namespace mcv

using namespace mcv;

extern "C" {

int mcv_silu_mul(const void* gate, const void* up, void* out, int64_t n, mcv_stream_t stream) {
    if (!gate || !up || !out) return fail(MCV_ERR_INVALID_ARG, "silu_mul: null pointer");
    if (n <= 0) return fail(MCV_ERR_SHAPE, "silu_mul: n must be positive (n=%lld)", (long long)n);
    int rc = require_device();
    if (rc != MCV_OK) return rc;
    const bool vec = (reinterpret_cast<uintptr_t>(gate) | reinterpret_cast<uintptr_t>(up) |
                      reinterpret_cast<uintptr_t>(out)) % 16 == 0;
    // (512 x 3584 3.9 us either way, 77 x 3584 1.9 / 2.1: fewer waves hide less)
    const bool chunked = vec && n >= (int64_t(1) << 21);
    const int64_t want = ceil_div(chunked ? ceil_div(n, 8) : n, 256);
    const int64_t blocks = want < 4096 ? want : 4096;
    hipLaunchKernelGGL(chunked ? silu_mul_kernel<true> : silu_mul_kernel<false>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, static_cast<hipStream_t>(stream),
                       static_cast<const uint16_t*>(gate), static_cast<const uint16_t*>(up), static_cast<uint16_t*>(out), n);
    return check_launch("silu_mul_kernel");
}

int mcv_argmax_f16(const void* x, int64_t M, int64_t N, int64_t* idx, mcv_stream_t stream) {
    if (!x || !idx) return fail(MCV_ERR_INVALID_ARG, "argmax: null pointer");
    if (M <= 0 || N <= 0 || M > 0x7fffffff || N > 0xffffffffll)
        return fail(MCV_ERR_SHAPE, "argmax: bad shape M=%lld N=%lld", (long long)M, (long long)N);
    int rc = require_device();
    if (rc != MCV_OK) return rc;
    hipLaunchKernelGGL((N <= 8 * kArgThreads ? argmax_kernel<1> : argmax_kernel<4>), dim3(static_cast<unsigned>(M)),
                       dim3(kArgThreads), 0, static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(x), N, idx);
    return check_launch("argmax_kernel");
}

}  // extern "C"

extern "C" int mcv_rms_norm(const void* x, const void* gamma, int64_t M, int64_t H, double eps, void* out,
                            mcv_stream_t stream) {
    if (!x || !gamma || !out) return fail(MCV_ERR_INVALID_ARG, "rms_norm: null pointer");
    if (M <= 0 || H <= 0 || M > 0x7fffffff || H > 0x7fffffff || !(eps >= 0.0))
        return fail(MCV_ERR_SHAPE, "rms_norm: bad shape M=%lld H=%lld or eps", (long long)M, (long long)H);
    int rc = require_device();
    if (rc != MCV_OK) return rc;
    launch_rms<false>(static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(gamma), M, H, static_cast<float>(eps),
                      static_cast<uint16_t*>(out), nullptr, nullptr, nullptr, static_cast<hipStream_t>(stream));
    return check_launch("rms_row_kernel");
}
