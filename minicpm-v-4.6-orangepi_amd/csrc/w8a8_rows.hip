// w8a8_rows.hip -- W8A8 matmul for a few activation rows on int8 MFMA over the
// tiled weight layout (MCV_W8_TILED), gfx950: batched decode, short prompts.
//
// acc[m][n] = sum_k xq[m][k] w[k][n] in int32 (exact), out int32 or the fused
// fp16 RNE((float(acc) * ws[n]) * xs[m]).  The integer sums are exact in any
// order, so every result is bit-identical to the GEMV's and the GEMM's.
//
// v_mfma_i32_16x16x64_i8 takes 16 bytes of k per lane from each operand: row or
// column lane % 16, k 16 j .. + 15 with j = lane / 16.  A 1 KiB line of the layout
// holds 32 columns x 32 k as two k-halves of 32 x 16 bytes, so lane (c, j) of a
// 16-column block reads 16 bytes of line kb + j / 2, half j % 2: four 256-byte
// pieces per load.  x rows pass through LDS: loaded 128 contiguous bytes a row
// and read back in operand order (chunk q of row m at q ^ (m / 2), so that
// neither side conflicts).
//
// w8a8_rows_kernel: the waves of a workgroup split K in groups of 128, each over
// 16 CB columns and 16 MB rows; the partial sums meet in LDS.  The GEMM it
// replaces ran 64-row tiles whose grid covers a few CUs and whose waves walk all
// of K.  w8a8_rows_wide_kernel: the vocabulary; x staged once per workgroup, each
// wave walks 32 columns over all of K on its own.
#include <cstdio>
#include <string>

#include "common.h"

namespace mcv {
namespace {

constexpr int kLine8 = 1024;                             // one 32-column x 32-k line

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_8(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), 0x00020000);
}

// Byte of 16-byte chunk q of row m of a 16-row block in a staged group (2 KiB).
__device__ __forceinline__ int x8_at(int m, int q) { return m * 128 + ((q ^ (m >> 1)) << 4); }

struct Rows8Args {
    const int8_t* xq;
    const int8_t* w;
    void* out;
    const void* xs;
    const void* ws;
    int xs16, ws16;
    int M, K, N, KB, nslab;
};

__device__ __forceinline__ float scale_at(const void* p, int is16, int i) {
    return is16 ? h2f(static_cast<const uint16_t*>(p)[i]) : static_cast<const float*>(p)[i];
}

template <bool F16>
__device__ __forceinline__ void store_out8(const Rows8Args& a, int m, int n, int acc, float xs, float ws) {
    const size_t o = static_cast<size_t>(m) * a.N + n;
    if constexpr (F16) static_cast<uint16_t*>(a.out)[o] = f2h(__fmul_rn(__fmul_rn(static_cast<float>(acc), ws), xs));
    else static_cast<int32_t*>(a.out)[o] = acc;
}

// LDS bytes of one wave: a staged group per 16 rows, or its partial sums.
constexpr int rows8_wave_lds(int mb, int cb) { return mb * 1024 * (cb > 2 ? cb : 2); }

// grid (column units of 16 CB, blocks of 16 MB rows).
template <int MB, int CB, int TR, bool F16>
__global__ __launch_bounds__(1024) void w8a8_rows_kernel(Rows8Args a) {
    constexpr int E = MB * CB * 4 * 64;                  // partial sums of one wave
    constexpr int R = rows8_wave_lds(MB, CB);
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int KS = static_cast<int>(blockDim.x >> 6);
    const int j = lane >> 4;
    const int G = a.KB / 4;                              // groups of 128 k (the weight is padded to whole ones)
    const int c0 = static_cast<int>(blockIdx.x) * 16 * CB, m0 = static_cast<int>(blockIdx.y) * 16 * MB;
    const int rows = a.M - m0;
    const __amdgpu_buffer_rsrc_t xr = rsrc_8(a.xq + static_cast<size_t>(m0) * a.K,
                                             static_cast<uint32_t>(rows < 16 * MB ? rows : 16 * MB) * a.K);
    const __amdgpu_buffer_rsrc_t wr = rsrc_8(a.w, static_cast<uint32_t>(a.nslab) * a.KB * 2 * kLine8);
    // x loads: rows 8 t + lane / 8 of a 16-row block, 128 bytes a row; k past K
    // meets zero weights, rows past M are not used.  The whole offset is the
    // vector one: where K is not whole groups of 128 the last row's last chunks
    // lie past x, and the scalar offset is not part of the range check.
    const uint32_t xoff = static_cast<uint32_t>(lane >> 3) * a.K + 16u * (lane & 7);
    uint8_t* const mine = lds + wave * R;
    uint32_t woff[CB];
#pragma unroll
    for (int c = 0; c < CB; ++c) {
        const int n = c0 + 16 * c + (lane & 15);
        woff[c] = ((static_cast<uint32_t>(n / kSlab) * a.KB + (j >> 1)) * 2 + ((n >> 5) & 1)) * kLine8 +
                  ((j & 1) * 32 + (n & 31)) * 16u;
    }
    int4_t acc[MB][CB];
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
        for (int c = 0; c < CB; ++c) acc[b][c] = int4_t{0, 0, 0, 0};

    // TR groups per trip, their loads all out before the first wait; a group
    // past the last reads zeros (out of range)
    for (int g0 = wave; g0 < G; g0 += KS * TR) {
        int4_t xv[TR][MB][2], wv[TR][CB][2];
#pragma unroll
        for (int u = 0; u < TR; ++u) {
            const int g = g0 + u * KS, gc = g < G ? g : 0;
            const uint32_t dead = static_cast<uint32_t>(g >= G) << 31;
#pragma unroll
            for (int c = 0; c < CB; ++c)
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    wv[u][c][i] = __builtin_bit_cast(
                        int4_t, __builtin_amdgcn_raw_buffer_load_b128(wr, woff[c] | dead, (gc * 4 + 2 * i) * 2 * kLine8, 2));
#pragma unroll
            for (int b = 0; b < MB; ++b)
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    xv[u][b][t] = __builtin_bit_cast(
                        int4_t, __builtin_amdgcn_raw_buffer_load_b128(xr, (xoff + (16 * b + 8 * t) * a.K + gc * 128) | dead, 0, 0));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < TR; ++u) {
#pragma unroll
            for (int b = 0; b < MB; ++b)
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    *reinterpret_cast<int4_t*>(mine + b * 2048 + x8_at(8 * t + (lane >> 3), lane & 7)) = xv[u][b][t];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int b = 0; b < MB; ++b) {
                    const int4_t xo = *reinterpret_cast<const int4_t*>(mine + b * 2048 + x8_at(lane & 15, 4 * i + j));
#pragma unroll
                    for (int c = 0; c < CB; ++c)
                        acc[b][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xo, wv[u][c][i], acc[b][c], 0, 0, 0);
                }
        }
    }

    int* const part = reinterpret_cast<int*>(mine);
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
        for (int c = 0; c < CB; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[((b * CB + c) * 4 + r) * 64 + lane] = acc[b][c][r];
    __syncthreads();
    // register r of lane l in block (b, c): row 16 b + 4 (l / 16) + r, column 16 c + l % 16
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
        const int l = e & 63, r = (e >> 6) & 3, c = (e >> 8) % CB, b = (e >> 8) / CB;
        const int m = m0 + 16 * b + 4 * (l >> 4) + r, n = c0 + 16 * c + (l & 15);
        if (m >= a.M || n >= a.N) continue;
        const float xs = F16 ? scale_at(a.xs, a.xs16, m) : 0.f, ws = F16 ? scale_at(a.ws, a.ws16, n) : 0.f;
        int v = 0;
        for (int w = 0; w < KS; ++w) v += reinterpret_cast<const int*>(lds)[w * (R / 4) + e];
        store_out8<F16>(a, m, n, v, xs, ws);
    }
}

// Units of 32 columns (one half of a slab), one per wave and trip.
template <int MB, int D, bool F16>
__global__ __launch_bounds__(512) void w8a8_rows_wide_kernel(Rows8Args a) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];   // [group][mb] x8_at()
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int NW = static_cast<int>(blockDim.x >> 6);
    const int j = lane >> 4;
    const int G = a.KB / 4, units = a.nslab * 2;
    const __amdgpu_buffer_rsrc_t xr = rsrc_8(a.xq, static_cast<uint32_t>(a.M) * a.K);
    const __amdgpu_buffer_rsrc_t wr = rsrc_8(a.w, static_cast<uint32_t>(a.nslab) * a.KB * 2 * kLine8);
    uint32_t woff[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) woff[c] = (j >> 1) * 2 * kLine8 + ((j & 1) * 32 + 16 * c + (lane & 15)) * 16u;
    int4_t w[D][2][2];
    auto load_w = [&](int slot, int unit, int g) {
        const uint32_t dead = static_cast<uint32_t>(g >= G) << 31;
        const int gc = g < G ? g : 0;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int c = 0; c < 2; ++c)
                w[slot][i][c] = __builtin_bit_cast(
                    int4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                wr, woff[c] | dead, (((unit >> 1) * a.KB + gc * 4 + 2 * i) * 2 + (unit & 1)) * kLine8, 2));
    };
    const int unit = static_cast<int>(blockIdx.x) * NW + wave;
    if (unit < units) {
#pragma unroll
        for (int d = 0; d < D; ++d) load_w(d, unit, d);
    }
    for (int t = wave; t < G * MB * 2; t += NW) {         // eight rows of one group
        const int g = t / (2 * MB), m = 8 * (t % (2 * MB)) + (lane >> 3);
        const int4_t v = __builtin_bit_cast(
            int4_t, __builtin_amdgcn_raw_buffer_load_b128(xr, static_cast<uint32_t>(m) * a.K + 16u * (lane & 7) + g * 128, 0, 0));
        *reinterpret_cast<int4_t*>(lds + (g * MB + (m >> 4)) * 2048 + x8_at(m & 15, lane & 7)) = v;
    }
    __syncthreads();
    if (unit >= units) return;
    const int n0 = unit * 32 + (lane & 15);
    float ws[2] = {0.f, 0.f};
    if constexpr (F16)
#pragma unroll
        for (int c = 0; c < 2; ++c) ws[c] = n0 + 16 * c < a.N ? scale_at(a.ws, a.ws16, n0 + 16 * c) : 0.f;
    int4_t acc[MB][2];
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
        for (int c = 0; c < 2; ++c) acc[b][c] = int4_t{0, 0, 0, 0};
    for (int g0 = 0; g0 < G; g0 += D) {
#pragma unroll
        for (int u = 0; u < D; ++u) {
            const int g = g0 + u, gx = g < G ? g : G - 1;                // past G: zero weights
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int b = 0; b < MB; ++b) {
                    const int4_t xo = *reinterpret_cast<const int4_t*>(lds + (gx * MB + b) * 2048 + x8_at(lane & 15, 4 * i + j));
#pragma unroll
                    for (int c = 0; c < 2; ++c)
                        acc[b][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xo, w[u][i][c], acc[b][c], 0, 0, 0);
                }
            load_w(u, unit, g + D);
        }
    }
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = 16 * b + 4 * j + r;
            if (m >= a.M) continue;
            const float xs = F16 ? scale_at(a.xs, a.xs16, m) : 0.f;
#pragma unroll
            for (int c = 0; c < 2; ++c)
                if (n0 + 16 * c < a.N) store_out8<F16>(a, m, n0 + 16 * c, acc[b][c][r], xs, ws[c]);
        }
}

struct Rows8Cfg {
    int mb, cb, ks, wide;
};

int rows8_ks(int64_t G) { return static_cast<int>(ceil_div(G, ceil_div(G, 16))); }

// Whether and how these kernels run M x K x N.  MI355X, rotated weights, us, the
// GEMV (M <= 4) or GEMM they replace / here:
//   one row on a long K (the GEMV's two trips) up to 64 slabs: K=3584 N=1024 M=1 5.0 /
//   3.9, N=4608 5.1 / 5.9; two rows, M=2 6.5 / 3.9; M=2 K=1024 N=3584 3.2 / 3.0 but N=6144 3.4 / 3.5; M=4 N=248094
//   51.7 / 39.8;
//   up to 32 rows everywhere: K=1024 N=3584 M=5 5.1 / 3.0, M=32 5.2 / 3.5; K=3584
//   N=1024 M=32 11.7 / 4.5; N=31012 M=32 11.3 / 8.9;
//   more rows while the grid stays near a workgroup per CU: K=3584 N=1024 M=64
//   11.8 / 4.5, M=256 10.5 / 6.6; K=1024 N=3584 M=64 5.3 / 4.0, but M=256 4.8 / 6.6,
//   N=1024 M=256 3.8 / 3.9.
// Blocks grow from 16 rows x 16 columns until the grid fits a workgroup per CU
// (K=3584 N=1024 M=64: 256 of 16 x 16 4.5, 64 of 32 x 32 6.7).  The waves that split K
// also write the output, so the larger the block the more groups of 128 it takes
// to pay, GEMV or GEMM / here, mean of weights cold and in cache: one wave K=128
// N=3584 M=64 3.4 / 6.0 (32 x 32), N=1024 M=96 3.3 / 4.2 (16 x 32); two K=256 N=4608
// M=8 3.4 / 3.5, N=3072 M=64 3.5 / 4.8; six K=768 N=2048 M=96 4.1 / 4.5; eight K=1024
// N=3072 M=48 4.6 / 4.2.  A grid of several workgroups per CU hides more of it, but
// past K = 2048 the GEMM's wider tiles read x less often (K=512 N=31012 M=32 8.4 /
// 7.4; K=3584 23.8 / 26.7).
// The wide kernel: N=248094 M=6 50.2 / 40.6, M=16 55.8 / 44.1, M=32 63.3 / 50.6,
// M=64 85 / 61; at N=62024 it is level with the split kernel (M=32 15.7 both) and
// behind the GEMM at M=64 (18.6 / 19.7), as it is past 32 rows from K = 1536 on (N=124000
// M=48 40.5 / 45.8).
bool pick_rows8(int64_t M, int64_t K, int64_t N, Rows8Cfg& c) {
    const int64_t nslab = ceil_div(N, kSlab), G = ceil_div(K, 128);
    if (M < 1 || M > 512 || nslab * G * 8192 >= (int64_t(1) << 31) || M * K >= (int64_t(1) << 31)) return false;
    if (M == 1 && !(nslab <= 64 && K > 2048)) return false;
    if (M == 2 && nslab >= 64) return false;
    const int mb = M <= 16 ? 1 : (M <= 32 ? 2 : 4);
    c.ks = rows8_ks(G);
    c.wide = M <= 64 && nslab >= (mb == 1 ? 2000 : (mb == 2 ? 900 : 1200)) && G * mb * 2048 <= 160 * 1024 &&
             (mb < 4 || G < 12);
    c.mb = mb;
    c.cb = 2;
    if (c.wide) return true;
    if ((M > 32 && nslab * 2 * ceil_div(M, 32) > 256) || (M > 200 && K <= 1024)) return false;
    auto grid = [&](int rows, int cols) { return ceil_div(M, 16 * rows) * (nslab * 4 / cols); };
    c.mb = c.cb = 1;
    if (grid(1, 1) > 256) c.cb = 2;
    if (grid(1, 2) > 256 && M > 16) c.mb = 2;
    const int64_t wgs = grid(c.mb, c.cb);
    if (c.mb == 2) return wgs <= 512 ? G >= 7 : G >= 4 && G <= 16;
    if (c.cb == 2) return G > 2 || wgs > (G == 2 ? 512 : 900);
    return G > 1 || M > 4;
}

template <int MB, int CB, bool F16>
void launch_split8(const Rows8Args& a, int ks, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>(a.nslab * 4 / CB), static_cast<unsigned>(ceil_div(a.M, 16 * MB)));
    const size_t lds = size_t(ks) * rows8_wave_lds(MB, CB);
    if (a.KB / 4 > ks)
        hipLaunchKernelGGL((w8a8_rows_kernel<MB, CB, 2, F16>), grid, dim3(64 * ks), lds, stream, a);
    else
        hipLaunchKernelGGL((w8a8_rows_kernel<MB, CB, 1, F16>), grid, dim3(64 * ks), lds, stream, a);
}

template <int MB, bool F16>
void launch_wide8(const Rows8Args& a, hipStream_t stream) {
    constexpr int kWaves = 8, kDepth = 4;
    hipLaunchKernelGGL((w8a8_rows_wide_kernel<MB, kDepth, F16>), dim3(static_cast<unsigned>(ceil_div(a.nslab * 2, kWaves))),
                       dim3(64 * kWaves), size_t(a.KB / 4) * MB * 2048, stream, a);
}

template <bool F16>
int launch_cfg8(const Rows8Args& a, const Rows8Cfg& c, hipStream_t stream) {
    if (c.wide && c.mb == 1) launch_wide8<1, F16>(a, stream);
    else if (c.wide && c.mb == 2) launch_wide8<2, F16>(a, stream);
    else if (c.wide) launch_wide8<4, F16>(a, stream);
    else if (c.mb == 2) launch_split8<2, 2, F16>(a, c.ks, stream);
    else if (c.cb == 2) launch_split8<1, 2, F16>(a, c.ks, stream);
    else launch_split8<1, 1, F16>(a, c.ks, stream);
    return check_launch("w8a8_rows_kernel");
}

}  // namespace

bool w8a8_uses_rows(int64_t M, int64_t K, int64_t N) {
    Rows8Cfg c;
    return pick_rows8(M, K, N, c);
}

// The kernel these launches take, as text (report labels).
std::string w8a8_rows_name(int64_t M, int64_t K, int64_t N, bool f16) {
    Rows8Cfg c{};
    pick_rows8(M, K, N, c);
    char buf[128];
    if (c.wide) std::snprintf(buf, sizeof(buf), "w8a8_rows_wide_kernel<%d, 4, %s>", c.mb, f16 ? "true" : "false");
    else
        std::snprintf(buf, sizeof(buf), "w8a8_rows_kernel<%d, %d, %d, %s> (%d waves splitting K)", c.mb, c.cb,
                      ceil_div(K, 128) > c.ks ? 2 : 1, f16 ? "true" : "false", c.ks);
    return buf;
}

// As launch_w8a8_tiled (w8a8_tiled.hip), for the calls w8a8_uses_rows names.
int launch_w8a8_rows(const int8_t* xq, int64_t M, int64_t K, int64_t N, const int8_t* w, void* out, bool f16,
                     const void* xs, int xs16, const void* ws, int ws16, hipStream_t stream) {
    Rows8Cfg c{};
    if (!pick_rows8(M, K, N, c)) return fail(MCV_ERR_INVALID_ARG, "w8a8 rows: not a call for these kernels");
    const Rows8Args a{xq, w, out, xs, ws, xs16, ws16, static_cast<int>(M), static_cast<int>(K), static_cast<int>(N),
                      static_cast<int>(ceil_div(K, 128) * 4), static_cast<int>(ceil_div(N, kSlab))};
    return f16 ? launch_cfg8<true>(a, c, stream) : launch_cfg8<false>(a, c, stream);
}

}  // namespace mcv
