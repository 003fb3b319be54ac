// w4a16_rows.hip -- W4A16 matmul for a few activation rows (2 <= M <= 64) on
// fp16 MFMA, gfx950: batched decode, drafted tokens, short prompts.
//
// out[M][N] = x[M][K] . W[K][N], W in the slab-64 int4 layout, fp32
// accumulation, fp16 RNE output.  Like the GEMV it is bound by one pass over
// the packed weights (large N) or by the launch and one memory round trip
// (the decoder's projections); unlike the GEMV it reads and widens each weight
// once for all rows instead of once per row.
//
// v_mfma_f32_16x16x32_f16 takes rows 0-15 and k octet j = lane / 16 of x from
// one operand, column lane % 16 and the same k octet of W from the other.
// Which k an octet means is free as long as both agree, so lane (c, j) loads
// the 16 packed bytes of column c in chunk j of a quantisation group (32 k,
// four words of 8): word w of all lanes is then the weight operand for k =
// 32 j + 8 w .. + 7, four MFMAs cover the group's 128 k, and no lane needs
// another lane's weights.  x's operand is 16 contiguous bytes of one row.
//
// A word widens exactly: (word & mask) | 0x6400 is 1024 + q, minus 1024 + z;
// or 1024 + 16 q, times 1/16 minus 64 + z in one packed fma (64 + q is exact).
// Each group's sum over q - z leaves the MFMAs in fp32 and meets its scale in
// one fma, as in the GEMV: nothing is rounded before the output.  9 VALU per
// 8 weights and 16 MB rows, against the GEMV's 13 per row.
//
// Workgroup: KS waves split the groups (wave w takes w, w + KS, ...), each
// over 16 CB columns and 16 MB rows; the fp32 partial sums meet in LDS and are
// added in wave order.  KS is the same for every launch with the same K, so
// here a weight's output does not depend on what else the launch computes.
//
// x passes through LDS: loaded row by row (16 lanes read 256 contiguous bytes)
// and read back in operand order, because the operand's own order touches 32
// lines per load (K=3584 N=1024: M=16 6.0 -> 5.0 us, M=32 8.9 -> 6.1; M=2, with
// little to gather, 4.27 -> 4.46).
//
// MI355X, rotated weights, us per call against one GEMV row per activation row:
// K=3584 N=1024 M=6 4.6 / 5.2, M=32 6.1 / 9.2; K=1024 N=3584 M=5 3.3 / 3.8; qkv
// and z together (8192 columns) M=5 3.9 / 5.2, M=16 4.1 / 11.0; gate + up M=5
// 4.2 / 5.5, M=16 4.4 / 10.3; the vocabulary (K=1024 N=248094) M=6 27.1 / 124,
// M=16 29.1 / 66, M=32 37.1 / 79, M=64 53 / 105 (the last three the GEMM).
#include <algorithm>
#include <cstdio>
#include <string>

#include "common.h"
#include "w4a16_rows.h"

namespace mcv {
namespace {

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_r(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), 0x00020000);
}

// One wave's operands of one quantisation group.
template <int MB, int CB>
struct RowsGroup {
    uint4 w[CB];
    uint32_t z[CB];
    uint32_t s[CB];
    int4_t x[MB][4];       // rows 16 b + 4 t + lane / 16, one 16-byte chunk each
};

// Byte of 16-byte chunk q of row m of 16-row block b in a staged group.
__device__ __forceinline__ int x_at(int b, int m, int q) { return b * 4096 + m * 256 + ((q ^ m) << 4); }

// LDS bytes of one wave: its staged x rows or its partial sums.
constexpr int rows_wave_lds(int mb, int cb, int nw) { return mb * 1024 * (nw * cb > 4 ? nw * cb : 4); }

// Waves of a workgroup: the fewest that finish the groups in as many trips as
// 16 would.
int rows_ks(int64_t G) {
    const int64_t trips = ceil_div(G, 16);
    return static_cast<int>(ceil_div(G, trips));
}

template <int MB, int CB, int TR, bool SILU>
__global__ __launch_bounds__(1024) void w4a16_gemv_kernel_rows(const uint16_t* __restrict__ x, int M, int K,
                                                                              W4Parts parts, uint16_t* __restrict__ act) {
    constexpr int NW = SILU ? 2 : 1;                     // weights per workgroup
    constexpr int E = MB * CB * 4 * 64;                  // partial sums of one wave and weight
    // per wave: a group's x rows, then the wave's partial sums
    // [weight][mb][cb][register][lane]
    constexpr int R = rows_wave_lds(MB, CB, NW);
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int KS = static_cast<int>(blockDim.x >> 6);
    const int j = lane >> 4;
    const int G = K / kGroup, C = K / kChunkK;
    // this workgroup's weight and columns (constant indices only: the kernel
    // arguments stay in SGPRs)
    W4Part P[NW];
    P[0] = parts.p[0];
    if constexpr (SILU) P[1] = parts.p[1];
    int unit = blockIdx.x;
    if constexpr (!SILU) {
        int first = 0;
#pragma unroll
        for (int i = 1; i < kMaxParts; ++i)
            if (i < parts.count && unit >= parts.p[i - 1].end) {
                P[0] = parts.p[i];
                first = parts.p[i - 1].end;
            }
        unit -= first;
    }
    const int c0 = unit * 16 * CB;
    const int Npad = P[0].Npad;

    const __amdgpu_buffer_rsrc_t xr = rsrc_r(x, static_cast<uint32_t>(M) * K * 2u);
    __amdgpu_buffer_rsrc_t qr[NW], sr[NW], zr[NW];
#pragma unroll
    for (int t = 0; t < NW; ++t) {
        qr[t] = rsrc_r(P[t].qw, static_cast<uint32_t>(Npad) * (K / 2));
        sr[t] = rsrc_r(P[t].scales, static_cast<uint32_t>(G) * Npad * 2u);
        zr[t] = rsrc_r(P[t].zeros, static_cast<uint32_t>(G) * (Npad >> 3) * 4u);
    }
    // x loads: rows 4 t + lane / 16 of 16-row block b, 256 contiguous bytes a
    // row; rows past M are out of range and read zero
    const uint32_t xoff = static_cast<uint32_t>(j) * K * 2u + 16u * (lane & 15);
    uint8_t* const mine = lds + wave * R;
    uint32_t woff[CB];
#pragma unroll
    for (int b = 0; b < CB; ++b) {
        const int n = c0 + 16 * b + (lane & 15);
        woff[b] = ((static_cast<uint32_t>(n / kSlab) * C + j) * kSlab + (n & (kSlab - 1))) * 16u;
    }

    uint32_t vmagic;
    asm("v_mov_b32 %0, 0x64006400" : "=v"(vmagic));
    const uint32_t mlo = __builtin_amdgcn_readfirstlane(0x000F000Fu);
    const uint32_t mhi = __builtin_amdgcn_readfirstlane(0x00F000F0u);
    const half2_t sixteenth = as_h2(0x2C002C00u);        // half2(1/16)

    float4_t acc[NW][MB][CB];
#pragma unroll
    for (int t = 0; t < NW; ++t)
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int c = 0; c < CB; ++c) acc[t][b][c] = float4_t{0.f, 0.f, 0.f, 0.f};

    auto load_x = [&](int g, int4_t (&d)[MB][4]) {
        const uint32_t dead = static_cast<uint32_t>(g >= G) << 31;
        const int gc = g < G ? g : 0;
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                d[b][t] = __builtin_bit_cast(
                    int4_t, __builtin_amdgcn_raw_buffer_load_b128(xr, (xoff + (16 * b + 4 * t) * K * 2u) | dead, gc * 256, 0));
    };
    // the group's rows into this wave's LDS, chunk q of row m at q ^ m, where
    // 16 lanes write one row and 16 rows' lanes read one q without conflicts
    auto put_x = [&](const int4_t (&d)[MB][4]) {
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                *reinterpret_cast<int4_t*>(mine + x_at(b, 4 * t + j, lane & 15)) = d[b][t];
    };
    auto load_w = [&](int t, int g, RowsGroup<MB, CB>& d) {
        const uint32_t dead = static_cast<uint32_t>(g >= G) << 31;
        const int gc = g < G ? g : 0;
#pragma unroll
        for (int c = 0; c < CB; ++c)
            d.w[c] = __builtin_bit_cast(
                uint4, __builtin_amdgcn_raw_buffer_load_b128(qr[t], woff[c] | dead, gc * 4 * kSlab * 16, 2));
#pragma unroll
        for (int c = 0; c < CB; ++c) {
            const uint32_t n = static_cast<uint32_t>(c0 + 16 * c + (lane & 15));
            d.s[c] = __builtin_amdgcn_raw_buffer_load_b16(sr[t], (n * 2u) | dead, gc * Npad * 2, 0);
            d.z[c] = __builtin_amdgcn_raw_buffer_load_b32(zr[t], ((n >> 3) * 4u) | dead, gc * (Npad >> 3) * 4, 0);
        }
    };
    auto sum = [&](int t, const RowsGroup<MB, CB>& a) {
#pragma unroll
        for (int c = 0; c < CB; ++c) {
            const int n = c0 + 16 * c + (lane & 15);
            const uint32_t zq = ((a.z[c] >> ((n & 7) * 4)) & 15u) + P[t].zero_bias;
            const half2_t zlo = as_h2((0x6400u + zq) * 0x10001u);            // 1024 + z
            const half2_t zhi = as_h2((0xD400u + (zq << 4)) * 0x10001u);     // -(64 + z)
            const uint32_t words[4] = {a.w[c].x, a.w[c].y, a.w[c].z, a.w[c].w};
            float4_t ga[MB];
#pragma unroll
            for (int b = 0; b < MB; ++b) ga[b] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const half8_t wv = widen_exact(words[i], zlo, zhi, mlo, mhi, vmagic, sixteenth);
#pragma unroll
                for (int b = 0; b < MB; ++b)
                    ga[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        *reinterpret_cast<const half8_t*>(mine + x_at(b, lane & 15, 4 * j + i)), wv, ga[b], 0, 0, 0);
            }
            const float sc = h2f(static_cast<uint16_t>(a.s[c]));
#pragma unroll
            for (int b = 0; b < MB; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[t][b][c][r] = fmaf(ga[b][r], sc, acc[t][b][c][r]);
        }
    };

    // TR groups per trip, their loads all out before the first wait; a group
    // past the last reads zeros (out of range) and adds nothing
    for (int g0 = wave; g0 < G; g0 += KS * TR) {
        RowsGroup<MB, CB> a[TR][NW];
#pragma unroll
        for (int u = 0; u < TR; ++u) {
#pragma unroll
            for (int t = 0; t < NW; ++t) load_w(t, g0 + u * KS, a[u][t]);
            load_x(g0 + u * KS, a[u][0].x);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < TR; ++u) {
            put_x(a[u][0].x);
#pragma unroll
            for (int t = 0; t < NW; ++t) sum(t, a[u][t]);
        }
    }
    float* const part = reinterpret_cast<float*>(mine);

#pragma unroll
    for (int t = 0; t < NW; ++t)
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int c = 0; c < CB; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    part[t * E + ((b * CB + c) * 4 + r) * 64 + lane] = acc[t][b][c][r];
    __syncthreads();
    // register r of lane l in block (b, c): row 16 b + 4 (l / 16) + r, column 16 c + l % 16
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
        const int l = e & 63, r = (e >> 6) & 3, c = (e >> 8) % CB, b = (e >> 8) / CB;
        const int m = 16 * b + 4 * (l >> 4) + r, n = c0 + 16 * c + (l & 15);
        if (m >= M || n >= P[0].N) continue;
        uint16_t h[NW];
#pragma unroll
        for (int t = 0; t < NW; ++t) {
            const float* sums = reinterpret_cast<const float*>(lds) + t * E + e;
            float v = sums[0];
            for (int w = 1; w < KS; ++w) v += sums[w * (R / 4)];
            h[t] = f2h(v);
        }
        if constexpr (SILU) act[static_cast<size_t>(m) * P[0].N + n] = silu_mul_f16(h[0], h[1]);
        else P[0].out[static_cast<size_t>(m) * P[0].N + n] = h[0];
    }
}

// ---- wide outputs (the lm_head over a few rows): HBM bound, so no split and
// no exchange.  x is staged once per workgroup in LDS in MFMA operand order
// (1 KiB per group, word and 16 rows); each wave then takes one unit of 16 CB
// columns over all of K, with the next D groups' weights in flight, and stores
// its columns straight from the accumulators.  Its groups add up one after
// another, the split kernel's per wave and then over the waves, so the last
// bits of the two differ.  A group's scales and zero words come in as one load
// each for the unit's columns (the lanes past them load nothing) and reach the
// lanes of each 16-column block through ds_bpermute.  MI355X, K=1024, us, split
// kernel / this one with 32 columns a unit, two groups in flight, 8 waves: M=6
// V=31012 6.6 / 8.8, 62024 11.2 / 10.2, 124047 19.6 / 15.4, 248094 35.3 / 27.1
// (64 columns 28.6; four groups in flight 29.3; 4 waves 29.2; 16 waves of 64
// columns 30.1); M=32 V=31012 11.2 / 10.7, 62024 20.5 / 12.4.
template <int MB, int CB, int D, int T>
__global__ __launch_bounds__(T) void w4a16_rows_wide_kernel(const uint16_t* __restrict__ x, int M, int K, W4Part P,
                                                               int units) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t xl[];   // [group] x_at()
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int NW = static_cast<int>(blockDim.x >> 6);
    const int j = lane >> 4;
    const int G = K / kGroup, C = K / kChunkK;
    const int Npad = P.Npad;
    const __amdgpu_buffer_rsrc_t xr = rsrc_r(x, static_cast<uint32_t>(M) * K * 2u);
    const __amdgpu_buffer_rsrc_t qr = rsrc_r(P.qw, static_cast<uint32_t>(Npad) * (K / 2));
    const __amdgpu_buffer_rsrc_t sr = rsrc_r(P.scales, static_cast<uint32_t>(G) * Npad * 2u);
    const __amdgpu_buffer_rsrc_t zr = rsrc_r(P.zeros, static_cast<uint32_t>(G) * (Npad >> 3) * 4u);

    uint32_t woff[CB];
#pragma unroll
    for (int c = 0; c < CB; ++c) woff[c] = static_cast<uint32_t>(j * kSlab + 16 * c + (lane & 15)) * 16u;
    const uint32_t soff = wide_scale_offset(lane, CB), zoff = wide_zero_offset(lane, CB);
    uint4 w[D][CB];
    uint32_t s[D], z[D];
    auto load_w = [&](int slot, int unit, int g) {
        // unit = 16 CB columns: column base n0 = 16 CB unit, inside slab n0 / 64
        const int n0 = unit * 16 * CB, slab = n0 / kSlab, in = n0 % kSlab;
        const uint32_t dead = static_cast<uint32_t>(g >= G) << 31;       // out of range: reads zero
        const int gc = g < G ? g : 0;
#pragma unroll
        for (int c = 0; c < CB; ++c)
            w[slot][c] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
                                                       qr, woff[c] | dead, (slab * C + gc * 4) * 1024 + in * 16, 2));
        s[slot] = __builtin_amdgcn_raw_buffer_load_b16(sr, soff | dead, wide_scale_base(gc, Npad, n0), 0);
        z[slot] = __builtin_amdgcn_raw_buffer_load_b32(zr, zoff | dead, wide_zero_base(gc, Npad, n0), 0);
    };
    const int unit = static_cast<int>(blockIdx.x) * NW + wave;
    if (unit < units) {
#pragma unroll
        for (int d = 0; d < D; ++d) load_w(d, unit, d);
    }
    for (int t = wave; t < G * 4 * MB; t += NW) {         // four rows of one group
        const int g = t / (4 * MB), m = 4 * (t % (4 * MB)) + j;
        const int4_t v = __builtin_bit_cast(
            int4_t, __builtin_amdgcn_raw_buffer_load_b128(xr, static_cast<uint32_t>(m) * K * 2u + 16u * (lane & 15), g * 256, 0));
        *reinterpret_cast<int4_t*>(xl + g * MB * 4096 + x_at(m >> 4, m & 15, lane & 15)) = v;
    }
    __syncthreads();
    if (unit >= units) return;

    uint32_t vmagic;
    asm("v_mov_b32 %0, 0x64006400" : "=v"(vmagic));
    const uint32_t mlo = __builtin_amdgcn_readfirstlane(0x000F000Fu);
    const uint32_t mhi = __builtin_amdgcn_readfirstlane(0x00F000F0u);
    const half2_t sixteenth = as_h2(0x2C002C00u);        // half2(1/16)

    float4_t acc[MB][CB];
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
        for (int c = 0; c < CB; ++c) acc[b][c] = float4_t{0.f, 0.f, 0.f, 0.f};
    for (int g0 = 0; g0 < G; g0 += D) {
#pragma unroll
        for (int u = 0; u < D; ++u) {
            const int g = g0 + u;                    // past G: zero weights and scales, x of the last group
            const int gx = g < G ? g : G - 1;
            // scale (low half) and zero (high half) of this lane's column of the slab
            const uint32_t sz = (s[u] & 0xffffu) | ((((z[u] >> ((lane & 7) * 4)) & 15u) + P.zero_bias) << 16);
            half8_t xv[MB][4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int b = 0; b < MB; ++b)
                    xv[b][i] = *reinterpret_cast<const half8_t*>(xl + gx * MB * 4096 + x_at(b, lane & 15, 4 * j + i));
#pragma unroll
            for (int c = 0; c < CB; ++c) {
                const uint32_t v = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(
                    (16 * c + (lane & 15)) * 4, static_cast<int>(sz)));
                const uint32_t zq = v >> 16;
                const half2_t zlo = as_h2((0x6400u + zq) * 0x10001u);            // 1024 + z
                const half2_t zhi = as_h2((0xD400u + (zq << 4)) * 0x10001u);     // -(64 + z)
                const uint32_t words[4] = {w[u][c].x, w[u][c].y, w[u][c].z, w[u][c].w};
                float4_t ga[MB];
#pragma unroll
                for (int b = 0; b < MB; ++b) ga[b] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const half8_t wv = widen_exact(words[i], zlo, zhi, mlo, mhi, vmagic, sixteenth);
#pragma unroll
                    for (int b = 0; b < MB; ++b) ga[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv[b][i], wv, ga[b], 0, 0, 0);
                }
                const float sc = h2f(static_cast<uint16_t>(v));
#pragma unroll
                for (int b = 0; b < MB; ++b)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[b][c][r] = fmaf(ga[b][r], sc, acc[b][c][r]);
            }
            load_w(u, unit, g + D);
        }
    }
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = 16 * b + 4 * j + r;
#pragma unroll
            for (int c = 0; c < CB; ++c) {
                const int n = (unit * CB + c) * 16 + (lane & 15);
                if (m < M && n < P.N) P.out[static_cast<size_t>(m) * P.N + n] = f2h(acc[b][c][r]);
            }
        }
}

struct RowsCfg {
    int mb;
    int cb;
    int ks;
};

// 16-row blocks by M; columns per workgroup: the most (64, 32, 16) that still
// leave about one workgroup per CU, unless fewer would make more than one
// (65-95 slabs on 16 columns: two rounds; K=2560 N=4608 M=2 6.5 us, on 32 5.1).
RowsCfg choose_rows(int64_t M, int64_t K, int64_t cols, int nw) {
    RowsCfg c;
    c.mb = M <= 16 ? 1 : 2;
    c.ks = rows_ks(K / kGroup);
    c.cb = 4;
    while (c.cb > 1 && ((cols / (16 * c.cb) < 192 && cols / (8 * c.cb) <= 256) || c.mb * c.cb * nw > 4)) c.cb /= 2;
    return c;
}

// Wide outputs, from where their free-running waves pay for each walking all of
// K alone (the figures at the kernel); LDS holds x, 4 KiB per group and 16 rows.
bool rows_wide(int64_t M, int64_t K, int64_t nslab) {
    const int mb = M <= 16 ? 1 : (M <= 32 ? 2 : 4);
    return nslab >= (mb == 1 ? 800 : 400) && (K / kGroup) * mb * 4096 <= 160 * 1024;
}

template <int MB, int CB, int TR, bool SILU>
int launch_rows(const void* x, int64_t M, int64_t K, const W4Parts& parts, void* act, int64_t units, int ks,
                hipStream_t stream) {
    const size_t lds = size_t(ks) * rows_wave_lds(MB, CB, SILU ? 2 : 1);
    hipLaunchKernelGGL((w4a16_gemv_kernel_rows<MB, CB, TR, SILU>), dim3(static_cast<unsigned>(units)), dim3(64 * ks), lds,
                       stream, static_cast<const uint16_t*>(x), static_cast<int>(M), static_cast<int>(K), parts,
                       static_cast<uint16_t*>(act));
    return check_launch("w4a16_gemv_kernel_rows");
}

template <bool SILU>
int launch_any(const void* x, int64_t M, int64_t K, W4Parts& parts, void* act, hipStream_t stream) {
    int64_t cols = 0;
    const int n = SILU ? 1 : parts.count;
    for (int i = 0; i < n; ++i) cols += parts.p[i].Npad;
    const RowsCfg c = choose_rows(M, K, cols, SILU ? 2 : 1);
    int64_t units = 0;
    for (int i = 0; i < n; ++i) {
        units += parts.p[i].Npad / (16 * c.cb);
        parts.p[i].end = static_cast<int>(units);
    }
#define MCV_ROWS(MB_, CB_) \
    if (c.mb == MB_ && c.cb == CB_)                                                                       \
        return K / kGroup > c.ks && MB_ * CB_ <= 2                                                          \
                   ? launch_rows<MB_, CB_, (MB_ * CB_ <= 2 ? 2 : 1), SILU>(x, M, K, parts, act, units, c.ks, stream) \
                   : launch_rows<MB_, CB_, 1, SILU>(x, M, K, parts, act, units, c.ks, stream);
    MCV_ROWS(1, 1) MCV_ROWS(1, 2) MCV_ROWS(2, 1)
    if constexpr (!SILU) { MCV_ROWS(1, 4) MCV_ROWS(2, 2) }
#undef MCV_ROWS
    return fail(MCV_ERR_INVALID_ARG, "w4a16 rows: no kernel for %d x %d blocks", c.mb, c.cb);
}

template <int MB, int CB>
int launch_wide(const void* x, int64_t M, int64_t K, const W4Part& p, hipStream_t stream) {
    constexpr int kWaves = 8;
    const int64_t units = p.Npad / (16 * CB);
    const size_t lds = size_t(K / kGroup) * MB * 4096;
    hipLaunchKernelGGL((w4a16_rows_wide_kernel<MB, CB, 2, 64 * kWaves>), dim3(static_cast<unsigned>(ceil_div(units, kWaves))),
                       dim3(64 * kWaves), lds, stream, static_cast<const uint16_t*>(x), static_cast<int>(M),
                       static_cast<int>(K), p, static_cast<int>(units));
    return check_launch("w4a16_rows_wide_kernel");
}

thread_local std::string g_rows_name;

}  // namespace

bool w4a16_rows_ok(const void* x, int64_t M, int64_t K, const W4Parts& parts) {
    if (M < 2 || reinterpret_cast<uintptr_t>(x) % 16 != 0 || M * K * 2 >= (int64_t(1) << 31)) return false;
    int64_t cols = 0;
    for (int i = 0; i < parts.count; ++i) {
        cols += parts.p[i].Npad;
        if (int64_t(parts.p[i].Npad) * (K / 2) >= (int64_t(1) << 31)) return false;
    }
    return cols / 16 <= 0x7fffffff;
}

// Against the GEMV, whose grid is one workgroup per slab and row.  That grid
// costs little until it exceeds a workgroup per CU, and its rows need no LDS; the
// few-row kernel's time hardly depends on M within a 16-row block.  MI355X, us,
// GEMV / here, mean of weights cold and in cache (measured over K = 128..8192, N =
// 64..12288, M = 2..32):
//   grid > 256: K=3584 N=1000 M=32 9.0 / 6.4; but one or two groups leave neither a K
//   to split, and the GEMV starts sooner: K=128 N=6144 M=5 2.7 / 3.5, K=256 N=6144 M=8
//   3.2 / 3.5, M=12 3.6 / 3.5; four: N=2048 M=8 2.9 / 3.1; more than 128 slabs on a
//   short K, where 64-column units are the narrowest to fit a round: K=1024 N=10240
//   M=2 4.3 / 5.1, M=5 6.2 / 5.1;
//   grid <= 256, up to 16 rows: past K = 2048 the GEMV's second trip over K loses
//   (K=3584 N=1000 M=2 5.3 / 4.8) unless its slabs are many (N=4608 5.6 / 5.9); a
//   shorter K from 32 slabs and 100 workgroups on unless its groups are four or
//   eight, one per GEMV wave (K=768 N=3584 M=3 3.8 / 3.5, K=1024 3.4 / 3.7);
//   17 to 32 rows: K=1024 N=512 M=32 3.3 / 3.9, K=2048 N=256 4.0 / 4.7; but one
//   narrow weight (up to three slabs): K=1152 N=136 M=20 4.0 / 3.6.  Gate and up
//   together do not (K=2048 N=136 M=32 5.0 / 5.8).
// Past 32 rows only wide outputs.
bool w4a16_rows_pays(int64_t M, int64_t K, int64_t nslab, int kind) {
    if (M < 2 || M > 64) return false;
    const int64_t G = K / kGroup, grid = M * nslab;
    if (G <= 2 && M <= 3) return false;
    if (kind == kOne && rows_wide(M, K, nslab)) return true;
    if (M > 32) return false;
    if (G == 1) return grid > 4096;
    if (G == 2) return grid > (kind == kParts ? 640 : 960);
    if (grid > 256) return (G != 4 || grid > 512) && (M > 16 || nslab <= 128 || grid * K > 500000);
    if (M > 16) return kind == kOne && nslab < 4;
    return nslab <= 64 && (K > 2048 || (G != 4 && G != 8 && nslab >= 32 && grid > 100));
}

// Against the GEMM, for outputs too large for the GEMV.  17 to 32 rows of 32-column
// units take a second round past 128 slabs, where the GEMM's tiles of 32 x 128 do not
// (K=3584 N=10240 M=32 15.5 us here / 11.8 GEMM) unless an odd group count leaves it
// one k-part (K=3968 M=17 14.6 / 18.4); one or two groups leave the waves here
// nothing to split (K=256 N=6144 M=24 4.4 / 4.0, N=4096 3.5 / 4.1).
bool w4a16_rows_trail_gemm(int64_t M, int64_t K, int64_t nslab) {
    if (rows_wide(M, K, nslab)) return false;
    const int64_t G = K / kGroup;
    if (G <= 2) return G == 1 || nslab > (M <= 16 ? 128 : 64);
    return M > 16 && G % 2 == 0 && (nslab > 128 || K > 6144);
}

int launch_w4a16_rows(const void* x, int64_t M, int64_t K, W4Parts parts, hipStream_t stream) {
    if (parts.count == 1 && rows_wide(M, K, parts.p[0].Npad / kSlab)) {
        if (M <= 16) return launch_wide<1, 2>(x, M, K, parts.p[0], stream);
        if (M <= 32) return launch_wide<2, 2>(x, M, K, parts.p[0], stream);
        return parts.p[0].Npad / kSlab >= 1536 ? launch_wide<4, 4>(x, M, K, parts.p[0], stream)
                                               : launch_wide<4, 2>(x, M, K, parts.p[0], stream);
    }
    return launch_any<false>(x, M, K, parts, nullptr, stream);
}

int launch_w4a16_rows_silu(const void* x, int64_t M, int64_t K, W4Parts parts, void* act, hipStream_t stream) {
    return launch_any<true>(x, M, K, parts, act, stream);
}

const char* w4a16_rows_name(int64_t M, int64_t K, int64_t nslab, int kind) {
    char buf[128];
    if (kind == kOne && rows_wide(M, K, nslab)) {
        std::snprintf(buf, sizeof(buf), "w4a16_rows_wide_kernel<%d, %d, 2, 512>", M <= 16 ? 1 : (M <= 32 ? 2 : 4),
                      M > 32 && nslab >= 1536 ? 4 : 2);
    } else {
        const RowsCfg c = choose_rows(M, K, nslab * kSlab, kind == kSilu ? 2 : 1);
        std::snprintf(buf, sizeof(buf), "w4a16_gemv_kernel_rows<%d, %d, %d, %s> (%lld workgroups of %d waves)", c.mb, c.cb,
                      K / kGroup > c.ks && c.mb * c.cb <= 2 ? 2 : 1, kind == kSilu ? "true" : "false", (long long)(nslab * 4 / c.cb),
                      c.ks);
    }
    g_rows_name = buf;
    return g_rows_name.c_str();
}

}  // namespace mcv
