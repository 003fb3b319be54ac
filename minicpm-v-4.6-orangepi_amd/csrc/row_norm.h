// row_norm.h -- RMSNorm of fp16 rows, alone (elementwise.hip) or followed by
// the W8A8 activation quantisation (w8a8.hip); one 256-thread workgroup per row.
#pragma once

#include "common.h"

namespace mcv {

// Two halves of 16 bytes at a time, element e of a chunk.
__device__ __forceinline__ uint16_t chunk_get(const uint4& v, int e) {
    const uint32_t w = e < 4 ? (e < 2 ? v.x : v.y) : (e < 6 ? v.z : v.w);
    return static_cast<uint16_t>(w >> (16 * (e & 1)));
}

// The normed values of a chunk; MAX: m becomes the largest magnitude among them and m.
template <bool MAX>
__device__ __forceinline__ uint4 rms_chunk(const uint4& x, const uint4& g, float rstd, float& m) {
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        const uint16_t a = rms_apply(chunk_get(x, e), rstd, chunk_get(g, e));
        const uint16_t b = rms_apply(chunk_get(x, e + 1), rstd, chunk_get(g, e + 1));
        w[e / 2] = a | (static_cast<uint32_t>(b) << 16);
        if constexpr (MAX) {
            const float va = fabsf(h2f(a)), vb = fabsf(h2f(b));
            m = va > m ? va : m;
            m = vb > m ? vb : m;
        }
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// normed = fp16((x * rstd) * gamma), rstd = 1 / sqrt(mean(x^2) + eps); QUANT:
// then the row's int8 values and scale, from the same fp16 values.  Every step
// is an explicitly rounded fp32 operation, and thread t sums the squares of
// elements t, t + 256, ... in that order, so the result does not depend on PER,
// VEC or QUANT.
//
// A row is one memory round trip: every load goes out before the first use
// (PER strided elements a thread for the sum; VEC: x again and gamma as 16-byte
// chunks, chunk t + 256 c, for the output, whose stores are then 16 bytes of
// fp16 and 8 of int8 a thread).  Reloading x and gamma element by element
// after the sum made two and more.  MI355X, us before / after: M=1 H=1024 2.7 /
// 2.4, H=3584 5.1 / 3.6, M=1100 H=1024 4.1 / 3.4, M=3000 7.5 / 6.4; with the
// quantisation M=1 H=1024 3.5 / 3.1, H=2048 4.9 / 3.5.  PER = 0: rows longer than
// 256 * 32, strided loops, each with only the loads and stores it needs (with the
// store conditional inside: M=1 H=16384 27.8 us, now 26.3, as before PER).
template <int PER, bool VEC, bool QUANT>
__global__ __launch_bounds__(256) void rms_row_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ gamma,
                                                      int H, float eps, uint16_t* __restrict__ normed,
                                                      int8_t* __restrict__ xq, float* __restrict__ s32,
                                                      uint16_t* __restrict__ s16) {
    const int row = blockIdx.x;
    const int t = threadIdx.x;
    const uint16_t* xr = x + static_cast<size_t>(row) * H;
    uint16_t* nr = normed ? normed + static_cast<size_t>(row) * H : nullptr;
    int8_t* qr = QUANT ? xq + static_cast<size_t>(row) * H : nullptr;
    float m = 0.f;
    float scale = 0.f;
    if constexpr (PER > 0) {
        constexpr int NC = VEC ? (PER + 7) / 8 : 1;
        uint16_t xs[PER], gs[VEC ? 1 : PER];
        uint4 xv[NC], gv[NC];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int i = t + 256 * j;
            xs[j] = i < H ? xr[i] : uint16_t(0);
            if constexpr (!VEC) gs[j] = i < H ? gamma[i] : uint16_t(0);
        }
        if constexpr (VEC)
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const int i = 8 * (t + 256 * c);
                xv[c] = i < H ? *reinterpret_cast<const uint4*>(xr + i) : make_uint4(0, 0, 0, 0);
                gv[c] = i < H ? *reinterpret_cast<const uint4*>(gamma + i) : make_uint4(0, 0, 0, 0);
            }
        // x may be `normed`: no load may be in flight when another thread stores
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const float v = h2f(xs[j]);                  // zero past the row: adds nothing
            ss = fmaf(v, v, ss);
        }
        const float rstd = block_rstd(ss, H, eps);
        if constexpr (VEC) {
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const int i = 8 * (t + 256 * c);
                xv[c] = rms_chunk<QUANT>(xv[c], gv[c], rstd, m);          // now the normed chunk
                if (i < H && nr) *reinterpret_cast<uint4*>(nr + i) = xv[c];
            }
        } else {
#pragma unroll
            for (int j = 0; j < PER; ++j) {
                const int i = t + 256 * j;
                xs[j] = rms_apply(xs[j], rstd, gs[j]);
                if (i < H && nr) nr[i] = xs[j];
                if constexpr (QUANT) {
                    const float v = i < H ? fabsf(h2f(xs[j])) : 0.f;
                    m = v > m ? v : m;
                }
            }
        }
        if constexpr (QUANT) {
            scale = act_scale(row_absmax(m));
            const float inv = __fdiv_rn(1.0f, scale);
            if constexpr (VEC) {
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    const int i = 8 * (t + 256 * c);
                    if (i < H) *reinterpret_cast<uint2*>(qr + i) = act_quant8(xv[c], inv);
                }
            } else {
#pragma unroll
                for (int j = 0; j < PER; ++j) {
                    const int i = t + 256 * j;
                    if (i < H) qr[i] = act_quant(xs[j], inv);
                }
            }
        }
    } else {
        const float rstd = row_rstd(xr, H, eps);
        if constexpr (!QUANT) {
            for (int i = t; i < H; i += blockDim.x) nr[i] = rms_apply(xr[i], rstd, gamma[i]);
        } else {
            auto each = [&](auto&& use) {
                for (int i = t; i < H; i += blockDim.x) use(i, rms_apply(xr[i], rstd, gamma[i]));
            };
            auto largest = [&](uint16_t h) {
                const float v = fabsf(h2f(h));
                m = v > m ? v : m;
            };
            if (nr) each([&](int i, uint16_t h) { largest(h); nr[i] = h; });
            else each([&](int, uint16_t h) { largest(h); });
            scale = act_scale(row_absmax(m));
            const float inv = __fdiv_rn(1.0f, scale);
            // the normed row again, from memory only where x is gone (in place)
            if (nr == xr) for (int i = t; i < H; i += blockDim.x) qr[i] = act_quant(nr[i], inv);
            else each([&](int i, uint16_t h) { qr[i] = act_quant(h, inv); });
        }
    }
    if constexpr (QUANT) {
        if (t == 0) {
            if (s32) s32[row] = scale;
            if (s16) s16[row] = f2h(scale);
        }
    }
}

using RmsFn = void (*)(const uint16_t*, const uint16_t*, int, float, uint16_t*, int8_t*, float*, uint16_t*);

// Launches the kernel for M rows of H; VEC needs whole 16-byte chunks: H a
// multiple of 8 and aligned rows, and more than one element a thread: up to 256
// it loads x twice where the strided form has everything in one load each
// (M=50000 H=128 33.3 us in chunks, 24.3 strided; M=8192 H=256 7.8 / 6.3).  (A wave per row, without barriers, was slower
// below 8192 rows: M=512 H=1024 3.9 us against 3.1, M=2000 H=2048 13.6 / 7.9.)
template <bool QUANT>
void launch_rms(const uint16_t* x, const uint16_t* gamma, int64_t M, int64_t H, float eps, uint16_t* normed, int8_t* xq,
                float* s32, uint16_t* s16, hipStream_t stream) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(gamma) |
                         reinterpret_cast<uintptr_t>(normed) | (reinterpret_cast<uintptr_t>(xq) << 1);
    const bool vec = H % 8 == 0 && at % 16 == 0;
    const int h = static_cast<int>(H);
    RmsFn fn = rms_row_kernel<0, false, QUANT>;
    if (H <= 256) fn = rms_row_kernel<1, false, QUANT>;
    else if (H <= 1024) fn = vec ? rms_row_kernel<4, true, QUANT> : rms_row_kernel<4, false, QUANT>;
    else if (H <= 2048) fn = vec ? rms_row_kernel<8, true, QUANT> : rms_row_kernel<8, false, QUANT>;
    else if (H <= 4096) fn = vec ? rms_row_kernel<16, true, QUANT> : rms_row_kernel<16, false, QUANT>;
    else if (H <= 8192) fn = vec ? rms_row_kernel<32, true, QUANT> : rms_row_kernel<32, false, QUANT>;
    hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>(M)), dim3(256), 0, stream, x, gamma, h, eps, normed, xq, s32, s16);
}

}  // namespace mcv
