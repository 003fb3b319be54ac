// w4a16_rows.h -- launch interfaces shared by the W4A16 entry points that take
// several activation rows: the few-row kernel (w4a16_rows.hip), and the list of
// weights that share one x.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mcv {

// Up to four slab-64 weights read by one launch over the same x.
constexpr int kMaxParts = 4;
struct W4Part {
    const uint4* qw;
    const uint16_t* scales;
    const uint32_t* zeros;
    uint16_t* out;         // fp16 [M][N]
    int N;
    int Npad;
    int end;               // running total of the launch's column units up to and including this part
    uint32_t zero_bias;
};
struct W4Parts {
    W4Part p[kMaxParts];
    int count;
};

// The wide kernel's loads of a group's scales (fp16 [G][Npad]) and zero words
// (u32 [G][Npad / 8]): lane l < 16 cb takes column n0 + l of the unit, by a
// vector offset and a scalar base.  The buffer range check covers the vector
// offset alone, so the base plus the last taking lane's offset has to lie in
// the buffer, and a lane past the unit's columns gets an offset the check
// refuses: in the last unit of the last group it would read past the tensors.
constexpr uint32_t kLoadNothing = 0x80000000u;
__host__ __device__ constexpr uint32_t wide_scale_offset(int lane, int cb) {
    return lane < 16 * cb ? static_cast<uint32_t>(lane) * 2u : kLoadNothing;
}
__host__ __device__ constexpr uint32_t wide_zero_offset(int lane, int cb) {
    return lane < 16 * cb ? static_cast<uint32_t>(lane >> 3) * 4u : kLoadNothing;
}
__host__ __device__ constexpr int wide_scale_base(int g, int Npad, int n0) { return (g * Npad + n0) * 2; }
__host__ __device__ constexpr int wide_zero_base(int g, int Npad, int n0) { return (g * (Npad >> 3) + n0 / 8) * 4; }

// What a launch computes: one weight's out = x . W; several weights' over the
// same x; silu(x . gate) * (x . up).
constexpr int kOne = 0, kParts = 1, kSilu = 2;

// True where the few-row kernels are faster than the GEMV for M rows over `nslab`
// slabs in all (kSilu: of gate and of up each).
bool w4a16_rows_pays(int64_t M, int64_t K, int64_t nslab, int kind);

// True where the GEMM is faster than they are, on an output too large for the
// GEMV (one weight).
bool w4a16_rows_trail_gemm(int64_t M, int64_t K, int64_t nslab);

// True where the few-row kernels can run this call: at least 2 rows, x
// 16-byte aligned, x and every packed weight below 2 GiB (32-bit buffer
// offsets).
bool w4a16_rows_ok(const void* x, int64_t M, int64_t K, const W4Parts& parts);

// out_i = x . W_i for every part (`end` is set here).
int launch_w4a16_rows(const void* x, int64_t M, int64_t K, W4Parts parts, hipStream_t stream);

// act = silu(x . gate) * (x . up): parts.p[0] is gate, p[1] up, both [K][N];
// the sums are launch_w4a16_rows' and round to fp16 before silu_mul_f16.
int launch_w4a16_rows_silu(const void* x, int64_t M, int64_t K, W4Parts parts, void* act, hipStream_t stream);

// The kernel's configuration for M x K over `nslab` slabs, as text.
const char* w4a16_rows_name(int64_t M, int64_t K, int64_t nslab, int kind);

}  // namespace mcv
