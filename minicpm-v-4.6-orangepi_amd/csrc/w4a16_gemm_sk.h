// w4a16_gemm_sk.h -- launch interface of the half-slab W4A16 GEMM with an
// in-launch K split (w4a16_gemm_sk.hip), shared with the dispatcher.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "w4a16_rows.h"

namespace mcv {

// Tile TM rows x 32 * nwv columns (nwv half-slabs of 32 columns), ns stages
// in flight, K split `splits` ways across workgroups, kg quantisation groups
// (128 k each) per stage (kg must divide the groups of every split:
// K / 128 / splits), kw k-parts: nwv * kw waves, k-part j taking group j of
// every stage (kw = 2 needs kg = 2), their sums added in LDS at the end.
struct SkConfig {
    int tm;
    int nwv;
    int ns;
    int splits;
    int kg = 1;
    int kw = 1;
    int wr = 0;             // 1: each wave loads its weights, zeros and scales into registers (LDS holds x only)
    int order = 0;          // tile order: 0 by operand bytes (2 or 3), 1 along the rows, 2 down the
                            // columns, 3 down the columns of groups of tile rows
};

// The workspace starts with the tile arrival counters, a fixed region for
// every shape (so calls of different shapes may share one workspace), then
// the partial tiles.  A split call may have at most kSkMaxSplitTiles tiles.
constexpr int kSkMaxSplitTiles = 1024;
constexpr uint32_t kSkCounterBytes = kSkMaxSplitTiles * 4;

int64_t w4a16_sk_tiles(int64_t M, int64_t N, const SkConfig& c);
// Workspace bytes of a call (0 without a split): tile arrival counters
// (zero-filled once, left zero by every call) and the fp32 partial tiles.
int64_t w4a16_sk_workspace_bytes(int64_t M, int64_t N, const SkConfig& c);
bool w4a16_sk_config_valid(int64_t M, int64_t K, int64_t N, const SkConfig& c);
int launch_w4a16_gemm_sk(const void* x, int64_t M, int64_t K, int64_t N, const void* qw, const void* scales,
                         const void* zeros, int zero_bias, void* out, const SkConfig& c, void* ws, int64_t ws_bytes,
                         hipStream_t stream);

// Several weights over one x (no K split): out_i = x . W_i per part, or with
// `act` part 0 the gate and part 1 the up weight of silu(x . gate) * (x . up).
int launch_w4a16_gemm_sk_parts(const void* x, int64_t M, int64_t K, const W4Parts& parts, void* act, const SkConfig& c,
                               hipStream_t stream);
// The kernel's configuration as text: its first six template arguments, KIND (0
// one weight, 1 several, 2 gate and up) and whether its weight operands are the
// exact q - z or the rounded (q - z) s.
std::string w4a16_sk_name(const SkConfig& c, int kind, int64_t workgroups);
// True where the GEMM's 32-bit buffer offsets cover this call.
bool w4a16_sk_fits(int64_t M, int64_t K, const W4Parts& parts);
// The configuration the dispatch (w4a16_gemm.hip) takes for M x K x N; `exact`:
// for launch_w4a16_gemm_sk_parts.
SkConfig choose_gemm(int64_t M, int64_t K, int64_t N, bool can_split, bool exact = false);
// True where several weights over one x (`nslab` slabs in all) or, with `silu`,
// gate and up of `nslab` slabs each, run the GEMV rather than that GEMM.
bool w4a16_parts_prefer_gemv(int64_t M, int64_t K, int64_t nslab, bool silu);

}  // namespace mcv
