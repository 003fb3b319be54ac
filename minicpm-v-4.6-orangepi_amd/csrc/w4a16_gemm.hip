// w4a16_gemm.hip -- the W4A16 matmul dispatch for any M, gfx950.
//
// out[M][N] = x[M][K] . W[K][N], W in the slab-64 int4 layout.  One row streams
// the weights through the GEMV (w4a16_gemv.hip; one grid row per activation row
// where a few rows of a small weight are as fast that way); a few rows run the
// kernels that widen every weight once for all of them (w4a16_rows.hip); larger M
// runs the half-slab MFMA GEMM (w4a16_gemm_sk.hip), which reuses each widened
// weight operand across TM rows, in the tile shape and K split picked here.
//
// The reference has no M > 1 quantised path: its matmul_w4a16 is M = 1 only
// (src/csrc/lib/ops.cpp:1030-1095) and its prefill runs dense fp16 aclnnMm
// through matmul_b_transposed (src/csrc/lib/decoder_layer.cpp:459-462,
// 656-659, 857-860; src/csrc/lib/ops.cpp:159-322).
#include <cstdio>
#include <string>

#include "common.h"
#include "w4a16_gemm_sk.h"

namespace mcv {

int launch_w4a16_gemv(const void* x, int64_t M, int64_t K, int64_t N, const void* qw, const void* scales,
                      const void* zeros, int zero_bias, void* out, hipStream_t stream);
int gemv_ksplit(int64_t G, int64_t blocks);

// The few-row kernels aside (w4a16_rows_pays comes first): the GEMV streams the
// weights once per row and still beats the MFMA GEMM, whose tile count is M/TM
// * N/TN, until the output reaches about 64K elements.
bool small_output(int64_t M, int64_t N) { return M >= 1 && (M < 8 || M * N < 65536); }

// The GEMM's configuration for M x K x N.  First the largest tile whose grid
// gives 200-256 workgroups, one tile each (a workgroup per CU): 128 x 256
// (eight waves), 64 x 128, 64 x 64, 32 x 128, 32 x 64; past 256
// tiles of even the smallest, the least of a cost table: what a CU's tiles take
// depends on how many it gets (a shape just past 256 takes two rounds) and on
// whether another workgroup on the CU covers a tile's start and end.  Against
// the largest tile that reached 200 workgroups, us: M=8192 K=1024 N=3584 65.2 ->
// 61.8 (128 x 128, two per CU), M=1100 K=1024 N=8192 30.3 -> 24.9 and N=3584 15.6
// -> 12.1, M=577 N=8192 21.2 -> 15.9, M=1600 N=3584 22.5 -> 16.6, M=1100 K=3584
// N=1024 22.2 -> 15.5, M=4096 37.2 -> 32.9.  Failing that (few rows and N =
// 1024-like widths), with a workspace, K is split across workgroups on 32 x 64
// tiles: the most ways that keep the grid within one workgroup per CU and
// leave each workgroup at least 7 quantisation groups on average (splits are
// cut in whole stages, so they differ by at most one) -- the partial tiles'
// exchange costs ~1-2 us, which a shorter loop does not pay back.  A
// tile of four half-slabs takes two k-parts (eight waves, two groups per
// stage) when its workgroups' group count is even and at least 8 (32 x 128 at
// M=130 K=1024 N=3584 6.1 us against 6.8 with one k-part); the 32 x 64 and 64 x 64 tiles (two
// half-slabs) whenever K/128 is even: two waves per SIMD cover each other's
// copy issue.  The 64-
// and 32-row tiles load their weights, zeros and scales straight into
// registers (each wave's columns are its own; LDS then stages x only): 0-9 %
// faster than staging them in LDS in two sweeps, never slower; the 128 x 256
// tile measured the same either way and keeps the LDS path.  Measured on
// MI355X (rotated weights, us per call, back to back; the same launch varies
// by up to +-7 % from one 200-launch region to the next on the long shapes):
// M=2048 K=1024 N=3584 128x256 20.0-20.6 (64x128 24-25); M=2048 K=3584 N=1024
// 64x128 two k-parts 19.6-22.3 (LDS weights 20.1-21.6, one k-part 21.6-22.6);
// M=512 K=1024 N=3584 64x128 two k-parts 8.3-8.5 (32x64 10.0-11.6); M=512
// K=3584 N=1024 32x64 two k-parts 10.1 (32x128 split 2 ways 11.4-12.1, 64x64
// split 2 ways 10.8); M=128 K=1024 N=3584 32x64 two k-parts 5.5 (one k-part
// 6.6, 32x128 6.7-7.0); M=128 K=3584 N=1024 32x64 split 4 ways, two k-parts
// 7.96 (3 ways 7.93, 2 ways 8.8; one k-part 4 ways 9.7; 32x128 split 4 ways
// 9.6-9.8); M=64 K=3584 N=1024 32x64 split 4 ways 7.2 (3 ways 7.4, 8 ways
// 8.0); M=128 K=2048 N=1024 2 ways 7.1 (3 ways 6.85); 64x64 two
// k-parts against 32x128 at 224-256 tiles: M=256 K=1024 N=3584 6.6 / 7.3,
// M=1024 K=3584 N=1024 13.9 / 15.6, M=512 K=1024 N=2048 6.5 / 7.1, M=1024
// K=2048 N=1024 9.3 / 9.9, M=512 K=3584 N=2048 14.1 / 15.9; at 288-384
// tiles 64x64 is 0.1-2 us slower.  Against the
// rule before the 32 x 64 tile, over M = 48..512 and (K, N) = (1024, 3584),
// (3584, 1024), (1024, 6144), (1024, 2048), (2048, 1024): 10-25 % faster
// where it changes the configuration, except 0.05-0.15 us slower where its
// grid passes 256 workgroups (M = 96-192 at N = 3584-6144).
SkConfig choose_gemm(int64_t M, int64_t K, int64_t N, bool can_split, bool exact) {
    // us per quantisation group of K with n tiles on the fullest CU, n = 1, 2 and
    // each further one, fitted to sweeps at M = 300..8192, N = 1024..8192, K = 1024,
    // 2048 and 3584 (a call adds ~3 us): MI355X.
    struct Cost {
        SkConfig c;
        double one, two, more;
    };
    static const Cost kCosts[] = {
        {{128, 8, 3, 1}, 1.85, 3.8, 2.1},                      // 128 x 256
        {{128, 4, 2, 1, 1, 1, 1}, 1.17, 1.85, 1.05},           // 128 x 128, two workgroups per CU
        {{128, 4, 3, 1, 1, 1, 0}, 1.15, 2.25, 1.1},            // 128 x 128 through LDS
        {{64, 4, 2, 1, 1, 1, 1}, 0.8, 1.2, 0.6},               // 64 x 128, three
        {{64, 4, 3, 1}, 0.6, 1.2, 0.75},                       // 64 x 128, two k-parts
        {{64, 2, 3, 1}, 0.42, 0.75, 0.4},                      // 64 x 64
        {{32, 4, 3, 1}, 0.42, 0.65, 0.55},                     // 32 x 128
        {{32, 2, 3, 1}, 0.3, 0.47, 0.27},                      // 32 x 64
    };
    constexpr SkConfig kRound[] = {{128, 8, 3, 1}, {64, 4, 3, 1}, {64, 2, 3, 1}, {32, 4, 3, 1}, {32, 2, 3, 1}};
    const int64_t G = K / kGroup;
    auto finish = [&](SkConfig c) {
        if (G % 2 == 0 && (c.nwv == 2 || (c.nwv == 4 && G >= 8)))
            c.kg = c.kw = 2;
        c.wr = c.tm != 128;
        return c;
    };
    // one tile per workgroup and one workgroup per CU where a tile fits that
    // (200-256 tiles); exact operands (several weights) leave the 128 x 256 tile
    // out, whose registers they fill (gate + up M=1100 21.4 us and here 21.4-21.9, qkv + z 30.1 and 26.3)
    for (const SkConfig& c : kRound) {
        if (exact && c.nwv == 8) continue;
        const int64_t t = w4a16_sk_tiles(M, N, c);
        if (t >= 200 && t <= 256) return finish(c);
    }
    SkConfig c{32, 2, 3, 1};
    const int64_t tiles = w4a16_sk_tiles(M, N, c);
    if (tiles > 256) {
        SkConfig best = c;
        double least = 0;
        for (const Cost& k : kCosts) {
            if (exact && k.c.nwv == 8) continue;
            const int64_t tk = w4a16_sk_tiles(M, N, k.c), n = ceil_div(tk, 256);
            // (a round that leaves CUs idle leaves the others more bandwidth and clock:
            // 128 x 256 at K=3584 37.4 us with 72 tiles, 44.9 with 184, 52.8 with 240)
            const double t = n == 1 ? k.one * (0.6 + 0.4 * static_cast<double>(tk) / 256)
                                    : k.two + static_cast<double>(n - 2) * k.more;
            if (least == 0 || t < least) {
                least = t;
                best = k.c;
            }
        }
        // the 128 x 128 and three-per-CU shapes are what the table says
        return best.ns == 2 || (best.tm == 128 && best.nwv == 4) ? best : finish(best);
    }
    static_assert(kSkCounterBytes + 256 * 32 * 64 * 4 == MCV_W4A16_GEMM_WORKSPACE_MAX, "tiles * splits <= 256");
    if (!can_split) return finish(c);
    // the K split: the most ways within 256 workgroups that leave at least 7
    // groups per workgroup on average, cut in whole stages (two groups each
    // where K/128 is even)
    const int64_t U = G % 2 == 0 ? G / 2 : G;
    for (int64_t s = 2; s <= U && s <= 64; ++s)
        if (tiles * s <= 256 && G >= 7 * s) c.splits = static_cast<int>(s);
    return finish(c);
}

bool w4a16_parts_prefer_gemv(int64_t M, int64_t K, int64_t nslab, bool silu) {
    // The GEMV's grid at which the GEMM, a row tile or two of few workgroups and
    // without a K split, catches up: the shorter K, the larger; with an odd group
    // count, which leaves the GEMM one k-part, half as much again.  MI355X, us,
    // GEMV / GEMM: N=1024 + 1024 M=32 K=128 3.0 / 3.9; N=512 M=33 K=1152 4.4 / 7.0,
    // K=3072 7.8 / 9.2; gate + up N=512 M=64 K=256 3.8 / 4.5, M=33 K=3584 13.4 / 10.6.
    // Gate + up of up to 32 rows never runs the GEMM, so that its bits stay two GEMV
    // calls'.
    if (M < 8 || (silu && M <= 32)) return true;
    const int64_t limit = silu ? 192 + 131072 / K : 512 + 196608 / K;
    return M * nslab <= ((K / kGroup) % 2 != 0 && K > 1024 ? limit + limit / 2 : limit);
}

namespace {

// One weight, the few-row kernels aside.  Past 32 rows and K = 1024 the GEMV's
// grid has to stay near two workgroups per CU (one where the GEMM splits K); where
// an odd group count leaves the GEMM one k-part, any small output up to K = 1408
// and three workgroups per CU without a split.  MI355X, us, GEMV / GEMM, mean of
// weights cold and in cache: K=1152 N=512 M=64 4.5 / 6.9; K=1536 N=512 M=64 4.9 / 6.3,
// N=1000 M=40 6.1 / 6.7, K=1280 M=48 5.7 / 6.1, M=64 6.6 / 6.1; K=2048 N=1000 M=40 8.4 /
// 7.3 split, 7.5 unsplit; K=3584 12.4 / 7.9, 10.4; K=3968 N=512 M=33 9.4 / 8.3, 15.9.
bool prefers_gemv(int64_t M, int64_t K, int64_t N, bool can_split) {
    if (!small_output(M, N)) return false;
    if (M <= 32 || K <= 1024) return true;
    const int64_t grid = M * ceil_div(N, kSlab);
    if ((K / kGroup) % 2 != 0) {
        if (K <= 1408) return true;
        if (!can_split) return grid <= 768;
    }
    return grid <= (K <= 1536 ? 640 : can_split && K > 2304 ? 256 : 512);
}

// The few-row kernels by speed: ahead of the GEMV and, where that does not take
// the call, of the GEMM.
bool prefers_rows(int64_t M, int64_t K, int64_t N) {
    const int64_t nslab = ceil_div(N, kSlab);
    return w4a16_rows_pays(M, K, nslab, kOne) && (small_output(M, N) || !w4a16_rows_trail_gemm(M, K, nslab));
}

// The GEMV or (through launch_w4a16_gemv) the few-row kernels take this call.
// The few-row kernels and the GEMM need an aligned x and 32-bit offsets; a small
// output without them runs the GEMV, which needs neither.
bool takes_gemv(const void* x, int64_t M, int64_t K, int64_t N, bool can_split) {
    if (x == nullptr || M < 2 || K <= 0 || K % kGroup != 0 || N <= 0 || N > (int64_t(1) << 30)) return small_output(M, N);
    if (prefers_gemv(M, K, N, can_split)) return true;
    W4Parts parts{};
    parts.count = 1;
    parts.p[0].Npad = static_cast<int>(ceil_div(N, kSlab) * kSlab);
    if (prefers_rows(M, K, N) && w4a16_rows_ok(x, M, K, parts)) return true;
    return small_output(M, N) && (reinterpret_cast<uintptr_t>(x) % 16 != 0 || !w4a16_sk_fits(M, K, parts));
}

int check_gemm_args(const void* x, int64_t M, int64_t K, int64_t N, const void* qw, const void* scales,
                    const void* zeros, int zero_bias, const void* out, const char* who) {
    if (!x || !out || !qw || !scales || !zeros) return fail(MCV_ERR_INVALID_ARG, "%s: null pointer", who);
    if (zero_bias != 0 && zero_bias != 1) return fail(MCV_ERR_INVALID_ARG, "%s: zero_bias must be 0 or 1", who);
    if (K <= 0 || K % kGroup != 0 || K > (int64_t(1) << 24))
        return fail(MCV_ERR_SHAPE, "%s: K must be a positive multiple of 128 (K=%lld)", who, (long long)K);
    if (N <= 0 || N > (int64_t(1) << 30) || M <= 0 || M > (int64_t(1) << 30))
        return fail(MCV_ERR_SHAPE, "%s: bad M/N (M=%lld N=%lld)", who, (long long)M, (long long)N);
    if (reinterpret_cast<uintptr_t>(x) % 16 != 0) return fail(MCV_ERR_INVALID_ARG, "%s: x must be 16-byte aligned", who);
    return require_device();
}

// The MFMA GEMM with the configuration above; a split only into a caller's
// workspace that holds it (else unsplit).
int launch_w4a16_gemm_mfma(const void* x, int64_t M, int64_t K, int64_t N, const void* qw, const void* scales,
                           const void* zeros, int zero_bias, void* out, hipStream_t stream, void* ws,
                           int64_t ws_bytes) {
    int rc = check_gemm_args(x, M, K, N, qw, scales, zeros, zero_bias, out, "mcv_w4a16_gemm_mfma");
    if (rc != MCV_OK) return rc;
    SkConfig c = choose_gemm(M, K, N, ws != nullptr);
    if (c.splits > 1 && (ws_bytes < w4a16_sk_workspace_bytes(M, N, c) || (reinterpret_cast<uintptr_t>(ws) & 255) != 0))
        c = choose_gemm(M, K, N, false);
    return launch_w4a16_gemm_sk(x, M, K, N, qw, scales, zeros, zero_bias, out, c, ws, ws_bytes, stream);
}

thread_local std::string g_kernel_name;

}  // namespace

}  // namespace mcv

using namespace mcv;

extern "C" {

int mcv_w4a16_gemm_mfma(const void* x, int64_t M, int64_t K, int64_t N, const void* qw, const void* scales,
                        const void* zeros, int zero_bias, void* out, mcv_stream_t stream) {
    return launch_w4a16_gemm_mfma(x, M, K, N, qw, scales, zeros, zero_bias, out, static_cast<hipStream_t>(stream),
                                  nullptr, 0);
}

int64_t mcv_w4a16_gemm_workspace_bytes(int64_t M, int64_t K, int64_t N) {
    if (M < 1 || K <= 0 || N <= 0 || K % kGroup != 0 || prefers_gemv(M, K, N, true) || prefers_rows(M, K, N)) return 0;
    return w4a16_sk_workspace_bytes(M, N, choose_gemm(M, K, N, true));
}

int64_t mcv_stream_capture_id(mcv_stream_t stream) {
    if (stream == nullptr) return 0;                     // the default stream cannot be captured
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    if (hipStreamGetCaptureInfo(static_cast<hipStream_t>(stream), &status, &id) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return status == hipStreamCaptureStatusNone ? 0 : static_cast<int64_t>(id + 1);
}

// mcv_w4a16_gemm with a caller-owned workspace, which lets the MFMA path
// split K across workgroups where the tile grid is small.
int mcv_w4a16_gemm_ws(const void* x, int64_t M, int64_t K, int64_t N, const void* qw, const void* scales,
                      const void* zeros, int zero_bias, void* out, void* workspace, int64_t workspace_bytes,
                      mcv_stream_t stream) {
    if (takes_gemv(x, M, K, N, workspace != nullptr))
        return launch_w4a16_gemv(x, M, K, N, qw, scales, zeros, zero_bias, out, static_cast<hipStream_t>(stream));
    return launch_w4a16_gemm_mfma(x, M, K, N, qw, scales, zeros, zero_bias, out, static_cast<hipStream_t>(stream),
                                  workspace, workspace_bytes);
}

// Decode-sized M streams the weights once per row through the GEMV; larger M
// goes to the MFMA kernel, which reuses each dequantised operand across rows.
int mcv_w4a16_gemm(const void* x, int64_t M, int64_t K, int64_t N, const void* qw, const void* scales,
                   const void* zeros, int zero_bias, void* out, mcv_stream_t stream) {
    if (takes_gemv(x, M, K, N, false))
        return launch_w4a16_gemv(x, M, K, N, qw, scales, zeros, zero_bias, out, static_cast<hipStream_t>(stream));
    return launch_w4a16_gemm_mfma(x, M, K, N, qw, scales, zeros, zero_bias, out, static_cast<hipStream_t>(stream),
                                  nullptr, 0);
}

const char* mcv_w4a16_gemm_kernel_name(int64_t M, int64_t K, int64_t N, int with_workspace) {
    char buf[160];
    if (M < 1 || K <= 0 || N <= 0 || K % kGroup != 0) {
        g_kernel_name = "none (bad shape)";
    } else if (prefers_rows(M, K, N)) {
        g_kernel_name = w4a16_rows_name(M, K, ceil_div(N, kSlab), kOne);
    } else if (prefers_gemv(M, K, N, with_workspace != 0)) {
        std::snprintf(buf, sizeof(buf), "w4a16_gemv_kernel<%d, 1, 0> (grid %lld x %lld)",
                      gemv_ksplit(K / kGroup, ceil_div(N, kSlab) * M), (long long)ceil_div(N, kSlab), (long long)M);
        g_kernel_name = buf;
    } else {
        const SkConfig c = choose_gemm(M, K, N, with_workspace != 0);
        g_kernel_name = w4a16_sk_name(c, kOne, w4a16_sk_tiles(M, N, c) * c.splits);
        if (!w4a16_sk_config_valid(M, K, N, c)) g_kernel_name += " NOT VALID";
    }
    return g_kernel_name.c_str();
}

const char* mcv_w4a16_parts_kernel_name(int64_t M, int64_t K, int64_t nslab, int n_parts, int gate_up) {
    const int kind = gate_up ? kSilu : (n_parts == 1 ? kOne : kParts);
    if (M < 1 || K <= 0 || K % kGroup != 0 || nslab <= 0 || n_parts < 1 || n_parts > kMaxParts || (gate_up && n_parts != 2)) {
        g_kernel_name = "none (bad shape)";
    } else if (w4a16_rows_pays(M, K, nslab, kind)) {
        g_kernel_name = w4a16_rows_name(M, K, nslab, kind);
    } else if (w4a16_parts_prefer_gemv(M, K, nslab, gate_up != 0)) {
        g_kernel_name = gate_up ? "w4a16_gate_up_silu_kernel" : "w4a16_gemv_multi_kernel";
    } else {
        g_kernel_name = w4a16_sk_name(choose_gemm(M, K, (gate_up ? 2 : 1) * nslab * kSlab, false, true),
                                      gate_up ? kSilu : kParts, 0);
    }
    return g_kernel_name.c_str();
}

}  // extern "C"
