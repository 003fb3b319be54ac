// The scale and zero loads of the wide few-row W4A16 kernel (w4a16_rows.hip),
// on the CPU: every lane of every unit and group either reads inside the tensor
// or is refused by the buffer range check, which covers the vector offset
// alone, and the lanes whose values are used read their own column.
#include "w4a16_rows.h"

#include <cstdio>

using namespace mcv;

namespace {

int bad = 0;

// One load of `size` bytes; want < 0: a lane whose value is not used.
void load(const char* what, int64_t bytes, uint32_t voff, int64_t base, int size, int64_t want, int n0, int lane, int cb) {
    const bool clipped = static_cast<int64_t>(voff) + size > bytes;
    const int64_t at = base + voff;
    if (!clipped && at + size > bytes) {
        if (bad++ < 8)
            std::printf("%s: unit of %d columns at %d, lane %d reads bytes %lld.. of %lld\n", what, 16 * cb, n0, lane,
                        static_cast<long long>(at), static_cast<long long>(bytes));
    } else if (want >= 0 && (clipped || at != want)) {
        if (bad++ < 8)
            std::printf("%s: unit at %d, lane %d reads byte %lld, wants %lld\n", what, n0, lane,
                        static_cast<long long>(at), static_cast<long long>(want));
    }
}

}  // namespace

int main() {
    for (int cb : {2, 4})
        for (int Npad : {64, 128, 192, 25600, 51328})
            for (int G : {1, 2, 8}) {
                const int64_t sbytes = int64_t(G) * Npad * 2, zbytes = int64_t(G) * (Npad / 8) * 4;
                for (int n0 = 0; n0 < Npad; n0 += 16 * cb)
                    for (int g = 0; g < G; ++g)
                        for (int lane = 0; lane < 64; ++lane) {
                            const bool used = lane < 16 * cb;
                            load("scales", sbytes, wide_scale_offset(lane, cb), wide_scale_base(g, Npad, n0), 2,
                                 used ? (int64_t(g) * Npad + n0 + lane) * 2 : -1, n0, lane, cb);
                            load("zeros", zbytes, wide_zero_offset(lane, cb), wide_zero_base(g, Npad, n0), 4,
                                 used ? (int64_t(g) * (Npad / 8) + (n0 + lane) / 8) * 4 : -1, n0, lane, cb);
                        }
            }
    std::printf(bad ? "%d bad loads\n" : "ok\n", bad);
    return bad ? 1 : 0;
}
