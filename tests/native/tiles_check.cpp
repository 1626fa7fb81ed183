// Host check of the spread tile shapes the library accepts (spread_impl.h,
// spread_tile_ok) against what the kernels can hold, for every shape up to
// 16 x 16, every even fine grid up to 4096 cells, both precisions, real and
// complex strengths:
//   the x FFT of the kernel the tile runs on (2E cells per thread in the
//   narrow kernel, E in the wide one; rows in pairs where they are real),
//   the queue entries of a queued FP32 tile's passes, one pass in FP64, and
//   passes that cover every row.
// Prints "ok" or the first failure.
#include <cstdio>

#include "spread_impl.h"

using namespace mpsq;

template <typename R> static int check(bool real)
{
    const bool f32 = sizeof(R) == 4;
    int most = 0;
    for (int n1 = 4; n1 <= SpreadCfg<R>::E * SpreadCfg<R>::NT; n1 += 2)
        for (int by = 1; by <= 16; ++by)
            for (int bz = 1; bz <= 16; ++bz) {
                if (!spread_tile_ok<R>(by, bz, n1, real)) continue;
                const int rows = by * bz;
                const bool pairs = real && (!f32 || rows % 2 == 0);
                auto ffts = [&](int r) { return pairs ? (r + 1) / 2 : r; };
                const int G = spread_group_rows<R>(by, bz, n1, pairs), np = rows / G;
                const char *what = nullptr;
                if (f32 && ffts(rows) * n1 > 2 * NarrowCfg::E * NarrowCfg::NT) what = "narrow x FFT";
                if (G > 1 && ffts(G) * n1 > SpreadCfg<R>::E * SpreadCfg<R>::NT) what = "wide x FFT";
                if (G * np != rows || (G >= by ? (G % by || bz % (G / by)) : by % G)) what = "passes cover the tile";
                if (np > (f32 ? MAX_WIDE_PASSES : 1)) what = "passes";
                if (what) {
                    std::printf("FAIL %s: fp%d real %d n1 %d tile %d x %d\n", what, f32 ? 32 : 64, (int)real, n1, by, bz);
                    return 1;
                }
                most = np > most ? np : most;
            }
    // the shapes that tests and programs ask for stay accepted
    if (!spread_tile_ok<R>(1, 1, 512, real) || !spread_tile_ok<R>(4, 2, 512, real) || !spread_tile_ok<R>(5, 3, 128, real)) {
        std::printf("FAIL refused\n");
        return 1;
    }
    return 0;
}

int main()
{
    if (check<float>(false) || check<float>(true) || check<double>(false) || check<double>(true)) return 1;
    std::printf("ok\n");
    return 0;
}
