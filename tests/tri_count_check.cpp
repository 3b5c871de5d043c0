// Host check of tri_tile_count (clgpu_amd/csrc/level3_tiles.hpp) against the tiles that
// tri_tile_row lists, for outputs of any shape with both triangles whole and, square, in
// bands. Exits non-zero on a mismatch. Built and run by tests/test_tri_count_cpu.py.
#include "level3_tiles.hpp"
#include "kernel_abi.h"
#include <cstdio>
int main()
{
    const int sizes[] = {1, 31, 32, 33, 64, 100, 255, 256, 257, 500, 512, 513, 1000, 3008};
    const int tiles[][2] = {{32, 32}, {64, 64}, {128, 128}, {256, 256}, {256, 128}, {128, 256}, {128, 64}, {64, 128}};
    long bad = 0, cases = 0;
    for (int M : sizes)
        for (int N : sizes)
            for (auto& t : tiles)
                for (int tri : {ICL_TRI_LOWER, ICL_TRI_UPPER})
                    for (int band : {0, (int)ICL_TRI_OFF_BAND, (int)ICL_TRI_BAND}) {
                        if (band && M != N) continue;
                        const int tiles_n = (N + t[1] - 1) / t[1];
                        long count = 0;
                        for (int tm = 0; tm < (M + t[0] - 1) / t[0]; ++tm) {
                            int lo, cnt;
                            icl::tri_tile_row(tri | band, tm, tiles_n, t[0], t[1], lo, cnt);
                            count += cnt;
                        }
                        ++cases;
                        if (count == icl::tri_tile_count(M, N, tri | band, t[0], t[1])) continue;
                        if (++bad < 10) std::printf("%d x %d, tile %d x %d, %d: %ld\n", M, N, t[0], t[1], tri | band, count);
                    }
    std::printf("%ld cases, %ld mismatches\n", cases, bad);
    return bad != 0;
}
