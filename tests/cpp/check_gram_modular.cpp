// Walks the tile order and the plan of the modular Gram product on the CPU: every tile on or above the diagonal once,
// row passes and tile ranges that cover everything, parts of the workspace that do not overlap, sums that stay below
// 2^30 and row ranges that are even.
#include <cstdio>
#include <vector>
#include "gram_modular.h"

int main() {
    for (int nt = 1; nt <= 140; ++nt) {
        std::vector<int> seen((size_t)nt * nt, 0);
        for (int t = 0; t < nt * (nt + 1) / 2; ++t) {
            int ti = -1, tj = -1;
            modular_tile(t, nt, ti, tj);
            if (ti < 0 || ti > tj || tj >= nt || seen[(size_t)ti * nt + tj]++) {
                std::printf("nt=%d t=%d: tile (%d,%d)\n", nt, t, ti, tj);
                return 1;
            }
        }
    }
    for (int nt = 1; nt <= 70; ++nt)                 // the first tile rows only: each of their tiles once
        for (int rows = 1; rows <= (nt < 3 ? nt : 3); ++rows) {
            std::vector<int> seen((size_t)nt * nt, 0);
            int expect = 0;
            for (int i = 0; i < rows; ++i) expect += nt - i;
            bool ok = expect == modular_band_tiles(rows, nt);
            for (int t = 0; t < expect; ++t) {
                int ti = -1, tj = -1;
                modular_band_tile(t, rows, ti, tj);
                ok = ok && ti >= 0 && ti < rows && ti <= tj && tj < nt && !seen[(size_t)ti * nt + tj]++;
            }
            if (!ok) {
                std::printf("band of %d tile rows of %d\n", rows, nt);
                return 1;
            }
        }
    const int Ms[] = {1, 64, 127, 128, 129, 768, 1000, 5001, 32000, 65536, 65537, 200000, 1000003};
    const int Fs[] = {1, 24, 255, 256, 257, 512, 1000, 4096, 8200, 16384, 32768, 65536, 131072};
    for (int M : Ms)
        for (int F : Fs) {
            const ModularPlan p = modular_plan(M, F);
            bool ok = p.Fp >= F && p.Fp % 256 == 0 && p.Fp == p.nt * 256;
            ok = ok && p.rows % 128 == 0 && p.rows > 0 && p.rows <= MODULAR_MAX_ROWS;
            ok = ok && (size_t)GRAM_MODULI * p.rows * p.Fp <= (8ull << 30) + (size_t)GRAM_MODULI * 128 * p.Fp;
            ok = ok && p.range > 0 && p.range <= p.tiles && p.pieces >= 1 && p.pieces <= 8;
            ok = ok && (size_t)p.pieces * GRAM_MODULI * p.range * 65536 <= (1ull << 30);
            ok = ok && p.expo >= 4 && p.scale >= p.expo + 4 * (size_t)p.Fp && p.parts >= p.scale + 8 * (size_t)p.Fp;
            ok = ok && p.planes >= p.parts + 16 * (size_t)p.max_parts * F && p.max_parts * (long long)NORM_ROWS >= p.rows;
            ok = ok && p.results >= p.planes + (size_t)GRAM_MODULI * p.rows * p.Fp && p.planes % 1024 == 0 && p.results % 1024 == 0;
            ok = ok && p.bytes == p.results + (size_t)p.pieces * GRAM_MODULI * p.range * 65536;
            ok = ok && 128ll * 128 * p.rows <= (1ll << 30);
            if (!ok) {
                std::printf("plan of M=%d F=%d\n", M, F);
                return 1;
            }
        }
    std::printf("ok\n");
    return 0;
}
