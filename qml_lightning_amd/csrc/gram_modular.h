// Sizes, workspace and tile order of the modular Gram product (gram_modular.hip), as plain C++ so that a test on
// the host can walk them.
#pragma once
#include <stddef.h>
#include "gram_tiles.h"     // QMLL_HD

// moduli, and gamma: columns are scaled to a norm in (2^(gamma-1), 2^gamma].  Products over rows that are large or small in all columns
// alike, as training rows are, lose more to the rounding of an fp64 sum than to operands rounded to 2^-54 of the norm; the rows of a
// Cholesky factor do not (entries far below their column's norm, sums that nearly vanish), and need the four bits that one modulus
// more gives.
constexpr int GRAM_MODULI = 14, CHOL_MODULI = 15;
constexpr int modular_gamma(int moduli) { return moduli == 14 ? 54 : 58; }
constexpr int NORM_ROWS = 512;     // rows per partial sum of the column norms
constexpr int MODULAR_MIN_ROWS = 768;
constexpr int MODULAR_CUS = 256;
// residues are below 128 in magnitude and a sum must stay below 2^30
constexpr int MODULAR_MAX_ROWS = 65536;

// number t of a 256 x 256 tile on or above the diagonal of nt x nt: bands of four tile rows, the tiles of a band
// column by column, so that 32 consecutive tiles share 4 + 8 panels
QMLL_HD void modular_tile(int t, int nt, int& ti, int& tj) {
    int r = 0;
    for (;;) {
        const int h = nt - r < 4 ? nt - r : 4;
        const int tri = h * (h + 1) / 2, n = tri + 4 * (nt - r - h);
        if (t < n || h < 4) {
            if (t < tri) {
                int c = 0;
                while (t > c) { t -= c + 1; ++c; }      // column c of the triangle holds c + 1 tiles
                ti = r + t;
                tj = r + c;
            } else {
                ti = r + (t - tri) % 4;
                tj = r + 4 + (t - tri) / 4;
            }
            return;
        }
        t -= n;
        r += 4;
    }
}

// the same for the first `rows` tile rows of the nt x nt upper triangle, column by column
QMLL_HD void modular_band_tile(int t, int rows, int& ti, int& tj) {
    const int tri = rows * (rows + 1) / 2;
    if (t < tri) {
        int c = 0;
        while (t > c) { t -= c + 1; ++c; }
        ti = t;
        tj = c;
    } else {
        ti = (t - tri) % rows;
        tj = rows + (t - tri) / rows;
    }
}
QMLL_HD int modular_band_tiles(int rows, int nt) { return rows * (rows + 1) / 2 + rows * (nt - rows); }

// row ranges a product of nk 64-row steps is cut into, so that few tiles fill the CUs: a workgroup costs its steps and about 12
// more for filling the stages and for its residues
inline int modular_pieces(int moduli, long long tiles, int nk, int most) {
    int pieces = 1;
    double best = 0.0;
    for (int c = 1; c <= 8 && c * tiles <= most && (c == 1 || nk >= 4 * c); ++c) {
        const long long items = tiles * moduli * c;
        const double cost = (double)((items + MODULAR_CUS - 1) / MODULAR_CUS) * ((nk + c - 1) / c + 12.0);
        if (c == 1 || cost < 0.97 * best) {
            best = cost;
            pieces = c;
        }
    }
    return pieces;
}
constexpr int modular_tiles_at_once(int moduli) { return (int)((1ll << 30) / (moduli * 65536ll)); }     // results of at most 1 GiB

struct ModularPlan {
    int Fp;            // features rounded up to whole tiles
    int nt, tiles;     // tiles per edge, tiles on or above the diagonal
    int rows;          // rows per pass
    int range;         // tiles per launch
    int pieces;        // row ranges a tile's product is cut into
    int max_parts;
    size_t expo, scale, parts, planes, results, bytes;     // offsets in the workspace, and its size
};

inline ModularPlan modular_plan(int M, int F) {
    ModularPlan p;
    p.nt = (F + 255) / 256;
    p.Fp = p.nt * 256;
    p.tiles = p.nt * (p.nt + 1) / 2;
    // planes of at most 8 GiB, results of at most 1 GiB at a time
    long long rows = (8ll << 30) / ((long long)GRAM_MODULI * p.Fp) / 128 * 128;
    if (rows > MODULAR_MAX_ROWS) rows = MODULAR_MAX_ROWS;
    if (rows < 128) rows = 128;
    const long long passes = (M + rows - 1) / rows;
    p.rows = (int)(((M + passes - 1) / passes + 127) / 128 * 128);
    const int launches = (p.tiles + modular_tiles_at_once(GRAM_MODULI) - 1) / modular_tiles_at_once(GRAM_MODULI);
    p.range = (p.tiles + launches - 1) / launches;
    p.pieces = modular_pieces(GRAM_MODULI, p.range, p.rows / 64, modular_tiles_at_once(GRAM_MODULI));
    p.max_parts = (p.rows + NORM_ROWS - 1) / NORM_ROWS;
    auto up = [](size_t v) { return (v + 1023) / 1024 * 1024; };
    p.expo = 1024;
    p.scale = p.expo + up((size_t)p.Fp * 4);
    p.parts = p.scale + up((size_t)p.Fp * 8);
    p.planes = p.parts + up((size_t)2 * p.max_parts * F * 8);
    p.results = p.planes + up((size_t)GRAM_MODULI * p.rows * p.Fp);
    p.bytes = p.results + (size_t)p.pieces * GRAM_MODULI * p.range * 65536;
    return p;
}
