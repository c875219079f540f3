// gemm_slices.h — which tiles of the prompt GEMM's grid each XCD takes.
//
// The grid of mt vector tiles x nt row tiles is cut into ga x (8 / ga) slices
// of mts x nts tiles, one per XCD.  A slice per vector tile keeps the most of
// the operand in each L2 (4 MiB; a tile's operand is 16 KiB per block quad), but
// where the tiles do not divide, the last slices are short or empty: six vector
// tiles in four slices of two leave two XCDs without work.  So fewer vector
// slices are taken when they shorten the fullest XCD by more than a fifteenth,
// an eighth where its operand then outgrows the L2, counted once in work-groups
// and once in rounds of its CUs (a CU with one work-group more than the others
// holds them up); for a sixteenth, some products were 5 % slower.
// Q4_0, us in eight slices (one per vector tile up to eight) / as taken here:
// 22016 rows x 2048 inputs, 160 vectors 62.6 / 47.3 (one slice), 188 59.9 /
// 53.5 (two), 300 106 / 70.9 (two), 400 104 / 90 (one), 600 156 / 133 (four),
// 1600 343 / 325 (four; two 341); 2048 x 11008, 300 61.6 / 46.9 (two); 3072 x
// 2048, 300 26.6 / 19.6 (two), 1300 53.4 / 47.1 (two), 1800 61.4 (eight, taken;
// one 64.3).
#pragma once

struct GemmSlices {
    int ga = 1, mts = 1, nts = 1;
};

// ks k ranges of kq block quads; cus: CUs of an XCD.
static inline GemmSlices gemm_slices(int mt, int nt, int ks, int kq, int cus)
{
    GemmSlices s;
    long best = 0;
    for (int ga = 8; ga >= 1; ga >>= 1) {
        if (ga > mt && ga > 1) continue;
        const int mts = (mt + ga - 1) / ga, nts = (nt + 8 / ga - 1) / (8 / ga);
        const long wgs = (long)mts * nts * ks, cost = wgs + (wgs + cus - 1) / cus * cus;
        const bool fits = (long)mts * kq <= 256;
        if (best && (fits ? 15 * cost >= 14 * best : 8 * cost >= 7 * best)) continue;
        best = cost;
        s.ga = ga;
        s.mts = mts;
        s.nts = nts;
    }
    return s;
}
