// rows_rule.hpp -- which kernel solves with a factor of order <= 512: the row
// solver (trsv_rows.hpp) or the tile solver (tile_solve.hpp); and how a blocked
// solve of a larger order is launched.  Same operations per row, same bits.
// Host code, no HIP.
//
// The tile solver works on 16 right-hand sides and whole 32-row blocks whatever
// the call has; the row solver on what is there, in smaller workgroups that
// keep more systems in flight, but slower for one system.  So rows win in large
// batches of few right-hand sides, the earlier the less of the last 32-row
// block the order fills.
//
// The lines come from timing both at about 110 orders and 25 batches per type
// and op.  Over those the chosen kernel is within 1.15 of the faster one (but for
// launches of a few us, and FP32 potrs of n <= 2 with 9 to 16 right-hand sides,
// 1.3) and mostly the faster one; the wrong one costs up to 3.5 times.
#pragma once

#include <cstddef>
#include <cstdint>

namespace rsa
{

// One line of a table: for orders up to `order`, beyond how many systems per
// CU rows are taken with 1, 2..4 and 5..8 right-hand sides.
struct RowsFrom
{
    int order;
    int one, few, more;
};
constexpr int NEVER = 1 << 23; // times ROWS_CUS: more than a batch holds
constexpr int ROWS_CUS = 256;

template <size_t K>
inline bool rows_win(const RowsFrom (&table)[K], int n, int nrhs, int bc)
{
    for(const RowsFrom& l : table)
        if(n <= l.order)
        {
            const int per_cu = nrhs <= 1 ? l.one : nrhs <= 4 ? l.few : nrhs <= 8 ? l.more : NEVER;
            return bc > int64_t(ROWS_CUS) * per_cu;
        }
    return false;
}

// getrs, 64 < n <= 512.  On both sides of the lines, rows against tiles
// in us (order x systems, right-hand sides):
//   op N, FP64: 65 x 512, 1: 31 against 34; 65 x 2048, 1: 42 against 77; 128 x
//     8192, 4: 340 against 416; 256 x 1024, 4: 165 against 177; 304 x 2904, 8:
//     1012 against 1109; but 96 x 512, 4: 44 against 34
//   op N, FP32: 65 x 512, 1: 28 against 34; 128 x 8192, 4: 203 against 222;
//     304 x 640, 4: 129 against 163; but 304 x 1024, 4: 229 against 198
//   op T, FP64: 97 x 8192, 4: 360 against 403; 129 x 1024, 1: 83 against 108;
//     but 128 x 8192, 4: 498 against 439
//   op T, FP32: 65 x 8192, 1: 125 against 198; 83 x 8192, 4: 173 against 202;
//     but 96 x 8192, 4: 256 against 211
// In op T a row's entries are a column of A, which a thread reads alone: there
// rows win only where the last 32-row block holds few rows.
template <typename T>
inline bool getrs_by_rows(bool trans, int n, int nrhs, int bc)
{
    static constexpr RowsFrom N64[] = {{72, 1, 3, NEVER},
                                       {128, 2, 4, NEVER},
                                       {256, 2, 2, NEVER},
                                       {512, 1, 1, 3}};
    static constexpr RowsFrom T64[] = {{76, 2, 4, NEVER},
                                       {104, 4, 4, NEVER},
                                       {128, NEVER, NEVER, NEVER},
                                       {152, 2, 2, NEVER}};
    static constexpr RowsFrom N32[] = {{84, 0, 1, NEVER},
                                       {96, 1, 6, NEVER},
                                       {108, 1, 1, NEVER},
                                       {128, 1, 8, NEVER},
                                       {256, 2, 4, NEVER},
                                       {512, 2, 2, 8}};
    static constexpr RowsFrom T32[] = {{70, 0, 1, NEVER},
                                       {84, 1, 8, NEVER},
                                       {96, NEVER, NEVER, NEVER},
                                       {102, 1, 8, NEVER},
                                       {128, NEVER, NEVER, NEVER},
                                       {136, 4, 4, NEVER}};
    if(sizeof(T) == 8)
        return trans ? rows_win(T64, n, nrhs, bc) : rows_win(N64, n, nrhs, bc);
    // FP32 beyond n = 256: a CU holds two workgroups of tiles and three of
    // rows, so rows win between two and three systems per CU for any number of
    // right-hand sides up to 8, and tiles again up to four, where both take
    // two rounds
    if(!trans && n > 256 && nrhs <= 8 && bc > 2 * ROWS_CUS && bc <= 4 * ROWS_CUS)
        return bc <= 3 * ROWS_CUS;
    return trans ? rows_win(T32, n, nrhs, bc) : rows_win(N32, n, nrhs, bc);
}

// potrs, n <= 512.  On both sides of the lines, rows against tiles in us,
// lower storage (order x systems, right-hand sides):
//   FP64: 1 x 65536, 1: 154 against 533; 8 x 4096, 4: 32 against 44; 32 x 2048,
//     1: 22 against 28; 64 x 4096, 1: 64 against 86; 129 x 4096, 4: 351 against
//     406; 257 x 1280, 4: 436 against 458; but 32 x 1024, 1: 19 against 16; 64 x
//     4096, 4: 116 against 86; 512 x 1024, 4: 797 against 748
//   FP32: 1 x 65536, 1: 100 against 307; 8 x 4096, 4: 19 against 31; 33 x 4096,
//     4: 42 against 58; 65 x 3072, 4: 63 against 78; 129 x 3072, 1: 137 against
//     173; but 64 x 1536, 4: 44 against 31; 96 x 1024, 1: 44 against 36; 128 x
//     2048, 4: 94 against 71
template <typename T>
inline bool potrs_by_rows(int n, int nrhs, int bc)
{
    static constexpr RowsFrom R64[] = {{4, 0, 1, 6},
                                       {8, 1, 4, 6},
                                       {20, 1, 6, NEVER},
                                       {24, 4, 16, NEVER},
                                       {32, 6, NEVER, NEVER},
                                       {47, 3, 6, NEVER},
                                       {52, 4, 32, NEVER},
                                       {64, 6, NEVER, NEVER},
                                       {88, 2, 4, NEVER},
                                       {96, 4, 16, NEVER},
                                       {108, 2, 4, NEVER},
                                       {128, 4, 12, NEVER},
                                       {151, 2, 2, NEVER},
                                       {224, 2, 12, NEVER},
                                       {256, 12, NEVER, NEVER},
                                       {288, 1, 3, NEVER},
                                       {384, 1, 6, NEVER},
                                       {512, 12, NEVER, NEVER}};
    static constexpr RowsFrom R32[] = {{5, 0, 0, 4},
                                       {8, 0, 0, 8},
                                       {12, 0, 4, 12},
                                       {20, 0, 8, NEVER},
                                       {26, 4, 12, NEVER},
                                       {32, 4, NEVER, NEVER},
                                       {44, 0, 8, NEVER},
                                       {52, 4, 12, NEVER},
                                       {64, 12, NEVER, NEVER},
                                       {68, 1, 4, NEVER},
                                       {84, 4, 8, NEVER},
                                       {96, 8, NEVER, NEVER},
                                       {108, 6, 8, NEVER},
                                       {128, 32, NEVER, NEVER},
                                       {136, 4, 4, NEVER},
                                       {256, 32, NEVER, NEVER}};
    return sizeof(T) == 8 ? rows_win(R64, n, nrhs, bc) : rows_win(R32, n, nrhs, bc);
}

// Blocked solves (n > 512) of `tiles` tiles of 128 rows: whether the updates get
// launches of their own (gemm_sub_kernel, which shares its operands through
// LDS) and the solves up to 64 (FP64) or 128 right-hand sides per workgroup.
// Where there is work for the whole chip, a step is bound by the operands that
// every 32 right-hand sides read again, not by the launch that this costs.
// Same sums, same bits.
//
// Step by step against own launches, in ms (a launch per 64 rows with updates
// of their own, a thread per column, took 2.62, 4.98 and 1.45 in the first
// three): FP64 n = 513 x 300, op T, 100 right-hand sides 3.37 against 1.52; n =
// 800 x 64, op T, 600 6.53 against 2.62; n = 513 x 150, op N, 33 0.93 against
// 0.46; FP32 n = 800 x 64, op T, 600 4.58 against 1.66; but FP64 n = 513 x 1, op
// N, 2000 0.31 against 0.38, FP32 n = 2500 x 1, op N, 2000 1.58 against 2.03, n =
// 600 x 300, op N, 1 0.34 against 0.39, n = 1100 x 64, op T, 1 0.45 against 0.51.
// (FP32 takes half the time for the same steps, few systems share less.)
template <typename T>
inline bool trsm_many(bool trans, int tiles, int nrhs, int bc)
{
    const int64_t blocks = int64_t(tiles) * ((int64_t(nrhs) + 31) / 32) * bc;
    const bool few = bc < 16;
    if(sizeof(T) == 8)
        return blocks > (trans && nrhs > 16 ? 400 : !trans && few ? 800 : 600);
    if(trans)
        return blocks > (few ? 800 : nrhs <= 16 ? 600 : 400);
    return blocks > (few ? 2500 : nrhs <= 16 ? 2000 : 1400);
}

} // namespace rsa
