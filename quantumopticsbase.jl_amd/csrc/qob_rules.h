// Choices between kernels by sizes alone, in plain C++ (tests/rules_check.cpp
// compiles them without a GPU).
#pragma once
#include <cstdint>

namespace qob {

// Whether one launch does an m x n matrix on a vector (k_zgemv_one: 16 rows
// and all columns per workgroup) or columns are split over workgroups and
// their sums added by a second launch, which costs more than the better use
// of the CUs gains while both sides are short.  One / two launches, us:
// ComplexF32 (1536, 1536) 7.2 / 7.8, (64, 1024) 5.3 / 8.1, (64, 2048) 8.7 /
// 7.0, (64, 65536) 228 / 20, (1, 2^20) 3553 / 43; ComplexF64 (1536, 1536) 9.4 /
// 8.9, (200, 1024) 5.7 / 8.1, (200, 2048) 9.3 / 7.0, (512, 16384) 67 / 25;
// more rows: (2013, 2013) in ComplexF32 11.4 / 10.7.
inline bool zgemv_in_one(int64_t m, int64_t n) { return m <= 1536 && n <= 1536; }

// y = A^T x for a column-major k x m A, a wave per column (k_zgemv_t): loads in
// flight per lane and elements per load.  Four loads hide the latency of
// columns that come from the caches; a matrix that streams from HBM has enough
// in flight with one where it also has the waves (n x n, one / four, us:
// ComplexF64 2048 13.5 / 10.9, 3009 21.9 / 21.5, 3300 25.6 / 26.9, 4096 38.8 /
// 40.7, 6143 91.6 / 102.4; ComplexF32, half as many loads per column, 2048 6.9 /
// 5.1, 2896 11.3 / 11.4, 3300 13.7 / 14.9, 6143 51.2 / 54.2; fewer waves in
// ComplexF64: (16384, 512) 80 / 29, (16384, 2048) 146 / 95, (16384, 3072) 164 /
// 141, (2^20, 16) 5980 / 1930).  Columns that end within the first of four
// loads leave the others idle, and in ComplexF32 half of the lanes too: (16,
// 65536) four loads of two elements 13.0 us (31.5 with every load issued at the
// column's end), one of two 10.6, one of one 9.8; (128, 262144) 56.1, 48.8, 54.9.
struct GemvT {
    int loads, elems;
};
inline GemvT zgemv_t_form(bool c64, int64_t k, int64_t m) {
    const double mib = (double)k * m * (c64 ? 16 : 8) / (1 << 20);
    GemvT f{4, c64 ? 1 : 2};
    if (mib > (c64 ? 160 : 64) && m > 3072) f.loads = 1;
    if (!c64 && k < 256) f.loads = 1;
    if (!c64 && k < 128) f.elems = 1;
    return f;
}

// log2 of the tile of ncols states of nbits bits (k_qubit; a reduction has one
// column).  A larger tile reads fewer partner tiles from memory, a smaller one
// gives more workgroups and waits less in each: 2^10 states while the tiles
// are few or the partners are read from the caches.  2^10 / 2^11 / 2^12 tiles of
// chains, us.  ComplexF32, 2^11 above 2^20 elements: 18 sites 6.6 / 7.7 / 9.6,
// 12 sites of 256 columns (2^20) 7.9 / 8.2 / 8.1 and of 1024 25.7 / 19.0 / 20.2,
// 16 sites of 256 111 / 79 / 83.  ComplexF64, 2^12 from about 2^23 elements on, where
// input and output leave the Infinity Cache, later for shorter states, which
// have fewer partners: 18 sites of 16 columns 38.8 / 40.6 / 42.0, of 32 (2^23) 78.6 /
// 79.0 / 71.5, of 256 955 / 757 / 627; 16 sites of 128 62.5 / 60.3 / 64.4, of 256
// (2^24) 124 / 112 / 116; 14 sites of 1024 106 / 100 / 110, of 4096 587 / 544 / 513;
// 13 sites of 4096 (2^25) 251 / 247 / 240; expect of 25 sites 952 / 910 / 910.
// The first of two passes has fewer partners: 23 sites 120 / 127 / 129, 24 of 2
// columns (2^25) 666 / 658 / 624.
inline int qubit_state_tbits(int nbits, bool c64, int64_t ncols, bool two_pass) {
    int lg = nbits;  // log2 of all elements, rounded down
    while (ncols > 1) {
        ncols >>= 1;
        ++lg;
    }
    if (!c64) return nbits > 10 && lg > 20 ? 11 : 10;
    const int from = two_pass || nbits < 16 ? 25 : nbits < 18 ? 24 : 23;
    return nbits >= 12 && lg >= from ? 12 : 10;
}

// Rows of a tile of a site-group pass over n1 >= 16 rows of P elements in n3
// blocks (k_ltany): runs of 128 bytes.
// Too few tiles for the CUs: shorter runs, down to two rows, as long as the tiles
// stay one round (from the right on a rho that the MALL holds anyway; ComplexF64 /
// ComplexF32 (14, 9, 8): 8 / 16 rows 22.1 / 26.7 us, 4 rows and 252 tiles 17.7 /
// 18.5, 2 rows and 504 tiles 26.4 / 24.8).
// Small blocks: longer runs, up to 32 KiB of tile, while every CU still has a
// tile (from the right, us: ComplexF32 without the first site of (16, 4, 4), 1000
// rows, 256-row tiles 15.0, 64-row ones 9.7; (20, 3), 2469 rows, 64 / 32 / 16 rows
// 15.4 / 7.8 / 7.8; ComplexF64 the outer two of (3, 6, 7), 2298 rows, 16 / 8 rows
// 10.8 / 9.1).
inline int any_rows(bool c64, int64_t n1, int64_t P, int64_t n3, int64_t ncu) {
    const int64_t wmin = c64 ? 8 : 16, es = c64 ? 16 : 8;
    auto tiles = [&](int64_t w) { return (n1 + w - 1) / w; };
    int64_t W = wmin;
    while (W > 2 && 2 * tiles(W) * n3 <= ncu) W /= 2;
    if (W == wmin)
        while (W < 256 && W < n1 && 2 * W * P * es <= 32 * 1024 && tiles(2 * W) * n3 >= ncu)
            W *= 2;
    return (int)W;
}

// Whether blocks of P elements are too long for one site-group pass of so many
// modes over few rows: with tiles of two rows one tile's modes are the pass's
// time, and runs are 32 bytes, 16 in ComplexF32.  From the right, chain of modes /
// one group of all factors, us, factors at their sites of the shape: ComplexF32
// (8, 4, 5, 3, 5) at 1, 3, 5 on 54 rows 11.4 / 19.9, (7, 3, 4, 23) at 1, 2, 4 on 64
// 14.6 / 20.9, (36, 5, 7) on 64 17.0 / 18.9, (34, 5, 5), blocks of 850, on 55 16.4 /
// 14.9; ComplexF64 two factors (3, 32, 14) at 1, 3 on 38 8.4 / 12.0, (33, 8, 13) at
// 1, 3 on 138 20.1 / 26.8, (35, 5, 5), blocks of 875, at 1, 3 on 20 16.4 / 13.7, more
// factors (13, 8, 19) on 184 20.1 / 16.6, (12, 2, 7, 9) on 448 40.9 / 21.8, (9, 4, 28)
// on 52 15.6 / 18.2.  The factors then form several groups.
inline bool group_too_thin(bool c64, int64_t n1, int W, int64_t P, int modes) {
    return n1 > 1 && W <= 2 && P > 1024 && (!c64 || modes == 2);
}

// Whether one d x d factor on n1 x d x n3 (total elements) takes a mode kernel
// (k_mode_fib for n1 >= 16, else k_mode_chunk) and not a site-group pass of its
// own.  The mode kernels pad the factor to multiples of 16 both ways, the group
// kernel to multiples of 8 and 2, but each of its workgroups loads the factor and
// it needs tiles enough to hide that.  Up to width 16 the mode kernels run at
// copy speed.  Mode / group kernel, us, total 10^5, 10^6, 10^7:
//   ComplexF64 n1 = 1      17: 6.1 / 5.7, 15 / 12, 129 / 63;  25: 6.3 / 8.3, 14 /
//                          15, 108 / 104;  33: 9.6 / 10.6, 30 / 17, 264 / 107
//   ComplexF32 n1 = 1      20: 5.6 / 5.6, 9.3 / 8.9, 51 / 40;  21: 5.6 / 5.9, 8.2 /
//                          9.9, 49 / 49;  28: 5.8 / 7.1, 8.4 / 12.5, 40 / 67;
//                          33: 8.0 / 8.7, 13 / 12, 83 / 60
//   ComplexF32 n1 = 5      21: 7.3 / 5.9, 10 / 10.5, 57 / 49
//   n1 = 16                21: ComplexF64 7.1 / 6.7, 13 / 15, 80 / 111; ComplexF32
//                          5.7 / 5.8, 8.4 / 13, 45 / 93;  17: 7.1 / 5.8, 12 / 14,
//                          94 / 96; 5.7 / 5.3, 8.1 / 12, 52 / 83
//   n1 = 600               22: ComplexF64 7.2 / 6.7, 13 / 10, 81 / 67; ComplexF32
//                          5.7 / 5.7, 8.3 / 10, 45 / 40
inline bool one_factor_by_mode(bool c64, int64_t total, int64_t n1, int d) {
    if (d <= 16 || (total < (1 << 16) && (n1 == 1 || n1 >= 16))) return true;
    if (n1 >= 16) {
        if (d <= 20) return n1 < (c64 ? 20 : 32) && total >= (1 << 17);
        if (d <= 24) return n1 < 64 || total < (c64 ? 1 << 19 : 1 << 21);
        return true;
    }
    if (d <= 20) return false;
    if (c64) return total < (d <= 24 ? 1 << 19 : d <= 32 ? 1 << 20 : 1 << 18);
    if (d <= 24) return total < (1 << 21) && (n1 <= 2 || total >= (1 << 18));
    return d <= 32 || total < (1 << 19);
}

}  // namespace qob
