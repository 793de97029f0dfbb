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

}  // namespace qob
