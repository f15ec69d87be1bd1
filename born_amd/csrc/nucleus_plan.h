// Into how many parts the rows of a batch without a top-k cut go (nucleus_parts.h): a host decision without HIP.
#pragma once
#include <algorithm>

namespace born {

constexpr int PARTS_ROW_MAX = 32;             // parts of a row
constexpr int PARTS_LEAST = 4096;             // logits of a part, about: one 128-bit load per thread
// Parts pay where the logits that a row's own workgroup is spared, V - V / parts, reach a number, a larger one for few parts; two parts, whose batch keeps the device
// busy either way, only from twice the row.  us, one workgroup to a row and parts, top-p 0.95 at T = 0.8 (rows, and so parts: 1 of 32, 8 of 32, 32 of 8, 42 of 6, 64 of 4, 85 of 3,
// 128 of 2; a row has V / 4096 at most):
//               1            8            32           42           64           85           128
//     50 257    22.4 22.6    23.9 23.6    24.2 25.0    24.1 26.0    24.4 26.6    24.3 28.5    24.7 30.6
//     53 001    24.1 22.8    24.5 23.7    24.9 25.1    24.9 26.1    24.9 26.4    24.4 28.8    24.8 30.7
//     57 000    24.5 22.8    25.1 24.0    25.4 25.0    25.5 26.1    25.5 26.6    25.3 28.7    25.8 31.8
//     61 000    24.9 22.9    25.8 24.0    26.1 25.6    26.2 26.3    26.4 26.7    26.2 28.9    26.7 32.7
//     66 001    26.4 23.0    27.8 23.7    27.9 25.5    27.8 26.1    27.6 28.3    28.5 29.6    28.7 34.7
//     80 000    28.8 23.1    -    24.3    30.1 25.8    30.1 27.0    29.9 28.9    30.0 31.6    32.0 39.1
//    100 003    34.1 23.4    -    24.7    35.2 26.4    34.7 28.4    34.8 30.6    36.5 35.6    38.9 44.1
//    152 064    45.0 24.2    -    25.1    46.1 28.3    46.5 30.7    48.2 38.2    50.9 45.2    52.3 55.7
//    250 000    66.5 25.4    -    -       66.9 32.5    73.7 40.4    76.8 49.9    78.6 60.6    83.7 79.6
// Four launches, chains of memory and LDS round trips each.
constexpr int PARTS_SPARED = 50000, PARTS_FEW = 6, PARTS_SPARED_FEW = 60000, PARTS_TWO_FROM = 196608;

// most: parts of the batch.  0: not cut.
inline int row_parts(int V, int rows, int most) {
    const int parts = std::min(std::min(most / rows, PARTS_ROW_MAX), V / PARTS_LEAST);
    if (parts < 2 || V - V / parts < (parts < PARTS_FEW ? PARTS_SPARED_FEW : PARTS_SPARED) || (parts == 2 && V < PARTS_TWO_FROM)) return 0;
    return parts;
}

}  // namespace born
