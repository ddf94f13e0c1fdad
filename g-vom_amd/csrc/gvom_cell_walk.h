// The cell pass's walk from a cell of a column group to its column; also compiled for the host,
// where a test sweeps it over groups, map ends and what lies behind them.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

constexpr int CELL_LOADS = 4;     // 16 in flight: 0.4 to 0.9 us longer

// Column, counted from the group's first, of the group's r-th cell (from 0); r becomes the cell's
// place in that column.  cc: the cell counts of the group's gcols columns (a multiple of four),
// `left` of them or more up to the map's last column; the group has more than r cells.  The
// column is the first one with more cells than r up to and including it; four counts per load,
// CELL_LOADS loads in flight.  The last load may hold up to three words past the map's last column,
// which nothing writes: whatever they make of the sum, no column from `left` on is taken.
__host__ __device__ __forceinline__ int cell_column(const uint4 *cc, int gcols, int32_t left, uint32_t &r) {
    uint32_t sum = 0, skip = 0;
    int k = 0;
    for (int q0 = 0; q0 < gcols / 4 && sum <= r; q0 += CELL_LOADS) {
        uint4 m[CELL_LOADS];
#pragma unroll
        for (int u = 0; u < CELL_LOADS; ++u)
            m[u] = q0 + u < gcols / 4 && 4 * (q0 + u) < left ? cc[q0 + u] : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int u = 0; u < CELL_LOADS; ++u)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                sum += j == 0 ? m[u].x : j == 1 ? m[u].y : j == 2 ? m[u].z : m[u].w;
                if (sum <= r && 4 * (q0 + u) + j + 1 < left) {
                    skip = sum;
                    k = 4 * (q0 + u) + j + 1;
                }
            }
    }
    r -= skip;
    return k;
}
