// CPU check of the workspaces of the azimuth-ordered cast, the combine's cell pass and the slot
// clear: what their kernels index against what the C-ABI allocates, over the domain, and the
// launchers' refusals of buffers one word short or counts out of range.  Built by
// tests/test_workspaces.py with hipcc against libgvom_hip.so; every launcher call below is refused
// before it touches the device, so the program needs no GPU.
#include <stdio.h>

#include <algorithm>
#include <random>
#include <vector>

#include "gvom_kernels.h"

namespace P = gvom_plan;

static int fails = 0;
#define CHECK(cond, ...)                       \
    do {                                       \
        if (!(cond)) {                         \
            ++fails;                           \
            if (fails < 20) {                  \
                printf("FAIL %s: ", #cond);    \
                printf(__VA_ARGS__);           \
                printf("\n");                  \
            }                                  \
        }                                      \
    } while (0)
#define REFUSED(call, what) CHECK((call) == hipErrorInvalidValue, what)

static Geo geo(int xy, int z, int B) {
    Geo g{};
    g.xy_res = 0.4;
    g.z_res = 0.2;
    g.XY = xy;
    g.Z = z;
    g.X = (int64_t)xy * xy;
    g.V = g.X * z;
    g.B = B;
    g.VB = 24;
    return g;
}

// The rows of azimuth counts that a batch uses (a scan's part of a tile each): inside the rows
// the launchers ask for, and no row for two scans.
static void azimuth_rows(const std::vector<int64_t> &counts) {
    const int S = (int)counts.size();
    int64_t n = 0, last = -1;
    for (int64_t c : counts) n += c;
    int64_t beg = 0;
    for (int s = 0; s < S; ++s) {
        const int64_t end = beg + counts[s];
        if (end > beg) {
            const int64_t r0 = beg / P::RS_TILE + s, r1 = (end - 1) / P::RS_TILE + s;
            CHECK(r0 > last, "n %lld scan %d", (long long)n, s);
            CHECK(r1 < P::az_rows(n, S), "n %lld S %d scan %d row %lld", (long long)n, S, s, (long long)r1);
            last = r1;
        }
        beg = end;
    }
    CHECK(P::az_hist_words(n, S) <= P::alloc_az_hist_words(n), "n %lld S %d", (long long)n, S);
    // a buffer made for more points
    CHECK(P::az_hist_words(n, S) <= P::alloc_az_hist_words(n + 1), "n %lld S %d", (long long)n, S);
}

int main() {
    std::mt19937 rng(1);
    const int64_t sizes[] = {0, 1, 255, 256, 2047, 2048, 2049, 4096, 131072, 1000001};
    for (int S = 1; S <= P::MAX_BATCH; ++S)
        for (int k = 0; k < 40; ++k) {
            std::vector<int64_t> c(S);
            for (auto &v : c) v = sizes[rng() % (k < 20 ? 10 : 7)];
            azimuth_rows(c);
        }

    const int xys[] = {4, 5, 7, 8, 13, 37, 64, 100, 127, 128, 129, 151, 255, 256, 257, 512, 1024, 4096};
    const int zs[] = {4, 5, 8, 9, 16, 31, 32, 33, 48, 60, 64, 65, 72, 100, 128, 136, 176, 200, 250, 256};
    for (int xy : xys)
        for (int z : zs) {
            if (!P::params_in_domain(xy, z, 1)) continue;
            const Geo g = geo(xy, z, 1);
            const int64_t cols = comb_group_columns(g), groups = comb_groups(g);
            CHECK(cols % 4 == 0, "xy %d z %d: %lld columns", xy, z, (long long)cols);
            CHECK(groups * cols >= g.X && (groups - 1) * cols < g.X, "xy %d z %d", xy, z);
            // four counts at a time: of the groups, and of the columns from a group's first on
            CHECK((groups + 3) / 4 * 4 <= comb_group_words(g), "xy %d z %d", xy, z);
            CHECK((g.X + 3) / 4 * 4 <= P::alloc_col_count_words(g.X), "xy %d z %d", xy, z);
            if (comb_cells_direct(g)) CHECK(groups <= 8192, "xy %d z %d: %lld groups", xy, z, (long long)groups);
        }

    const Geo g = geo(256, 64, 8);
    const int64_t n = 131072, az = P::az_hist_words(n, 3), tables = P::alloc_slot_table_words(g.V, g.B);
    REFUSED(launch_prepare(GVOM_F32, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 3, n, g, nullptr, RAY_AZIMUTH,
                           nullptr, nullptr, 0, (uint32_t *)16, az - 1, nullptr),
            "azimuth bins one word short");
    REFUSED(launch_prepare(GVOM_F32, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 3, n, g, nullptr, RAY_AZIMUTH,
                           nullptr, nullptr, 0, nullptr, az, nullptr),
            "no azimuth bins");
    struct { int S; int64_t az, tables; int force; const char *what; } bad[] = {
        {3, az - 1, tables, -1, "azimuth counts one word short"}, {3, az, tables - 1, -1, "slot tables one word short"},
        {0, az, tables, -1, "no scan"}, {33, P::alloc_az_hist_words(n) * 2, tables, -1, "33 scans"},
        {1, az, g.V - 1, 0, "a tuner's table one word short"}};
    for (const auto &b : bad) {
        REFUSED(launch_az_order(nullptr, nullptr, nullptr, b.S, n, g, nullptr, nullptr, b.az, nullptr, nullptr, b.tables,
                                b.force, nullptr), b.what);
        REFUSED(launch_raycast_az(GVOM_F32, nullptr, nullptr, b.S, n, g, nullptr, nullptr, b.tables, nullptr, nullptr,
                                  b.az, 1, b.force, nullptr), b.what);
    }
    uint32_t *kout = nullptr, *vout = nullptr;
    const struct { int64_t words; int S; const char *what; } clears[] = {
        {tables - 1, 1, "a clear of tables one word short"}, {tables, 0, "a clear of no scan"},
        {tables, 33, "a clear of 33 scans"}};
    for (const auto &c : clears) {
        const SlotClear clear{nullptr, c.words, g.B, c.S, g.V};
        REFUSED(radix_sort(nullptr, nullptr, nullptr, nullptr, n, 26, 24, nullptr, P::radix_hist_words(n), nullptr, &kout,
                           &vout, nullptr, &clear), c.what);
        REFUSED(launch_clear_slots(nullptr, c.words, nullptr, c.S, g, nullptr), c.what);
    }
    const int64_t gw = comb_group_words(g);
    REFUSED(launch_comb_tables(g, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, gw - 1, nullptr, nullptr, nullptr,
                               nullptr), "group counts one word short");
    REFUSED(launch_comb_cells(g, nullptr, nullptr, nullptr, 0, nullptr, nullptr, 0, nullptr, g.X, nullptr, gw - 1,
                              nullptr, 0, nullptr, nullptr, nullptr, nullptr), "cells: group counts one word short");
    REFUSED(launch_comb_cells(g, nullptr, nullptr, nullptr, 0, nullptr, nullptr, 0, nullptr, g.X - 1, nullptr, gw,
                              nullptr, 0, nullptr, nullptr, nullptr, nullptr), "cells: column counts one word short");
    const Geo large = geo(257, 64, 8);
    REFUSED(launch_comb_cells(large, nullptr, nullptr, nullptr, 0, nullptr, nullptr, 0, nullptr, large.X, nullptr,
                              comb_group_words(large), nullptr, P::col_chunks(large.X), nullptr, nullptr, nullptr,
                              nullptr), "a large map without a list");
    ScanDesc d[1] = {};
    REFUSED(launch_set_descs(nullptr, d, 0, nullptr), "no descriptor");
    REFUSED(launch_set_descs(nullptr, d, GVOM_MAX_BATCH + 1, nullptr), "33 descriptors");
    REFUSED(launch_copy((void *)16, (void *)8, 64, nullptr), "a copy from an unaligned buffer");
    REFUSED(launch_debug_height(g, nullptr, 0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 5, nullptr, nullptr),
            "rows of five words");
    if (fails) {
        printf("%d failed\n", fails);
        return 1;
    }
    printf("ok\n");
    return 0;
}
