// CPU check of the combine's walk from a cell to its column (gvom_cell_walk.h): every cell of
// random groups in the middle and at the end of a map, against a walk of one column after
// another.  Behind the map's last column lie up to three words that nothing writes; here they
// hold zeros, large counts, and small negative numbers, which take a wrapped sum back below
// the cell's place.  Built by tests/test_cell_walk.py with hipcc; no device work.
#include <stdio.h>

#include <random>
#include <vector>

#include "gvom_cell_walk.h"

int main() {
    std::mt19937 rng(3);
    int fails = 0;
    long cells = 0;
    const int groups[] = {4, 8, 12, 20, 28, 32, 64, 84, 128, 256};
    for (int gcols : groups)
        for (int rep = 0; rep < 400; ++rep) {
            // columns from the group's first to the map's last
            const int left = rep % 2 ? 1 + (int)(rng() % gcols) : gcols + (int)(rng() % 5);
            const int cols = left < gcols ? left : gcols;
            std::vector<uint4> buf((cols + 3) / 4);
            uint32_t *count = reinterpret_cast<uint32_t *>(buf.data());
            uint32_t total = 0;
            for (int c = 0; c < cols; ++c) {
                count[c] = rng() % 3 ? 0u : rng() % 257;
                total += count[c];
            }
            for (size_t c = cols; c < 4 * buf.size(); ++c)
                count[c] = rep % 5 == 0 ? 0u : rep % 5 == 1 ? 0x7FFFFFFFu : 0u - (1u + rng() % (total + 2u));
            for (uint32_t id = 0; id < total; ++id) {
                int want = 0;
                uint32_t rest = id;
                while (rest >= count[want]) rest -= count[want++];
                uint32_t r = id;
                const int got = cell_column(buf.data(), gcols, left, r);
                ++cells;
                if (got == want && r == rest) continue;
                if (++fails < 10)
                    printf("FAIL %d columns, %d left, cell %u of %u: column %d place %u, want %d and %u\n", gcols, left,
                           id, total, got, r, want, rest);
            }
        }
    printf("%ld cells, %d failed\n%s\n", cells, fails, fails ? "failed" : "ok");
    return fails != 0;
}
