// Prints what csrc/qmm_route.h decides for each line of stdin (tests/test_route.py).
#include <cstdio>
#include <cstring>
#include <vector>

#include "qmm_route.h"

int main() {
    char what[32];
    while (std::scanf("%31s", what) == 1) {
        if (!std::strcmp(what, "rms_rows")) {  // M: rows on each XCD, rows missed or taken twice
            int M;
            if (std::scanf("%d", &M) != 1) return 1;
            const int per = qmm::rms_rows_per_xcd(M), grid = per ? 8 * per : M;
            std::vector<int> seen(M), xcd(8);
            int bad = 0;
            for (int b = 0; b < grid; ++b) {
                const int m = qmm::xcd_row(unsigned(b), per);
                if (m >= M) continue;
                ++seen[m];
                ++xcd[b % 8];
            }
            for (int m = 0; m < M; ++m) bad += seen[m] != 1;
            std::printf("%d", bad);
            for (int x : xcd) std::printf(" %d", x);
            std::printf("\n");
        } else if (!std::strcmp(what, "blocks")) {  // M, blocks: items missed or taken twice, waves with work on each XCD
            int M, nb;
            if (std::scanf("%d %d", &M, &nb) != 2) return 1;
            std::vector<int> seen(size_t(M) * nb), xcd(8);
            int bad = 0;
            const qmm::BlockMap map = qmm::block_map(M, nb);
            for (unsigned b = 0; b < map.grid; ++b)
                for (int wave = 0; wave < 4; ++wave) {
                    const qmm::BlockItem it = qmm::xcd_block(b, wave, map);
                    if (it.m < 0 || it.j < 0) return 1;
                    if (it.m >= M || it.j >= nb) continue;
                    ++seen[size_t(it.m) * nb + it.j];
                    ++xcd[b % 8];
                }
            for (int v : seen) bad += v != 1;
            std::printf("%d", bad);
            for (int x : xcd) std::printf(" %d", x);
            std::printf("\n");
        } else if (!std::strcmp(what, "prefill")) {  // format, K, M, CUs, tasks, rows of each: the kernel past 64 tokens
            int f, K, M, cus, n;
            if (std::scanf("%d %d %d %d %d", &f, &K, &M, &cus, &n) != 5) return 1;
            qmm::RowTiles r;
            for (int rows; n > 0; --n) {
                if (std::scanf("%d", &rows) != 1) return 1;
                r.add(rows);
            }
            std::printf("%c\n", char(qmm::prefill_kernel(qmm::KFormat(f - 4), r, K, M, cus)));
        } else if (!std::strcmp(what, "tall")) {  // format, rows, K, M, CUs: token tiles of the tall wave slabs
            int f, rows, K, M, cus;
            if (std::scanf("%d %d %d %d %d", &f, &rows, &K, &M, &cus) != 5) return 1;
            std::printf("%d\n", qmm::tall_tiles(qmm::KFormat(f - 4), (rows + 63) / 64, K, M, cus));
        } else {
            return 1;
        }
    }
    return 0;
}
