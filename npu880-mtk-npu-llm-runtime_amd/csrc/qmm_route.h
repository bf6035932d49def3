// qmm_route.h — which rows a producer's workgroup takes, as plain C++ (no
// HIP): the kernels and launchers use these rules, and a host program can
// check them without a device.
#pragma once

namespace qmm {

// Workgroup b of a launch runs on XCD b mod 8, so workgroups b, b + 8, ...
// given consecutive items meet in one XCD's L2. The rows of a one-row-per-
// workgroup producer: `per` consecutive ones on each XCD (0: row b).
constexpr int xcd_row(unsigned b, int per) { return per ? int(b % 8u) * per + int(b / 8u) : int(b); }

// Rows per XCD of the RMSNorm producer: from 256 rows on (two token tiles of
// 16 for each XCD) an eighth of them, consecutive; fewer rows spread one by
// one. Not rounded to whole token tiles: up to seven tiles then meet in two
// L2s, but no XCD takes a tile more than another or stays without rows (rows
// of 4096, M = 257 / 400 / 520: 6.5 / 6.9 / 8.25 -> 6.0 / 6.65 / 7.9 us; rows
// of 9728 13.2 / 13.9 / 17.2 -> 12.4 / 13.2 / 16.5).
constexpr int rms_rows_per_xcd(int M) { return M >= 256 ? (M + 7) / 8 : 0; }

// The SwiGLU producer's workgroups take one token's quad of 256-value blocks.
// A unit is one quad for 8 tokens, whose 16-B pieces of the tiles section fill
// whole 128-B lines: 8 workgroups in a row on one XCD, which meet in its L2.
// Units go round the XCDs, so no XCD takes more than one over another and the
// launch walks memory in order. Measured (us; unit by unit / an eighth of the
// 16-token tiles' quads to each XCD / blocks in order): 9728 columns at M = 17
// / 65 / 513 / 2048 2.6 / 3.9 / 15.7 / 60.5, 3.0 / 4.4 / 15.2 / 61, 2.9 / 4.4
// / 16.7 / 64.6; 9984 at M = 2048 61.6, 67.0, 64.3; 14336 88.9, 99.6, 98.8.
struct QuadItem {
    int m, q;  // token, quad
};
constexpr QuadItem xcd_quad(unsigned b, int nq) {
    const int i = int(b / 8u), u = (i >> 3) * 8 + int(b % 8u);
    return QuadItem{u / nq * 8 + (i & 7), u % nq};
}
constexpr unsigned xcd_quad_grid(int M, int nq) { return unsigned(((M + 7) / 8 * nq + 7) / 8 * 64); }

}  // namespace qmm
