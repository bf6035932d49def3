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

}  // namespace qmm
