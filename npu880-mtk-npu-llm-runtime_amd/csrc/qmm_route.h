// qmm_route.h — which rows a producer's workgroup takes, and which kernel a
// GEMM of k-quant rows takes, as plain C++ (no HIP): the kernels and launchers
// use these rules, and a host program can check them without a device.
#pragma once

#include <cstdint>

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

// The SwiGLU producer: a wave takes one 256-value block of one token, a
// workgroup of 4 waves a quad of blocks, or one of the nb % 4 last blocks for 4
// tokens, so that no wave is without a block. 8 workgroups in a row on one XCD
// make a unit: a quad for a group of 8 tokens, or a last block for 32 tokens.
// Their 16-B pieces of the tiles section fill whole 128-B lines in that XCD's
// L2. Units go round the XCDs (none takes more than one over another), four
// token groups' quads and then their last blocks: the launch walks memory in
// order. Measured (us; so / an eighth of the 16-token tiles' quads to each XCD,
// a last quad's waves without a block idle / blocks in order, every token's on
// all XCDs): 9728 columns at M = 17 / 65 / 513 / 2048 2.6 / 3.85 / 14.6 / 56.3,
// 3.0 / 4.4 / 15.2 / 61, 2.9 / 4.4 / 16.6 / 64.6; 9984 at M = 2048 59.8, 67.0,
// 64.3; 14336 88.8, 99.6, 98.8; 1280 at M = 2048 / 16384 8.5 / 60, 11.9 / 89,
// 9.8 / 72.
struct BlockMap {
    int nb, groups;  // blocks of a row, groups of 8 tokens
    uint32_t inv;    // 2^32 / nb, rounded up: a unit's u inv / 2^32 is u / nb or one more
    unsigned grid;   // workgroups
};
constexpr BlockMap block_map(int M, int nb) {
    const int groups = (M + 7) / 8, part = groups & 3;
    const int units = (groups >> 2) * nb + (part ? part * (nb >> 2) + (nb & 3) : 0);
    return BlockMap{nb, groups, uint32_t(0xFFFFFFFFu / unsigned(nb) + 1u), unsigned((units + 7) / 8) * 64u};
}
struct BlockItem {
    int m, j;  // token, block (either may lie past the rows)
};
constexpr BlockItem xcd_block(unsigned b, int wave, const BlockMap &o) {
    const int i = int(b / 8u), u = (i >> 3) * 8 + int(b % 8u), k = i & 7;
    int s = o.nb > 1 ? int(uint64_t(unsigned(u)) * o.inv >> 32) : u, v = u - s * o.nb;
    if (v < 0) --s, v += o.nb;
    const int q = o.nb >> 2, left = o.groups - 4 * s, quads = (left < 4 ? left : 4) * q;
    if (v < quads) {
        const int g = int(v >= q) + int(v >= 2 * q) + int(v >= 3 * q);
        return BlockItem{32 * s + 8 * g + k, 4 * (v - g * q) + wave};
    }
    return BlockItem{32 * s + 4 * k + wave, 4 * q + v - quads};
}

enum class KFormat { Q4, Q5, Q6 };

// a task group's row tiles of 16, 32, 64 and 128 rows (each task rounded up)
struct RowTiles {
    int r16 = 0, r32 = 0, r64 = 0, r128 = 0;
    void add(int rows) {
        r16 += (rows + 15) / 16;
        r32 += (rows + 31) / 32;
        r64 += (rows + 63) / 64;
        r128 += (rows + 127) / 128;
    }
};

// Past 64 tokens. Wave slabs (qmm_wslab.hip) of 128 rows x 96 tokens, 128 x 64
// and 64 x 64; decoded slabs (qmm_slab.hip) of 128 tokens (16 rows for Q6_K,
// 32 for Q5_K) and, for Q6_K, of 32 rows x 256 tokens; packed slabs of 64 x 32.
enum class Prefill : char { W128x96 = 'A', W128x64 = 'B', W64x64 = 'C', D128 = 'D', D256 = 'E', P64x32 = 'P' };

// The kernel with the least expected time per 256-value block, in nanoseconds.
// Wave slabs: a CU takes its share of the workgroups, rounded up; of the 8-wave
// shapes two run side by side, and one left alone takes 0.7 of a pair's time
// (64 x 64: its step has a floor that three side by side hide). A workgroup's
// time per block, a call's fixed 4 us taken off, from a sweep of 18 shapes (M =
// 192..2048). Measured (us, 128 x 96 / 128 x 64 / 64 x 64, chosen first): Q4_K
// 2 x 9728 x 2560 at M = 2048 264 / 272 / 303, at M = 512 (128 x 64) 75 / 70 /
// 75, at M = 192 (128 x 64) 40 / 32 / 36; 2560 x 4096 at M = 2048 60 / 63 / 66;
// Q5_K 6144 x 2560 at M = 2048 (128 x 64) 105 / 102 / 113, at M = 512 (64 x 64)
// 42 / 33 / 30; Q6_K 2560 x 9728 at M = 2048 156 / 187 / 186, 9728 x 2560 at M
// = 512 47 / 54 / 49.
// They are taken where that is at least 8 % below the slabs of 32 and 128
// tokens (or below those of 256 at all), which win where the workgroups are few
// (their steps are shorter, their tiles smaller). Fitted over the same sweep
// with w workgroups per CU: decoded Q6_K 16 x 128 0.1 + 0.56 w us (2560 x 9728
// at M = 512 / 1024 / 2048: 1.34 / 2.55 / 5.95), Q5_K 32 x 128 0.3 + 0.92 w
// (6144 x 2560 at M = 200 / 512 / 2048: 1.7 / 2.9 / 11.5, 3001 x 8192 at M =
// 777 2.6), packed 64 x 32 0.35 + 0.5 w (Q4_K 2560 x 4096 at M = 512 / 1024:
// 1.3 / 2.5, 2 x 9728 x 2560 at M = 65: 1.9).
// Q6_K and Q5_K decode in LDS (their decoding is costly next to their update)
// from 65 tokens, Q5_K where those workgroups number at least 5/8 of the CUs
// (QKV 6144 x 2560 at M = 65..127 17.4 -> 16.1 us; 4096 x 2560 at M = 128 12.8
// against 16.2, 1024 x 2560 12.3 against 15.8 on the packed slabs: there they
// stay). Q4_K stays packed: its update outweighs its decoding (2560 x 4096 at M
// = 512 25.1 against 26.9 us and more).
// Q6_K 32 x 256 (each block decoded once per 256 tokens, one workgroup per CU):
// 1.3 us a block while they make one round, 1.45 a round after that, but a
// longer start, so the time per block is not all. Over 8 heights, K = 512 /
// 1024 / 2560 / 4096 / 9728 and M = 65..2048, against the 16 x 128 slabs: in
// one round with w > 3 of those 0.89 / 0.86 / 0.77 / 0.73 / 0.66 of their time,
// with 2 < w <= 3 1.15 / 1.12 / 1.07 / 1.04 / 0.88..1.04: there only over K >=
// 8192 where their 128 tokens are in use (live: 2560 x 9728 at M = 512 52.8 ->
// 51.7 us, 6144 x 9728 at M = 256 56.2 -> 52.1; 5000 x 5120 at M = 400 61
// against 51); in several rounds 1.0..1.2 over K <= 1024.
inline Prefill prefill_kernel(KFormat f, const RowTiles &r, int K, int M, int cus) {
    const int i = int(f);
    constexpr int k96[] = {1750, 2040, 2100}, k64[] = {1290, 1650, 1800}, kC[] = {780, 900, 960};
    constexpr int kC0[] = {850, 1350, 1350}, kC1[] = {450, 400, 400};
    auto load = [&](int wgs) { return (wgs + cus - 1) / cus; };
    auto pairs = [&](int wgs, int64_t ns) {  // two per CU side by side
        const int l = load(wgs);
        return ns * (l & ~1) + (l & 1) * (ns * 27 / 20);
    };
    const int64_t a = pairs(r.r128 * ((M + 95) / 96), k96[i]), b = pairs(r.r128 * ((M + 63) / 64), k64[i]);
    const int64_t lc = load(r.r64 * ((M + 63) / 64)), c0 = lc * kC[i], c1 = kC0[i] + lc * kC1[i], c = c0 > c1 ? c0 : c1;
    const int64_t ab = b < a ? b : a, wave = c < ab ? c : ab;
    const Prefill w = c < ab ? Prefill::W64x64 : b < a ? Prefill::W128x64 : Prefill::W128x96;

    const int t16 = (M + 15) / 16, t32 = (M + 31) / 32, t128 = (M + 127) / 128;
    const bool q6 = f == KFormat::Q6, decoded = q6 || (f == KFormat::Q5 && 8 * r.r32 * t128 >= 5 * cus);
    const int64_t ns128 = q6        ? 100 + int64_t(560) * r.r16 * t128 / cus
                          : decoded ? 300 + int64_t(920) * r.r32 * t128 / cus
                                    : 350 + int64_t(500) * r.r64 * t32 / cus;
    if (q6) {
        const int rounds = load(r.r32 * ((M + 255) / 256));
        const int64_t ns256 = rounds == 1 ? 1300 : 1450 * int64_t(rounds);
        const int64_t live = int64_t(r.r16) * t16;  // (eight to a workgroup of 128 tokens)
        const bool pays = rounds > 1 ? K >= 2048 : load(r.r16 * t128) > 3 || (K >= 8192 && 10 * live >= 8 * 24 * int64_t(cus));
        if (pays && 100 * ns256 < 95 * ns128) return wave < ns256 ? w : Prefill::D256;
    }
    if (108 * wave < 100 * ns128) return w;
    return decoded ? Prefill::D128 : Prefill::P64x32;
}

// Up to 64 tokens: wave slabs of 64 rows and all the tokens, in 4 waves (their
// 16-token tiles; 0: the small-M kernels). Those read every token's codes again
// for each 16 rows (at 16-row tiles about 12 TB/s out of the L2s, their bound)
// and again the rows for each token group; here 64 rows share them. Measured (K
// = 2560 unless said, us, small-M kernel -> this): M = 48 at 19456 / 30000 /
// 100000 rows Q4_K 23.4 / 32.6 / 98.7 -> 21.1 / 22.1 / 68.7, Q6_K 27.3 / 40.7 /
// 121 -> 25.3 / 27.3 / 81.9, Q5_K 30000 x 4096 57.2 -> 36.3; M = 64 Q4_K 24.1 /
// 34.0 / 102 -> 23.5 / 24.7 / 74.3.
// Under one workgroup per CU (9728 rows at M = 37..64: 12.2..16 against
// 15.3..19) a step's latency shows and the small-M kernels stay. So they do
// where the last round of workgroups (one per CU each) is too empty, by how
// good they are at that K: 33..64 tokens, time against theirs at 1.0 / 1.06 /
// 1.19 / 1.25 / 1.38 / 2.02 workgroups per CU: K <= 1536 at most 0.94; K =
// 2560 0.9 / 1.05 / 0.95 / 0.95 / 0.9 / 0.95, Q5_K at 33 tokens 1.0 / 1.1 /
// 1.03 / 0.99 / 0.9 / 1.0; K = 3072 (the part kernel's best) 0.95 / 1.1 / 1.02 /
// 1.0 / 0.9 / 0.97; Q5_K and Q6_K past that at most 0.97; Q4_K at K = 3584..4096
// 0.9 / 1.0 / 0.85 / 0.85 / 0.8 / 0.85, past it 1.03 / 1.04 / 1.03 / 1.03 / 1.0 /
// 1.05 and 0.8 at 2.0. Q4_K over K > 2560 at exactly one round 1.06.
// At 17..32 tokens the small-M kernels take each 16-row tile's tokens at once:
// faster here only for Q4_K from 7/4 workgroups per CU (30000 / 100000 rows
// 20.6 / 55.2 -> 18.3 / 48.9). Time against theirs with the weights in HBM and
// 2 GB of others read since, at 2.0 / 2.44 / 2.69 / 3.01 / 6.11 workgroups per
// CU: K <= 1536 and K > 3072 at most 0.98, K = 2560 0.89 / 0.98 / 0.93 / 1.02 /
// 0.94, K = 3072 (the part kernel's best) 0.95 / 1.03 / 0.97 / 1.10 / 1.05.
// At 9..16 tokens Q6_K alone gains (decoding bound, one stage pair and four
// waves per SIMD; K = 1024 / 1536 / 4096 on 151936 rows warm 0.71 / 0.80 / 0.83
// of the part kernel's time, with the weights in HBM 0.73 / 0.85 / 0.83). Over
// K = 2048..3072 it gains 0..10 % warm only: with the weights in HBM 1.0..1.05,
// and 1.1..1.2 on buffers just written (a wave's 16 rows are 16 distant pieces
// a step; the part kernel's are contiguous): left to the part kernel.
inline int tall_tiles(KFormat f, int r64, int K, int M, int cus) {
    if (M <= 8 || M > 64 || r64 < cus) return 0;
    const int full = (r64 + cus - 1) / cus * cus;  // the rounds' slots
    auto filled = [&](int num, int den) { return int64_t(den) * r64 > int64_t(num) * full; };
    const bool q4 = f == KFormat::Q4;
    if (M <= 16) return f == KFormat::Q6 && r64 >= 4 * cus && (K < 2048 || K > 3072) ? 1 : 0;
    if (M <= 32) return q4 && 4 * r64 >= 7 * cus && (K <= 1536 || K > 3072 || (K <= 2560 && filled(4, 5))) ? 2 : 0;
    const bool ok = K <= 1536                         ? true
                    : K <= 2560 && f != KFormat::Q5   ? filled(7, 12)
                    : K <= 3072 || (q4 && K <= 4096) ? filled(5, 8)
                                                      : !q4 || filled(3, 4);
    if (!ok || (q4 && K > 2560 && r64 == cus)) return 0;
    return (M + 15) / 16;
}

}  // namespace qmm
