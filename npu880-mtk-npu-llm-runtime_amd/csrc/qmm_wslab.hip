// qmm_wslab.hip — prefill GEMM of many tokens over GGUF-packed k-quant rows
// (Q4_K, Q5_K, Q6_K) with int8 MFMA, gfx950: wave slabs.
//
// A workgroup is NW waves on 16 NW weight rows x T = 16 TT tokens; every wave
// owns 16 rows and ALL the workgroup's tokens. It decodes a 256-value block
// of its rows into MFMA operand registers (the two folded int8 planes of the
// slab kernel) and uses them for its TT token tiles, so no row is decoded by
// two waves and a block's decoding is paid once per 16 TT tokens. The tokens'
// codes, sums of 16 codes and block scales are staged in LDS one block ahead
// (two stages, shared by the NW waves); each wave's packed rows go through an
// LDS region of its own with one stage only — free again as soon as the wave
// has decoded it — which is what lets 96 tokens fit two workgroups of 8 waves
// on a CU (74..81 KB of LDS, <= 128 VGPRs: four waves per SIMD). At 96 tokens
// that bound costs 3 spilled registers in Q4_K and 5 in Q5_K (none elsewhere):
// transfer offsets reloaded from scratch inside the K loop, where the wait for
// a reload is one for the transfers issued before it too.
//
// What bounds it: VALU issue, then power. A 16 x 16 tile and block costs 8
// int8 MFMAs (128 cycles), 28 VALU of exact fp32 update (Q6_K: 20) and its
// share of the decoding (Q4_K 94, Q5_K ~170, Q6_K 230 VALU per 16 rows and
// block): Q4_K 19456 x 2560 at M = 2048 has 68 % of all VALU issue slots busy,
// the matrix core 42 %, and the clock at 1.8 GHz (Q6_K 2560 x 9728 59 and 26 %;
// at M = 512 33..50 % and 20 %). Shapes that trade these against each
// other (32 x 32 MFMA tiles in two waves per SIMD, 192 tokens, no operand
// reads at all) all land within 5 % of it. Measured (prequantized input,
// kernel alone): down Q6_K 2560 x 9728 at M = 2048 230 -> 155 us, gate + up
// Q4_K 2 x 9728 x 2560 at M = 2048 / 512 287 / 77 -> 264 / 67, QKV Q5_K 6144 x
// 2560 at M = 2048 / 512 120 / 33.7 -> 102 / 29.0.
//
// Arithmetic and results are the slab kernel's (qmm_slab.hip): exact integer
// sums per block, the reference's fp32 expression, blocks in order.
#include "qmm_slab.h"

namespace qmm {

// TT token tiles, NW waves, WPS waves per SIMD that the registers must allow,
// PD stages of the tokens' operands (and PD - 1 of the rows)
template <class F, int TT_, int NW_, int WPS_, int PD_ = 2>
struct WsCfg {
    static constexpr int TT = TT_, NW = NW_, WPS = WPS_, PD = PD_;
    static constexpr int R = 16 * NW, T = 16 * TT;
    static constexpr bool MIN = F::kMin;
    static constexpr int SB = F::BB;
    static constexpr bool ALIGNED = SB % 16 == 0;
    static constexpr int WCR = (ALIGNED ? SB / 16 : (SB + 30) / 16) | 1;  // 16-B units per staged row, odd
    static constexpr int WSU = 16 * WCR;                                  // units of a wave's rows
    static constexpr int NWW = (WSU + 63) / 64;                           // their transfers
    static constexpr int NAI = 4 * TT;            // code transfers (1 KB) per block
    static constexpr int NBI = MIN ? (TT + 1) / 2 : 0;      // transfers of the sums of 16 codes
    static constexpr int NDI = (T + 63) / 64;     // transfers of the block scales (256 B)
    static constexpr int OFF_B = NAI * 1024, OFF_D = OFF_B + NBI * 1024, STAGE = OFF_D + NDI * 256;
    static constexpr int OFF_W = PD * STAGE, WREG = WSU * 16;
    static constexpr int LDS = OFF_W + (PD - 1) * NW * WREG;
    // transfers that every wave issues per block at least (some issue more)
    static constexpr int L = NWW + NAI / NW + (NBI + NDI) / NW;
    static_assert(LDS <= 160 * 1024, "LDS");
    static_assert(PD >= 2 && (PD - 2) * L <= 63, "vmcnt range");
};

template <class C, class F>
__global__ __launch_bounds__(64 * C::NW, C::WPS) void wslab_kernel(MatGroup grp, Q8KView x, int ntg) {
    extern __shared__ __align__(16) uint8_t lds[];
    constexpr int TT = C::TT;
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nl = lane & 15, cl = lane >> 4;

    // workgroup -> (row slab, token group): consecutive slots of one XCD
    // take the token groups of one slab
    const int G = grp.wg0[grp.n] * ntg;
    const int per = (G + 7) / 8;
    const int lin = int(blockIdx.x % 8u) * per + int(blockIdx.x / 8u);
    if (lin >= G) return;
    const int rg = lin / ntg, tg = lin - rg * ntg;
    int bx;
    const MatArgs a = grp.t[group_task(grp, rg, bx)];
    if (scan_stopped(a.scan)) return;
    const int n0 = bx * C::R, m0 = tg * C::T;
    const int K = a.K, nbk = K / 256;
    const bool live = n0 + 16 * wid < a.N;  // (a wave past the rows only helps staging)

    const uintptr_t wstart = reinterpret_cast<uintptr_t>(a.w) + size_t(n0) * a.row_bytes;
    const uint32_t bl = uint32_t(wstart & 15);
    const int rows_valid = min(C::R, a.N - n0);
    const v4i32 rw = buf_rsrc(reinterpret_cast<const void *>(wstart - bl),
                              (bl + uint32_t(rows_valid) * uint32_t(a.row_bytes) + 15u) & ~15u);
    const uint32_t mpad = uint32_t((a.M + 15) & ~15);
    const v4i32 ra = buf_rsrc(x.qt, mpad * uint32_t(K));
    v4i32 rb = ra;
    if constexpr (C::MIN) rb = buf_rsrc(x.bh, mpad * uint32_t(K / 8));
    const v4i32 rd = buf_rsrc(x.d, uint32_t(a.M) * uint32_t(nbk) * 4u);
    const uint32_t lds0 = lds_addr(lds);

    // the wave's packed rows of block j into stage j mod (PD - 1) of its region
    auto wbase = [&](int j) __attribute__((always_inline)) {
        return uint32_t(C::OFF_W + (wid * (C::PD - 1) + (C::PD > 2 ? j % (C::PD - 1) : 0)) * C::WREG);
    };
    uint32_t wo[C::NWW];
#pragma unroll
    for (int s = 0; s < C::NWW; ++s) {
        const int p = s * 64 + lane, row = p / C::WCR, pc = p - row * C::WCR;
        wo[s] = uint32_t(16 * wid + row) * uint32_t(a.row_bytes) + bl;
        if constexpr (C::ALIGNED) wo[s] += 16u * uint32_t(pc);
    }
    auto issue_w = [&](int j) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < C::NWW; ++s) {
            if ((s + 1) * 64 > C::WSU && s * 64 + lane >= C::WSU) continue;
            if constexpr (C::ALIGNED) {
                dma16s(rw, wo[s], uint32_t(j) * uint32_t(C::SB), lds0 + wbase(j) + uint32_t(s * 1024));
            } else {
                const int p = s * 64 + lane, pc = p - p / C::WCR * C::WCR;
                dma16s(rw, ((wo[s] + uint32_t(j) * uint32_t(C::SB)) & ~15u) + 16u * uint32_t(pc), 0u,
                       lds0 + wbase(j) + uint32_t(s * 1024));
            }
        }
    };
    // the tokens' operands of block j into stage sg: transfer i by wave i % NW.
    // A code tile past the input repeats the last one (its tokens are not
    // stored): the block offsets are uniform and must stay inside the
    // descriptor's range. Sums and scales past their range read zeros.
    constexpr int NAW = (C::NAI + C::NW - 1) / C::NW, NXI = C::NBI + C::NDI, NXW = (NXI + C::NW - 1) / C::NW;
    const int tile0 = m0 / 16, tlast = int(mpad) / 16 - 1;
    uint32_t xo[NXW];
#pragma unroll
    for (int s = 0; s < NXW; ++s) {
        const int i = s * C::NW + wid;  // the sums of token tiles 2 i, 2 i + 1, then 64 tokens' scales each
        const int p = (i - C::NBI) * 64 + lane;
        if (i < C::NBI)
            xo[s] = uint32_t(tile0 + 2 * i + (lane >> 5)) * uint32_t(nbk) * 512u + 16u * uint32_t(lane & 31);
        else
            xo[s] = p < C::T ? uint32_t(m0 + p) * uint32_t(nbk) * 4u : kFar;
    }
    auto issue_a = [&](int j, int sg) __attribute__((always_inline)) {
        const uint32_t base = lds0 + uint32_t(sg * C::STAGE);
#pragma unroll
        for (int s = 0; s < NAW; ++s) {
            const int i = s * C::NW + wid;
            if (C::NAI % C::NW && i >= C::NAI) break;
            // quarter i % 4 of token tile i / 4
            const uint32_t tile = uint32_t(min(tile0 + (i >> 2), tlast));
            dma16s(ra, 16u * uint32_t(lane), (tile * uint32_t(nbk) + uint32_t(j)) * 4096u + 1024u * uint32_t(i & 3),
                   base + uint32_t(i * 1024));
        }
#pragma unroll
        for (int s = 0; s < NXW; ++s) {
            const int i = s * C::NW + wid;
            if (i < C::NBI) dma16s(rb, xo[s], uint32_t(j) * 512u, base + uint32_t(C::OFF_B + i * 1024));
            else if (i < NXI) dma4s(rd, xo[s], uint32_t(j) * 4u, base + uint32_t(C::OFF_D + (i - C::NBI) * 256));
        }
    };
    SlabB B;
    // waits for this wave's transfers of block j: the PD - 2 blocks after it may
    // be in flight (retired in order; near the end fewer were issued: all)
    auto decode = [&](int j) __attribute__((always_inline)) {
        if (C::PD > 2 && j + C::PD - 2 < nbk) wait_vmcnt<(C::PD - 2) * C::L>();
        else wait_vmcnt<0>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t mis =
            C::ALIGNED ? 0u : (uint32_t(16 * wid + nl) * uint32_t(a.row_bytes) + bl + uint32_t(j) * uint32_t(C::SB)) & 15u;
        slab_unpack<F>(lds + wbase(j) + nl * (C::WCR * 16) + mis, cl, B);
    };

    f32x4v acc[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[t] = f32x4v{};

#pragma unroll
    for (int p = 0; p + 1 < C::PD; ++p)
        if (p < nbk) {
            issue_w(p);
            issue_a(p, p);
        }
    decode(0);
    lds_barrier();
    for (int j = 0; j < nbk; ++j) {
        if (j + C::PD - 1 < nbk) {
            issue_w(j + C::PD - 1);
            issue_a(j + C::PD - 1, (j + C::PD - 1) % C::PD);
        }
        const uint8_t *sb = lds + (j % C::PD) * C::STAGE;
        const uint8_t *sa = sb + 16 * lane;
        const uint8_t *sm = sb + C::OFF_B + 8 * lane;
        const uint8_t *sd = sb + C::OFF_D + 16 * cl;
        if (live) {
            uint4 av[2][4];
            half4v bh[2];
            float4 dx[2];
            int4v D1[2], D2[2];
            f32x4v Mb[2];
            auto load_a = [&](int t, int buf) __attribute__((always_inline)) {
#pragma unroll
                for (int h = 0; h < 4; ++h) av[buf][h] = ld16(sa + t * 4096 + h * 1024);
                if constexpr (C::MIN) bh[buf] = __builtin_bit_cast(half4v, ld8(sm + t * 512));
            };
            auto load_d = [&](int t, int buf) __attribute__((always_inline)) { dx[buf] = *reinterpret_cast<const float4 *>(sd + t * 64); };
            auto mm = [&](int buf) __attribute__((always_inline)) {
                int4v d1 = {0, 0, 0, 0}, d2 = {0, 0, 0, 0};
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    d1 = mfma16x16x64(av[buf][h], B.b1[h], d1);
                    d2 = mfma16x16x64(av[buf][h], B.b2[h], d2);
                }
                D1[buf] = d1;
                D2[buf] = d2;
                f32x4v m = {0.0f, 0.0f, 0.0f, 0.0f};
                if constexpr (C::MIN) m = __builtin_amdgcn_mfma_f32_16x16x16f16(bh[buf], B.mh, m, 0, 0, 0);
                Mb[buf] = m;
            };
            auto epi = [&](int t, int buf) __attribute__((always_inline)) {
                const float dxq[4] = {dx[buf].x, dx[buf].y, dx[buf].z, dx[buf].w};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int Sx = (D1[buf][q] << F::kShift) + D2[buf][q];
                    if constexpr (C::MIN)
                        acc[t][q] += dxq[q] * (B.d * (float)Sx - B.dmin * Mb[buf][q]);  // E:11026 / E:11063
                    else
                        acc[t][q] += (B.d * dxq[q]) * (float)Sx;  // E:11101
                }
            };
            load_a(0, 0);
            load_d(0, 0);
            if (TT > 1) load_a(1, 1);
            mm(0);
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                if (t + 1 < TT) {
                    mm((t + 1) & 1);
                    load_d(t + 1, (t + 1) & 1);
                }
                if (t + 2 < TT) load_a(t + 2, t & 1);
                epi(t, t & 1);
                if (t + 1 < TT) {
#pragma unroll
                    for (int i = 0; i < (C::MIN ? 9 : 8); ++i) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
                    }
                }
            }
        }
        if (j + 1 < nbk) {
            decode(j + 1);
            lds_barrier();  // every wave's transfers of block j + 1 have landed, and stage j % PD is free
        }
    }

    const int n = n0 + 16 * wid + nl;
    if (n >= a.N) return;
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int tok = m0 + t * 16 + 4 * cl + r;
            if (tok >= a.M) continue;
            float v = acc[t][r];
            if (a.res) v = v + a.res[size_t(tok) * a.ldr + n];
            a.y[size_t(tok) * a.ldy + n] = v;
        }
}

template <class C, class F>
static hipError_t launch_wslab_t(const MatArgs *tasks, int n, const Q8KView &x, hipStream_t s) {
    MatGroup g{};
    g.n = n;
    g.wg0[0] = 0;
    for (int i = 0; i < n; ++i) {
        g.t[i] = tasks[i];
        g.wg0[i + 1] = g.wg0[i] + (tasks[i].N + C::R - 1) / C::R;
    }
    const int ntg = (tasks[0].M + C::T - 1) / C::T;
    const unsigned grid = unsigned((g.wg0[n] * ntg + 7) / 8 * 8);
    hipLaunchKernelGGL((wslab_kernel<C, F>), dim3(grid), dim3(64 * C::NW), size_t(C::LDS), s, g, x, ntg);
    return hipGetLastError();
}

int mfma_cu_count();

// 128 rows x 96 and 128 x 64 tokens in 8 waves (two workgroups per CU), 64 x
// 64 in 4 waves (three per CU); prefill_kernel chooses.
template <class F>
hipError_t launch_wslab(Prefill p, const MatArgs *tasks, int n, const Q8KView &x, hipStream_t s) {
    if (p == Prefill::W128x96) return launch_wslab_t<WsCfg<F, 6, 8, 4>, F>(tasks, n, x, s);
    if (p == Prefill::W128x64) return launch_wslab_t<WsCfg<F, 4, 8, 4>, F>(tasks, n, x, s);
    return launch_wslab_t<WsCfg<F, 4, 4, 3>, F>(tasks, n, x, s);
}

// Up to 64 tokens (tall_tiles): one group of all the tokens, 64 rows in 4
// waves, from 17 tokens three stages (two blocks in flight: a block's work is
// short).
template <class F>
hipError_t launch_wslab_tall(const MatArgs *tasks, int n, const Q8KView &x, hipStream_t s) {
    const int tt = tall_tiles(kformat<F>(), row_tiles(tasks, n).r64, tasks[0].K, tasks[0].M, mfma_cu_count());
    if (!tt || !slab_ok<F>(tasks, n, x)) return hipErrorNotSupported;
    if (tt == 4) return launch_wslab_t<WsCfg<F, 4, 4, 2, 3>, F>(tasks, n, x, s);
    if (tt == 3) return launch_wslab_t<WsCfg<F, 3, 4, 2, 3>, F>(tasks, n, x, s);
    if constexpr (std::is_same_v<F, MQ4KS>)
        if (tt == 2) return launch_wslab_t<WsCfg<F, 2, 4, 3, 3>, F>(tasks, n, x, s);
    if constexpr (std::is_same_v<F, MQ6KS>)
        if (tt == 1) return launch_wslab_t<WsCfg<F, 1, 4, 4, 2>, F>(tasks, n, x, s);
    return hipErrorNotSupported;
}

#define QMM_WSLAB(F)                                                                                     \
    template hipError_t launch_wslab<F>(Prefill, const MatArgs *, int, const Q8KView &, hipStream_t); \
    template hipError_t launch_wslab_tall<F>(const MatArgs *, int, const Q8KView &, hipStream_t);
QMM_WSLAB(MQ4KS)
QMM_WSLAB(MQ5KS)
QMM_WSLAB(MQ6KS)

}  // namespace qmm
