// qmm_slab.h — what the prefill kernels share (qmm_slab.hip, qmm_wslab.hip):
// a row tile's block unpacked from LDS into MFMA operand registers.
#pragma once

#include "qmm_kformats.h"
#include "qmm_route.h"

namespace qmm {

typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float f32x4v __attribute__((ext_vector_type(4)));

// B operands of one row tile for one block
struct SlabB {
    uint4 b1[4], b2[4];
    half4v mh;  // mins of the lane's groups (Q4_K / Q5_K)
    float d, dmin;
};

// the 4 mins (as fp16) a lane supplies for groups 4c .. 4c + 3: units 2c, 2c,
// 2c + 1, 2c + 1 (mw: the 8 mins four to a dword)
__device__ inline half4v mins_f16(const uint32_t (&mw)[2], int c) {
    // (a mask select: an index would put mw in scratch memory)
    const uint32_t sel = 0u - uint32_t((c >> 1) & 1);
    const uint32_t w = (mw[0] & ~sel) | (mw[1] & sel);
    const int b0 = 2 * (c & 1);
    const half2v bias = {(_Float16)1024.0f, (_Float16)1024.0f};
    // 0x6400 | m is the fp16 value 1024 + m (m < 64): subtract 1024, exactly
    const half2v lo = __builtin_bit_cast(half2v, __builtin_bit_cast(uint32_t, byte_pair(w, b0)) | 0x64006400u) - bias;
    const half2v hi =
        __builtin_bit_cast(half2v, __builtin_bit_cast(uint32_t, byte_pair(w, b0 + 1)) | 0x64006400u) - bias;
    return half4v{lo.x, lo.y, hi.x, hi.y};
}

template <class F>
__device__ inline void slab_unpack(const uint8_t *blk, int c, SlabB &o) {
    if constexpr (std::is_same_v<F, MQ6KS>) {
        const MQ6KS::W w = MQ6KS::load_lds(blk, c);
        SplitB sb;
        split_b(w, c, sb);
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            o.b1[h] = sb.b1[h];
            o.b2[h] = sb.b2[h];
        }
        o.d = fp16_bits_to_f32(w.d);
        o.dmin = 0.0f;
    } else {  // Q4_K / Q5_K folded
        const typename F::W w = F::load_lds(blk, c);
        uint32_t scp[2], mp[2];
        scales_k4_packed(w.h.y, w.h.z, w.h.w, scp, mp);
        SplitB sb;
        split_b(w, scp, mp, sb);
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            o.b1[h] = sb.b1[h];
            o.b2[h] = sb.b2[h];
        }
        o.mh = mins_f16(mp, c);
        o.d = fp16_bits_to_f32(w.h.x & 0xFFFFu);
        o.dmin = fp16_bits_to_f32(w.h.x >> 16);
    }
}

// whether the slab kernels apply: K a multiple of 256, the operand sections
// present, rows of an aligned format 16-B aligned, offsets inside the 32-bit
// buffer range
template <class F>
inline bool slab_ok(const MatArgs *tasks, int n, const Q8KView &x) {
    const MatArgs &a = tasks[0];
    if (a.K % 256 || !x.qt || (F::kMin && !x.bh)) return false;
    if (size_t((a.M + 15) & ~15) * size_t(a.K) >= (size_t(1) << 31)) return false;
    for (int i = 0; i < n; ++i) {
        if (F::BB % 16 == 0 && ((reinterpret_cast<uintptr_t>(tasks[i].w) | tasks[i].row_bytes) & 15)) return false;
        if (size_t(tasks[i].N) * tasks[i].row_bytes + 16 >= (size_t(1) << 31)) return false;
    }
    return true;
}

// up to 64 tokens on tall tensors; hipErrorNotSupported (nothing launched)
// where the small-M kernels are to run
template <class F>
hipError_t launch_wslab_tall(const MatArgs *tasks, int n, const Q8KView &x, hipStream_t s);

// a wave-slab shape (W128x96, W128x64 or W64x64)
template <class F>
hipError_t launch_wslab(Prefill p, const MatArgs *tasks, int n, const Q8KView &x, hipStream_t s);

template <class F>
constexpr KFormat kformat() {
    return std::is_same_v<F, MQ4KS> ? KFormat::Q4 : std::is_same_v<F, MQ5KS> ? KFormat::Q5 : KFormat::Q6;
}
inline RowTiles row_tiles(const MatArgs *tasks, int n) {
    RowTiles r;
    for (int i = 0; i < n; ++i) r.add(tasks[i].N);
    return r;
}

}  // namespace qmm
