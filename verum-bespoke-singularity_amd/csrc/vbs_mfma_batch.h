// vbs_mfma_batch.h — what the batched (skinny) matvec kernels share: the
// prepared form of x (f16 hi/lo planes, vbs_kern_mfma_batch.hip explains it),
// its per-block preparation and the byte-to-f16 helpers of the unpacks.
#pragma once

#include "vbs_mfma.h"

namespace vbs {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kBatchMax = 8;

// Prepared x: [cols/8][16 planes][8] f16 | [cols/256][16 planes][8] f16
// sub-block sums of x'/32 | int s[cols/256][8] (block, vector).
struct XbLayout {
    uint32_t msum, expo, bytes;
};
__host__ __device__ inline XbLayout xb_layout(uint32_t cols) {
    XbLayout L;
    L.msum = 32u * cols;
    L.expo = 33u * cols;
    L.bytes = 33u * cols + cols / 8u;
    return L;
}

// Block b of vector t (one wave, lane l: elements 4l..4l+3 of the block in v)
// into the prepared form: its exponent, f16 hi/lo planes 2t and 2t + 1 and the
// sub-block sums of x'/32.
__device__ __forceinline__ void xprep_block(const float v[4], uint32_t lane, uint32_t t, uint32_t b,
                                            uint32_t cols, uint8_t *xp) {
    const uint32_t e0 = 256u * b + 4u * lane;
    const float amax = wave_max(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
    int e = 0;
    (void)frexpf(amax, &e);  // amax < 2^e
    const int s = amax > 0.f ? 15 - e : 0;
    h2 hi[2], lo[2];
    float sum = 0.f;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const float xs2 = ldexpf(v[k], s);
        const _Float16 h = (_Float16)xs2;
        hi[k >> 1][k & 1] = h;
        lo[k >> 1][k & 1] = (_Float16)(xs2 - (float)h);
        sum += xs2;
    }
    const XbLayout L = xb_layout(cols);
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    // elements e0..e0+3: chunk e0 / 8, half lane & 1; planes 2t and 2t + 1
    _Float16 *ph = reinterpret_cast<_Float16 *>(xp) + 128u * (e0 >> 3) + 8u * (2u * t) + 4u * (lane & 1u);
    *reinterpret_cast<u32x2 *>(ph) = u32x2{__builtin_bit_cast(uint32_t, hi[0]), __builtin_bit_cast(uint32_t, hi[1])};
    *reinterpret_cast<u32x2 *>(ph + 8u) = u32x2{__builtin_bit_cast(uint32_t, lo[0]), __builtin_bit_cast(uint32_t, lo[1])};
    // sub-block sums of x'/32: eight lanes per 32 elements
    sum += __shfl_xor(sum, 1, 64);
    sum += __shfl_xor(sum, 2, 64);
    sum += __shfl_xor(sum, 4, 64);
    if ((lane & 7u) == 0) {
        const float m = sum * 0.03125f;
        const _Float16 h = (_Float16)m;
        _Float16 *pm = reinterpret_cast<_Float16 *>(xp + L.msum) + 128u * b + 8u * (2u * t) + lane / 8u;
        pm[0] = h;
        pm[8] = (_Float16)(m - (float)h);
    }
    if (lane == 0) reinterpret_cast<int *>(xp + L.expo)[8u * b + t] = s;
}

// This lane's A row: its plane's first eight elements and first eight
// sub-block sums; element chunk c of the plane is at plane + 128 c, block b's
// sums at msum + 128 b.
struct XbView {
    const _Float16 *plane, *msum;
    const int *expo;
};

// {1024 + byte, 1024 + byte'} as an f16 pair: bytes (0, 1) of w for sel
// 0x00050004, (2, 3) for 0x00070006, (k, k) for 0x00040004 + 0x00010001 k.
__device__ __forceinline__ h2 f16_bytes(uint32_t w, uint32_t sel) {
    return __builtin_bit_cast(h2, __builtin_amdgcn_perm(w, 0x64646464u, sel));
}
__device__ __forceinline__ h8 join8(h2 a, h2 b, h2 c, h2 d) {
    const u32x4 v = {__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                     __builtin_bit_cast(uint32_t, c), __builtin_bit_cast(uint32_t, d)};
    return __builtin_bit_cast(h8, v);
}
__device__ __forceinline__ h4 join4(h2 a, h2 b) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 v = {__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b)};
    return __builtin_bit_cast(h4, v);
}

}  // namespace vbs
