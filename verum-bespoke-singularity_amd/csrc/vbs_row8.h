// vbs_row8.h — eight consecutive weights of a packed row per lane, as the
// general linear kernel reads rows (k_rows, vbs_kern_linear.hip) and the batched
// matrix-core kernel takes single rows again (vbs_kern_mfma_batch_blk.hip).
#pragma once

#include "vbs_dev_common.h"

namespace vbs {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t __attribute__((aligned(2))) u32h;  // words at a 2-byte aligned address
typedef uint32_t u2h __attribute__((ext_vector_type(2), aligned(2)));

// A step's share of a row: a lane takes eight elements. Blocks of 32: lane l
// takes block l >> 2 of the step's sixteen, its quarter q = l & 3 being the
// elements lo(q) .. + 3 and hi(q) .. + 3 (the two nibbles of four bytes; else
// eight in a row). raw() loads the bytes, value() makes the eight weights.
template <int T> struct Row8;
typedef uint32_t u4h __attribute__((ext_vector_type(4), aligned(2)));
// K-quants (what the matrix cores do not take: bases off their alignment, rows
// past 32768 columns): the 32-element sub-blocks of a 256-element block are the
// blocks of 32, and the sub-block's scale is formed once per eight elements.
// Weights from HBM: Q4_K 4096 x 4096 9.9 us at a 2-byte base (per element through
// deq_elem 40.4, a lane per sub-block 13.4), 4096 x 40960 52 (388, 89); Q6_K 4096 x
// 4096 9.6 (20.6, 13.9).
template <> struct Row8<kQ4_K> {
    struct Raw {
        u4h h;  // d, dmin and the twelve scale bytes
        u2h q;
        uint32_t j;
    };
    static constexpr uint32_t E = 32;
    __device__ static uint32_t lo(uint32_t q) { return 8u * q; }
    __device__ static uint32_t hi(uint32_t q) { return 8u * q + 4u; }
    __device__ static Raw raw(const uint8_t *row, uint32_t u, uint32_t q) {
        const uint8_t *b = row + (uint64_t)(u >> 3) * 144u;
        const uint32_t j = u & 7u;
        return Raw{*reinterpret_cast<const u4h *>(b),
                   *reinterpret_cast<const u2h *>(b + 16u + 32u * (j >> 1) + 8u * q), j};
    }
    __device__ static void value(const Raw &r, float (&w)[8]) {
        const float d = h2f((uint16_t)r.h[0]), dmin = h2f((uint16_t)(r.h[0] >> 16));
        // (the scale bytes j mod 4, 4 + j mod 4 and 8 + j mod 4: q4k_scale_min)
        const uint32_t s = 8u * (r.j & 3u), a = r.h[1] >> s, b = r.h[2] >> s, c = r.h[3] >> s;
        const uint32_t sc = r.j < 4u ? a & 63u : (c & 15u) | ((a >> 6 & 3u) << 4);
        const uint32_t mn = r.j < 4u ? b & 63u : (c >> 4 & 15u) | ((b >> 6 & 3u) << 4);
        const float ds = __fmul_rn(d, (float)sc), dm = __fmul_rn(dmin, (float)mn);
        const uint32_t sh = 4u * (r.j & 1u);
#pragma unroll
        for (int k = 0; k < 8; k++)
            w[k] = __fsub_rn(__fmul_rn(ds, (float)(r.q[k >> 2] >> (8 * (k & 3) + sh) & 15u)), dm);
    }
};
template <> struct Row8<kQ6_K> {
    struct Raw {
        u2h l, h;
        uint32_t j;
        uint16_t d;
        int8_t s;
    };
    static constexpr uint32_t E = 32;
    __device__ static uint32_t lo(uint32_t q) { return 8u * q; }
    __device__ static uint32_t hi(uint32_t q) { return 8u * q + 4u; }
    __device__ static Raw raw(const uint8_t *row, uint32_t u, uint32_t q) {
        const uint8_t *b = row + (uint64_t)(u >> 3) * 210u;
        const uint32_t j = u & 7u, h = j >> 2;
        return Raw{*reinterpret_cast<const u2h *>(b + 64u * h + 32u * (j & 1u) + 8u * q),
                   *reinterpret_cast<const u2h *>(b + 128u + 32u * h + 8u * q), j & 3u, ld16(b + 208),
                   (int8_t)b[192u + 2u * j + (q >> 1)]};
    }
    __device__ static void value(const Raw &r, float (&w)[8]) {
        const float ds = __fmul_rn(h2f(r.d), (float)r.s);
        const uint32_t lsh = r.j & 2u ? 4u : 0u, hsh = 2u * r.j;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t lo = r.l[k >> 2] >> (8 * (k & 3) + lsh) & 15u, hi = r.h[k >> 2] >> (8 * (k & 3) + hsh) & 3u;
            w[k] = __fmul_rn(ds, (float)((int)(lo | hi << 4) - 32));
        }
    }
};
template <int T> struct Nib8 {  // Q4_0, Q4_1
    struct Raw {
        uint32_t q;
        uint16_t d, m;
    };
    static constexpr uint32_t E = 32;
    __device__ static uint32_t lo(uint32_t q) { return 4u * q; }
    __device__ static uint32_t hi(uint32_t q) { return 16u + 4u * q; }
    __device__ static Raw raw(const uint8_t *row, uint32_t u, uint32_t q) {
        const uint8_t *b = row + (uint64_t)u * Geo<T>::B;
        return Raw{*reinterpret_cast<const u32h *>(b + (T == kQ4_0 ? 2u : 4u) + 4u * q), ld16(b),
                   T == kQ4_0 ? (uint16_t)0 : ld16(b + 2)};
    }
    __device__ static void value(const Raw &r, float (&w)[8]) {
        const float d = h2f(r.d), m = h2f(r.m);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float n = (float)((r.q >> (8 * (k & 3) + (k >> 2) * 4)) & 15u);
            w[k] = T == kQ4_0 ? __fmul_rn(n - 8.0f, d) : __fadd_rn(__fmul_rn(d, n), m);
        }
    }
};
template <> struct Row8<kQ4_0> : Nib8<kQ4_0> {};
template <> struct Row8<kQ4_1> : Nib8<kQ4_1> {};
template <> struct Row8<kQ8_0> {
    struct Raw {
        uint32_t q[2];
        uint16_t d;
    };
    static constexpr uint32_t E = 32;
    __device__ static uint32_t lo(uint32_t q) { return 8u * q; }
    __device__ static uint32_t hi(uint32_t q) { return 8u * q + 4u; }
    __device__ static Raw raw(const uint8_t *row, uint32_t u, uint32_t q) {
        const uint8_t *b = row + (uint64_t)u * 34u;
        const u32h *p = reinterpret_cast<const u32h *>(b + 2u + 8u * q);
        return Raw{{p[0], p[1]}, ld16(b)};
    }
    __device__ static void value(const Raw &r, float (&w)[8]) {
        const float d = h2f(r.d);
#pragma unroll
        for (int k = 0; k < 8; k++)
            w[k] = __fmul_rn(d, (float)(int8_t)(r.q[k >> 2] >> (8 * (k & 3))));
    }
};
template <> struct Row8<kLNS8> {  // exp2f(code) * scale, as deq_elem<kLNS8>
    struct Raw {
        u2h q;
        float s;
    };
    static constexpr uint32_t E = 32;
    __device__ static uint32_t lo(uint32_t q) { return 8u * q; }
    __device__ static uint32_t hi(uint32_t q) { return 8u * q + 4u; }
    __device__ static Raw raw(const uint8_t *row, uint32_t u, uint32_t q) {
        const uint8_t *b = row + (uint64_t)u * 36u;
        return Raw{*reinterpret_cast<const u2h *>(b + 8u * q), *reinterpret_cast<const float *>(b + 32)};
    }
    __device__ static void value(const Raw &r, float (&w)[8]) {
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t c = (r.q[k >> 2] >> (8 * (k & 3))) & 255u;
            w[k] = __fmul_rn(c < 128u ? __uint_as_float((c + 127u) << 23) : INFINITY, r.s);
        }
    }
};
// F16, F32: lane l takes elements 8 l .. 8 l + 7 of the step's 512 ("blocks" of
// 8); rows may start at any element, so the loads are only element-aligned.
template <> struct Row8<kF16> {
    struct Raw {
        u4h v;
    };
    static constexpr uint32_t E = 8;
    __device__ static uint32_t lo(uint32_t) { return 0u; }
    __device__ static uint32_t hi(uint32_t) { return 4u; }
    __device__ static Raw raw(const uint8_t *row, uint32_t u, uint32_t) {
        return Raw{*reinterpret_cast<const u4h *>(row + 16ull * u)};
    }
    __device__ static void value(const Raw &r, float (&w)[8]) {
#pragma unroll
        for (int k = 0; k < 8; k++)
            w[k] = (float)__builtin_bit_cast(_Float16, (uint16_t)(r.v[k >> 1] >> (16 * (k & 1))));
    }
};
template <> struct Row8<kF32> {
    struct Raw {
        v4f a, b;
    };
    static constexpr uint32_t E = 8;
    __device__ static uint32_t lo(uint32_t) { return 0u; }
    __device__ static uint32_t hi(uint32_t) { return 4u; }
    __device__ static Raw raw(const uint8_t *row, uint32_t u, uint32_t) {
        const f4u *p = reinterpret_cast<const f4u *>(row + 32ull * u);
        return Raw{p[0], p[1]};
    }
    __device__ static void value(const Raw &r, float (&w)[8]) {
        w[0] = r.a.x, w[1] = r.a.y, w[2] = r.a.z, w[3] = r.a.w;
        w[4] = r.b.x, w[5] = r.b.y, w[6] = r.b.z, w[7] = r.b.w;
    }
};

}  // namespace vbs
