// vbs_kern_hot.hip — the CPU hot-kernel table's arithmetic (ABI v1,
// include/vbs_hotpath.h:38-57 of the reference) and the CPU model's Q8
// activation quantiser, on gfx950, bit-identical to the reference.
//
// The table's contract fixes the float order: one sum per row, added to block
// by block (element by element for F32/F16) in column order
// (src/hotkernels/vbs_hot_ref_impl.h:49-129). The kernels form the terms (what
// is exact: integer dots on v_dot4_i32_i8, each product rounded separately)
// with all lanes and leave them in LDS in column order; then one lane per row
// adds its row's terms in turn. Every product and sum is an explicitly rounded
// intrinsic, so nothing is fused.
#include <type_traits>

#include "vbs_dev_common.h"
#include "vbs_internal.h"

namespace vbs {

enum : int { HK_Q8_0 = 0, HK_Q4_0 = 1, HK_Q4_1 = 2, HK_F32 = 3, HK_F16 = 4 };

typedef uint32_t __attribute__((aligned(2))) w32h;  // a word at a 2-byte aligned address
typedef int i2w __attribute__((ext_vector_type(2), aligned(4)));
typedef float f4w __attribute__((ext_vector_type(4)));
typedef float f4e __attribute__((ext_vector_type(4), aligned(4)));
typedef uint16_t h4w __attribute__((ext_vector_type(4)));
typedef uint16_t h4e __attribute__((ext_vector_type(4), aligned(2)));

template <int CTRL>
__device__ __forceinline__ int dpp_add_i(int v) {
    return v + __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}

// sum += t[0], t[1], ... t[n - 1] in turn (t 16-byte aligned, in LDS, of which
// `size` >= 32 terms may be read), the next 32 requested while 32 are added.
__device__ __forceinline__ float add_in_order(float sum, const float *t, uint32_t n, uint32_t size) {
    f4w a[8], b[8];
    auto get = [&](uint32_t k0, f4w (&v)[8]) {
        const float *p = t + min(k0, size - 32u);
#pragma unroll
        for (uint32_t i = 0; i < 8u; i++) v[i] = *reinterpret_cast<const f4w *>(p + 4u * i);
    };
    auto add = [&](const f4w (&v)[8]) {
#pragma unroll
        for (uint32_t i = 0; i < 32u; i++) sum = __fadd_rn(sum, v[i >> 2][i & 3u]);
    };
    auto rest = [&](uint32_t k0, const f4w (&v)[8]) {
#pragma unroll
        for (uint32_t i = 0; i < 32u; i++)
            if (k0 + i < n) sum = __fadd_rn(sum, v[i >> 2][i & 3u]);
    };
    get(0u, a);
    uint32_t k0 = 0;
    for (; k0 + 64u <= n; k0 += 64u) {
        get(k0 + 32u, b);
        add(a);
        get(k0 + 64u, a);
        add(b);
    }
    if (k0 + 32u <= n) {
        get(k0 + 32u, b);
        add(a);
        rest(k0 + 32u, b);
    } else {
        rest(k0, a);
    }
    return sum;
}

__device__ __forceinline__ float lane_f(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// f16 bits -> f32: the hardware's conversion but for inf and NaN (h2f's bits).
__device__ __forceinline__ float hot_h2f(uint16_t h) {
    const float v = (float)__builtin_bit_cast(_Float16, h);
    return __builtin_expect((h & 0x7C00u) == 0x7C00u, 0) ? h2f(h) : v;
}

// Block types: a row per wave, four rows per workgroup, so that the sums of
// some workgroups run under the loads of others. A lane takes a quarter of a
// block (as k_rows, vbs_kern_linear.hip), sixteen blocks per step, the quads
// add their integer dots, and kHotBlocks blocks' terms at a time wait in LDS;
// rows of one or two steps (REG) need no LDS and no barrier: the wave adds its
// row's terms from the lanes that hold them, those past the row as +0, which
// leaves a sum that began at +0 its bits.
// Bound: the loads' latency, then HBM. Q8_0 4096 x 4096 10.2 -> 7.6 us (2.3
// TB/s), 1000 x 11008 17.9 -> 7.9, Q4_0 4096 x 4096 9.2 -> 6.2, Q4_1 11008 x 4096
// 26.2 -> 11.1 against the kernel before, which took a whole block per lane, in
// 2-byte pieces, and added every term on all lanes through lane reads.
constexpr uint32_t kHotBlocks = 512;

template <int K, uint32_t U, bool REG>
__global__ __launch_bounds__(256) void k_hot_blocks(const uint8_t *__restrict__ w, uint32_t rows,
                                                    uint32_t nblk, const int8_t *__restrict__ xq,
                                                    const float *__restrict__ qd,
                                                    const float *__restrict__ qsum,
                                                    float *__restrict__ y) {
    constexpr uint32_t kBytes = K == HK_Q8_0 ? 34u : K == HK_Q4_0 ? 18u : 20u;
    constexpr uint32_t N = K == HK_Q4_1 ? 2u : 1u;  // terms per block
    constexpr uint32_t kSize = kHotBlocks * N;
    __shared__ __align__(16) float terms[REG ? 1 : 4][REG ? 4 : kSize + 4u];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, q = lane & 3u;
    const uint32_t row = blockIdx.x * 4u + wave;
    const uint8_t *const rp = w + (uint64_t)min(row, rows - 1u) * nblk * kBytes;
    float sum = 0.0f;
    for (uint32_t c0 = 0; c0 < nblk; c0 += kHotBlocks) {
        const uint32_t n = min(kHotBlocks, nblk - c0);
        for (uint32_t b0 = 0; b0 < n; b0 += 16u * U) {  // (U steps' loads together)
            uint32_t p[U][K == HK_Q8_0 ? 2 : 1];
            int xw[U][2];
            uint16_t d[U], m[U];
            float xd[U], xs[U];
#pragma unroll
            for (uint32_t k = 0; k < U; k++) {
                const uint32_t u = c0 + min(b0 + 16u * k + (lane >> 2), n - 1u);
                const uint8_t *blk = rp + (uint64_t)u * kBytes;
                const int8_t *xb = xq + (uint64_t)u * 32u;
                if constexpr (K == HK_Q8_0) {
                    const w32h *wp = reinterpret_cast<const w32h *>(blk + 2u + 8u * q);
                    p[k][0] = wp[0], p[k][1] = wp[1];
                    const i2w xv = *reinterpret_cast<const i2w *>(xb + 8u * q);
                    xw[k][0] = xv.x, xw[k][1] = xv.y;
                } else {
                    p[k][0] = *reinterpret_cast<const w32h *>(blk + (K == HK_Q4_0 ? 2u : 4u) + 4u * q);
                    xw[k][0] = *reinterpret_cast<const int *>(xb + 4u * q);
                    xw[k][1] = *reinterpret_cast<const int *>(xb + 16u + 4u * q);
                }
                d[k] = ld16(blk);
                xd[k] = qd[u];
                if constexpr (K == HK_Q4_1) m[k] = ld16(blk + 2), xs[k] = qsum[u];
            }
#pragma unroll
            for (uint32_t k = 0; k < U; k++) {
                const uint32_t b = b0 + 16u * k + (lane >> 2);
                int dot = 0;
                if constexpr (K == HK_Q8_0) {
                    dot = __builtin_amdgcn_sdot4((int)p[k][0], xw[k][0], dot, false);
                    dot = __builtin_amdgcn_sdot4((int)p[k][1], xw[k][1], dot, false);
                } else {
                    // nibbles 0..15 are valid int8 lanes; Q4_0's "- 8" is applied as
                    // -8 * sum(xq), which is the same integer
                    dot = __builtin_amdgcn_sdot4((int)(p[k][0] & 0x0F0F0F0Fu), xw[k][0], dot, false);
                    dot = __builtin_amdgcn_sdot4((int)((p[k][0] >> 4) & 0x0F0F0F0Fu), xw[k][1], dot, false);
                    if constexpr (K == HK_Q4_0) {
                        int s8 = __builtin_amdgcn_sdot4(0x01010101, xw[k][0], 0, false);
                        s8 = __builtin_amdgcn_sdot4(0x01010101, xw[k][1], s8, false);
                        dot -= 8 * s8;
                    }
                }
                dot = dpp_add_i<0xB1>(dot);  // the block's four lanes
                dot = dpp_add_i<0x4E>(dot);
                const float t0 = __fmul_rn(__fmul_rn(hot_h2f(d[k]), xd[k]), (float)dot);
                if constexpr (REG) {
                    if (16u * k >= n) break;
                    float t1 = 0.0f;
                    if constexpr (K == HK_Q4_1) t1 = b < n ? __fmul_rn(hot_h2f(m[k]), xs[k]) : 0.0f;
                    const float t = b < n ? t0 : 0.0f;
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        sum = __fadd_rn(sum, lane_f(t, 4 * i));
                        if constexpr (K == HK_Q4_1) sum = __fadd_rn(sum, lane_f(t1, 4 * i));
                    }
                } else if (q == 0u && b < n) {
                    terms[wave][N * b] = t0;
                    if constexpr (K == HK_Q4_1) terms[wave][2u * b + 1u] = __fmul_rn(hot_h2f(m[k]), xs[k]);
                }
            }
        }
        if constexpr (REG) break;
        __syncthreads();
        if (threadIdx.x < 4u) sum = add_in_order(sum, terms[threadIdx.x], N * n, kSize);
        if (c0 + kHotBlocks < nblk) __syncthreads();
    }
    if constexpr (REG) {
        if (lane == 0u && row < rows) y[row] = sum;
    } else if (threadIdx.x < 4u && blockIdx.x * 4u + threadIdx.x < rows) {
        y[blockIdx.x * 4u + threadIdx.x] = sum;
    }
}

// F32 and F16: a term per element, so a row's sum is a chain of `cols` adds
// and bounds the kernel (~5 ns each: 2048 of them alone take 10 us). Sixteen
// rows per workgroup: four waves form the products of 256 columns (four rows
// each, kHotAhead tiles of loads under way), a fifth adds the tile before, a
// lane per row. 4096 x 4096 F32 161 -> 27 us, F16 170 -> 24; 3 x 2048 67 -> 12
// against the kernel before, which issued two instructions per term and row.
constexpr uint32_t kHotRows = 16, kHotCols = 256, kHotAhead = 4;

template <int K>
__global__ __launch_bounds__(320) void k_hot_float(const uint8_t *__restrict__ w, uint32_t rows,
                                                   uint32_t cols, const float *__restrict__ x,
                                                   float *__restrict__ y) {
    __shared__ __align__(16) float terms[2][kHotRows][kHotCols + 4u];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    typedef typename std::conditional<K == HK_F32, float, uint16_t>::type E;
    typedef typename std::conditional<K == HK_F32, f4w, h4w>::type Raw;
    typedef typename std::conditional<K == HK_F32, f4e, h4e>::type E4;
    const uint32_t row0 = blockIdx.x * kHotRows, full = cols / kHotCols, tail = cols % kHotCols;
    const bool maker = wave != 0u;
    const uint32_t mr = maker ? 4u * (wave - 1u) : 0u;  // a maker wave's first row of the sixteen
    const E *rp[4];
#pragma unroll
    for (uint32_t r = 0; r < 4u; r++)
        rp[r] = reinterpret_cast<const E *>(w) + (uint64_t)min(row0 + mr + r, rows - 1u) * cols;
    auto value = [](E v) {
        if constexpr (K == HK_F32) return v;
        else return hot_h2f(v);
    };
    Raw wv[kHotAhead][4];
    f4w xv[kHotAhead];
    auto load = [&](uint32_t t, Raw (&a)[4], f4w &b) {
        const uint32_t e0 = t * kHotCols + 4u * lane;
        b = *reinterpret_cast<const f4e *>(x + e0);
#pragma unroll
        for (uint32_t r = 0; r < 4u; r++) a[r] = *reinterpret_cast<const E4 *>(rp[r] + e0);
    };
    float sum = 0.0f;
    if (maker && full) {
#pragma unroll
        for (uint32_t k = 0; k < kHotAhead; k++) load(min(k, full - 1u), wv[k], xv[k]);
    }
    // round t: the makers write tile t (the last one, a part, one element at a
    // time), wave 0 adds tile t - 1
    const uint32_t tiles = full + (tail != 0u);
    for (uint32_t t0 = 0; t0 <= tiles; t0 += kHotAhead) {
#pragma unroll
        for (uint32_t k = 0; k < kHotAhead; k++) {
            const uint32_t t = t0 + k;
            if (t > tiles) break;
            if (maker) {
                if (t < full) {
#pragma unroll
                    for (uint32_t r = 0; r < 4u; r++) {
                        f4w p;
#pragma unroll
                        for (uint32_t e = 0; e < 4u; e++) p[e] = __fmul_rn(value(wv[k][r][e]), xv[k][e]);
                        *reinterpret_cast<f4w *>(&terms[t & 1u][mr + r][4u * lane]) = p;
                    }
                    load(min(t + kHotAhead, full - 1u), wv[k], xv[k]);
                } else if (t < tiles) {
                    for (uint32_t e = lane; e < tail; e += 64u) {
                        const float xe = x[t * kHotCols + e];
                        E v[4];
#pragma unroll
                        for (uint32_t r = 0; r < 4u; r++) v[r] = rp[r][t * kHotCols + e];
#pragma unroll
                        for (uint32_t r = 0; r < 4u; r++) terms[t & 1u][mr + r][e] = __fmul_rn(value(v[r]), xe);
                    }
                }
            } else if (t > 0u && lane < kHotRows) {
                sum = add_in_order(sum, terms[(t - 1u) & 1u][lane], t <= full ? kHotCols : tail, kHotCols);
            }
            __syncthreads();
        }
    }
    if (wave == 0u && lane < kHotRows && row0 + lane < rows) y[row0 + lane] = sum;
}

// One thread per 32-element block (src/vbs_cpu.c:166-182).
__global__ __launch_bounds__(256) void k_quantize_q8(const float *__restrict__ x, uint32_t nblk,
                                                     int8_t *__restrict__ xq,
                                                     float *__restrict__ qd,
                                                     float *__restrict__ qsum) {
    const uint32_t b = blockIdx.x * 256u + threadIdx.x;
    if (b >= nblk) return;
    const float *xb = x + (uint64_t)b * 32u;
    float v[32];
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; i++) {
        v[i] = xb[i];
        amax = fabsf(v[i]) > amax ? fabsf(v[i]) : amax;
    }
    const float d = __fdiv_rn(amax, 127.0f);
    const float inv = d != 0.0f ? __fdiv_rn(1.0f, d) : 0.0f;
    int total = 0;
    uint32_t packed[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        uint32_t word = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            int q = (int)roundf(__fmul_rn(v[4 * j + i], inv));
            q = q < -127 ? -127 : (q > 127 ? 127 : q);
            total += q;
            word |= ((uint32_t)q & 255u) << (8 * i);
        }
        packed[j] = word;
    }
    uint32_t *out = reinterpret_cast<uint32_t *>(xq + (uint64_t)b * 32u);
#pragma unroll
    for (int j = 0; j < 8; j++) out[j] = packed[j];
    qd[b] = h2f(vbs_f2h_rne(d));
    qsum[b] = h2f(vbs_f2h_rne(__fmul_rn((float)total, d)));
}

}  // namespace vbs

using namespace vbs;

static bool aligned(const void *p, uintptr_t a) { return ((uintptr_t)p & (a - 1)) == 0; }

extern "C" {

int vbs_gfx950_quantize_q8(const float *x, uint32_t cols, int8_t *xq, float *qd, float *qsum) {
    if (!rt_ready()) return 0;
    if (cols % 32u) return rt_fail("quantize_q8: cols %u not a multiple of 32", cols);
    if (cols == 0) return 1;
    if (!x || !xq || !qd || !qsum) return rt_fail("quantize_q8: null pointer");
    if (!aligned(x, 4) || !aligned(xq, 4) || !aligned(qd, 4) || !aligned(qsum, 4))
        return rt_fail("quantize_q8: buffers must be 4-byte aligned");
    const uint32_t nblk = cols / 32u;
    hipLaunchKernelGGL(k_quantize_q8, dim3((nblk + 255u) / 256u), dim3(256), 0, rt_stream(), x,
                       nblk, xq, qd, qsum);
    return rt_hip_ok(hipGetLastError(), "quantize_q8");
}

int vbs_gfx950_hot_matvec(int type, const void *w, uint32_t rows, uint32_t cols, const void *act,
                          const float *qd, const float *qsum, float *y) {
    if (!rt_ready()) return 0;
    int kind;
    switch (type) {
        case kQ8_0: kind = HK_Q8_0; break;
        case kQ4_0: kind = HK_Q4_0; break;
        case kQ4_1: kind = HK_Q4_1; break;
        case kF32: kind = HK_F32; break;
        case kF16: kind = HK_F16; break;
        default: return rt_fail("hot_matvec: type %d is not in the hot-kernel table", type);
    }
    const bool quant = kind <= HK_Q4_1;
    if (quant && cols % 32u) return rt_fail("hot_matvec: cols %u not a multiple of 32", cols);
    if (rows == 0) return 1;
    if (rows > 0x7FFFFFFFu) return rt_fail("hot_matvec: too many rows (%u)", rows);
    if (!y || (cols && (!w || !act))) return rt_fail("hot_matvec: null pointer");
    if (quant && cols && (!qd || (kind == HK_Q4_1 && !qsum)))
        return rt_fail("hot_matvec: null activation scales");
    if (!aligned(w, kind == HK_F32 ? 4 : 2) || !aligned(act, 4) || !aligned(y, 4) ||
        !aligned(qd, 4) || !aligned(qsum, 4))
        return rt_fail("hot_matvec: misaligned buffer");
    const uint8_t *wb = static_cast<const uint8_t *>(w);
    hipStream_t s = rt_stream();
    if (quant) {
        const dim3 grid((rows + 3u) / 4u), block(256);
        const int8_t *xq = static_cast<const int8_t *>(act);
        // loads of U steps of 16 blocks together: no more than short rows have (16000
        // x 320 Q8_0 6.3 us with one, 13.2 with eight; 4096 x 4096 12.9 / 7.6; 16000 x
        // 544 5.9 with two, 8.5 with four). Terms added from the lanes against LDS:
        // Q8_0 1 x 32 2.06 / 2.25, 16000 x 320 4.29 / 5.65, 4096 x 1024 3.17 / 3.53; but
        // of 64 blocks Q4_0 8000 x 2048 5.70 / 5.30, and of Q4_1's two terms a block
        // 16000 x 544 7.6 / 6.0 (256 x 544 2.47 / 2.68)
#define VBS_HOT_L(K, U, R) hipLaunchKernelGGL((k_hot_blocks<K, U, R>), grid, block, 0, s, wb, rows, cols / 32u, xq, qd, qsum, y)
#define VBS_HOT(K)                                               \
    do {                                                         \
        if (cols <= 512u) VBS_HOT_L(K, 1, true);                 \
        else if (cols <= 1024u) VBS_HOT_L(K, 2, K != HK_Q4_1);   \
        else if (cols <= 2048u) VBS_HOT_L(K, 4, false);          \
        else VBS_HOT_L(K, 8, false);                             \
    } while (0)
        if (kind == HK_Q8_0) VBS_HOT(HK_Q8_0);
        else if (kind == HK_Q4_0) VBS_HOT(HK_Q4_0);
        else VBS_HOT(HK_Q4_1);
#undef VBS_HOT
#undef VBS_HOT_L
    } else {
        const dim3 grid((rows + kHotRows - 1u) / kHotRows), block(320);
        const float *x = static_cast<const float *>(act);
        if (kind == HK_F32) hipLaunchKernelGGL(k_hot_float<HK_F32>, grid, block, 0, s, wb, rows, cols, x, y);
        else hipLaunchKernelGGL(k_hot_float<HK_F16>, grid, block, 0, s, wb, rows, cols, x, y);
    }
    return rt_hip_ok(hipGetLastError(), "hot_matvec");
}

}  // extern "C"
