// vbs_kern_linear.hip — the general linear (matvec) kernel, k_rows: every
// hot-path weight type, one vector or up to 16, any shape; and the dispatch
// of the linear entry points to the matrix-core kernels or to it.
//
// Semantics: vbs_host_linear_tile (src/vbs_host_math.h:223-267) —
// y[r] (+)= sum_c deq(W[r,c]) * x[c]. Each weight is dequantised with the
// reference's exact roundings (vbs_dev_common.h) and then accumulated in
// fp32 with fused multiply-adds; rows are reduced across the wavefront.
#include "vbs_dev_common.h"
#include "vbs_internal.h"
#include "vbs_lds_dma.h"
#include "vbs_row8.h"

namespace vbs {

namespace {

// The value that lane l ^ M holds.
template <uint32_t M>
__device__ __forceinline__ float xor_lane(float v) {
    if constexpr (M >= 16u) {
        return lane_xor<(int)M>(v);
    } else if constexpr (M == 4u) {  // (lanes of even quads from above, of odd ones from below)
        const int i = __builtin_bit_cast(int, v);
        const int t = __builtin_amdgcn_update_dpp(0, i, 0x104, 0xF, 0x5, false);
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(t, i, 0x114, 0xF, 0xA, false));
    } else {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                                                     M == 8u ? 0x128 : M == 2u ? 0x4E : 0xB1, 0xF, 0xF,
                                                                     false));
    }
}
// wave_sum of each of N values (a power of two), bit for bit: every lane of the
// k-th group of 64 / N gets the k-th sum. Each step halves the values a lane
// carries, so N of them take about 2 N exchanges instead of 6 N.
template <uint32_t N, uint32_t M = 32>
__device__ __forceinline__ float wave_sums(const float (&v)[N], uint32_t lane) {
    if constexpr (M == 0u) {
        return v[0];
    } else if constexpr (N == 1u) {
        const float t[1] = {v[0] + xor_lane<M>(v[0])};
        return wave_sums<1u, M / 2u>(t, lane);
    } else {
        float t[N / 2u];
#pragma unroll
        for (uint32_t i = 0; i < N / 2u; i++) {
            const float own = lane & M ? v[i + N / 2u] : v[i], send = lane & M ? v[i] : v[i + N / 2u];
            t[i] = own + xor_lane<M>(send);
        }
        return wave_sums<N / 2u, M / 2u>(t, lane);
    }
}

// R rows and NB vectors per group of S waves (S = 1: every wave has rows of its
// own; else the workgroup's S waves split the row's steps and add their sums
// in wave order). A step is 512 elements of a row; U steps' loads go out
// together. With NB > 1 the eight weights serve every vector.
//
// Bound: HBM for the large shapes, the latency of one row's loads for the
// small ones (so few rows are split over sixteen waves). Measured, weights
// from HBM, against the kernels it replaced (a block or a 2-byte element per
// lane): 11008 x 4128 F16 120.6 -> 17.5 us (5.2 TB/s), F32 74.5 -> 33.5 (5.4),
// Q4_0 29.3 -> 13.3, Q8_0 37.0 -> 14.7, LNS8 28.0 -> 15.2; 2049 x 5664 Q4_0 9.4
// -> 6.1; 256 x 4128 F16 55.2 -> 2.8, Q4_0 5.3 -> 2.5. Vectors of their own
// loads: F32 11008 x 4128, 4 vectors 179 -> 42, 16 vectors 521 -> 116.
template <int T, uint32_t R, uint32_t NB, uint32_t S, uint32_t U>
__global__ __launch_bounds__(S > 4 ? 64 * S : 256) void k_rows(const uint8_t *__restrict__ w,
                                                               const float *__restrict__ x, uint32_t xs,
                                                               float *__restrict__ y, uint32_t ys,
                                                               uint32_t cols, uint32_t rows, uint64_t rb,
                                                               uint32_t batch, int accumulate) {
    typedef Row8<T> P;
    constexpr uint32_t kWaves = S > 4u ? S : 4u, kGroups = kWaves / S, L = P::E / 8u;  // lanes per block
    // rows on one wave (short ones): all NB vectors are formed, without a branch
    // between their loads; those past the batch repeat its last and are dropped
    constexpr bool kAll = NB > 1u && R <= 2u && S == 1u;
    __shared__ float red[S > 1 ? kWaves : 1][R * NB];
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    const uint32_t part = S > 1u ? wave % S : 0u;
    const uint32_t row0 = (blockIdx.x * kGroups + (S > 1u ? wave / S : wave)) * R;
    // whole blocks; cols of F16 / F32 may have a tail (rows of at most 64 elements
    // are all tail: a lane per element)
    const uint32_t q = lane % L, nu = P::E == 8u && cols <= 64u ? 0u : cols / P::E;
    const uint8_t *rp[R];
#pragma unroll
    for (uint32_t r = 0; r < R; r++) rp[r] = w + (uint64_t)min(row0 + r, rows - 1u) * rb;
    float acc[R][NB];
#pragma unroll
    for (uint32_t r = 0; r < R; r++)
#pragma unroll
        for (uint32_t b = 0; b < NB; b++) acc[r][b] = 0.f;
    if (row0 < rows) {
        for (uint32_t u0 = lane / L + (64u / L) * part; u0 < nu; u0 += (64u / L) * S * U) {
            typename P::Raw raw[U][R];
            v4f xa[U], xb[U];
#pragma unroll
            for (uint32_t k = 0; k < U; k++) {
                const uint32_t u = min(u0 + (64u / L) * S * k, nu - 1u);  // (past the row: its last block)
#pragma unroll
                for (uint32_t r = 0; r < R; r++) raw[k][r] = P::raw(rp[r], u, q);
                if constexpr (NB == 1u) {
                    const float *xp = x + P::E * u;
                    xa[k] = *reinterpret_cast<const f4u *>(xp + P::lo(q));
                    xb[k] = *reinterpret_cast<const f4u *>(xp + P::hi(q));
                }
            }
#pragma unroll
            for (uint32_t k = 0; k < U; k++) {
                const uint32_t u = u0 + (64u / L) * S * k;
                if (u >= nu) break;
                float wv[R][8];
#pragma unroll
                for (uint32_t r = 0; r < R; r++) P::value(raw[k][r], wv[r]);
#pragma unroll
                for (uint32_t b = 0; b < NB; b++) {
                    if (NB > 1u && !kAll && b >= batch) break;  // (uniform)
                    v4f a, c;
                    if constexpr (NB == 1u) {
                        a = xa[k], c = xb[k];
                    } else {
                        const float *xp = x + (uint64_t)(kAll ? min(b, batch - 1u) : b) * xs + P::E * u;
                        a = *reinterpret_cast<const f4u *>(xp + P::lo(q));
                        c = *reinterpret_cast<const f4u *>(xp + P::hi(q));
                    }
                    const float xv[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
#pragma unroll
                    for (uint32_t r = 0; r < R; r++) {
                        float s = 0.f;
#pragma unroll
                        for (int e = 0; e < 8; e++) s = fmaf(wv[r][e], xv[e], s);
                        acc[r][b] += s;
                    }
                }
            }
        }
        if (P::E == 8u && part == 0u) {  // the tail of F16 / F32 rows
            const uint32_t c = 8u * nu + lane;
            if (c < cols) {
                float wv[R];
#pragma unroll
                for (uint32_t r = 0; r < R; r++) wv[r] = deq_elem<T>(rp[r], c);
#pragma unroll
                for (uint32_t b = 0; b < NB; b++) {
                    if (NB > 1u && !kAll && b >= batch) break;
                    const float xv = x[(uint64_t)(kAll ? min(b, batch - 1u) : b) * xs + c];
#pragma unroll
                    for (uint32_t r = 0; r < R; r++) acc[r][b] = fmaf(wv[r], xv, acc[r][b]);
                }
            }
        }
    }
    // row r of vector b ends in the lanes of group r NB + b (R NB <= 64), or in LDS first
    float v[R * NB];
#pragma unroll
    for (uint32_t k = 0; k < R * NB; k++) v[k] = acc[k / NB][k % NB];
    float mine = wave_sums<R * NB>(v, lane);
    constexpr uint32_t kGroup = 64u / (R * NB);
    const uint32_t k = lane / kGroup, r = k / NB, b = k % NB;
    if (S > 1u) {
        if (lane % kGroup == 0u) red[wave][k] = mine;
        __syncthreads();
        if (part != 0u) return;
        mine = 0.f;
        for (uint32_t i = 0; i < S; i++) mine += red[wave + i][k];
    }
    if (lane % kGroup == 0u && row0 + r < rows && b < batch) {
        float *dst = y + (uint64_t)b * ys + row0 + r;
        *dst = accumulate ? *dst + mine : mine;
    }
}

template <int T, uint32_t R, uint32_t NB, uint32_t S, uint32_t U>
hipError_t launch_rows_t(const uint8_t *w, const float *x, uint32_t xs, float *y, uint32_t ys, uint32_t cols,
                         uint32_t rows, uint32_t batch, int accumulate, hipStream_t s) {
    constexpr uint32_t waves = S > 4u ? S : 4u, per = waves / S * R;
    k_rows<T, R, NB, S, U><<<(rows + per - 1u) / per, 64u * waves, 0, s>>>(w, x, xs, y, ys, cols, rows,
                                                                        row_bytes(T, cols), batch, accumulate);
    return hipGetLastError();
}

// Few rows: one per workgroup of sixteen waves (256 x 4128 F16 2.8 us, four
// waves 3.5, one 6.5). Up to 3072 rows: two rows per workgroup of four waves
// (1000 x 10528 Q4_0 6.0 us; one row on sixteen 6.7, four rows 8.7; 2049 x 5664
// F16 6.7 / 10.3 / 6.4). Above, four rows share x (11008 x 4128 F16 17.5 us,
// two rows 18.7, one 20.8), by a wave each where a row is under four steps
// (32000 x 1056 Q4_0 12.0 us against 14.6). Several vectors alike: 4, 16 vectors,
// F32 256 x 4128 4.1, 7.3 us (a wave per row 10.5, 24.8), 1000 x 10528 13.5, 38.7
// (29.1, 100), 11008 x 4128 42.1, 115 (55.9, 147).
// Rows of no more steps than that split has waves leave waves idle, so short
// rows take fewer: one wave at a step (512 elements; two for one vector and
// 513-3072 rows), two rows a wave past 3072 rows (one vector past 16384 four:
// 32000 x 96 F16 4.4 us, two 4.7), with as many sums as there are
// vectors (us, before the split went by length -> now: F32 32000 x 32, 16 vectors
// 99.9 -> 9.4, x 256 104 -> 24.1, 5000 x 96, 8 vectors 11.8 -> 4.2; Q4_0 512 x 96
// one vector 2.69 -> 2.27, 1000 x 544 2.92 -> 2.56; one and four rows a wave
// at 32000 x 256 F32, 8 vectors 24.9 and 17.0, two 16.7), four at up to four
// steps of few rows (512 x 1024 F32, 16 vectors 7.2 -> 4.7; one wave 7.2).
template <int T>
hipError_t launch_rows(const uint8_t *w, const float *x, uint32_t xs, float *y, uint32_t ys, uint32_t cols,
                       uint32_t rows, uint32_t batch, int accumulate, hipStream_t s) {
#define VBS_ROWS(R, NB, S, U) \
    return launch_rows_t<T, R, NB, S, U>(w, x, xs, y, ys, cols, rows, batch, accumulate, s)
    if (batch == 1u) {
        if (cols <= (rows <= 512u ? 512u : rows <= 3072u ? 1024u : 0u)) VBS_ROWS(1, 1, 1, 1);
        if (rows <= 512u && cols <= 2048u) VBS_ROWS(1, 1, 4, 1);
        if (rows <= 512u) VBS_ROWS(1, 1, 16, 1);
        if (rows <= 3072u && cols <= 2048u) VBS_ROWS(2, 1, 4, 1);
        if (rows <= 3072u) VBS_ROWS(2, 1, 4, 2);
        if (cols <= 512u && rows <= 16384u) VBS_ROWS(2, 1, 1, 1);
        if (cols < 2048u) VBS_ROWS(4, 1, 1, 1);
        VBS_ROWS(4, 1, 4, 1);
    }
    if (cols <= 512u) {
        if (rows <= 3072u) {
            if (batch == 2u) VBS_ROWS(1, 2, 1, 1);
            if (batch <= 4u) VBS_ROWS(1, 4, 1, 1);
            if (batch <= 8u) VBS_ROWS(1, 8, 1, 1);
            VBS_ROWS(1, 16, 1, 1);
        }
        if (batch == 2u) VBS_ROWS(2, 2, 1, 1);
        if (batch <= 4u) VBS_ROWS(2, 4, 1, 1);
        if (batch <= 8u) VBS_ROWS(2, 8, 1, 1);
        VBS_ROWS(2, 16, 1, 1);
    }
    if (batch <= 4u) {
        if (rows <= 512u && cols <= 2048u) VBS_ROWS(1, 4, 4, 1);
        if (rows <= 512u) VBS_ROWS(1, 4, 16, 1);
        if (rows <= 3072u) VBS_ROWS(2, 4, 4, 1);
        VBS_ROWS(4, 4, 1, 1);
    }
    if (rows <= 512u && cols <= 2048u) VBS_ROWS(1, 16, 4, 1);
    if (rows <= 512u) VBS_ROWS(1, 16, 16, 1);
    VBS_ROWS(2, 16, 4, 1);
#undef VBS_ROWS
}

hipError_t launch_rows_any(int type, const uint8_t *w, const float *x, uint32_t xs, float *y, uint32_t ys,
                           uint32_t cols, uint32_t rows, uint32_t batch, int accumulate, hipStream_t s) {
    switch (type) {
        case kF32: return launch_rows<kF32>(w, x, xs, y, ys, cols, rows, batch, accumulate, s);
        case kF16: return launch_rows<kF16>(w, x, xs, y, ys, cols, rows, batch, accumulate, s);
        case kQ4_0: return launch_rows<kQ4_0>(w, x, xs, y, ys, cols, rows, batch, accumulate, s);
        case kQ4_1: return launch_rows<kQ4_1>(w, x, xs, y, ys, cols, rows, batch, accumulate, s);
        case kQ8_0: return launch_rows<kQ8_0>(w, x, xs, y, ys, cols, rows, batch, accumulate, s);
        case kQ4_K: return launch_rows<kQ4_K>(w, x, xs, y, ys, cols, rows, batch, accumulate, s);
        case kQ6_K: return launch_rows<kQ6_K>(w, x, xs, y, ys, cols, rows, batch, accumulate, s);
        case kLNS8: return launch_rows<kLNS8>(w, x, xs, y, ys, cols, rows, batch, accumulate, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t launch_linear(int type, const uint8_t *w, const float *x, float *y, uint32_t cols,
                         uint32_t rows, int accumulate, hipStream_t s) {
    if (rows == 0) return hipSuccess;
    if (type == kQ4_K || type == kQ6_K || type == kQ4_0 || type == kQ4_1 || type == kQ8_0) {
        hipError_t e = launch_kq_linear(type, w, x, y, cols, rows, accumulate, s);
        if (e != hipErrorNotSupported) return e;
    }
    if (type == kQ4_K) {
        hipError_t e = launch_q4k_fast(w, x, y, cols, rows, accumulate, s);
        if (e != hipErrorNotSupported) return e;
    }
    return launch_rows_any(type, w, x, cols, y, rows, cols, rows, 1u, accumulate, s);
}

hipError_t launch_linear_batch(int type, const uint8_t *w, const float *x, uint32_t xs, float *y,
                               uint32_t ys, uint32_t cols, uint32_t rows, uint32_t batch,
                               hipStream_t s) {
    if (rows == 0 || batch == 0) return hipSuccess;
    // K-quants: the matrix-core kernel, eight vectors per launch
    if (type == kQ4_K || type == kQ6_K) {
        hipError_t e = hipSuccess;
        for (uint32_t b0 = 0; b0 < batch && e == hipSuccess; b0 += 8u)
            e = launch_kq_linear_batch(type, w, x + (uint64_t)b0 * xs, xs, y + (uint64_t)b0 * ys, ys,
                                       cols, rows, min(8u, batch - b0), s);
        if (e != hipErrorNotSupported) return e;  // the shape check fails on the first launch
    }
    {  // Q4_0, Q4_1, Q8_0 and F16: the matrix cores again, all vectors in one launch
        const hipError_t e = launch_blk_linear_batch(type, 1u, &w, &rows, x, xs, &y, &ys, cols, batch, s);
        if (e != hipErrorNotSupported) return e;
    }
    return launch_rows_any(type, w, x, xs, y, ys, cols, rows, batch, 0, s);
}

}  // namespace vbs
