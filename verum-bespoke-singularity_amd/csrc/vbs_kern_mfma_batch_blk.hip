// vbs_kern_mfma_batch_blk.hip — batched (skinny) matvec on the f16 matrix
// cores for the 32-element block types (Q4_0, Q4_1, Q8_0) and F16 weights:
// k_mvbb, over the prepared x of vbs_mfma_batch.h.
//
// Y[t][r] = sum_c deq(W[r,c]) * X[t][c] (vbs_host_linear_tile once per vector,
// src/vbs_host_math.h:223-267), W read once for up to 8 (VG = 1) or 16 vectors
// (VG = 2: two groups of 16 planes). Eight GGUF blocks, 256 elements, are one
// unit as in the batch-1 kernel; here rows need only be a multiple of 32
// elements (8 for F16): the last unit of a row may be partial, its missing
// elements zero in the prepared x and their block scales taken as zero.
//
// MFMA m of a unit (v_mfma_f32_16x16x32_f16) takes elements 32 m .. 32 m + 31,
// one GGUF block: lane (n, g) holds elements 8 g .. 8 g + 7 of row n as B and
// the same elements of plane n as A (one 16-byte load; the sixteen lanes of a
// group read 256 contiguous bytes). The operand is the bare quant, exact in
// f16: q (Q8_0), nibble - 8 (Q4_0), nibble (Q4_1), the weight itself (F16). D
// is then the block's dot with each plane in fp32 and the block's d multiplies
// it: y += d D (F16: the unit's eight D are added up). Q4_1's
// d nib + m adds m times the block's sum of x by one more MFMA per unit, A the
// unit's eight sub-block sums (x'/32, hi and lo planes), B the eight mins.
//
// Work split: a workgroup owns T tiles of 16 rows, its waves split the rows
// by units (wave w: units w, w + nw, ...) and add their sums in wave order at
// the end; a unit's A operands serve the wave's T tiles. One item (tile, unit)
// is in flight per wave in registers while the one before it is computed
// from the wave's LDS slot (two in flight cost registers and were slower:
// 22016 x 4096 Q8_0 33.7 against 29.8 us).
//
// Bound: each wave's chain of load, LDS, unpack, MFMA and scale, with 1.3 to 1.6
// waves per SIMD in flight (Q8_0, 8 vectors: vector ALU 26-37% busy, LDS 6-9%, matrix
// cores 3-5%, 3.0 to 4.3 TB/s fetched). Measured
// with its x preparation, weights from HBM, 8 vectors, against the VALU kernel
// it replaced: Q8_0 4096 x 4096 72.5 -> 10.7 us, 11008 x 4096 251.7 -> 16.7
// (2.9 TB/s), 4096 x 11008 199.2 -> 18.9; Q4_0 11008 x 4096 170.4 -> 14.5; F16
// 11008 x 4096 315 -> 24.3 (3.7 TB/s); 16 vectors, Q8_0 11008 x 4096 445 -> 23.7.
// About 6 us of each is the fixed cost of the two launches.
// Error against 64 bits 0.7 to 1.3e-7 (the VALU kernel's 1.0 to 2.4e-7; F16 rows of 128
// to 256 elements 5% over its, 7.8 -> 8.2e-8: the 22 bits of x).
//
// Results that are not finite (an inf or NaN in x makes its whole block's
// planes NaN here) are computed again by a wave each in the general kernel's
// arithmetic, a row on one wave: such vectors and weights give the oracle's inf
// and NaN (a NaN in one of eight vectors: Q8_0 4096 x 4096 37 us; by one lane per
// result it took 1163).
#include "vbs_mfma_batch.h"
#include "vbs_row8.h"

namespace vbs {

namespace {

struct MbbArgs {
    const uint8_t *w[3];
    float *y[3];
    uint32_t ys[3], rows[3];
    uint32_t tile_end[3];  // cumulative 16-row tiles per matrix
    uint32_t nmat;
    const uint8_t *xp;     // prepared x: VG groups of xb_layout(pcols)
    const float *x;        // the vectors themselves, xs floats apart
    uint32_t xs, cols, batch;
};

// ---- x preparation: rows of any length, zero up to the next 256 -----------------------
__global__ __launch_bounds__(256) void k_xprep_r(const float *x, uint32_t xs, uint32_t cols,
                                                 uint32_t pcols, uint8_t *xp) {
    const uint32_t t = blockIdx.y, lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t b = blockIdx.x * 4u + wave;
    if (b >= pcols / 256u) return;
    const uint32_t e0 = 256u * b + 4u * lane;
    const float *xt = x + (uint64_t)t * xs;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    if (e0 + 4u <= cols) {
        typedef float4 __attribute__((aligned(4))) f4u;
        const float4 q = *reinterpret_cast<const f4u *>(xt + e0);
        v[0] = q.x, v[1] = q.y, v[2] = q.z, v[3] = q.w;
    } else {
#pragma unroll
        for (uint32_t k = 0; k < 4u; k++)
            if (e0 + k < cols) v[k] = xt[e0 + k];
    }
    xprep_block(v, lane, t % kBatchMax, b, pcols, xp + (uint64_t)(t / kBatchMax) * xb_layout(pcols).bytes);
}

// ---- weight types -----------------------------------------------------------------------
template <int BLK>
struct BlkB {
    static constexpr int TYPE = BLK;
    typedef KBlk<TYPE> K;
    static constexpr uint32_t BB = K::BB, QOFF = K::QOFF, BYTES = K::BYTES, CH = K::CH, NLD = K::NLD;
    static constexpr uint32_t SCRATCH = K::SCRATCH;
    static constexpr bool MINS = TYPE == kQ4_1;
    __device__ static void load(const Src &src, uint32_t u, uint32_t, uint32_t n, uint32_t g, u32x4 *r) {
        K::load(src, u, n, g, r);
    }
    __device__ static void stage(const u32x4 *r, uint8_t *scratch, uint32_t n, uint32_t g) {
        const uint32_t lane = 16u * g + n;
#pragma unroll
        for (uint32_t i = 0; i < NLD; i++) {
            const uint32_t c = lane + 64u * i;
            if (i + 1u < NLD || c < K::NCHUNK) *reinterpret_cast<u32x4 *>(scratch + 16u * c) = r[i];
        }
    }
    // D of each block by its scale d: acc[v][0] and [1] get vectors 2g and 2g + 1
    // of group v (before the exponent)
    template <uint32_t VG>
    __device__ static void dot(const u32x4 *, const uint8_t *scratch, const Src &src, uint32_t u,
                               uint32_t cols, uint32_t n, uint32_t g, const h8 (&A)[VG][8],
                               const h8 (&mn)[VG], float (&acc)[VG][2]) {
        const uint32_t o = ((uint32_t)(uintptr_t)src.w + src.row(n) + u * BYTES) & 15u;
        const uint8_t *row = scratch + 16u * CH * n;
        // this lane's eight quants of block m start at row byte qo + BB m (nibbles:
        // the 8 bytes of its half; the upper lane groups take the high nibbles)
        const uint32_t qo = o + QOFF + (TYPE == kQ8_0 ? 8u * g : 8u * (g & 1u));
        const uint32_t sh0 = qo & 3u, sh2 = (qo + 2u) & 3u;
        const uint32_t *r0 = reinterpret_cast<const uint32_t *>(row + (qo & ~3u));
        const uint32_t *r2 = reinterpret_cast<const uint32_t *>(row + ((qo + 2u) & ~3u));
        const uint32_t nsh = TYPE == kQ8_0 ? 0u : 4u * (g >> 1);
        const uint32_t valid = cols / 32u - 8u * u;  // blocks of this unit within the row
        const float off = TYPE == kQ8_0 ? -1152.f : TYPE == kQ4_0 ? -1032.f : -1024.f;
        const h2 bias = {(_Float16)off, (_Float16)off};
        const f4 z = {0.f, 0.f, 0.f, 0.f};
        uint32_t mb[8];
#pragma unroll
        for (uint32_t m = 0; m < 8u; m++) {
            constexpr uint32_t kOdd = BB & 3u;  // 2 (18, 34) or 0 (20)
            const bool half = kOdd && (m & 1u);
            const uint32_t *p = (half ? r2 : r0) + (BB * m - (half ? 2u : 0u)) / 4u;
            const uint32_t sh = half ? sh2 : sh0;
            uint32_t q0 = __builtin_amdgcn_alignbyte(p[1], p[0], sh);
            uint32_t q1 = __builtin_amdgcn_alignbyte(p[2], p[1], sh);
            if (TYPE == kQ8_0) {
                q0 ^= 0x80808080u;
                q1 ^= 0x80808080u;
            } else {
                q0 = (q0 >> nsh) & 0x0F0F0F0Fu;
                q1 = (q1 >> nsh) & 0x0F0F0F0Fu;
            }
            const h8 B = join8(f16_bytes(q0, 0x00050004u) + bias, f16_bytes(q0, 0x00070006u) + bias,
                               f16_bytes(q1, 0x00050004u) + bias, f16_bytes(q1, 0x00070006u) + bias);
            const uint32_t db = *reinterpret_cast<const uint16_t *>(row + o + BB * m);
            const float d = cvt_h(m < valid ? db : 0u);
#pragma unroll
            for (uint32_t v = 0; v < VG; v++) {
                const f4 D = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[v][m], B, z, 0, 0, 0);
                acc[v][0] = fmaf(d, D[0] + D[1], acc[v][0]);
                acc[v][1] = fmaf(d, D[2] + D[3], acc[v][1]);
            }
            if (MINS) {
                const uint32_t b = *reinterpret_cast<const uint16_t *>(row + o + BB * m + 2u);
                mb[m] = m < valid ? b : 0u;
            }
        }
        if (MINS) {
            const u32x4 bw = {mb[0] | (mb[1] << 16), mb[2] | (mb[3] << 16), mb[4] | (mb[5] << 16),
                              mb[6] | (mb[7] << 16)};
            const h8 B = __builtin_bit_cast(h8, bw);
#pragma unroll
            for (uint32_t v = 0; v < VG; v++) {
                const f4 D = __builtin_amdgcn_mfma_f32_16x16x32_f16(mn[v], B, z, 0, 0, 0);
                acc[v][0] = fmaf(32.f, D[0] + D[1], acc[v][0]);
                acc[v][1] = fmaf(32.f, D[2] + D[3], acc[v][1]);
            }
        }
    }
};

// F16 rows of a multiple of 8 elements at 16-byte alignment: the operands are
// loaded where they are used, no LDS. Each MFMA has a sum of its own, added in a
// tree: chained, the rounding of short rows was larger than that of the VALU kernel
// before (256 and 512 columns, error against 64 bits 7.8 and 8.6e-8 there, two chains
// 9.5 and 9.9, now 8.2 and 8.7; the general kernel's 8.1 and 8.6), for no time.
struct F16B {
    static constexpr int TYPE = kF16;
    static constexpr uint32_t BYTES = 512, NLD = 8, SCRATCH = 0;
    static constexpr bool MINS = false;
    __device__ static void load(const Src &src, uint32_t u, uint32_t cols, uint32_t n, uint32_t g,
                                u32x4 *r) {
        const uint32_t rb = src.row(n), last = cols / 8u - 1u;
#pragma unroll
        for (uint32_t m = 0; m < 8u; m++) r[m] = lda4(src.w + rb + 16u * min(32u * u + 4u * m + g, last));
    }
    __device__ static void stage(const u32x4 *, uint8_t *, uint32_t, uint32_t) {}
    template <uint32_t VG>
    __device__ static void dot(const u32x4 *r, const uint8_t *, const Src &, uint32_t u, uint32_t cols,
                               uint32_t, uint32_t g, const h8 (&A)[VG][8], const h8 (&)[VG],
                               float (&acc)[VG][2]) {
        f4 D[VG][8];
#pragma unroll
        for (uint32_t m = 0; m < 8u; m++) {
            const u32x4 z = {0u, 0u, 0u, 0u};
            const h8 B = __builtin_bit_cast(h8, 256u * u + 32u * m + 8u * g < cols ? r[m] : z);
#pragma unroll
            for (uint32_t v = 0; v < VG; v++)
                D[v][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[v][m], B, f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        }
#pragma unroll
        for (uint32_t v = 0; v < VG; v++) {
#pragma unroll
            for (uint32_t w = 4u; w; w /= 2u)
#pragma unroll
                for (uint32_t k = 0; k < w; k++) D[v][k] += D[v][k + w];
            const f4 S = D[v][0];
            acc[v][0] += S[0] + S[1];
            acc[v][1] += S[2] + S[3];
        }
    }
};

// A row times x in f32 by the whole wave, as k_rows has a row on one wave.
template <int T>
__device__ __forceinline__ float row_whole(const uint8_t *row, const float *x, uint32_t cols, uint32_t lane) {
    typedef Row8<T> R;
    constexpr uint32_t L = R::E / 8u;
    const uint32_t q = lane % L;
    float acc = 0.f;
#pragma unroll 2
    for (uint32_t u = lane / L; u < cols / R::E; u += 64u / L) {
        const f4u *x0 = reinterpret_cast<const f4u *>(x + R::E * u + R::lo(q));
        const f4u *x1 = reinterpret_cast<const f4u *>(x + R::E * u + R::hi(q));
        const typename R::Raw raw = R::raw(row, u, q);
        const v4f a = *x0, b = *x1;
        float w[8], s = 0.f;
        R::value(raw, w);
        const float xv[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int e = 0; e < 8; e++) s = fmaf(w[e], xv[e], s);
        acc += s;
    }
    return wave_sum(acc);
}

template <class P, uint32_t T, uint32_t VG>
__global__ __launch_bounds__(512) void k_mvbb(const MbbArgs a) {
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t cols = a.cols, nu = (cols + 255u) >> 8, pcols = 256u * nu;
    const uint32_t rb = P::SCRATCH ? (uint32_t)(cols / 32u * (P::BYTES / 8u)) : 2u * cols;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const uint32_t nw = blockDim.x >> 6, n = lane & 15u, g = lane >> 4;
    const XbLayout L = xb_layout(pcols);
    const uint32_t total = a.tile_end[a.nmat - 1u];
    // (planes past the batch re-read its last one and are never stored)
    const uint8_t *plane[VG], *expo[VG];
#pragma unroll
    for (uint32_t v = 0; v < VG; v++) {
        const uint32_t nb = min(kBatchMax, a.batch - kBatchMax * v);
        plane[v] = a.xp + v * L.bytes + 16u * min(n, 2u * nb - 1u);
        expo[v] = a.xp + v * L.bytes + L.expo + 8u * g;
    }
    Src src[T];
    uint32_t mt[T], lt[T];
#pragma unroll
    for (uint32_t j = 0; j < T; j++) {
        const uint32_t gt = min(blockIdx.x * T + j, total - 1u);
        const uint32_t m = (uint32_t)(gt >= a.tile_end[0]) + (uint32_t)(a.nmat > 2u && gt >= a.tile_end[1]);
        mt[j] = m;
        lt[j] = gt - (m == 0u ? 0u : m == 1u ? a.tile_end[0] : a.tile_end[1]);
        const uint32_t rows = m == 0u ? a.rows[0] : m == 1u ? a.rows[1] : a.rows[2];
        src[j] = Src{m == 0u ? a.w[0] : m == 1u ? a.w[1] : a.w[2], rows * rb, rb, lt[j] * 16u, rows};
    }
    uint8_t *const scratch = lds + wave * P::SCRATCH;
    float acc[T][VG][2];
#pragma unroll
    for (uint32_t j = 0; j < T; j++)
#pragma unroll
        for (uint32_t v = 0; v < VG; v++) acc[j][v][0] = acc[j][v][1] = 0.f;

    // a unit's A operands: two sets, the next unit's requested before the
    // current one's last tile, or one (VG = 2)
    constexpr uint32_t NA = VG == 1u ? 2u : 1u;
    h8 A[NA][VG][8], mn[NA][VG];
    int2 es[NA][VG];
    auto load_a = [&](uint32_t u, auto set) {
        constexpr uint32_t S = decltype(set)::value % NA;
#pragma unroll
        for (uint32_t v = 0; v < VG; v++) {
#pragma unroll
            for (uint32_t m = 0; m < 8u; m++)
                A[S][v][m] = *reinterpret_cast<const h8 *>(plane[v] + 256u * (32u * u + 4u * m + g));
            es[S][v] = *reinterpret_cast<const int2 *>(expo[v] + 32u * u);
            if (P::MINS) {
                const h8 t = *reinterpret_cast<const h8 *>(plane[v] + L.msum + 256u * u), z = {};
                mn[S][v] = g == 0u ? t : z;
            }
        }
    };
    u32x4 W[P::NLD];  // the next item's weights
    // the T tiles of unit u with A set `set`
    auto unit = [&](uint32_t u, auto set) {
        constexpr uint32_t S = decltype(set)::value % NA;
        unroll_for<0u, T>([&](auto jc) {
            constexpr uint32_t j = decltype(jc)::value;
            P::stage(W, scratch, n, g);
            __builtin_amdgcn_wave_barrier();
            u32x4 B[P::NLD];
#pragma unroll
            for (uint32_t i = 0; i < P::NLD; i++) B[i] = W[i];
            const uint32_t un = j + 1u < T ? u : u + nw;
            if (un < nu) P::load(src[(j + 1u) % T], un, cols, n, g, W);
            if (NA == 2u && j + 1u == T && u + nw < nu)
                load_a(u + nw, std::integral_constant<uint32_t, (S + 1u) % NA>{});
            float part[VG][2];
#pragma unroll
            for (uint32_t v = 0; v < VG; v++) part[v][0] = part[v][1] = 0.f;
            P::template dot<VG>(B, scratch, src[j], u, cols, n, g, A[S], mn[S], part);
#pragma unroll
            for (uint32_t v = 0; v < VG; v++) {
                acc[j][v][0] += ldexpf(part[v][0], -es[S][v].x);
                acc[j][v][1] += ldexpf(part[v][1], -es[S][v].y);
            }
            __builtin_amdgcn_wave_barrier();
        });
        if (NA == 1u && u + nw < nu) load_a(u + nw, set);
    };
    const std::integral_constant<uint32_t, 0u> set0{};
    const std::integral_constant<uint32_t, 1u> set1{};
    uint32_t u = wave;
    if (u < nu) {
        load_a(u, set0);
        P::load(src[0], u, cols, n, g, W);
        for (;;) {
            unit(u, set0);
            u += nw;
            if (u >= nu) break;
            unit(u, set1);
            u += nw;
            if (u >= nu) break;
        }
    }

    // partial sums [T][nw][lane][2] of one vector group at a time, added in
    // wave order; lane (n, g) holds row n for vectors 2g and 2g + 1
    float *const red = reinterpret_cast<float *>(lds);
#pragma unroll
    for (uint32_t v = 0; v < VG; v++) {
        __syncthreads();
#pragma unroll
        for (uint32_t j = 0; j < T; j++) {
            red[(j * nw + wave) * 128u + 2u * lane] = acc[j][v][0];
            red[(j * nw + wave) * 128u + 2u * lane + 1u] = acc[j][v][1];
        }
        __syncthreads();
        for (uint32_t q = threadIdx.x; q < T * 128u; q += blockDim.x) {  // (a wave's q are 64 in a row)
            const uint32_t j = q >> 7, l = (q >> 1) & 63u, tk = q & 1u;
            float s = 0.f;
            for (uint32_t w = 0; w < nw; w++) s += red[(j * nw + w) * 128u + 2u * l + tk];
            const uint32_t gt = blockIdx.x * T + j;
            const uint32_t m = (uint32_t)(gt >= a.tile_end[0]) + (uint32_t)(a.nmat > 2u && gt >= a.tile_end[1]);
            const uint32_t row = 16u * (gt - (m == 0u ? 0u : m == 1u ? a.tile_end[0] : a.tile_end[1])) + (l & 15u);
            const uint32_t rows = m == 0u ? a.rows[0] : m == 1u ? a.rows[1] : a.rows[2];
            const uint32_t t = kBatchMax * v + 2u * (l >> 4) + tk;
            const bool ours = gt < total && row < rows && t < a.batch;
            for (uint64_t bad = __ballot(ours && !(fabsf(s) <= 3.4028235e38f)); __builtin_expect(bad != 0u, 0); bad &= bad - 1u) {
                const int who = __ffsll((unsigned long long)bad) - 1;
                const uint32_t bm = __builtin_amdgcn_readlane(m, who), br = __builtin_amdgcn_readlane(row, who);
                const uint32_t bt = __builtin_amdgcn_readlane(t, who);
                const float again = row_whole<P::TYPE>((bm == 0u ? a.w[0] : bm == 1u ? a.w[1] : a.w[2]) + (uint64_t)br * rb,
                                                       a.x + (uint64_t)bt * a.xs, cols, lane);
                if ((int)lane == who) s = again;
            }
            if (ours)
                (m == 0u ? a.y[0] : m == 1u ? a.y[1] : a.y[2])[(uint64_t)t * (m == 0u ? a.ys[0] : m == 1u ? a.ys[1] : a.ys[2]) + row] = s;
        }
    }
}

template <class P, uint32_t T, uint32_t VG>
hipError_t launch_mvbb_t(const MbbArgs &a, uint32_t nw, hipStream_t s) {
    const uint32_t tiles = a.tile_end[a.nmat - 1u];
    const size_t slots = (size_t)nw * P::SCRATCH, red = (size_t)T * nw * 128u * sizeof(float);
    const size_t lds = slots > red ? slots : red;  // (at most 8 x 4608 bytes)
    k_mvbb<P, T, VG><<<(tiles + T - 1u) / T, 64u * nw, lds, s>>>(a);
    return hipGetLastError();
}

// Tiles per workgroup: the tiles per CU up to three, so that a unit's A
// operands (8 KB, twice a Q8_0 item's bytes) are read once for as many tiles
// as still leave every CU a workgroup (Q8_0, 8 vectors, T = 1 / 2 / 3: 4096 x
// 4096 10.7 / 12.9 / 14.8 us, 6144 x 4096 15.7 / 13.5 / 15.5, 22016 x 4096
// 38.0 / 32.8 / 29.8; four tiles spill). Eight waves: twelve or sixteen on
// the one-tile shapes changed nothing (4096 x 11008 19.2 / 19.0 us) and four
// were slower, but for sixteen vectors over more than two tiles per CU, where
// two workgroups of four waves share a CU (11008 x 4096 26.7 -> 23.7 us,
// 22016 x 4096 48.3 -> 39.9; 4096 x 4096 12.3 -> 12.5).
template <class P>
hipError_t launch_mvbb(const MbbArgs &a, hipStream_t s) {
    const uint32_t nu = (a.cols + 255u) / 256u, tiles = a.tile_end[a.nmat - 1u], cus = device_cus();
    if (a.batch > kBatchMax) return launch_mvbb_t<P, 1, 2>(a, min(tiles > 2u * cus ? 4u : 8u, nu), s);
    if (tiles <= cus) return launch_mvbb_t<P, 1, 1>(a, min(8u, nu), s);
    if (tiles <= 2u * cus) return launch_mvbb_t<P, 2, 1>(a, min(8u, nu), s);
    return launch_mvbb_t<P, 3, 1>(a, min(8u, nu), s);
}

// Where the general kernel's one launch (k_rows) ends before this path's two
// for one matrix. Times of the general kernel over this path's, graph replays
// with weights from HBM (Q4_0 / Q8_0 / F16):
// * one vector: 0.2 to 0.8 at any size;
// * two to four: 2048 x 14336 0.7-0.9 / 0.6-0.9 / 0.5-0.7, 5000 x 2048 0.9-1.0 /
//   0.8-0.9 / 0.7-0.9 (Q4_1 1.0-1.15); but 4096 x 4096 1.2-1.4 / 1.2 / 0.9-1.0, 8192 x 11008 2.0-2.2 /
//   1.5-1.6 / 0.9-1.0, 4096 x 14336 2.1-2.4 / 1.8-1.9 / 1.0-1.6;
// * five to eight: up to 2048 x 2048 0.5-0.9, 1024 x 4096 0.7-0.8, 2048 x 4096 0.8-1.05;
//   but 3072 x 1024 0.9-1.3, 4096 x 4096 1.2-1.8, 1024 x 11008 1.0-1.2 (F16 0.7-0.9);
//   nine to sixteen: 1024 x 4096 0.8-1.0, 1536 x 4096 0.9-1.15, 8192 x 4096 1.7-2.7;
// * rows of one step of the general kernel, five to eight vectors 16384 x 512
//   0.8-0.9 / 0.8-0.9 / 1.0, 32000 x 512 1.3; more 4096 x 512 0.8-0.9 (F16 1.0), 8192 x
//   512 1.1-1.2; F16 of 32 columns 32000 rows 0.9 and 1.3.
bool general_sooner(int type, uint32_t rows, uint32_t cols, uint32_t batch) {
    const bool f16 = type == kF16;
    if (batch == 1u) return true;
    if (batch <= 4u) {
        if (f16 && batch == 2u) return true;
        if (rows < 3072u || (rows == 3072u && (batch == 2u || cols < 8192u))) return true;
        return cols < (f16 ? 8192u : type == kQ4_1 ? 2048u : 3072u);
    }
    if (cols <= 512u) {
        if (f16) return cols < 64u ? batch <= 8u || rows < 24576u : rows < (batch <= 8u ? 16384u : 3072u);
        return rows < (batch <= 8u ? 24576u : 8192u);
    }
    if (rows >= 3072u || (cols >= 2048u && rows * batch >= 32768u)) return false;
    if (rows < 1024u || cols < 4096u) return true;
    return rows * batch < (cols < 8192u ? 15360u : f16 ? 12288u : 5120u);
}

// The same for two or three matrices, a launch of the general kernel (or its own
// matrix-core pair) each, against this path's two launches for all. Over their
// times (us, of this path / one by one; two matrices of R rows each):
// * two to four vectors: R = 512 x 14336 Q4_0 15.2 / 10.6 and 15.4 / 14.6, R = 1024 x
//   2048 7.4 / 6.3 and 7.5 / 7.0, R = 4096 x 512 7.2 / 5.8 and 7.3 / 6.8; but R = 2048 x
//   2048 7.7 / 7.4 and 7.7 / 7.9, R = 1024 x 8192 11.3 / 12.2 and 11.3 / 13.3; F16, two
//   vectors R = 1024 x 8192 16.0 / 12.5, R = 8192 x 4096 38.5 / 30.7, R = 4096 x 4096 18.9 / 22.5;
// * one vector: R = 1024 x 14336 16.9 / 14.1, R = 2048 x 4096 9.0 / 8.1, but R = 4096 x 4096
//   11.6 / 12.7, R = 2048 x 8192 12.9 / 13.6; R = 8192 x 4096 23.0 / 18.2 (Q8_0 26.3 / 21.1),
//   R = 28672 x 8192 94 / 97 (Q4_1 R = 11008 x 4096 23.7 / 25.1); F16 4.6 / 3.9 to 185 / 153;
// * five to eight: R = 64 x 4096 8.1 / 6.8, R = 256 x 8192 11.4 / 9.7, but R = 512 x 8192 11.4 /
//   14.5, R = 256 x 2048 6.8 / 6.7; nine and more 300 + 70 rows x 5664 11.4 / 12.6;
// * three matrices: 300 + 70 + 20 rows x 8192, one to four vectors 11.4 / 8.5, 9.9, 11.8
//   (F16 14.0 / 8.3, 10.0, 12.0), F16 of one vector 2048 + 512 + 512 x 2048 7.8 / 9.2, 8192 + 1024 + 1024 x 8192 40 / 35.
bool general_sooner_multi(int type, uint32_t nmat, uint64_t rows, uint32_t cols, uint32_t batch) {
    const bool f16 = type == kF16;
    if (nmat == 3u) {
        if (rows <= 512u && cols >= 4096u) return batch <= (f16 ? 4u : 2u);
        return f16 && batch == 1u && rows >= 4096u && cols >= 4096u;
    }
    if (batch > 4u) return batch <= 8u && rows <= 512u && cols >= 4096u;
    if (rows <= 1024u || cols <= 512u || (rows <= 2048u && (cols <= 2048u || (f16 && batch == 2u)))) return true;
    if (batch == 1u)
        return f16 || rows <= 2048u || (rows <= 4096u && cols <= 4096u) ||
               (type != kQ4_1 && rows >= 16384u && cols <= 4096u);
    return f16 && batch == 2u && rows >= 16384u;
}

}  // namespace

hipError_t launch_blk_linear_batch(int type, uint32_t nmat, const uint8_t *const w[], const uint32_t rows[],
                                   const float *x, uint32_t xs, float *const y[], const uint32_t ys[],
                                   uint32_t cols, uint32_t batch, hipStream_t s) {
    const bool f16 = type == kF16;
    if (!f16 && type != kQ4_0 && type != kQ4_1 && type != kQ8_0) return hipErrorNotSupported;
    if (nmat == 0u || nmat > 3u || batch == 0u || batch > 2u * kBatchMax) return hipErrorNotSupported;
    if (cols == 0u || cols % (f16 ? 8u : 32u) || cols > (1u << 20) || ((uintptr_t)x & 3u)) return hipErrorNotSupported;
    MbbArgs a{};
    uint32_t tiles = 0;
    for (uint32_t m = 0; m < nmat; m++) {
        if (rows[m] == 0u || ((uintptr_t)w[m] & (f16 ? 15u : 1u)) ||
            (uint64_t)rows[m] * row_bytes(type, cols) + 1024u >= (1ull << 32))
            return hipErrorNotSupported;
        a.w[m] = w[m];
        a.y[m] = y[m];
        a.ys[m] = ys[m];
        a.rows[m] = rows[m];
        tiles += (rows[m] + 15u) / 16u;
        a.tile_end[m] = tiles;
    }
    uint64_t all_rows = 0;
    for (uint32_t m = 0; m < nmat; m++) all_rows += rows[m];
    if (nmat == 1u ? general_sooner(type, rows[0], cols, batch) : general_sooner_multi(type, nmat, all_rows, cols, batch))
        return hipErrorNotSupported;
    const uint32_t pcols = (cols + 255u) & ~255u;
    hipError_t why;
    const size_t need = (size_t)((batch + kBatchMax - 1u) / kBatchMax) * xb_layout(pcols).bytes;
    uint8_t *xp = static_cast<uint8_t *>(rt_scratch_or_captured(need, s, &why));
    if (!xp) return hipErrorNotSupported;  // (no memory for it: the general kernel needs none)
    a.nmat = nmat;
    a.xp = xp;
    a.x = x;
    a.xs = xs;
    a.cols = cols;
    a.batch = batch;
    k_xprep_r<<<dim3((pcols / 256u + 3u) / 4u, batch), 256, 0, s>>>(x, xs, cols, pcols, xp);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (type == kQ4_0) return launch_mvbb<BlkB<kQ4_0>>(a, s);
    if (type == kQ4_1) return launch_mvbb<BlkB<kQ4_1>>(a, s);
    if (type == kQ8_0) return launch_mvbb<BlkB<kQ8_0>>(a, s);
    return launch_mvbb<F16B>(a, s);
}

}  // namespace vbs
