// vbs_kern_attn.hip — single-query GQA attention over the f16 KV cache,
// split along the sequence ("flash decoding").
//
// Reference: vbs_host_attention (src/vbs_host_math.h:170-209): for every q
// head h (kv head h / group), score_s = (float)(double dot(q_h, k_s)) * scale,
// then a sequential online softmax over s < seq_len and out = acc * (1/l).
//
// Each workgroup takes a chunk of positions of one kv head and produces, per
// q head of that kv head, the chunk maximum m, the sum l of exp(score - m)
// and acc[d] = sum exp(score - m) * v[d]; the chunks are merged with
// log-sum-exp rescaling: out = sum_c acc_c * e^(m_c-M) / sum_c l_c * e^(m_c-M).
// The chunk length follows the sequence (attn_split) so that about
// kMfmaTargetWgs (vbs_attn_common.h) workgroups of the matrix-core kernel, or
// kTargetWgs of k_attn_solo, share it at any length; the generic kernel's is
// kChunk. A second kernel merges (a hand-off inside one kernel, through
// device-scope stores, loads and an arrival count, measured slower than the
// kernel boundary on this part); short sequences take one launch that does
// both, the chunks of a kv head on the waves of one workgroup (k_attn_one).
//
// head_dim 32, 64, 96 and 128 with at most eight q heads per kv head take the
// matrix-core chunk kernel, but one q head per kv head of 32 or 64 dims past the
// one-launch lengths k_attn_solo; other shapes the generic one (double dot, one
// position per four threads).
#include <type_traits>

#include "vbs_attn_common.h"
#include "vbs_dev_common.h"
#include "vbs_internal.h"

namespace vbs {

constexpr uint32_t kChunk = 64;  // positions per workgroup of the generic kernel
constexpr uint32_t kMaxGroup = 16;
constexpr uint32_t kTargetWgs = 512;      // workgroups k_attn_solo's split aims for

// (attn_split, the matrix-core split's constants and the exponentials: vbs_attn_common.h)
// Chunks per kv head of any split of a sequence of at most max_seq (every
// len >= 64 or len >= seq * nkh / target, target <= kMfmaTargetWgs).
inline uint32_t attn_max_chunks(uint32_t max_seq, uint32_t nkh) {
    const uint32_t a = (kMfmaTargetWgs + nkh - 1u) / nkh, b = (max_seq + 63u) / 64u;
    return a > b ? a : b;
}

// f16 bits -> f32 with the hardware converter (exact for every finite value).
__device__ __forceinline__ float hcvt(uint32_t bits16) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16);
}

// ---- generic chunk kernel ------------------------------------------------------
__global__ __launch_bounds__(256) void k_attn_partial(const float *__restrict__ q,
                                                      const uint16_t *__restrict__ kc,
                                                      const uint16_t *__restrict__ vc,
                                                      float *__restrict__ part,
                                                      uint32_t seq_len, const uint32_t *pos_dev,
                                                      uint64_t layer_off, uint32_t nkh, uint32_t hd,
                                                      uint32_t group, float scale,
                                                      uint32_t n_chunks) {
    extern __shared__ float lds[];
    float *qs = lds;                       // [group][hd]
    float *ps = qs + group * hd;           // [group][kChunk]
    float *red = ps + group * kChunk;      // [256 / hd][group][hd] partial acc

    const uint32_t chunk = blockIdx.x, kvh = blockIdx.y, t = threadIdx.x;
    // graph replays take the position from device memory: seq_len = pos + 1
    if (pos_dev) seq_len = pos_dev[0] + 1u;
    const uint32_t s0 = chunk * kChunk;
    if (s0 >= seq_len) return;  // chunk past the current sequence (grid sized for the maximum)
    const uint32_t valid = min(kChunk, seq_len - s0);

    for (uint32_t i = t; i < group * hd; i += 256u) qs[i] = q[(uint64_t)kvh * group * hd + i];
    __syncthreads();

    // Scores: four threads per position, each a quarter of the head dim.
    {
        const uint32_t sl = t >> 2, quarter = t & 3u;
        double dot[kMaxGroup];
#pragma unroll
        for (uint32_t g = 0; g < kMaxGroup; g++) dot[g] = 0.0;
        if (sl < valid) {
            const uint16_t *kr = kc + layer_off + ((uint64_t)(s0 + sl) * nkh + kvh) * hd;
            uint32_t d0 = (hd / 4u) * quarter, d1 = quarter == 3u ? hd : d0 + hd / 4u;
            for (uint32_t d = d0; d < d1; d++) {
                double kv = (double)h2f(kr[d]);
#pragma unroll
                for (uint32_t g = 0; g < kMaxGroup; g++)
                    if (g < group) dot[g] = fma((double)qs[g * hd + d], kv, dot[g]);
            }
        }
#pragma unroll
        for (uint32_t g = 0; g < kMaxGroup; g++) {
            if (g < group) {
                double v = dot[g];
                v += __shfl_xor(v, 1, 64);
                v += __shfl_xor(v, 2, 64);
                if (quarter == 0)
                    ps[g * kChunk + sl] = sl < valid ? __fmul_rn((float)v, scale) : -INFINITY;
            }
        }
    }
    __syncthreads();

    // Chunk softmax statistics, one wavefront per q head.
    const uint32_t wave = t >> 6, lane = t & 63u;
    for (uint32_t g = wave; g < group; g += 4u) {
        float sc = ps[g * kChunk + lane];
        float m = wave_max(sc);
        float e = lane < valid ? expf(sc - m) : 0.f;
        float l = wave_sum(e);
        ps[g * kChunk + lane] = e;
        if (lane == 0) {
            float *dst = part + ((uint64_t)(kvh * group + g) * n_chunks + chunk) * (hd + 2u);
            dst[0] = m;
            dst[1] = l;
        }
    }
    __syncthreads();

    // acc[g][d] = sum_s p[g][s] * v[s][d]; threads split (d, s-slice).
    const uint32_t nsl = 256u / hd, d = t % hd, sg = t / hd;
    float acc[kMaxGroup];
#pragma unroll
    for (uint32_t g = 0; g < kMaxGroup; g++) acc[g] = 0.f;
    if (sg < nsl) {
        for (uint32_t sl = sg; sl < valid; sl += nsl) {
            float v = h2f(vc[layer_off + ((uint64_t)(s0 + sl) * nkh + kvh) * hd + d]);
#pragma unroll
            for (uint32_t g = 0; g < kMaxGroup; g++)
                if (g < group) acc[g] = fmaf(ps[g * kChunk + sl], v, acc[g]);
        }
#pragma unroll
        for (uint32_t g = 0; g < kMaxGroup; g++)
            if (g < group) red[(sg * group + g) * hd + d] = acc[g];
    }
    __syncthreads();
    for (uint32_t i = t; i < group * hd; i += 256u) {
        uint32_t g = i / hd, dd = i % hd;
        float sum = 0.f;
        for (uint32_t k = 0; k < nsl; k++) sum += red[(k * group + g) * hd + dd];
        part[((uint64_t)(kvh * group + g) * n_chunks + chunk) * (hd + 2u) + 2u + dd] = sum;
    }
}


// ---- one q head per kv head (head_dim 32, 64) on the vector ALU -----------------
// Four waves; lanes of a wave split a position's head_dim into 8-element slices
// (16-byte K and V loads), so one wave step covers 64 / (HD / 8) positions
// ("slots"). A wave loads kSteps steps at a time (up to kBatches such batches;
// the next batch's K rows are requested once the scores are taken, its V rows
// once they are used). The partial dot of a slice is an fp32 FMA chain and the
// slices are added with DPP row operations, which leaves every lane of a slot
// with its score. Each slot keeps a running softmax state (max, sum, acc); the
// slots of a wave are combined with lane shuffles and the four waves in LDS.
// With a single q head the matrix cores' columns stand empty and its scores and
// weights cost the same as eight heads': past the one-launch lengths this
// kernel is ahead (8 heads of 64, 300, 3001 and 9000 positions 6.6, 7.2 and 8.1 us
// against 6.9, 8.3 and 11.0; 32 heads 3001 8.3 against 11.5; at two q heads per
// kv head the matrix cores are, 16 over 8 3001 8.5 against 9.4).
constexpr uint32_t kWaves = 4, kSteps = 4, kBatches = 4;
template <uint32_t HD>
struct ChunkShape {
    static constexpr uint32_t LPP = HD / 8, PPW = 64 / LPP, GRAN = kWaves * PPW,
                              LMAX = kBatches * kSteps * GRAN;
};

template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
    return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                                                     CTRL, 0xF, 0xF, false));
}
// Sum over each aligned group of L lanes (L = 4, 8), for every lane of it.
template <uint32_t L>
__device__ __forceinline__ float group_sum(float v) {
    v = dpp_add<0xB1>(v);                         // quad_perm [1,0,3,2]
    v = dpp_add<0x4E>(v);                         // quad_perm [2,3,0,1]
    if constexpr (L >= 8) v = dpp_add<0x141>(v);  // row_half_mirror
    return v;
}

template <uint32_t HD>
__global__ __launch_bounds__(64 * kWaves) void k_attn_solo(
    const float *__restrict__ q, const uint16_t *__restrict__ kc, const uint16_t *__restrict__ vc,
    float *__restrict__ part, uint32_t seq_len, const uint32_t *__restrict__ pos_dev, uint64_t layer_off,
    uint32_t nh, float scale, uint32_t stride_chunks) {
    using S = ChunkShape<HD>;
    constexpr uint32_t LPP = S::LPP, PPW = S::PPW;
    __shared__ __align__(16) float red[kWaves][HD];
    __shared__ float sm[kWaves], sl[kWaves];
    const uint32_t chunk = blockIdx.x, h = blockIdx.y, t = threadIdx.x;
    const uint32_t wave = t >> 6, lane = t & 63u, slot = lane / LPP, c = lane % LPP;
    if (pos_dev) seq_len = pos_dev[0] + 1u;  // graph replay: the device holds the position
    const AttnSplit sp = attn_split(seq_len, nh, S::GRAN, S::LMAX, kTargetWgs);
    if (chunk >= sp.n) return;  // past the sequence (the grid covers the longest split)
    const uint32_t s0 = chunk * sp.len, valid = min(sp.len, seq_len - s0);
    const uint32_t pw = sp.len / kWaves, ns = pw / PPW;  // positions and steps per wave
    const uint32_t nb = (ns + kSteps - 1u) / kSteps;     // batches of kSteps steps
    const uint64_t rstride = (uint64_t)nh * HD;
    const uint64_t base = layer_off + (uint64_t)s0 * rstride + (uint64_t)h * HD + 8u * c;

    // position of step i of this lane's slot; positions past the chunk re-read
    // its last row and are masked (score -inf, v zero)
    auto pos_of = [&](uint32_t i) { return wave * pw + i * PPW + slot; };
    uint4 kr[kSteps], vr[kSteps];
    auto load_k = [&](uint32_t bi) {
#pragma unroll
        for (uint32_t b = 0; b < kSteps; b++)
            if (bi * kSteps + b < ns)
                kr[b] = *reinterpret_cast<const uint4 *>(
                    kc + base + (uint64_t)min(pos_of(bi * kSteps + b), valid - 1u) * rstride);
    };
    auto load_v = [&](uint32_t bi) {
#pragma unroll
        for (uint32_t b = 0; b < kSteps; b++) {
            const uint32_t i = bi * kSteps + b;
            if (i < ns) {
                vr[b] = *reinterpret_cast<const uint4 *>(vc + base + (uint64_t)min(pos_of(i), valid - 1u) * rstride);
                if (pos_of(i) >= valid) vr[b] = make_uint4(0u, 0u, 0u, 0u);
            }
        }
    };
    load_k(0);
    load_v(0);
    float qv[8];
    {
        const float4 *qp = reinterpret_cast<const float4 *>(q + (uint64_t)h * HD + 8u * c);
        const float4 a = qp[0], b = qp[1];
        qv[0] = a.x, qv[1] = a.y, qv[2] = a.z, qv[3] = a.w;
        qv[4] = b.x, qv[5] = b.y, qv[6] = b.z, qv[7] = b.w;
    }

    // per slot: running max m, sum l of e^(s - m), acc of e^(s - m) v
    float m = -INFINITY, l = 0.f, acc[8] = {};
    for (uint32_t bi = 0; bi < nb; bi++) {
        float sc[kSteps];  // every lane of a slot holds its position's score
#pragma unroll
        for (uint32_t b = 0; b < kSteps; b++) {
            const uint32_t i = bi * kSteps + b;
            float p = 0.f;
            if (i < ns) {
                const uint32_t kw[4] = {kr[b].x, kr[b].y, kr[b].z, kr[b].w};
#pragma unroll
                for (uint32_t j = 0; j < 8; j++) p = fmaf(qv[j], hcvt(kw[j >> 1] >> (16u * (j & 1u))), p);
                p = group_sum<LPP>(p);
            }
            sc[b] = i < ns && pos_of(i) < valid ? __fmul_rn(p, scale) : -INFINITY;
        }
        if (bi + 1u < nb) load_k(bi + 1u);  // the K registers are free again
        float mb = sc[0];
#pragma unroll
        for (uint32_t b = 1; b < kSteps; b++) mb = fmaxf(mb, sc[b]);
        const float mn = fmaxf(m, mb);
        const float r = m == -INFINITY ? 0.f : fast_exp(__fsub_rn(m, mn));
        l *= r;
#pragma unroll
        for (uint32_t j = 0; j < 8; j++) acc[j] *= r;
#pragma unroll
        for (uint32_t b = 0; b < kSteps; b++) {
            if (bi * kSteps + b < ns) {
                const float e = sc[b] == -INFINITY ? 0.f : fast_exp(__fsub_rn(sc[b], mn));
                const uint32_t vw[4] = {vr[b].x, vr[b].y, vr[b].z, vr[b].w};
                l += e;
#pragma unroll
                for (uint32_t j = 0; j < 8; j++) acc[j] = fmaf(e, hcvt(vw[j >> 1] >> (16u * (j & 1u))), acc[j]);
            }
        }
        m = mn;
        if (bi + 1u < nb) load_v(bi + 1u);
    }

    // the wave's slots combined (lanes of equal c): M = max m, weights e^(m - M)
    // (0 for an empty slot), then sums; slot 0 stores them
    float M = m;
#pragma unroll
    for (uint32_t off = LPP; off < 64u; off <<= 1) M = fmaxf(M, __shfl_xor(M, off, 64));
    const float f = m == -INFINITY ? 0.f : fast_exp(__fsub_rn(m, M));
    float L = l * f;
#pragma unroll
    for (uint32_t j = 0; j < 8; j++) acc[j] *= f;
#pragma unroll
    for (uint32_t off = LPP; off < 64u; off <<= 1) {
        L += __shfl_xor(L, off, 64);
#pragma unroll
        for (uint32_t j = 0; j < 8; j++) acc[j] += __shfl_xor(acc[j], off, 64);
    }
    if (slot == 0) {
        float4 *dst = reinterpret_cast<float4 *>(&red[wave][8u * c]);
        dst[0] = make_float4(acc[0], acc[1], acc[2], acc[3]);
        dst[1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
        if (c == 0) sm[wave] = M, sl[wave] = L;
    }
    __syncthreads();

    // the waves combined: M = max m_w, weights e^(m_w - M) (0 for empty waves)
    if (t < HD) {
        float Mw = sm[0], a = 0.f, Lw = 0.f;
#pragma unroll
        for (uint32_t w = 1; w < kWaves; w++) Mw = fmaxf(Mw, sm[w]);
#pragma unroll
        for (uint32_t w = 0; w < kWaves; w++) {
            const float fw = sm[w] == -INFINITY ? 0.f : fast_exp(__fsub_rn(sm[w], Mw));
            a = fmaf(red[w][t], fw, a);
            Lw = fmaf(sl[w], fw, Lw);
        }
        float *dst = part + ((uint64_t)h * stride_chunks + chunk) * (HD + 2u);
        dst[2u + t] = a;
        if (t == 0) dst[0] = Mw, dst[1] = Lw;
    }
}

// ---- matrix-core chunk kernel (head_dim 32, 64, 96, 128; group <= 8) -------------
// One wave per chunk of up to kMfmaTiles tiles of 32 positions, on
// v_mfma_f32_16x16x32_f16:
// * scores, S = K q^T: A = 16 positions x 32 head dims of K (the cache's f16,
//   exact), B = 32 dims x 16 columns: column n holds q' of head n & 7, its
//   f16 hi part for n < 8 and lo part (q' - hi) for n >= 8, with q' = q 2^s_h
//   scaled so that the head's largest |q| lies in [2^14, 2^15). Columns n and
//   n + 8 add up (a DPP row rotation) to the fp32 dot of k with q' to ~2^-22;
//   the score is that times 2^-s_h * scale. Lane (n, g) then holds the scores
//   of head n & 7 at positions 16 hf + 4 g + r (hf, r: the two 16-position
//   halves of the tile, the four D rows).
// * online softmax per head over the tiles (running max m, sum l).
// * P V: A = P, rows n: e^(s - m) of head n & 7 (f16 hi for n < 8, lo for
//   n >= 8), k slots = exactly the lane's own eight positions; B = V with the
//   same k slots and column n of dim tile t standing for head dim D n + t (D =
//   HD / 16), so lane (n, g) takes its B operands from eight V rows it loaded
//   itself (dims Dn..Dn+D-1 of its eight positions) and no transpose is needed.
//   D rows 0-7 (hi) and 8-15 (lo) add up at the end.
// Bound: latency (one or a few tiles per wave) up to HBM at long contexts.
// Measured (chunk + merge) against the vector-ALU kernel that took head_dim 32
// and 64 before and the generic one that took 96: 32 q heads over 8 kv heads,
// 3001 positions, head_dim 32 14.1 -> 8.5 us, 64 13.6 -> 9.1, 96 39.2 -> 9.9; 41
// positions 9.3 -> 3.9, 8.7 -> 4.3, 28.5 -> 4.8 (one launch). Head_dim 128 over one
// kv head, 16000 positions 37.4 -> 21.1 (the merge's later rows sixteen at a time).
// The most chunks the matrix-core split gives any sequence of at most max_seq
// positions: the chunk count grows with the sequence while the chunk length
// stays put, so the maximum lies at the longest sequence of some chunk length
// (32 k positions for sequences of at most 32 k * target / nkh, the last
// length open-ended) or at max_seq itself. The chunk launch's grid: a graph
// replay reads the position on the device, so the grid covers every
// position up to max_seq, and workgroups beyond the current split exit at
// once (each costs dispatch time, so the grid is no larger than this).
template <uint32_t HD = 128>
inline uint32_t mfma_grid_chunks(uint32_t max_seq, uint32_t nkh, uint32_t target = kMfmaTargetWgs) {
    uint32_t best = 0;
    for (uint32_t k = 1; k <= kMfmaTiles; k++) {
        uint64_t hi = max_seq;
        if (k < kMfmaTiles) {
            hi = (uint64_t)kMfmaGran * k * target / nkh;
            const uint64_t cap = (uint64_t)kMfmaGran * k * kFineChunks;
            if (HD != 128u && hi > cap) hi = cap;
        }
        const uint32_t s = (uint32_t)(hi < max_seq ? hi : max_seq);
        if (s == 0) continue;
        const uint32_t c = mfma_split<HD>(s, nkh, target).n;
        best = c > best ? c : best;
    }
    return best;
}

typedef _Float16 ah8 __attribute__((ext_vector_type(8)));
typedef float af4 __attribute__((ext_vector_type(4)));
typedef uint32_t au4 __attribute__((ext_vector_type(4)));

// One wave's chunk: positions [s0, s0 + valid) of kv head kvh (valid >= 1,
// nt tiles of 32) against the q heads of its group. On return every lane
// holds, for head n & 7 of its lane n = lane & 15, the chunk maximum m and
// l = sum e^(s - m); and a[dt][r] = the sum of e^(s - m) v[HD / 16 n + dt] of head
// 4 (lane >> 4) + r (rows hi + lo added; lane groups 0 and 1 carry them).
__device__ __forceinline__ float score_max(float a, float b) { return fmaxf(a, b); }
__device__ __forceinline__ double score_max(double a, double b) { return fmax(a, b); }
template <int M>
__device__ __forceinline__ float score_xor(float v) {
    return lane_xor<M>(v);
}
template <int M>
__device__ __forceinline__ double score_xor(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t h = lane_xor<M>((uint32_t)(b >> 32)), l = lane_xor<M>((uint32_t)b);
    return __builtin_bit_cast(double, (uint64_t)h << 32 | l);
}

constexpr uint32_t kOneChunks = 8;  // k_attn_one's waves

// JOINT (one tile per wave, head sizes but 128): the workgroup's n_joint waves
// take one maximum per head over all their positions, through joint[wave][8]
// and a barrier (none if n_joint is 0), so that its position and every chunk weigh
// exactly 1. Short contexts are then as exact as whole f32 products, one position
// exact: a whole power of two as the chunk's maximum left 6e-8 there (error figures
// below). It takes 0.2 to 0.5 us (32 q heads over 8 kv heads of 64, 41 positions 3.9 ->
// 4.25 us, 256 5.3 -> 6.0).
template <uint32_t HD, bool JOINT = false>
__device__ __forceinline__ void attn_mfma_wave(const float *__restrict__ q,
                                               const uint16_t *__restrict__ kc,
                                               const uint16_t *__restrict__ vc, uint64_t layer_off,
                                               uint32_t s0, uint32_t valid, uint32_t nt,
                                               uint32_t nkh, uint32_t kvh, uint32_t group,
                                               float scale, uint32_t lane, float &m_out,
                                               float &l_out, float (&a)[HD / 16][4],
                                               double (*joint)[8] = nullptr, uint32_t n_joint = 0,
                                               uint32_t wave = 0) {
    constexpr uint32_t KK = HD / 32u, DPL = HD / 16u, VW = DPL / 2u;  // K slices; V dims and words per lane
    constexpr bool FINE = HD != 128u;
    typedef std::conditional_t<FINE, double, float> Score;
    constexpr float PS = FINE ? 16384.f : 1.f;  // P's scale (f16 would drop lo bits of small weights)
    const uint32_t n = lane & 15u, g = lane >> 4;
    const uint64_t rstride = (uint64_t)nkh * HD;
    const uint64_t base = layer_off + (uint64_t)s0 * rstride + (uint64_t)kvh * HD;

    // ---- tile loads: K rows (A operand: position 16 hf + n, dims 32 kk + 8 g ..),
    // V rows (position p_j of this lane group, dims DPL n ..); positions past the
    // chunk re-read its last row and are masked
    auto pos_of = [&](uint32_t t, uint32_t j) { return 32u * t + 16u * (j >> 2) + 4u * g + (j & 3u); };
    au4 kr[2][KK];
    uint32_t vr[8][VW];
    auto load_k = [&](uint32_t t) {
#pragma unroll
        for (uint32_t hf = 0; hf < 2; hf++) {
            const uint32_t p = min(32u * t + 16u * hf + n, valid - 1u);
#pragma unroll
            for (uint32_t kk = 0; kk < KK; kk++)
                kr[hf][kk] = *reinterpret_cast<const au4 *>(kc + base + (uint64_t)p * rstride +
                                                            32u * kk + 8u * g);
        }
    };
    auto load_v = [&](uint32_t t) {
#pragma unroll
        for (uint32_t j = 0; j < 8; j++) {
            const uint16_t *p = vc + base + (uint64_t)min(pos_of(t, j), valid - 1u) * rstride + DPL * n;
            typedef uint32_t vw __attribute__((ext_vector_type(VW == 3u ? 2u : VW), aligned(4)));
            const vw w = *reinterpret_cast<const vw *>(p);
#pragma unroll
            for (uint32_t i = 0; i < (VW == 3u ? 2u : VW); i++) vr[j][i] = w[i];
            if (VW == 3u) vr[j][VW - 1u] = reinterpret_cast<const uint32_t *>(p)[VW - 1u];
        }
    };
    // ---- q' of head n & 7 (heads past the group repeat head 0 and are not stored)
    const uint32_t h = n & 7u, hq = h < group ? h : 0u;
    float qv[KK][8];
    {
        const float4 *qp = reinterpret_cast<const float4 *>(q + ((uint64_t)kvh * group + hq) * HD);
#pragma unroll
        for (uint32_t kk = 0; kk < KK; kk++) {
            const float4 a = qp[(32u * kk + 8u * g) / 4u], b = qp[(32u * kk + 8u * g) / 4u + 1u];
            qv[kk][0] = a.x; qv[kk][1] = a.y; qv[kk][2] = a.z; qv[kk][3] = a.w;
            qv[kk][4] = b.x; qv[kk][5] = b.y; qv[kk][6] = b.z; qv[kk][7] = b.w;
        }
    }
    // the first tile's K and V rows go out with q's loads: one memory round
    // trip before the first MMA instead of two (the scheduler may not sink
    // them below q's arithmetic)
    load_k(0);
    load_v(0);
    __builtin_amdgcn_sched_barrier(0);
    float amax = 0.f;
#pragma unroll
    for (uint32_t kk = 0; kk < KK; kk++)
#pragma unroll
        for (uint32_t j = 0; j < 8; j++) amax = fmaxf(amax, fabsf(qv[kk][j]));
    amax = fmaxf(amax, lane_xor<16>(amax));
    amax = fmaxf(amax, lane_xor<32>(amax));
    int e2 = 0;
    (void)frexpf(amax, &e2);  // amax < 2^e2
    const int sq = amax > 0.f ? 15 - e2 : 0;
    const float csc = ldexpf(scale, -sq);
    // FINE (head sizes whose scores were double dots, or sums of eight dims per
    // lane, before this kernel took them): each dot is a double sum of one
    // product per 16 dims and of the hi and lo columns, the scores (times log2 e)
    // stay double until the maximum is taken off them, that is rounded up to a whole
    // number (or JOINT), and l adds the weights as they multiply V. Error against 64
    // bits over 1 to 32 q heads (of the kernels before; of f32 scores -> now), at 2, 7, 45, 228,
    // 3000 positions, in 1e-8: head_dim 32 6.3, 9.5, 13.4, 16.3, 19.3; 7.8, 10.1, 13.1, 15.7, 19.2
    // -> 5.8, 8.3, 11.0, 13.0, 17.4; 64 6.5, 9.4, 12.6, 15.0, 18.3; 7.8, 9.7, 13.0, 14.7, 18.5 -> 5.8,
    // 8.3, 10.5, 11.9, 17.0; 96 5.7, 8.2, 13.4, 15.8, 19.3; 7.9, 10.2, 13.5, 14.9, 19.1 -> 5.9, 8.7,
    // 11.2, 12.6, 17.7.
    const double c2 = (double)csc * 1.4426950408889634;
    ah8 Qb[KK];
#pragma unroll
    for (uint32_t kk = 0; kk < KK; kk++)
#pragma unroll
        for (uint32_t j = 0; j < 8; j++) {
            const float x = ldexpf(qv[kk][j], sq);
            const _Float16 hi = (_Float16)x;
            Qb[kk][j] = n < 8u ? hi : (_Float16)(x - (float)hi);
        }


    Score m = -INFINITY;
    float l = 0.f;
    af4 acc[DPL];
#pragma unroll
    for (uint32_t t = 0; t < DPL; t++) acc[t] = af4{0.f, 0.f, 0.f, 0.f};
    auto tile = [&](uint32_t t) {
        af4 S[2][FINE ? 2u * KK : 1u];
#pragma unroll
        for (uint32_t hf = 0; hf < 2; hf++) {
            if constexpr (FINE) {  // a sum of its own per 16 dims, added in double below
                typedef _Float16 ah4 __attribute__((ext_vector_type(4)));
                typedef uint32_t au2 __attribute__((ext_vector_type(2)));
                const af4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (uint32_t kk = 0; kk < KK; kk++)
#pragma unroll
                    for (uint32_t v = 0; v < 2u; v++) {
                        const au2 ka = {kr[hf][kk][2u * v], kr[hf][kk][2u * v + 1u]};
                        const au4 qq = __builtin_bit_cast(au4, Qb[kk]);
                        const au2 qa = {qq[2u * v], qq[2u * v + 1u]};
                        S[hf][2u * kk + v] = __builtin_amdgcn_mfma_f32_16x16x16f16(
                            __builtin_bit_cast(ah4, ka), __builtin_bit_cast(ah4, qa), z, 0, 0, 0);
                    }
            } else {
                S[hf][0] = af4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (uint32_t kk = 0; kk < KK; kk++)
                    S[hf][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(ah8, kr[hf][kk]),
                                                                  Qb[kk], S[hf][0], 0, 0, 0);
            }
        }
        if (t + 1u < nt) load_k(t + 1u);  // the K registers are free again
        // scores of positions p_j: hi + lo columns (lane n and n ^ 8), scaled, masked
        Score sc[8], mt = -INFINITY;
#pragma unroll
        for (uint32_t j = 0; j < 8; j++) {
            const bool in = pos_of(t, j) < valid;
            if constexpr (FINE) {
                double d = 0.0;
#pragma unroll
                for (uint32_t k = 0; k < 2u * KK; k++) d += (double)S[j >> 2][k][j & 3u];
                const uint64_t b = __builtin_bit_cast(uint64_t, d);
                const uint32_t h = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x128, 0xF, 0xF, false);
                const uint32_t l = __builtin_amdgcn_update_dpp(0, (int)b, 0x128, 0xF, 0xF, false);
                sc[j] = in ? (d + __builtin_bit_cast(double, (uint64_t)h << 32 | l)) * c2 : -INFINITY;
            } else {
                const float v = S[j >> 2][0][j & 3u];
                const float w = v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                                                                  0, __builtin_bit_cast(int, v), 0x128,
                                                                  0xF, 0xF, false));  // row_ror:8
                sc[j] = in ? __fmul_rn(w, csc) : -INFINITY;
            }
            mt = score_max(mt, sc[j]);
        }
        mt = score_max(mt, score_xor<16>(mt));
        mt = score_max(mt, score_xor<32>(mt));
        if constexpr (FINE) {
            if (JOINT && n_joint) {
                if (lane < 8u) joint[wave][lane] = mt;
                __syncthreads();
                double v[kOneChunks];
#pragma unroll
                for (uint32_t w = 0; w < kOneChunks; w++) v[w] = joint[w][n & 7u];
#pragma unroll
                for (uint32_t w = 0; w < kOneChunks; w++) mt = w < n_joint ? score_max(mt, v[w]) : mt;
            } else if (fabs(mt) < 0x1p23) {  // (past that a float has no room for the difference)
                mt = ceil(mt);
            }
        }
        const Score mn = score_max(m, mt);
        const float rs = m == -INFINITY ? 0.f : merge_exp<HD>((float)(m - mn));
        m = mn;
        l *= rs;
        ah8 P;
#pragma unroll
        for (uint32_t j = 0; j < 8; j++) {
            float e;
            if constexpr (FINE) {  // 2^(n + x), |x| <= 1/2
                const double d = sc[j] - mn, n = rint(d);
                e = ldexpf(exp2_fast((float)(d - n)), (int)n);
            } else {
                e = fast_exp(__fsub_rn(sc[j], mn));
            }
            if (sc[j] == -INFINITY) e = 0.f;
            const float es = e * PS;
            const _Float16 hi = (_Float16)es, lo = (_Float16)(es - (float)hi);
            l += FINE ? (float)hi + (float)lo : e;  // (FINE: the sum of the weights as they multiply V)
            P[j] = n < 8u ? hi : lo;
        }
        // D rows 4 g + r of the P V accumulators belong to head (4 g + r) & 7
        float rsr[4];
#pragma unroll
        for (uint32_t r = 0; r < 4; r++) rsr[r] = __shfl(rs, (4u * g + r) & 7u, 64);
#pragma unroll
        for (uint32_t dt = 0; dt < DPL; dt++) {
            // B: element dt (head dim DPL n + dt) of each of the lane's eight V rows
            const uint32_t sel = (dt & 1u) ? 0x07060302u : 0x05040100u;
            au4 b;
#pragma unroll
            for (uint32_t i = 0; i < 4; i++)
                b[i] = __builtin_amdgcn_perm(vr[2 * i + 1][dt >> 1], vr[2 * i][dt >> 1], sel);
            af4 a = acc[dt];
#pragma unroll
            for (uint32_t r = 0; r < 4; r++) a[r] *= rsr[r];
            acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(P, __builtin_bit_cast(ah8, b), a, 0, 0, 0);
        }
        if (t + 1u < nt) load_v(t + 1u);
    };
    tile(0);  // peeled, so that its loads and uses share the entry block with q's
    for (uint32_t t = 1; t < nt; t++) tile(t);

    // ---- the chunk's partial: l summed over the lane groups of a head, rows
    // hi + lo of acc (lane groups g and g + 2), stored by lane groups 0 and 1
    l += lane_xor<16>(l);
    l += lane_xor<32>(l);
#pragma unroll
    for (uint32_t dt = 0; dt < DPL; dt++)
#pragma unroll
        for (uint32_t r = 0; r < 4; r++) a[dt][r] = (acc[dt][r] + lane_xor<32>(acc[dt][r])) * (1.f / PS);
    m_out = (float)m;
    l_out = l * (1.f / PS);
}

// A chunk's (m, l, acc) to its partials row (chunk rows `stride` apart per q
// head; HD + 2 floats each).
template <uint32_t HD>
__device__ __forceinline__ void attn_mfma_store(float *pk, uint32_t stride, uint32_t chunk, uint32_t group,
                                                uint32_t lane, float m, float l, const float (&a)[HD / 16][4]) {
    constexpr uint32_t DPL = HD / 16u;
    const uint32_t n = lane & 15u, g = lane >> 4;
    if (g < 2u) {
#pragma unroll
        for (uint32_t r = 0; r < 4; r++) {
            const uint32_t hh = 4u * g + r;
            if (hh < group) {
                float *dst = pk + ((uint64_t)hh * stride + chunk) * part_row<HD> + 2u + DPL * n;
#pragma unroll
                for (uint32_t i = 0; i < DPL / 2u; i++)
                    reinterpret_cast<float2 *>(dst)[i] = make_float2(a[2 * i][r], a[2 * i + 1][r]);
            }
        }
    }
    if (g == 0 && n < group) {
        float *dst = pk + ((uint64_t)n * stride + chunk) * part_row<HD>;
        dst[0] = m;
        dst[1] = l;
    }
}

// Head sizes but 128: one q head (qh) over `valid` <= kMfmaLmax positions from
// base on, in whole f32 products: scores as double dots, a lane per position;
// on return o[dt] = the sum of 2^(s log2 e - m) v[DPL n + dt] in every lane group.
// For heads whose sums are not finite: an infinite score or value meets the hi
// and lo halves of attn_mfma_wave as inf - inf or 0 * inf. Here, as in the
// sequential softmax, -inf scores weigh 0, +inf and NaN give NaN, and an infinite
// value of positive weight gives inf. About 2.5 us per 64 positions.
template <uint32_t HD>
__device__ __forceinline__ void attn_head_whole(const float *__restrict__ qh, const uint16_t *__restrict__ kc,
                                                const uint16_t *__restrict__ vc, uint64_t base, uint32_t valid,
                                                uint64_t rstride, float scale, uint32_t lane, float &m_out,
                                                float &l_out, float (&o)[HD / 16]) {
    constexpr uint32_t DPL = HD / 16u, NP = kMfmaLmax / 64u;  // positions per lane
    const uint32_t n = lane & 15u;
    float sc[NP], e[NP], mt = -INFINITY, l = 0.f;
#pragma unroll
    for (uint32_t i = 0; i < NP; i++) {
        const uint32_t p = lane + 64u * i;
        double d = 0.0;
        if (64u * i < valid) {
            const uint16_t *kr = kc + base + (uint64_t)min(p, valid - 1u) * rstride;
#pragma unroll
            for (uint32_t c = 0; c < HD; c += 8u) {
                const au4 kw = *reinterpret_cast<const au4 *>(kr + c);
#pragma unroll
                for (uint32_t k = 0; k < 8u; k++)
                    d = fma((double)qh[c + k], (double)hcvt(kw[k >> 1] >> (16u * (k & 1u))), d);
            }
        }
        sc[i] = p < valid ? __fmul_rn((float)d, scale) : -INFINITY;
        mt = fmaxf(mt, __fmul_rn(sc[i], 1.44269504088896341f));
    }
    const float mn = ceilf(wave_max(mt));  // (a whole power of two, as attn_mfma_wave's)
#pragma unroll
    for (uint32_t i = 0; i < NP; i++) {
        const float p = __fmul_rn(sc[i], 1.44269504088896341f), r = rintf(p);
        const float err = fmaf(sc[i], 1.92596299e-8f, fmaf(sc[i], 1.44269504088896341f, -p));
        e[i] = ldexpf(exp2_fast((p - r) + __builtin_amdgcn_fmed3f(err, -0.5f, 0.5f)), (int)(r - mn));
        if (sc[i] == -INFINITY) e[i] = 0.f;
        l += e[i];
    }
    m_out = mn;
    l_out = wave_sum(l);
#pragma unroll
    for (uint32_t dt = 0; dt < DPL; dt++) o[dt] = 0.f;
#pragma unroll
    for (uint32_t i = 0; i < NP; i++)
        for (uint32_t p0 = 64u * i; p0 < min(valid, 64u * (i + 1u)); p0 += 8u) {
            uint16_t vr[8][DPL];  // (eight rows requested at a time)
#pragma unroll
            for (uint32_t k = 0; k < 8u; k++)
#pragma unroll
                for (uint32_t dt = 0; dt < DPL; dt++)
                    vr[k][dt] = vc[base + (uint64_t)min(p0 + k, valid - 1u) * rstride + DPL * n + dt];
#pragma unroll
            for (uint32_t k = 0; k < 8u; k++) {
                const float w = __shfl(e[i], (int)((p0 + k) & 63u), 64);
                if (p0 + k < valid) {
#pragma unroll
                    for (uint32_t dt = 0; dt < DPL; dt++) o[dt] = fmaf(w, hcvt(vr[k][dt]), o[dt]);
                }
            }
        }
}

// The heads of a chunk whose sums (l, a: what attn_mfma_store has just stored) are
// not finite once more. The test hides behind those stores.
template <uint32_t HD>
__device__ __forceinline__ void attn_heads_again(const float *__restrict__ q, const uint16_t *__restrict__ kc,
                                                 const uint16_t *__restrict__ vc, uint64_t layer_off, uint32_t s0,
                                                 uint32_t valid, uint32_t nkh, uint32_t kvh, uint32_t group,
                                                 float scale, uint32_t lane, float *pk, uint32_t stride,
                                                 uint32_t chunk, float l, const float (&a)[HD / 16][4]) {
    constexpr uint32_t DPL = HD / 16u;
    const uint32_t n = lane & 15u, g = lane >> 4;
    float t[4] = {0.f, 0.f, 0.f, 0.f};  // NaN where a head's sums are not finite
#pragma unroll
    for (uint32_t dt = 0; dt < DPL; dt++)
#pragma unroll
        for (uint32_t r = 0; r < 4; r++) t[r] = fmaf(a[dt][r], 0.f, t[r]);
    if (__builtin_expect(!__ballot(fmaf(l, 0.f, (t[0] + t[1]) + (t[2] + t[3])) != 0.f), 1)) return;
    const uint64_t rstride = (uint64_t)nkh * HD, base = layer_off + (uint64_t)s0 * rstride + (uint64_t)kvh * HD;
#pragma unroll 1
    for (uint32_t hh = 0; hh < group; hh++) {
        bool bad = (n & 7u) == hh && !(fabsf(l) <= 3.4028235e38f);
#pragma unroll
        for (uint32_t r = 0; r < 4; r++) bad |= 4u * (g & 1u) + r == hh && t[r] != 0.f;
        if (!__ballot(bad)) continue;
        float mw, lw, o[DPL];
        attn_head_whole<HD>(q + ((uint64_t)kvh * group + hh) * HD, kc, vc, base, valid, rstride, scale, lane, mw, lw,
                            o);
        // (by the lanes that stored the head's row before)
        float *dst = pk + ((uint64_t)hh * stride + chunk) * part_row<HD>;
        if (g == hh >> 2) {
#pragma unroll
            for (uint32_t i = 0; i < DPL / 2u; i++)
                reinterpret_cast<float2 *>(dst + 2u + DPL * n)[i] = make_float2(o[2 * i], o[2 * i + 1]);
        }
        if (g == 0u && n == hh) {
            dst[0] = mw;
            dst[1] = lw;
        }
    }
}

// A chunk from its positions to its partials row.
template <uint32_t HD>
__device__ __forceinline__ void attn_mfma_chunk(const float *__restrict__ q, const uint16_t *__restrict__ kc,
                                                const uint16_t *__restrict__ vc, uint64_t layer_off, uint32_t s0,
                                                uint32_t valid, uint32_t nt, uint32_t nkh, uint32_t kvh,
                                                uint32_t group, float scale, uint32_t lane, float *pk,
                                                uint32_t stride, uint32_t chunk) {
    float m, l, a[HD / 16][4];
    attn_mfma_wave<HD>(q, kc, vc, layer_off, s0, valid, nt, nkh, kvh, group, scale, lane, m, l, a);
    attn_mfma_store<HD>(pk, stride, chunk, group, lane, m, l, a);
    if constexpr (HD != 128u)
        attn_heads_again<HD>(q, kc, vc, layer_off, s0, valid, nkh, kvh, group, scale, lane, pk, stride, chunk, l, a);
}

// A chunk per workgroup: one wave, or (MULTI, head sizes but 128) the chunk's
// tiles split over up to kFineWaves waves, whose sums are joined in LDS: their
// maxima are whole powers of two, so the weights are exact.
template <uint32_t HD, bool MULTI = false>
__global__ __launch_bounds__(MULTI ? 64 * kFineWaves : 64) void k_attn_mfma(const float *__restrict__ q,
                                                  const uint16_t *__restrict__ kc,
                                                  const uint16_t *__restrict__ vc,
                                                  float *__restrict__ part, uint32_t seq_len,
                                                  const uint32_t *__restrict__ pos_dev,
                                                  uint64_t layer_off, uint32_t nkh, uint32_t group,
                                                  float scale, uint32_t stride_chunks,
                                                  uint32_t q_bstride, uint64_t kv_bstride,
                                                  uint64_t part_bstride, uint32_t target,
                                                  uint32_t *__restrict__ clear, uint32_t nclear,
                                                  uint32_t clear_stride) {
    const uint32_t chunk = blockIdx.x, kvh = blockIdx.y, lane = threadIdx.x & 63u, bz = blockIdx.z;
    // the merging launch that follows (k_mvl_attn) starts from cleared flags
    if (clear && chunk == 0u && kvh == 0u && bz == 0u)
        for (uint32_t i = lane; i < nclear; i += 64u) clear[(uint64_t)i * clear_stride] = 0u;
    // sequence bz of a batch: its q, caches, position and partials
    q += (uint64_t)bz * q_bstride;
    kc += bz * kv_bstride;
    vc += bz * kv_bstride;
    part += bz * part_bstride;
    if (pos_dev) seq_len = pos_dev[bz] + 1u;  // graph replay: the device holds the position
    const AttnSplit sp = mfma_split<HD>(seq_len, nkh, target);
    if (chunk >= sp.n) return;  // past the sequence (the grid covers the longest split)
    const uint32_t s0 = chunk * sp.len, valid = min(sp.len, seq_len - s0);
    float *const pk = part + (uint64_t)kvh * group * stride_chunks * part_row<HD>;
    if constexpr (!MULTI) {
        attn_mfma_chunk<HD>(q, kc, vc, layer_off, s0, valid, sp.len / kMfmaGran, nkh, kvh, group, scale, lane, pk,
                            stride_chunks, chunk);
    } else {
        extern __shared__ __align__(16) float joint[];  // [group][waves][HD + 2]
        const uint32_t nw = blockDim.x >> 6, wave = threadIdx.x >> 6;
        const uint32_t tiles = (valid + kMfmaGran - 1u) / kMfmaGran, tpw = (tiles + nw - 1u) / nw;
        const uint32_t used = (tiles + tpw - 1u) / tpw, w0 = kMfmaGran * tpw * wave;
        if (wave < used) {
            const uint32_t v = min(kMfmaGran * tpw, valid - w0);
            attn_mfma_chunk<HD>(q, kc, vc, layer_off, s0 + w0, v, (v + kMfmaGran - 1u) / kMfmaGran, nkh, kvh, group,
                                scale, lane, joint, nw, wave);
        }
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < group * (HD / 2u); i += blockDim.x) {
            const uint32_t hh = i / (HD / 2u), d = 2u * (i % (HD / 2u));
            const float *row = joint + hh * nw * part_row<HD>;
            float M = row[0];
            for (uint32_t w = 1; w < used; w++) M = fmaxf(M, row[w * part_row<HD>]);
            float l = 0.f, ax = 0.f, ay = 0.f;
            for (uint32_t w = 0; w < used; w++) {
                const float *rw = row + w * part_row<HD>;
                const float wt = rw[0] == -INFINITY ? 0.f : ldexpf(1.f, (int)(rw[0] - M));
                l = fmaf(rw[1], wt, l);
                ax = fmaf(rw[2u + d], wt, ax);
                ay = fmaf(rw[3u + d], wt, ay);
            }
            float *dst = pk + ((uint64_t)hh * stride_chunks + chunk) * part_row<HD>;
            *reinterpret_cast<float2 *>(dst + 2u + d) = make_float2(ax, ay);
            if (d == 0u) *reinterpret_cast<float2 *>(dst) = make_float2(M, l);
        }
    }
}

// Short sequences (at most kOneChunks chunks) in one launch: workgroup kvh
// takes the kv head's chunks one per wave, as k_attn_mfma does (bit-identical:
// the same split, arithmetic and merge), leaves the partials in LDS and merges
// its q heads there.

template <uint32_t HD>
__global__ __launch_bounds__(64 * kOneChunks) void k_attn_one(
    const float *__restrict__ q, const uint16_t *__restrict__ kc, const uint16_t *__restrict__ vc,
    float *__restrict__ out, uint32_t seq_len, const uint32_t *__restrict__ pos_dev, uint64_t layer_off,
    uint32_t nkh, uint32_t group, float scale) {
    extern __shared__ __align__(16) float part[];  // [group][kOneChunks][HD + 2]
    const uint32_t nw = blockDim.x >> 6, kvh = blockIdx.x, lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    if (pos_dev) seq_len = pos_dev[0] + 1u;
    // (mfma_split's bound on the chunk count is not met at such lengths)
    const AttnSplit sp = attn_split(seq_len, nkh, kMfmaGran, kMfmaLmax, kMfmaTargetWgs);
    __shared__ double joint[HD == 128u ? 1 : kOneChunks][8];
    const bool is_joint = HD != 128u && sp.len == kMfmaGran;
    if (wave < sp.n) {
        const uint32_t s0 = wave * sp.len, valid = min(sp.len, seq_len - s0);
        float m, l, a[HD / 16][4];
        attn_mfma_wave<HD, HD != 128u>(q, kc, vc, layer_off, s0, valid, sp.len / kMfmaGran, nkh, kvh, group, scale, lane,
                                       m, l, a, joint, is_joint ? sp.n : 0u, wave);
        attn_mfma_store<HD>(part, kOneChunks, wave, group, lane, m, l, a);
    } else if (is_joint) {
        __syncthreads();  // (attn_mfma_wave's)
    }
    __syncthreads();
    uint32_t again = 0;  // heads whose results are not finite (attn_head_whole)
    for (uint32_t h = wave; h < group; h += nw) {
        const float2 o = merge_one_wave<kOneChunks, HD>(part + h * kOneChunks * part_row<HD>, sp.n, lane);
        if (HD == 128u || lane < HD / 2u)
            *reinterpret_cast<float2 *>(out + ((uint64_t)kvh * group + h) * HD + 2u * lane) = o;
        if (HD != 128u && __ballot(lane < HD / 2u && fmaf(o.x, 0.f, o.y * 0.f) != 0.f)) again |= 1u << h;
    }
    if constexpr (HD != 128u) {
        if (__builtin_expect(again != 0u, 0)) {
            constexpr uint32_t DPL = HD / 16u;
            // dims 2 lane and 2 lane + 1 go to the lane that stored them before
            const uint32_t at = 2u * (lane % (HD / 2u)), src = at / DPL, d0 = at % DPL;
#pragma unroll 1
            for (uint32_t h = wave; h < group; h += nw) {
                if (!((again >> h) & 1u)) continue;
                // (many kv heads have longer chunks, and more positions than attn_head_whole takes at once)
                float m = -INFINITY, l = 0.f, w[DPL] = {};
#pragma unroll 1
                for (uint32_t p0 = 0; p0 < seq_len; p0 += kMfmaLmax) {
                    float mp, lp, wp[DPL];
                    attn_head_whole<HD>(q + ((uint64_t)kvh * group + h) * HD, kc, vc,
                                        layer_off + ((uint64_t)p0 * nkh + kvh) * HD, min(kMfmaLmax, seq_len - p0),
                                        (uint64_t)nkh * HD, scale, lane, mp, lp, wp);
                    const float mn = fmaxf(m, mp);
                    const float r = m == -INFINITY ? 0.f : ldexpf(1.f, (int)(m - mn));
                    const float rp = mp == -INFINITY ? 0.f : ldexpf(1.f, (int)(mp - mn));
                    m = mn;
                    l = fmaf(lp, rp, l * r);
#pragma unroll
                    for (uint32_t dt = 0; dt < DPL; dt++) w[dt] = fmaf(wp[dt], rp, w[dt] * r);
                }
                float2 r = make_float2(0.f, 0.f);
#pragma unroll
                for (uint32_t i = 0; i < DPL / 2u; i++) {
                    const float x = __shfl(w[2 * i], (int)src, 64), y = __shfl(w[2 * i + 1], (int)src, 64);
                    if (d0 == 2u * i) r = make_float2(x, y);
                }
                if (lane < HD / 2u)
                    *reinterpret_cast<float2 *>(out + ((uint64_t)kvh * group + h) * HD + 2u * lane) =
                        make_float2(r.x / l, r.y / l);
            }
        }
    }
}

// ---- merge of the chunks -------------------------------------------------------
// One workgroup of kMergeThreads per q head; every global load is issued up
// front: thread (d, slice) loads acc_c[d] of its chunks c = slice, slice + ns,
// ... and thread t also m_t and l_t. Then M = max_c m_c (block maximum),
// weights w_c = e^(m_c - M) in LDS, L = sum_c l_c w_c, and the slices'
// weighted sums are added in LDS in a fixed order.
constexpr uint32_t kMergeThreadBatch = 32;     // chunks per thread held in registers at once
constexpr uint32_t kMergeThreads = 512;  // (measured 2-8% faster than 1024 and than 256)

__global__ __launch_bounds__(kMergeThreads) void k_attn_merge(const float *__restrict__ part,
                                                    float *__restrict__ out, uint32_t hd,
                                                    uint32_t n_chunks, uint32_t stride_chunks,
                                                    const uint32_t *__restrict__ pos_dev,
                                                    uint32_t nkh, uint32_t gran, uint32_t lmax) {
    extern __shared__ __align__(16) uint8_t merge_lds[];
    float *w = reinterpret_cast<float *>(merge_lds);  // [stride_chunks]
    float *sl = w + stride_chunks;                    // [kMergeThreads]
    constexpr uint32_t NW = kMergeThreads / 64u;
    __shared__ float red[2 * NW];
    const uint32_t h = blockIdx.x, t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    if (pos_dev) n_chunks = attn_split(pos_dev[0] + 1u, nkh, gran, lmax, kTargetWgs).n;  // seq = pos + 1
    const float *ph = part + (uint64_t)h * stride_chunks * (hd + 2u);
    const uint32_t ns = kMergeThreads / hd;
    const uint32_t d = t % hd, s = t / hd;
    float av[kMergeThreadBatch];
#pragma unroll
    for (uint32_t k = 0; k < kMergeThreadBatch; k++) {
        const uint32_t c = s + k * ns;
        av[k] = (s < ns && c < n_chunks) ? ph[(uint64_t)c * (hd + 2u) + 2u + d] : 0.f;
    }
    // this thread's chunks' (m, l): c = t, t + kMergeThreads, ...; the first
    // pair is loaded with the acc values, before any reduction
    float m0 = -INFINITY, l0 = 0.f;
    if (t < n_chunks) {
        m0 = ph[(uint64_t)t * (hd + 2u)];
        l0 = ph[(uint64_t)t * (hd + 2u) + 1u];
    }
    float M = m0;
    for (uint32_t c = t + kMergeThreads; c < n_chunks; c += kMergeThreads)
        M = fmaxf(M, ph[(uint64_t)c * (hd + 2u)]);
    M = wave_max(M);
    if (lane == 0) red[wave] = M;
    __syncthreads();
    M = red[0];
    for (uint32_t i = 1; i < NW; i++) M = fmaxf(M, red[i]);
    float L = 0.f;
    if (t < n_chunks) {
        const float wc = m0 == -INFINITY ? 0.f : fast_exp(__fsub_rn(m0, M));
        w[t] = wc;
        L = fmaf(l0, wc, L);
    }
    for (uint32_t c = t + kMergeThreads; c < n_chunks; c += kMergeThreads) {
        const float *pc = ph + (uint64_t)c * (hd + 2u);
        const float mc = pc[0], wc = mc == -INFINITY ? 0.f : fast_exp(__fsub_rn(mc, M));
        w[c] = wc;
        L = fmaf(pc[1], wc, L);
    }
    L = wave_sum(L);
    if (lane == 0) red[NW + wave] = L;
    __syncthreads();
    L = 0.f;
    for (uint32_t i = 0; i < NW; i++) L += red[NW + i];
    float a = 0.f;
    if (s < ns) {
#pragma unroll
        for (uint32_t k = 0; k < kMergeThreadBatch; k++) {
            const uint32_t c = s + k * ns;
            if (c < n_chunks) a = fmaf(av[k], w[c], a);
        }
        for (uint32_t c = s + kMergeThreadBatch * ns; c < n_chunks; c += ns)
            a = fmaf(ph[(uint64_t)c * (hd + 2u) + 2u + d], w[c], a);
    }
    sl[t] = a;
    __syncthreads();
    if (t < hd) {
        float acc = 0.f;
        for (uint32_t k = 0; k < ns; k++) acc += sl[k * hd + t];
        out[(uint64_t)h * hd + t] = __fmul_rn(acc, __fdiv_rn(1.0f, L));
    }
}

// Merge of the matrix-core chunk kernel's partials: one
// workgroup of four waves per q head (grid y: the sequences of a batch). Every
// wave forms M, L and the chunk weights itself from all chunks' (m, l); wave r
// takes residue r of the chunks (vbs_attn_common.h), its acc rows loaded at
// once, and one LDS pass adds the four sums in order. No loads wait on a
// reduction and one barrier ends it (the general merge above has four).
template <uint32_t HD>
__global__ __launch_bounds__(64 * kMergeRes) void k_attn_merge_hd(
    const float *__restrict__ part, float *__restrict__ out, uint32_t stride_chunks,
    const uint32_t *__restrict__ pos_dev, uint32_t seq_len, uint32_t nkh, uint32_t q_bstride,
    uint64_t part_bstride, uint32_t target) {
    __shared__ float2 red[kMergeRes][64];
    const uint32_t h = blockIdx.x, bz = blockIdx.y, lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    part += bz * part_bstride;
    out += (uint64_t)bz * q_bstride;
    if (pos_dev) seq_len = pos_dev[bz] + 1u;  // seq = pos + 1
    const uint32_t nc = mfma_split<HD>(seq_len, nkh, target).n;
    const float *ph = part + (uint64_t)h * stride_chunks * part_row<HD>;
    float2 av[kMergeBatch];
    merge_residue_load<HD>(ph, nc, wave, lane, av);  // with the (m, l) loads: one round trip
    const MergeStats st = merge_stats<HD>(ph, nc, lane, merge_ml_load<HD>(ph, nc, lane));
    red[wave][lane] = merge_residue_sum<HD>(ph, nc, st, wave, lane, av);
    __syncthreads();
    if (wave == 0) {
        float2 a[kMergeRes];
#pragma unroll
        for (uint32_t r = 0; r < kMergeRes; r++) a[r] = red[r][lane];
        if (HD == 128u || lane < HD / 2u)
            *reinterpret_cast<float2 *>(out + (uint64_t)h * HD + 2u * lane) = merge_finish<HD>(a, st.L);
    }
}

size_t attention_partial_bytes(uint32_t max_seq, uint32_t nqh, uint32_t nkh, uint32_t hd) {
    return (size_t)nqh * attn_max_chunks(max_seq, nkh) * (hd + 2u) * sizeof(float);
}

// The general merge after k_attn_partial or k_attn_solo.
static hipError_t launch_merge(const float *part, float *out, uint32_t seq_len, const uint32_t *pos_dev,
                               uint32_t nqh, uint32_t nkh, uint32_t hd, uint32_t gran, uint32_t lmax,
                               hipStream_t s) {
    const uint32_t stride = attn_max_chunks(seq_len, nkh);
    const size_t lds = ((size_t)stride + kMergeThreads) * sizeof(float);
    k_attn_merge<<<nqh, kMergeThreads, lds, s>>>(part, out, hd, attn_split(seq_len, nkh, gran, lmax, kTargetWgs).n,
                                                 stride, pos_dev, nkh, gran, lmax);
    return hipGetLastError();
}

// The matrix-core path of one sequence: one launch up to kOneChunks chunks
// (seq_len is the longest that the launch must cover), else chunks and merge.
template <uint32_t HD>
static hipError_t launch_mfma_hd(const float *q, const uint16_t *kc, const uint16_t *vc, float *out,
                                 float *part, uint32_t seq_len, const uint32_t *pos_dev, uint64_t layer_off,
                                 uint32_t nkh, uint32_t group, float scale, hipStream_t s) {
    const uint32_t chunks = mfma_grid_chunks<HD>(seq_len, nkh), stride = attn_max_chunks(seq_len, nkh);
    // One launch: 41 positions of 8 kv heads 3.7-4.8 us (chunks and merge 6.4-7.5),
    // 256 of head_dim 64 5.4-6.0 (6.4-7.0); at head_dim 128 and eight q heads per kv head
    // 256 positions are too many for one workgroup (7.9 against 7.1), 96 alike.
    if (chunks <= (HD <= 64u ? kOneChunks : kOneChunks / 2u)) {
        const uint32_t nw = chunks > group ? chunks : group;  // a wave per chunk, then per q head
        const size_t lds = (size_t)group * kOneChunks * part_row<HD> * sizeof(float);
        k_attn_one<HD><<<nkh, 64u * nw, lds, s>>>(q, kc, vc, out, seq_len, pos_dev, layer_off, nkh, group,
                                                     scale);
        return hipGetLastError();
    }
    if constexpr (HD == 32u || HD == 64u) {
        if (group == 1u) {  // (k_attn_solo: why)
            using S = ChunkShape<HD>;
            const uint32_t n = pos_dev ? stride : attn_split(seq_len, nkh, S::GRAN, S::LMAX, kTargetWgs).n;
            k_attn_solo<HD><<<dim3(n, nkh), 64u * kWaves, 0, s>>>(q, kc, vc, part, seq_len, pos_dev, layer_off, nkh,
                                                                  scale, stride);
            const hipError_t e = hipGetLastError();
            return e != hipSuccess ? e : launch_merge(part, out, seq_len, pos_dev, nkh, nkh, HD, S::GRAN, S::LMAX, s);
        }
    }
    // Long chunks of few kv heads are split over waves (4 q heads over 2 kv heads,
    // head_dim 64, 16000 positions 10.9 -> 9.0 us, 16 over 4 11.4 -> 10.6); with more
    // workgroups than this the chip is full of waves (32 over 8 14.2, split 15.9).
    // Two tiles pay for joining two waves' sums only below a workgroup per CU
    // (6000 positions, 4 over 2 8.6 -> 8.2, 16 over 4 8.8 -> 9.6).
    const uint32_t tiles = mfma_split<HD>(seq_len, nkh).len / kMfmaGran, wgs = chunks * nkh;
    const bool multi = HD != 128u && tiles > 1u && wgs <= (tiles > 2u ? 512u : 256u);
    if constexpr (HD != 128u) {
        const uint32_t nw = tiles < kFineWaves ? tiles : kFineWaves;
        if (multi)
            k_attn_mfma<HD, true><<<dim3(chunks, nkh), 64u * nw, (size_t)group * nw * part_row<HD> * sizeof(float), s>>>(
                q, kc, vc, part, seq_len, pos_dev, layer_off, nkh, group, scale, stride, 0u, 0ull, 0ull,
                kMfmaTargetWgs, nullptr, 0u, 0u);
    }
    if (!multi)
        k_attn_mfma<HD><<<dim3(chunks, nkh), 64, 0, s>>>(q, kc, vc, part, seq_len, pos_dev, layer_off, nkh, group,
                                                        scale, stride, 0u, 0ull, 0ull, kMfmaTargetWgs, nullptr, 0u,
                                                        0u);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    k_attn_merge_hd<HD><<<nkh * group, 64 * kMergeRes, 0, s>>>(part, out, stride, pos_dev, seq_len, nkh, 0u, 0ull,
                                                             kMfmaTargetWgs);
    return hipGetLastError();
}

hipError_t launch_attention(const float *q, const uint16_t *kc, const uint16_t *vc, float *out,
                            uint32_t seq_len, const uint32_t *pos_dev, float *part,
                            uint64_t layer_off, uint32_t nqh, uint32_t nkh, uint32_t hd,
                            float scale, hipStream_t s) {
    if (seq_len == 0 || nkh == 0 || nqh % nkh != 0 || hd == 0 || hd > 256 || (hd & 1u))
        return hipErrorInvalidValue;
    const uint32_t group = nqh / nkh;
    if (group > kMaxGroup) return hipErrorInvalidValue;
    // with pos_dev, seq_len is the largest sequence the grid must cover
    const uint32_t stride = attn_max_chunks(seq_len, nkh);
    if (!part) {
        hipError_t why;
        part = (float *)rt_scratch(attention_partial_bytes(seq_len, nqh, nkh, hd), s, &why);
        if (!part) return why;
    }
    if (group <= 8u && ((uintptr_t)q & 15u) == 0 && ((uintptr_t)kc & 15u) == 0 && ((uintptr_t)vc & 15u) == 0) {
#define VBS_ATTN_HD(HD)                                                                                \
    case HD:                                                                                           \
        return launch_mfma_hd<HD>(q, kc, vc, out, part, seq_len, pos_dev, layer_off, nkh, group, scale, s)
        switch (hd) {
            VBS_ATTN_HD(32);
            VBS_ATTN_HD(64);
            VBS_ATTN_HD(96);
            VBS_ATTN_HD(128);
            default: break;
        }
#undef VBS_ATTN_HD
    }
    const size_t lds = ((size_t)group * hd + (size_t)group * kChunk + (size_t)(256u / hd) * group * hd) *
                       sizeof(float);
    k_attn_partial<<<dim3(stride, nkh), 256, lds, s>>>(q, kc, vc, part, seq_len, pos_dev, layer_off, nkh, hd,
                                                       group, scale, stride);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_merge(part, out, seq_len, pos_dev, nqh, nkh, hd, kChunk, kChunk, s);
}

uint32_t attention_chunk_stride(uint32_t max_seq, uint32_t nkh) { return attn_max_chunks(max_seq, nkh); }

// The matrix-core chunk launch alone (head_dim 128, group <= 8), for a merge
// done by the launch that follows it (k_mvl_attn): the partials at part with
// attention_chunk_stride(seq_len, nkh) chunks per q head, and the words
// clear[i stride], i < nclear, zeroed for that launch's exchange.
hipError_t launch_attention_chunks(const float *q, const uint16_t *kc, const uint16_t *vc,
                                   uint32_t seq_len, const uint32_t *pos_dev, float *part,
                                   uint64_t layer_off, uint32_t nqh, uint32_t nkh, uint32_t hd,
                                   float scale, uint32_t *clear, uint32_t nclear, uint32_t stride,
                                   hipStream_t s) {
    if (seq_len == 0 || nkh == 0 || nqh % nkh != 0 || hd != 128u || nqh / nkh > 8u || !part ||
        ((uintptr_t)q & 15u) || ((uintptr_t)kc & 15u) || ((uintptr_t)vc & 15u))
        return hipErrorNotSupported;
    k_attn_mfma<128><<<dim3(mfma_grid_chunks(seq_len, nkh), nkh), 64, 0, s>>>(
        q, kc, vc, part, seq_len, pos_dev, layer_off, nkh, nqh / nkh, scale, attn_max_chunks(seq_len, nkh),
        0u, 0ull, 0ull, kMfmaTargetWgs, clear, nclear, stride);
    return hipGetLastError();
}

bool attn_mfma_batch_fits(const float *q, const uint16_t *kc, const uint16_t *vc, uint32_t nqh,
                          uint32_t nkh, uint32_t hd, uint32_t q_stride, uint64_t kv_stride) {
    return nkh != 0u && nqh % nkh == 0u && hd == 128u && nqh / nkh <= 8u && ((uintptr_t)q & 15u) == 0 &&
           ((uintptr_t)kc & 15u) == 0 && ((uintptr_t)vc & 15u) == 0 && (q_stride % 4u) == 0 &&
           (kv_stride % 8u) == 0;
}

hipError_t launch_attention_batch(const float *q, const uint16_t *kc, const uint16_t *vc,
                                  float *out, uint32_t max_seq, const uint32_t *pos_dev,
                                  float *part, uint64_t layer_off, uint32_t nqh, uint32_t nkh,
                                  uint32_t hd, float scale, uint32_t batch, uint32_t q_stride,
                                  uint64_t kv_stride, hipStream_t s) {
    if (batch == 0 || !part || !pos_dev) return hipErrorInvalidValue;
    if (!out && !attn_mfma_batch_fits(q, kc, vc, nqh, nkh, hd, q_stride, kv_stride))
        return hipErrorNotSupported;
    if (max_seq == 0 || nkh == 0 || nqh % nkh != 0) return hipErrorInvalidValue;
    const uint64_t pstride = attention_partial_bytes(max_seq, nqh, nkh, hd) / sizeof(float);
    const uint32_t group = nqh / nkh;
    const bool mfma = attn_mfma_batch_fits(q, kc, vc, nqh, nkh, hd, q_stride, kv_stride);
    if (!mfma) {  // one sequence at a time through the single-sequence path
        for (uint32_t b = 0; b < batch; b++) {
            const hipError_t e = launch_attention(q + (uint64_t)b * q_stride, kc + b * kv_stride,
                                                  vc + b * kv_stride, out + (uint64_t)b * q_stride,
                                                  max_seq, pos_dev + b, part + b * pstride, layer_off,
                                                  nqh, nkh, hd, scale, s);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    const uint32_t stride = attn_max_chunks(max_seq, nkh), target = attn_batch_target(batch);
    k_attn_mfma<128><<<dim3(mfma_grid_chunks(max_seq, nkh, target), nkh, batch), 64, 0, s>>>(
        q, kc, vc, part, max_seq, pos_dev, layer_off, nkh, group, scale, stride, q_stride, kv_stride,
        pstride, target, nullptr, 0u, 0u);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || !out) return e;  // (no out: the caller merges the partials itself)
    k_attn_merge_hd<128><<<dim3(nqh, batch), 64 * kMergeRes, 0, s>>>(part, out, stride, pos_dev,
                                                                     max_seq, nkh, q_stride, pstride,
                                                                     target);
    return hipGetLastError();
}

}  // namespace vbs
