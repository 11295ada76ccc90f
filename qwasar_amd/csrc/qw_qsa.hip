// qw_qsa.hip -- Qwen Sparse Attention on gfx950: the indexer's block scores,
// the stored block keys, top-k block selection and attention over the
// selected positions (reference contract qwasar_gpu.h:617-646, CPU semantics
// qwasar_flash_cpu.c:347-478).
//
// Block key (k_qsa_scores phase 1, k_qsa_pool): a wave per block, lane l
// owning dims l, l+64, ...: the serial mean of the block's `ratio` raw keys,
// the rms norm with the k_layernorm gain, then the rotary pair (j, j+32) of
// the first 64 dims at the block's first position -- lanes j and j+32, one
// swizzle apart.
//
// Score: up to 16 query heads of up to 128 dims on the fp32 matrix cores
// (k_qsa_scores_mx, below); else (k_qsa_scores phase 2) the keys are transposed through LDS so that a thread owns
// one block's key in registers; the row's query heads sit in LDS and are read
// as broadcast float4s.  Thread (wave w, lane l) scores block l against heads
// w, w+4, ...: per head a serial fma chain over the dims, the positive dots
// summed in head order; the four waves' partials meet as (p0 + p1) + (p2 +
// p3), then / sqrt(d).  Either way the arithmetic does not depend on how many
// rows or blocks a call has, and the pooled path runs the same sums on stored
// keys, so scores and pooled scores agree bit for bit.
//
// Selection (k_qsa_select): a workgroup of 1024 threads per query.  Scores
// map to 32-bit keys that order as the floats do (-0 as +0; -FLT_MAX, -inf
// and NaN, which the reference's scan never picks, to 0).  A radix search
// over key - kmin (the selectable keys' range), 8 bits a pass from the
// range's top bit and counted into per-wave histograms, finds the exact key
// T of the last block taken (scores of similar size share their leading
// bits: counted from bit 31 they would pile into a few bins and serialise
// the atomics); keys above T are taken and the rest of the budget comes from keys
// equal to T in block order.  One wave sums the bins and finds the cut with a
// suffix scan over its lanes; a pass whose cut bin holds exactly the blocks
// still needed ends the search.  Each thread owns a contiguous run of blocks,
// its keys loaded at once into registers, so block order is thread order and
// the position list is one prefix sum.
//
// Masked attention (k_attn_masked<G>): a workgroup per (query row, kv head,
// split of the position list) with its G query heads.  Positions go 32 at a
// time, 8 a wave: eight lanes per position score its fp16 key row against
// the G heads, each wave's maxima and weights (2^(s - max), scores in log2
// units) update its own online softmax, and the wave accumulates its
// positions' value rows with lanes over dims (each value row one coalesced
// 512-byte read); the four waves' states meet at the end.  When rows x kv heads alone would leave
// the chip idle (decode), the list is split over enough workgroups to fill
// it and k_attn_merge combines the splits' softmax states in a fixed order.
#include "qw_device.h"
#include "qw_kernels.h"

#include <float.h>

#define QS_BLK 64
#define QS_THREADS 256
#define QS_ROWS 8          // query rows a scoring workgroup walks
#define QS_ROTARY 64

// ---- block keys ---------------------------------------------------------------

template <int M>   // dims per lane: d <= 64 * M
__device__ __forceinline__ void qs_block_key(float (&kn)[M], const float *__restrict__ ikeys,
                                             const uint16_t *__restrict__ kw, const float *__restrict__ inv_freq,
                                             int b, int d, int ratio, float eps, int lane)
{
    float ss = 0.0f;
#pragma unroll
    for (int m = 0; m < M; m++) {
        const int dim = lane + 64 * m;
        kn[m] = 0.0f;
        if (dim < d) {
            const float *p = ikeys + (size_t)b * ratio * d + dim;
            float acc = p[0];
            for (int t = 1; t < ratio; t++) acc += p[(size_t)t * d];
            kn[m] = acc / (float)ratio;
            ss = __builtin_fmaf(kn[m], kn[m], ss);
        }
    }
    ss = qw_xor_sum<64>(ss);
    const float inv = 1.0f / sqrtf(ss / (float)d + eps);
#pragma unroll
    for (int m = 0; m < M; m++) {
        const int dim = lane + 64 * m;
        if (dim < d) kn[m] = kn[m] * inv * qw_bf16(kw[dim]);
    }
    const float partner = __shfl_xor(kn[0], 32, 64);
    const float ang = (float)(b * ratio) * inv_freq[lane & 31];
    const float c = cosf(ang), s = sinf(ang);
    // written as explicit fmas so every kernel inlining this rounds alike
    kn[0] = lane < 32 ? __builtin_fmaf(kn[0], c, -(partner * s)) : __builtin_fmaf(kn[0], c, partner * s);
}

// ---- scores ---------------------------------------------------------------------

// phase 2 over one WG's QS_BLK keys (LDS, row stride D + 4) for rows r0.. of
// the tile; `kl` holds the keys, `ql` one row's heads, `part` the partials.
template <int D>
__device__ __forceinline__ void qs_score_rows(float *__restrict__ scores, const float *__restrict__ qn,
                                              const float *kl, float *ql, float *part, int b0, int r0, int rows,
                                              int nq, int d, int ratio, int base_pos, int max_blocks)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float kr[D];
#pragma unroll
    for (int i = 0; i < D; i += 4) {
        const float4 v = *reinterpret_cast<const float4 *>(kl + lane * (D + 4) + i);
        kr[i] = v.x; kr[i + 1] = v.y; kr[i + 2] = v.z; kr[i + 3] = v.w;
    }
    // keeps the key in registers: without this the compiler re-reads it from
    // LDS inside every head's dot
#pragma unroll
    for (int i = 0; i < D; i++) asm volatile("" : "+v"(kr[i]));
    const float rs = sqrtf((float)d);
    for (int r = r0; r < min(r0 + QS_ROWS, rows); r++) {
        const int nb = (base_pos + r + 1) / ratio;
        if (nb <= b0) continue;                      // uniform: nothing of this row here
        __syncthreads();                             // ql free
        const float *qr = qn + (size_t)r * nq * d;
        for (int i = tid; i < nq * D; i += QS_THREADS) {
            const int h = i / D, j = i % D;
            ql[i] = j < d ? qr[(size_t)h * d + j] : 0.0f;
        }
        __syncthreads();
        float p = 0.0f;
        for (int h = wave; h < nq; h += QS_THREADS / 64) {
            const float4 *q4 = reinterpret_cast<const float4 *>(ql + h * D);
            float dot = 0.0f;
#pragma unroll
            for (int i = 0; i < D / 4; i++) {
                const float4 qv = q4[i];
                dot = __builtin_fmaf(qv.x, kr[4 * i], dot);
                dot = __builtin_fmaf(qv.y, kr[4 * i + 1], dot);
                dot = __builtin_fmaf(qv.z, kr[4 * i + 2], dot);
                dot = __builtin_fmaf(qv.w, kr[4 * i + 3], dot);
            }
            if (dot > 0.0f) p += dot;
        }
        part[wave * QS_BLK + lane] = p;
        __syncthreads();
        const int b = b0 + lane;
        if (wave == 0 && b < nb) {
            const float s = (part[lane] + part[QS_BLK + lane]) + (part[2 * QS_BLK + lane] + part[3 * QS_BLK + lane]);
            scores[(size_t)r * max_blocks + b] = s / rs;
        }
    }
}

// Phase 1: the workgroup's QS_BLK block keys into LDS, row stride D + 4, dims
// past d and blocks from nb_hi on zero.
template <int D, bool POOLED>
__device__ __forceinline__ void qs_keys_to_lds(float *kl, const float *__restrict__ src, const uint16_t *__restrict__ kw,
                                               const float *__restrict__ inv_freq, int b0, int nb_hi, int d,
                                               int ratio, float eps)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (POOLED) {
        for (int i = tid; i < QS_BLK * (D / 4); i += QS_THREADS) {
            const int bl = i / (D / 4), j = 4 * (i % (D / 4));
            float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            const int b = b0 + bl;
            if (b < nb_hi && j < d)   // d % 32 == 0: a float4 is wholly in or out
                v = *reinterpret_cast<const float4 *>(src + (size_t)b * d + j);
            *reinterpret_cast<float4 *>(kl + bl * (D + 4) + j) = v;
        }
    } else {
        for (int bl = wave; bl < QS_BLK; bl += QS_THREADS / 64) {
            const int b = b0 + bl;
            float kn[D / 64];
            if (b < nb_hi) qs_block_key<D / 64>(kn, src, kw, inv_freq, b, d, ratio, eps, lane);
            else {
#pragma unroll
                for (int m = 0; m < D / 64; m++) kn[m] = 0.0f;
            }
#pragma unroll
            for (int m = 0; m < D / 64; m++) kl[bl * (D + 4) + lane + 64 * m] = kn[m];
        }
    }
}

template <int D, bool POOLED>
__global__ void __launch_bounds__(QS_THREADS) __attribute__((amdgpu_waves_per_eu(1, 2))) k_qsa_scores(float *__restrict__ scores, const float *__restrict__ qn,
                                                           const float *__restrict__ src,
                                                           const uint16_t *__restrict__ kw,
                                                           const float *__restrict__ inv_freq, int rows, int nq,
                                                           int d, int ratio, int base_pos, int max_blocks, float eps)
{
    extern __shared__ float4 qs_lds[];
    float *kl = reinterpret_cast<float *>(qs_lds);            // [QS_BLK][D + 4]
    float *part = kl + QS_BLK * (D + 4);                       // [4][QS_BLK]
    float *ql = part + 4 * QS_BLK;                             // [nq][D]
    const int b0 = blockIdx.x * QS_BLK, r0 = blockIdx.y * QS_ROWS;
    const int nb_hi = (base_pos + min(r0 + QS_ROWS, rows)) / ratio;   // blocks any row of the tile sees
    if (nb_hi <= b0) return;                                   // uniform
    qs_keys_to_lds<D, POOLED>(kl, src, kw, inv_freq, b0, nb_hi, d, ratio, eps);
    __syncthreads();
    qs_score_rows<D>(scores, qn, kl, ql, part, b0, r0, rows, nq, d, ratio, base_pos, max_blocks);
}

// The scores on the fp32 matrix cores (nq <= 16, D <= 128).  The query heads
// are the rows of an MFMA tile (heads past nq zero: a zero dot, never summed)
// and 16 blocks its columns, so one query row fills the instruction
// (v_mfma_f32_16x16x4_f32) and a decode step takes the same kernel, and the
// same bits, as a chunk's rows.  Lane (ln, kg) holds dims 16 j + 4 kg .. + 3
// of head ln (A) and of block ln (B), element e feeding step e of the four, so
// both sides list the same dims.  A lane's accumulators are block ln's dots
// with heads 4 kg .. 4 kg + 3: their positive ones are summed in order, then
// over kg by two xor shuffles.
// A workgroup has NW waves of 16 TB blocks, whose keys stay in registers
// while it walks its rows; the rows' heads pass through LDS eight rows at a
// time (one row alone is read straight from memory).
// 512 rows at 16K: 127 us with K = 1 MFMAs in the serial chain's order, 102
// here; one row of 8192 blocks: 10.0 us with a thread a block,
// 4.1 here.  What bounds it: many rows, the fp32 MFMA's issue (35 cycles each,
// 60 of the 102) and the staging between groups of rows; one row, the trip to
// memory.
#define QM_ROWS 32                                 // the most rows a workgroup walks
#define QM_GROUP 8                                 // rows staged at once
template <int D, bool POOLED, int TB, int NW, bool ONE>
__global__ void __launch_bounds__(64 * NW, ONE ? 1 : 2) k_qsa_scores_mx(
    float *__restrict__ scores, const float *__restrict__ qn, const float *__restrict__ src,
    const uint16_t *__restrict__ kw, const float *__restrict__ inv_freq, int rows, int nq, int d, int ratio,
    int base_pos, int max_blocks, float eps, int wg_rows)
{
    typedef float f4v __attribute__((ext_vector_type(4)));
    static_assert(POOLED || (16 * TB * NW == QS_BLK && 64 * NW == QS_THREADS), "direct keys: qs_keys_to_lds's workgroup");
    constexpr int QST = 16 * (D + 4), NJ = D / 16;             // floats a staged row; float4s a lane a head
    constexpr int LQ = ONE ? 0 : QM_GROUP * QST, LK = POOLED ? 0 : QS_BLK * (D + 4), LN = LQ > LK ? LQ : LK;
    __shared__ float4 lds4[LN / 4 + 1];
    float *lds = reinterpret_cast<float *>(lds4);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ln = lane & 15, kg = lane >> 4;
    const int b0 = blockIdx.x * (16 * TB * NW), r0 = blockIdx.y * wg_rows;
    const int rend = min(r0 + wg_rows, rows), wb = b0 + wave * 16 * TB;
    const int nb_hi = (base_pos + rend) / ratio;
    if (nb_hi <= b0) return;                                   // uniform
    const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 key[TB][NJ];
    if (POOLED) {
        // every load issued, at a clamped place; dims past d zeroed after (d % 32 == 0: whole float4s)
#pragma unroll
        for (int t = 0; t < TB; t++)
#pragma unroll
            for (int j = 0; j < NJ; j++)
                key[t][j] = *reinterpret_cast<const float4 *>(src + (size_t)min(wb + 16 * t + ln, nb_hi - 1) * d +
                                                              min(16 * j + 4 * kg, d - 4));
    } else {
        qs_keys_to_lds<D, false>(lds, src, kw, inv_freq, b0, nb_hi, d, ratio, eps);
        __syncthreads();
#pragma unroll
        for (int t = 0; t < TB; t++)
#pragma unroll
            for (int j = 0; j < NJ; j++)
                key[t][j] = *reinterpret_cast<const float4 *>(lds + (wave * 16 * TB + 16 * t + ln) * (D + 4) + 16 * j + 4 * kg);
    }
    float4 one[ONE ? NJ : 1];
    if (ONE) {
#pragma unroll
        for (int j = 0; j < NJ; j++)
            one[j] = *reinterpret_cast<const float4 *>(qn + ((size_t)r0 * nq + min(ln, nq - 1)) * d + min(16 * j + 4 * kg, d - 4));
#pragma unroll
        for (int j = 0; j < NJ; j++)
            if (ln >= nq || 16 * j + 4 * kg >= d) one[j] = z4;
    }
    if (POOLED) {
#pragma unroll
        for (int t = 0; t < TB; t++)
#pragma unroll
            for (int j = 0; j < NJ; j++)
                if (16 * j + 4 * kg >= d) key[t][j] = z4;
    }
    const float rs = sqrtf((float)d);
    auto score = [&](const float4 (&a)[NJ], int r) __attribute__((always_inline)) {
        f4v acc[TB];
#pragma unroll
        for (int t = 0; t < TB; t++) acc[t] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const float av[4] = {a[j].x, a[j].y, a[j].z, a[j].w};
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int t = 0; t < TB; t++) {
                    const float kv[4] = {key[t][j].x, key[t][j].y, key[t][j].z, key[t][j].w};
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[e], kv[e], acc[t], 0, 0, 0);
                }
        }
        float mine = 0.0f;
#pragma unroll
        for (int t = 0; t < TB; t++) {
            float p = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (acc[t][e] > 0.0f) p += acc[t][e];
            p = p + __shfl_xor(p, 16, 64);
            p = p + __shfl_xor(p, 32, 64);
            if (t == kg) mine = p;
        }
        const int b = wb + 16 * kg + ln;
        if (kg < TB && b < (base_pos + r + 1) / ratio) scores[(size_t)r * max_blocks + b] = mine / rs;
    };
    if (ONE) {
        if constexpr (ONE) score(one, r0);
        return;
    }
    for (int g0 = r0; g0 < rend; g0 += QM_GROUP) {
        const int gl = min(g0 + QM_GROUP, rend);
        if ((base_pos + gl) / ratio <= b0) continue;           // uniform: no row of the group sees these blocks
        __syncthreads();                                       // the keys are in registers / the last group is done
        for (int i = tid; i < QM_GROUP * 16 * (D / 4); i += 64 * NW) {
            const int t = i / (16 * (D / 4)), h = (i / (D / 4)) % 16, j = 4 * (i % (D / 4)), r = g0 + t;
            float4 v = z4;
            if (r < gl && h < nq && j < d) v = *reinterpret_cast<const float4 *>(qn + ((size_t)r * nq + h) * d + j);
            *reinterpret_cast<float4 *>(lds + t * QST + h * (D + 4) + j) = v;
        }
        __syncthreads();
        for (int r = g0; r < gl; r++) {
            float4 a[NJ];
#pragma unroll
            for (int j = 0; j < NJ; j++)
                a[j] = *reinterpret_cast<const float4 *>(lds + (r - g0) * QST + ln * (D + 4) + 16 * j + 4 * kg);
            score(a, r);
        }
    }
}

template <int M>
__global__ void __launch_bounds__(QS_THREADS) k_qsa_pool(float *__restrict__ pool, const float *__restrict__ ikeys,
                                                         const uint16_t *__restrict__ kw,
                                                         const float *__restrict__ inv_freq, int d, int ratio,
                                                         int b0, int n, float eps)
{
    const int lane = threadIdx.x & 63;
    const int i = blockIdx.x * (QS_THREADS / 64) + (threadIdx.x >> 6);
    if (i >= n) return;
    const int b = b0 + i;
    float kn[M];
    qs_block_key<M>(kn, ikeys, kw, inv_freq, b, d, ratio, eps, lane);
#pragma unroll
    for (int m = 0; m < M; m++)
        if (lane + 64 * m < d) pool[(size_t)b * d + lane + 64 * m] = kn[m];
}

// ---- selection ------------------------------------------------------------------

#define QS_SEL_THREADS 1024
#define QS_SEL_WAVES (QS_SEL_THREADS / 64)
#define QS_SEL_MAX_BLOCKS 65536

__device__ __forceinline__ uint32_t qs_key(float v)
{
    if (!(v > -FLT_MAX)) return 0u;                 // never picked (also NaN)
    const uint32_t u = __float_as_uint(v + 0.0f);   // -0 -> +0
    return (u >> 31) ? ~u : (u | 0x80000000u);
}

// Exclusive prefix sum of one value per thread over the workgroup, thread
// order; *total gets the sum.  Every thread calls it.
__device__ __forceinline__ uint32_t qs_scan(uint32_t v, uint32_t *wt, uint32_t *total)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) wt[wave] = x;
    __syncthreads();
    if (wave == 0) {
        uint32_t t = lane < QS_SEL_WAVES ? wt[lane] : 0u, s = t;
#pragma unroll
        for (int o = 1; o < QS_SEL_WAVES; o <<= 1) {
            const uint32_t y = __shfl_up(s, o, 64);
            if (lane >= o) s += y;
        }
        if (lane < QS_SEL_WAVES) wt[lane] = s - t;
        if (lane == QS_SEL_WAVES - 1) *total = s;
    }
    __syncthreads();
    const uint32_t r = x - v + wt[wave];
    __syncthreads();
    return r;
}


#define QS_SEL_KREG 8      // keys a thread keeps in registers (up to 8192 blocks)

// A thread's contiguous run of blocks [lo, hi): its keys, from registers
// when the run fits, else from the scores.
#define QS_RUN(body)                                                              \
    if (in_regs) {                                                                \
        _Pragma("unroll") for (int i = 0; i < QS_SEL_KREG; i++)                   \
            if (lo + i < hi) { const int b = lo + i; const uint32_t k = kr[i]; body } \
    } else {                                                                      \
        for (int b = lo; b < hi; b++) { const uint32_t k = qs_key(sc[b]); body }  \
    }

// The count, minimum and maximum of the selectable keys over the workgroup
// (one barrier); every thread gets all three.
__device__ __forceinline__ void qs_reduce3(uint32_t &cnt, uint32_t &mn, uint32_t &mx, uint4 *wt3)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        cnt += (uint32_t)__shfl_xor((int)cnt, o, 64);
        mn = min(mn, (uint32_t)__shfl_xor((int)mn, o, 64));
        mx = max(mx, (uint32_t)__shfl_xor((int)mx, o, 64));
    }
    if (lane == 0) wt3[wave] = make_uint4(cnt, mn, mx, 0u);
    __syncthreads();
    cnt = 0; mn = 0xFFFFFFFFu; mx = 0u;
#pragma unroll
    for (int w = 0; w < QS_SEL_WAVES; w++) {
        const uint4 v = wt3[w];
        cnt += v.x; mn = min(mn, v.y); mx = max(mx, v.z);
    }
}

__global__ void __launch_bounds__(QS_SEL_THREADS) k_qsa_select(uint8_t *__restrict__ mask, uint32_t *__restrict__ list,
                                                               const float *__restrict__ scores, int ratio,
                                                               int base_pos, int block_topk, int max_ctx,
                                                               int max_blocks, int cap)
{
    extern __shared__ uint8_t sel[];
    // a histogram per wave (no cross-wave atomics), two sets: a pass counts
    // into one while it clears the other for the next pass
    __shared__ uint32_t hist[2][QS_SEL_WAVES][256];
    __shared__ uint32_t wt[QS_SEL_WAVES];
    __shared__ uint4 wt3[QS_SEL_WAVES];
    __shared__ uint32_t sh_total, sh_bin, sh_need, sh_exact;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = blockIdx.x;
    const int n_keys = base_pos + r + 1, nb = n_keys / ratio;
    const float *sc = scores + (size_t)r * max_blocks;
    const int per = (nb + QS_SEL_THREADS - 1) / QS_SEL_THREADS;
    const int lo = min(tid * per, nb), hi = min(lo + per, nb);
    const bool in_regs = per <= QS_SEL_KREG;
    // every load of the run issued before the first use (in-range addresses
    // for the lanes past the run, whose keys are then dropped)
    uint32_t kr[QS_SEL_KREG];
    if (in_regs && nb > 0) {
        float v[QS_SEL_KREG];
        if (per == QS_SEL_KREG && (reinterpret_cast<uintptr_t>(sc) & 15) == 0 && lo + QS_SEL_KREG <= max_blocks) {
            // two 16-byte loads (the run starts at a multiple of 8 blocks)
            const float4 a = reinterpret_cast<const float4 *>(sc + lo)[0];
            const float4 b = reinterpret_cast<const float4 *>(sc + lo)[1];
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
            v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        } else {
#pragma unroll
            for (int i = 0; i < QS_SEL_KREG; i++) v[i] = sc[min(lo + i, nb - 1)];
        }
#pragma unroll
        for (int i = 0; i < QS_SEL_KREG; i++) kr[i] = lo + i < hi ? qs_key(v[i]) : 0u;
    } else {
#pragma unroll
        for (int i = 0; i < QS_SEL_KREG; i++) kr[i] = 0u;
    }
    uint4 *h0 = reinterpret_cast<uint4 *>(&hist[0][0][0]);
    h0[tid] = make_uint4(0u, 0u, 0u, 0u);   // 16 x 256 words: one uint4 a thread

    uint32_t S = 0, mn = 0xFFFFFFFFu, mx = 0u;
    QS_RUN(if (k) { S++; mn = min(mn, k); mx = max(mx, k); })
    qs_reduce3(S, mn, mx, wt3);
    const uint32_t take = min((uint32_t)max(block_topk, 0), S);
    // blocks taken: key > T, then the first `need` blocks whose key equals T
    uint32_t T = 0u, need = 0u;
    if (take == 0) {
        T = 0xFFFFFFFFu;
    } else if (take < S) {
        // the key of the take-th largest.  The passes count u = key - kmin
        // (kmin, kmax: the selectable keys' range), 8 bits at a time from
        // the range's top bit, so even scores that share their leading bits
        // spread over the bins.  A pass whose bin holds exactly the blocks
        // still needed ends the search: the bin's lowest key bounds the take.
        const uint32_t range = mx - mn;
        const int nbits = range ? 32 - __builtin_clz(range) : 0;
        uint32_t prefix = 0;
        bool exact = false;
        int prev = 32, shift = nbits > 8 ? nbits - 8 : 0, cur = 0;
        need = take;
        while (true) {
            const uint32_t bmask = prev - shift >= 32 ? 0xFFFFFFFFu : ((1u << (prev - shift)) - 1u);
            const uint32_t hp = prev >= 32 ? 0u : prefix >> prev;
            reinterpret_cast<uint4 *>(&hist[cur ^ 1][0][0])[tid] = make_uint4(0u, 0u, 0u, 0u);
            QS_RUN(if (k) {
                const uint32_t u = k - mn;
                if ((prev >= 32 ? 0u : u >> prev) == hp) atomicAdd(&hist[cur][wave][(u >> shift) & bmask], 1u);
            })
            __syncthreads();
            if (wave == 0) {
                // lane l: bins 4l .. 4l+3 summed over the waves; counts above
                // a lane's bins are a suffix sum over the lanes
                uint4 c = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
                for (int w = 0; w < QS_SEL_WAVES; w++) {
                    const uint4 v = reinterpret_cast<const uint4 *>(&hist[cur][w][0])[lane];
                    c.x += v.x; c.y += v.y; c.z += v.z; c.w += v.w;
                }
                const uint32_t tl = c.x + c.y + c.z + c.w;
                uint32_t sfx = tl;
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const uint32_t y = (uint32_t)__shfl_down((int)sfx, o, 64);
                    if (lane + o < 64) sfx += y;
                }
                uint32_t a = sfx - tl;
                const uint32_t cj[4] = {c.w, c.z, c.y, c.x};
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if (a < need && a + cj[j] >= need) {
                        sh_bin = (uint32_t)(4 * lane + 3 - j);
                        sh_need = need - a;
                        sh_exact = a + cj[j] == need;
                    }
                    a += cj[j];
                }
            }
            __syncthreads();
            prefix |= sh_bin << shift;
            need = sh_need;
            exact = sh_exact != 0u;
            if (exact || shift == 0) break;
            prev = shift;
            shift = shift > 8 ? shift - 8 : 0;
            cur ^= 1;
        }
        T = prefix + mn;   // back from the range's offset to the key
        if (exact) { T -= 1u; need = 0u; }   // T >= kmin >= 1
    }
    uint32_t selm = 0, eq = 0;
    if (in_regs) {
#pragma unroll
        for (int i = 0; i < QS_SEL_KREG; i++) {
            if (lo + i < hi) {
                if (kr[i] > T) selm |= 1u << i;
                else eq += kr[i] == T;
            }
        }
    } else {
        for (int b = lo; b < hi; b++) {
            const uint32_t k = qs_key(sc[b]);
            sel[b] = k > T;
            eq += k == T;
        }
    }
    if (need > 0u) {   // uniform
        uint32_t rank = qs_scan(eq, wt, &sh_total);
        QS_RUN(if (k == T && rank < need) {
            if (in_regs) selm |= 1u << (b - lo); else sel[b] = 1;
            rank++;
        })
    }
    uint32_t mine = 0;
    if (in_regs) {
#pragma unroll
        for (int i = 0; i < QS_SEL_KREG; i++)
            if (lo + i < hi) sel[lo + i] = (uint8_t)((selm >> i) & 1u);
        mine = __builtin_popcount(selm);
    } else {
        for (int b = lo; b < hi; b++) mine += sel[b];
    }
    const uint32_t first = qs_scan(mine, wt, &sh_total);   // its barriers publish sel
    const uint32_t n_sel = sh_total;
    uint32_t *lr = list + (size_t)r * (1 + cap);
    uint32_t at = 1 + first * ratio;
    if (in_regs) {
#pragma unroll
        for (int i = 0; i < QS_SEL_KREG; i++)
            if ((selm >> i) & 1u)
                for (int t = 0; t < ratio; t++) lr[at++] = (uint32_t)((lo + i) * ratio + t);
    } else {
        for (int b = lo; b < hi; b++)
            if (sel[b])
                for (int t = 0; t < ratio; t++) lr[at++] = (uint32_t)(b * ratio + t);
    }
    if (tid == 0) {
        uint32_t n = n_sel * ratio;
        for (int t = nb * ratio; t < n_keys; t++) lr[1 + n++] = (uint32_t)t;
        lr[0] = n;
    }
    uint8_t *mr = mask + (size_t)r * max_ctx;
    int t0 = 0;
    if (ratio == 4 && (reinterpret_cast<uintptr_t>(mr) & 15) == 0) {
        // four blocks (16 positions) a 16-byte store
        const int n4 = nb >> 2;
        for (int w = tid; w < n4; w += QS_SEL_THREADS) {
            const uint32_t x = reinterpret_cast<const uint32_t *>(sel)[w];
            reinterpret_cast<uint4 *>(mr)[w] = make_uint4((x & 1u) * 0x01010101u, ((x >> 8) & 1u) * 0x01010101u,
                                                          ((x >> 16) & 1u) * 0x01010101u, (x >> 24) * 0x01010101u);
        }
        t0 = n4 * 16;
    }
    for (int t = t0 + tid; t < n_keys; t += QS_SEL_THREADS) mr[t] = t >= nb * ratio ? 1 : sel[t / ratio];
}
#undef QS_RUN

// ---- masked attention -------------------------------------------------------------

#define QA_D 256
#define QA_P 32            // positions a workgroup takes per pass
#define QA_QPOS(i) ((i) + (i) / 8)   // float4 i of a head in its padded LDS row
#define QA_QROW (QA_D / 4 + QA_D / 32)

#define QA_LOG2E 1.44269504088896340736f

// 2^x by the hardware's exp2 (v_exp_f32); results below the normal range
// flush to zero, which a softmax weight relative to the maximum can afford
__device__ __forceinline__ float qa_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ float qa_f16(uint32_t bits)
{
    return (float)__builtin_bit_cast(_Float16, (unsigned short)bits);
}

// A workgroup per (query row, kv head, split): the split's share of the
// row's listed positions, QA_P at a time.  With one split it writes the
// output; otherwise its softmax state (max, sum, unnormalised output per
// head) goes to `part` and k_attn_merge combines the splits.
template <int G>
struct qa_masked_lds {
    // the G heads, pre-scaled; each 32-dim piece padded by 16 bytes so the
    // eight pieces a score reads at once start in different banks
    float4 qs4[G][QA_QROW];
    float ps[G][QA_P];                // a pass's weights (wave w: [8w, 8w + 8))
    float wm[4][G], wl[4][G];         // the waves' softmax states
    float wbuf[G][QA_D];              // the waves' partial outputs meet here
};

template <int G>
__device__ __forceinline__ void qa_masked(qa_masked_lds<G> &sh, float *__restrict__ out, const float *__restrict__ gate,
                                          const float *__restrict__ q, const uint16_t *__restrict__ kc,
                                          const uint16_t *__restrict__ vc, const uint32_t *__restrict__ list,
                                          int q_heads, int kv_heads, int max_ctx, float scale, int cap,
                                          int nsplit, float *__restrict__ part)
{
    auto &qs4 = sh.qs4;
    auto &ps = sh.ps;
    auto &wm = sh.wm, &wl = sh.wl;
    auto &wbuf = sh.wbuf;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int split = blockIdx.x % nsplit, rk = blockIdx.x / nsplit;
    const int row = rk / kv_heads, kvh = rk % kv_heads;
    const uint32_t *lr = list + (size_t)row * (1 + cap);
    // the splits divide the list's capacity, so a split knows its range
    // before the list's length arrives: its first pass's entries are
    // requested with the length (entries past the length are not positions
    // and are clamped to a valid row, then dropped)
    const int per = ((cap + QA_P - 1) / QA_P + nsplit - 1) / nsplit;
    const int j_lo = min(split * per * QA_P, cap), j_cap = min(j_lo + per * QA_P, cap);
    const int jb = (QA_P / 4) * wave, jj = tid >> 3, kp = tid & 7;
    uint32_t vi[QA_P / 4], ki = 0;
    auto load_list = [&](int j0) {
#pragma unroll
        for (int i = 0; i < QA_P / 4; i++) vi[i] = lr[1 + min(j0 + jb + i, cap - 1)];
        ki = lr[1 + min(j0 + jj, cap - 1)];
    };
    const int n_sel = (int)lr[0];
    if (j_lo < j_cap) load_list(j_lo);
    const int j_hi = min(j_cap, n_sel);
    const float4 *qp = reinterpret_cast<const float4 *>(q + ((size_t)row * q_heads + (size_t)kvh * G) * QA_D);
    const float sl2 = scale * QA_LOG2E;   // scores in log2 units: weights are 2^(s - max)
    {
        constexpr int NQ = (G * QA_D / 4 + 255) / 256;
        float4 qv[NQ];
#pragma unroll
        for (int u = 0; u < NQ; u++)
            if (tid + 256 * u < G * QA_D / 4) qv[u] = qp[tid + 256 * u];
#pragma unroll
        for (int u = 0; u < NQ; u++) {
            const int f = tid + 256 * u;
            if (f < G * QA_D / 4)
                qs4[f / (QA_D / 4)][QA_QPOS(f % (QA_D / 4))] =
                    make_float4(qv[u].x * sl2, qv[u].y * sl2, qv[u].z * sl2, qv[u].w * sl2);
        }
    }
    const uint16_t *kbase = kc + (size_t)kvh * max_ctx * QA_D;
    const uint16_t *vbase = vc + (size_t)kvh * max_ctx * QA_D;

    float m[G], l[G], acc[G][4];
#pragma unroll
    for (int g = 0; g < G; g++) {
        m[g] = -FLT_MAX; l[g] = 0.0f;
        acc[g][0] = acc[g][1] = acc[g][2] = acc[g][3] = 0.0f;
    }
    __syncthreads();
    for (int j0 = j_lo; j0 < j_hi; j0 += QA_P) {
        const int n = min(QA_P, j_hi - j0), nj = max(0, min(QA_P / 4, n - jb));
        if (j0 != j_lo) load_list(j0);
        // every key and value row of the pass at once, the keys first
#pragma unroll
        for (int i = 0; i < QA_P / 4; i++) vi[i] = min(vi[i], (uint32_t)(max_ctx - 1));
        ki = min(ki, (uint32_t)(max_ctx - 1));
        uint4 kv[4];
        {
            const uint4 *kr = reinterpret_cast<const uint4 *>(kbase + (size_t)ki * QA_D + 32 * kp);
#pragma unroll
            for (int c = 0; c < 4; c++) kv[c] = kr[c];
        }
        uint2 vv[QA_P / 4];
#pragma unroll
        for (int i = 0; i < QA_P / 4; i++)
            vv[i] = *reinterpret_cast<const uint2 *>(vbase + (size_t)vi[i] * QA_D + 4 * lane);
        // the key rows, issued before the value rows, are waited for here
        // (the value rows stay in flight through the scores)
#pragma unroll
        for (int c = 0; c < 4; c++) asm volatile("" : "+v"(kv[c].x), "+v"(kv[c].y), "+v"(kv[c].z), "+v"(kv[c].w));
        // scores: eight threads per position, 32 dims each (one 64-byte
        // piece of the fp16 key row); the eight partial dots meet in the xor
        // tree of their 8-lane run.  Wave w scores positions 8w .. 8w+7 of
        // the pass, the ones its values take below, so the pass needs no
        // barrier: each wave runs its own softmax state
        const bool valid = jj < n;
        float sg[G];
#pragma unroll
        for (int g = 0; g < G; g++) sg[g] = 0.0f;
        if (valid) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const uint32_t w[4] = { kv[c].x, kv[c].y, kv[c].z, kv[c].w };
                const int d0 = 32 * kp + 8 * c;
                float kf[8];
#pragma unroll
                for (int e = 0; e < 4; e++) { kf[2 * e] = qa_f16(w[e] & 0xFFFFu); kf[2 * e + 1] = qa_f16(w[e] >> 16); }
#pragma unroll
                for (int g = 0; g < G; g++) {
                    const float4 a = qs4[g][QA_QPOS(d0 / 4)], b = qs4[g][QA_QPOS(d0 / 4) + 1];
                    sg[g] = __builtin_fmaf(a.x, kf[0], sg[g]);
                    sg[g] = __builtin_fmaf(a.y, kf[1], sg[g]);
                    sg[g] = __builtin_fmaf(a.z, kf[2], sg[g]);
                    sg[g] = __builtin_fmaf(a.w, kf[3], sg[g]);
                    sg[g] = __builtin_fmaf(b.x, kf[4], sg[g]);
                    sg[g] = __builtin_fmaf(b.y, kf[5], sg[g]);
                    sg[g] = __builtin_fmaf(b.z, kf[6], sg[g]);
                    sg[g] = __builtin_fmaf(b.w, kf[7], sg[g]);
                }
            }
        }
        // per head: the wave's maximum over its positions (lane bits 3-5),
        // the online rescale, the weights (into this wave's slice of ps) and
        // their sum in a fixed tree.  The 8 lanes of a position hold one
        // value, so the xor steps 8, 16, 32 are a row mirror (it pairs
        // position 2r with 2r + 1, as xor 8 does) and the row sums read from
        // lanes 0, 16, 32, 48, added (0 + 16) + (32 + 48) as xor 16 then 32
        // add them: the same bits, in the VALU (a shuffle goes through LDS)
#pragma unroll
        for (int g = 0; g < G; g++) {
            const float sc = qw_xor_sum<8>(sg[g]);
            float cm = valid ? sc : -FLT_MAX;
            cm = fmaxf(cm, qw_dpp<QW_DPP_MIRROR>(cm));
            cm = fmaxf(fmaxf(qw_lane(cm, 0), qw_lane(cm, 16)), fmaxf(qw_lane(cm, 32), qw_lane(cm, 48)));
            const float mn = fmaxf(m[g], cm);
            const float rs = qa_exp2(m[g] - mn);
            m[g] = mn;
            float e = valid ? qa_exp2(sc - mn) : 0.0f;
            if (kp == 0) ps[g][jj] = e;
            e = e + qw_dpp<QW_DPP_MIRROR>(e);
            e = (qw_lane(e, 0) + qw_lane(e, 16)) + (qw_lane(e, 32) + qw_lane(e, 48));
            l[g] = l[g] * rs + e;
#pragma unroll
            for (int i = 0; i < 4; i++) acc[g][i] *= rs;
        }
        // values: lane dims 4l..4l+3 of the wave's positions (their rows
        // were requested with the keys); the weights come back from the
        // wave's own slice of ps (its writes above, in program order)
#pragma unroll
        for (int i = 0; i < QA_P / 4; i++) {
            if (i < nj) {
                const float v0 = qa_f16(vv[i].x & 0xFFFFu), v1 = qa_f16(vv[i].x >> 16);
                const float v2 = qa_f16(vv[i].y & 0xFFFFu), v3 = qa_f16(vv[i].y >> 16);
#pragma unroll
                for (int g = 0; g < G; g++) {
                    const float p = ps[g][jb + i];
                    acc[g][0] = __builtin_fmaf(p, v0, acc[g][0]);
                    acc[g][1] = __builtin_fmaf(p, v1, acc[g][1]);
                    acc[g][2] = __builtin_fmaf(p, v2, acc[g][2]);
                    acc[g][3] = __builtin_fmaf(p, v3, acc[g][3]);
                }
            }
        }
    }
    // the four waves' states meet: the common maximum, each wave's factor,
    // the sums (w0 + w1) + (w2 + w3), and the outputs in the same tree
    // through wbuf and the query array (no longer read)
    if (lane == 0) {
#pragma unroll
        for (int g = 0; g < G; g++) { wm[wave][g] = m[g]; wl[wave][g] = l[g]; }
    }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < G; g++) {
        const float M = fmaxf(fmaxf(wm[0][g], wm[1][g]), fmaxf(wm[2][g], wm[3][g]));
        const float f = qa_exp2(m[g] - M);
#pragma unroll
        for (int i = 0; i < 4; i++) acc[g][i] *= f;
        if (wave == 0) {
            l[g] = (wl[0][g] * qa_exp2(wm[0][g] - M) + wl[1][g] * qa_exp2(wm[1][g] - M)) +
                   (wl[2][g] * qa_exp2(wm[2][g] - M) + wl[3][g] * qa_exp2(wm[3][g] - M));
            m[g] = M;
        }
    }
    float *bufA = &wbuf[0][0], *bufB = reinterpret_cast<float *>(&qs4[0][0]);
    __syncthreads();                                 // every wave's scores are done with qs4
    if (wave == 1 || wave == 3) {
        float *dst = wave == 1 ? bufA : bufB;
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
            for (int i = 0; i < 4; i++) dst[g * QA_D + 4 * lane + i] = acc[g][i];
    }
    __syncthreads();
    if (wave == 0 || wave == 2) {
        const float *src = wave == 0 ? bufA : bufB;
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[g][i] = acc[g][i] + src[g * QA_D + 4 * lane + i];
    }
    __syncthreads();
    if (wave == 2) {
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
            for (int i = 0; i < 4; i++) bufA[g * QA_D + 4 * lane + i] = acc[g][i];
    }
    __syncthreads();
    if (wave != 0) return;
    if (nsplit == 1) {
        // the gate rows requested together, before the first is used
        float4 gv[G];
        if (gate) {
#pragma unroll
            for (int g = 0; g < G; g++)
                gv[g] = *reinterpret_cast<const float4 *>(gate + ((size_t)row * q_heads + (size_t)kvh * G + g) * QA_D + 4 * lane);
        }
#pragma unroll
        for (int g = 0; g < G; g++) {
            const size_t ob = ((size_t)row * q_heads + (size_t)kvh * G + g) * QA_D + 4 * lane;
            const float gg[4] = {gv[g].x, gv[g].y, gv[g].z, gv[g].w};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float s = acc[g][i] + bufA[g * QA_D + 4 * lane + i];
                float o = l[g] > 0.0f ? s / l[g] : 0.0f;
                if (gate) o *= 1.0f / (1.0f + expf(-gg[i]));
                out[ob + i] = o;
            }
        }
    } else {
        float *pr = part + (size_t)blockIdx.x * G * (QA_D + 2);
#pragma unroll
        for (int g = 0; g < G; g++) {
            if (lane == 0) { pr[g] = m[g]; pr[G + g] = l[g]; }
#pragma unroll
            for (int i = 0; i < 4; i++) pr[2 * G + g * QA_D + 4 * lane + i] = acc[g][i] + bufA[g * QA_D + 4 * lane + i];
        }
    }
}

template <int G>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) k_attn_masked(float *__restrict__ out, const float *__restrict__ gate,
                                                     const float *__restrict__ q, const uint16_t *__restrict__ kc,
                                                     const uint16_t *__restrict__ vc, const uint32_t *__restrict__ list,
                                                     int q_heads, int kv_heads, int max_ctx, float scale, int cap,
                                                     int nsplit, float *__restrict__ part)
{
    __shared__ qa_masked_lds<G> sh;
    qa_masked<G>(sh, out, gate, q, kc, vc, list, q_heads, kv_heads, max_ctx, scale, cap, nsplit, part);
}

// ---- masked attention on the matrix cores -------------------------------------------
//
// The same split of the work (a workgroup a row, kv head and split) for many
// query heads a kv head, where k_attn_masked's multiply-adds bind it (G = 12:
// 26 GFLOP of fp32 vector work for 512 rows of 2052 positions, 850 us).  Both
// products run on f16 MFMAs with nothing rounded to 16 bits: the caches are
// f16 as they are, and each fp32 operand is cut into three f16 parts, a part a
// MFMA, the second and third times 2^12 and summed apart (f16's smallest step
// would cut the small ones off), all sums in fp32:
//   q   scaled a head by the power of two that puts its largest magnitude in
//       [2^14, 2^15); the parts stay in LDS for the row.  All 24 bits of
//       elements down to 2^-27 of the largest, 2^-51 of it below
//   p   the softmax weights 2^(s - m), at most 2^4 (below), times 2^11.  All
//       24 bits down to 2^-23 of the state's unit; what the parts leave of
//       smaller ones (a dominant position whose values are near zero makes
//       them count) is added by further turns where it could come to half a
//       unit of a sum's last place
// The scores are computed transposed, S'[position][head] = K q': a lane then
// holds its head's weights for positions 4 kg .. 4 kg + 3 of two tiles of 16,
// which is an A operand of the second product as it stands if the MFMA's k
// slots 8 kg .. are taken to be those positions.  V's operand must list the
// same positions of one dim a lane: a lane loads 8 dims (16 bytes) of each of
// its 8 positions and takes column t of that 8 x 8 block, by v_perm, as tile
// t's operand, so tile t holds dims 8 n + t.  No value passes through LDS.
// A wave takes 32 positions a pass and keeps its own softmax state; the
// reference maximum moves only when a score passes it by 4 (a weight is then
// at most 2^4 of the state's unit), so the sums are seldom rescaled.  The four
// waves' states meet in LDS at the end, as (w0 + w1) + (w2 + w3).
// Scores sum their first parts in four chains met in a tree, and their factor
// carries what rounding it to fp32 cuts off.  512 rows of 2052 positions at
// 16K, 24 / 2 heads, k_attn_masked -> this, for scores with a deviation of 1 /
// 4 / 24: 810 / 821 / 822 -> 180 / 201 / 216 us, error against 64 bits 4.4e-7 /
// 5.8e-7 / 9.4e-7 -> 2.2e-7 / 4.7e-7 / 9.1e-7 (two serial sums and a plain
// factor: 3.1e-7 / 7.1e-7 / 12.4e-7).  What bounds it: the gathered rows, 1 KB
// a position and kv head, 2.1 GB for that call: 11.6 TB/s through the L1s.
typedef _Float16 qa_h8 __attribute__((ext_vector_type(8)));
typedef float qa_f4 __attribute__((ext_vector_type(4)));
typedef unsigned short qa_us2 __attribute__((ext_vector_type(2)));
#define QAM_HEADS 16                      // a MFMA tile of heads (G of them real)
#define QAM_QST (QA_D + 8)                // halfs a head's row takes in LDS
#define QAM_OST (QA_D + 4)                // floats
#define QAM_STEP 32                       // positions a wave takes a pass
#define QAM_SLACK 4.0f                    // what a weight's exponent may be above its state's unit
#define QAM_P_UNIT 0x1p11f                // 2^(15 - QAM_SLACK)

// x (up to 2^15) as f16 parts, x = a + (b + c + r) 2^-12; r, at most 2^-25, is
// zero where x has no bit below 2^-36
__device__ __forceinline__ float qa_split(float x, _Float16 &a, _Float16 &b, _Float16 &c)
{
    a = (_Float16)x;
    float r = (x - (float)a) * 4096.0f;
    b = (_Float16)r;
    r = r - (float)b;
    c = (_Float16)r;
    return r - (float)c;
}

template <int G>
__global__ void __launch_bounds__(256, 2) k_attn_mx(float *__restrict__ out, const float *__restrict__ gate,
                                                    const float *__restrict__ q, const uint16_t *__restrict__ kc,
                                                    const uint16_t *__restrict__ vc, const uint32_t *__restrict__ list,
                                                    int q_heads, int kv_heads, int max_ctx, float scale, int cap,
                                                    int nsplit, float *__restrict__ part)
{
    constexpr int QB = 3 * QAM_HEADS * QAM_QST * 2, OB = 4 * QAM_HEADS * QAM_OST * 4, MB = sizeof(qa_masked_lds<G>);
    static_assert(MB <= OB && QB <= OB, "one place for all three");
    __shared__ __align__(16) uint8_t lds[OB];
    __shared__ float2 qf[QAM_HEADS];                  // a head's score factor and what it lacks
    __shared__ float wm[4][QAM_HEADS], wl[4][QAM_HEADS];
    _Float16 (*qp)[QAM_HEADS][QAM_QST] = reinterpret_cast<_Float16 (*)[QAM_HEADS][QAM_QST]>(lds);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), ln = lane & 15, kg = lane >> 4;
    const int split = blockIdx.x % nsplit, rk = blockIdx.x / nsplit;
    const int row = rk / kv_heads, kvh = rk % kv_heads;
    const uint32_t *lr = list + (size_t)row * (1 + cap);
    const int per = ((cap + QA_P - 1) / QA_P + nsplit - 1) / nsplit;
    const int j_lo = min(split * per * QA_P, cap), j_cap = min(j_lo + per * QA_P, cap);
    const int j_hi = min(j_cap, (int)min(lr[0], (uint32_t)cap));

    // the heads, a wave four: lane l dims 4 l ..
#pragma unroll
    for (int u = 0; u < QAM_HEADS / 4; u++) {
        const int g = 4 * u + wave;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (g < G) v = reinterpret_cast<const float4 *>(q + ((size_t)row * q_heads + (size_t)kvh * G + g) * QA_D)[lane];
        const float mx = qw_wave_max(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        // (any finite head: -113 .. 163.  A factor that leaves fp32's range
        // stands for scores that do.)
        const int sh = mx > 0.0f && mx <= FLT_MAX ? 15 - __builtin_amdgcn_frexp_expf(mx) : 0;
        const float f[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            _Float16 a, b, c;
            qa_split(__builtin_ldexpf(f[i], sh), a, b, c);
            qp[0][g][4 * lane + i] = a;
            qp[1][g][4 * lane + i] = b;
            qp[2][g][4 * lane + i] = c;
        }
        if (lane == 0) {
            // (a score of 100 units times log2 e's own rounding is 1e-6 of its weight)
            const double f64 = (double)scale * 1.4426950408889634;
            const float f32 = (float)f64;
            qf[g] = make_float2(__builtin_ldexpf(f32, -sh), __builtin_ldexpf((float)(f64 - (double)f32), -sh));
        }
    }
    __syncthreads();

    const uint16_t *kbase = kc + (size_t)kvh * max_ctx * QA_D + 8 * kg;      // K: dims 32 s + 8 kg of position ln
    const uint16_t *vbase = vc + (size_t)kvh * max_ctx * QA_D + 8 * ln;      // V: dims 8 ln (and 128 on) of 8 positions
    const float fac = qf[ln].x, fac2 = qf[ln].y;
    float m = -FLT_MAX, l = 0.0f;
    qa_f4 acc[16];
#pragma unroll
    for (int t = 0; t < 16; t++) acc[t] = qa_f4{0.f, 0.f, 0.f, 0.f};

    // list entries of a pass from j0 (past the range: its last again, with weight zero)
    auto at = [&](int j) { return min(lr[1 + min(j, j_hi - 1)], (uint32_t)(max_ctx - 1)); };
    uint32_t ki[2], vi[8];
    auto entries = [&](int j0) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 2; t++) ki[t] = at(j0 + 16 * t + ln);
#pragma unroll
        for (int i = 0; i < 8; i++) vi[i] = at(j0 + 16 * (i >> 2) + 4 * kg + (i & 3));
    };
    uint4 kv[2][8];
    auto load_k = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const uint4 *p = reinterpret_cast<const uint4 *>(kbase + (size_t)ki[t] * QA_D);
#pragma unroll
            for (int s = 0; s < 8; s++) kv[t][s] = p[4 * s];
        }
    };
    int j0 = j_lo + QAM_STEP * wave;
    if (j0 < j_hi) {
        entries(j0);
        load_k();
    }
    for (; j0 < j_hi; j0 += 4 * QAM_STEP) {
        // Half of the values' dims are requested ahead of the scores, half
        // after them (in the keys' registers), the next pass's keys ahead of
        // the second half's product.
        uint4 v0[8], v1[8];
        const uint16_t *vp[8];
#pragma unroll
        for (int i = 0; i < 8; i++) vp[i] = vbase + (size_t)vi[i] * QA_D;
        entries(j0 + 4 * QAM_STEP);                            // the next pass's, ahead of this one's values
#pragma unroll
        for (int i = 0; i < 8; i++) v0[i] = *reinterpret_cast<const uint4 *>(vp[i]);
        // scores: the first parts in four sums, the others in another
        qa_f4 hi[2][4], lo[2];
#pragma unroll
        for (int t = 0; t < 2; t++) hi[t][0] = hi[t][1] = hi[t][2] = hi[t][3] = lo[t] = qa_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 8; s++) {
            qa_h8 b[3];
#pragma unroll
            for (int p = 0; p < 3; p++) b[p] = *reinterpret_cast<const qa_h8 *>(&qp[p][ln][32 * s + 8 * kg]);
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const qa_h8 a = __builtin_bit_cast(qa_h8, kv[t][s]);
                hi[t][s >> 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[0], hi[t][s >> 1], 0, 0, 0);
                lo[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[2], lo[t], 0, 0, 0);
                lo[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[1], lo[t], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 8; i++) v1[i] = *reinterpret_cast<const uint4 *>(vp[i] + 128);
        float sc[8], cm = -FLT_MAX;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int j = j0 + 16 * (i >> 2) + 4 * kg + (i & 3);
            const qa_f4 *h = hi[i >> 2];
            sc[i] = __builtin_fmaf(lo[i >> 2][i & 3], 0x1p-12f,
                                   (h[0][i & 3] + h[1][i & 3]) + (h[2][i & 3] + h[3][i & 3]));
            cm = fmaxf(cm, j < j_hi ? sc[i] * fac : -FLT_MAX);
        }
        cm = fmaxf(cm, __shfl_xor(cm, 16, 64));
        cm = fmaxf(cm, __shfl_xor(cm, 32, 64));
        const bool up = cm > m + QAM_SLACK;                    // (at first m + 4 is -FLT_MAX itself)
        if (__ballot(up)) {
            const float mn = up ? cm : m, f = qa_exp2(m - mn);
            m = mn;
            l *= f;
            float fr[4];
#pragma unroll
            for (int e = 0; e < 4; e++) fr[e] = __shfl(f, 4 * kg + e, 64);
#pragma unroll
            for (int t = 0; t < 16; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[t][e] *= fr[e];
        }
        qa_h8 pa[3];
        float rem[8];
        bool left = false;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            // (a select: where no score is above -FLT_MAX, neither is m)
            const bool in = j0 + 16 * (i >> 2) + 4 * kg + (i & 3) < j_hi;
            const float p = in ? qa_exp2(__builtin_fmaf(sc[i], fac, __builtin_fmaf(sc[i], fac2, -m))) : 0.0f;
            l += p;
            _Float16 a, b, c;
            rem[i] = qa_split(p * QAM_P_UNIT, a, b, c);
            pa[0][i] = a;
            pa[1][i] = b;
            pa[2][i] = c;
            left |= fabsf(rem[i]) > 0.0f;
        }
        const bool deep = __ballot(left) != 0;                 // uniform
        // column t of the lane's 8 positions x 8 dims
        auto column = [&](const uint4 (&vv)[8], int t) __attribute__((always_inline)) {
            uint32_t c[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t x = reinterpret_cast<const uint32_t *>(&vv[2 * i])[t / 2];
                const uint32_t y = reinterpret_cast<const uint32_t *>(&vv[2 * i + 1])[t / 2];
                c[i] = __builtin_amdgcn_perm(y, x, t & 1 ? 0x07060302u : 0x05040100u);
            }
            return __builtin_bit_cast(qa_h8, make_uint4(c[0], c[1], c[2], c[3]));
        };
        auto values = [&](const uint4 (&vv)[8], int t0) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const qa_h8 b = column(vv, t);
                qa_f4 &o = acc[t0 + t];
                qa_f4 u = {0.f, 0.f, 0.f, 0.f};
                u = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa[2], b, u, 0, 0, 0);
                u = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa[1], b, u, 0, 0, 0);
                o = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa[0], b, o, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = __builtin_fmaf(u[e], 0x1p-12f, o[e]);
            }
            if (!deep) return;
            // What the parts left of small weights (32 of at most 2^-37) counts
            // where it may come to 2^-25 of a sum, half a unit of its last place
            float least = FLT_MAX;
            qa_us2 big = {0, 0};
#pragma unroll
            for (int t = 0; t < 8; t++) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    least = fminf(least, fabsf(acc[t0 + t][e]));
                    big = __builtin_elementwise_max(
                        big, __builtin_bit_cast(qa_us2, reinterpret_cast<const uint32_t *>(&vv[t])[e] & 0x7FFF7FFFu));
                }
            }
            float vm = fmaxf(qa_f16(big[0]), qa_f16(big[1]));
            vm = fmaxf(vm, __shfl_xor(vm, 16, 64));
            vm = fmaxf(vm, __shfl_xor(vm, 32, 64));
            if (!__ballot(!(least >= vm * 0x1p-7f))) return;
            float r[8], dn = 0x1p-12f;
#pragma unroll
            for (int i = 0; i < 8; i++) r[i] = rem[i];
#pragma unroll 1
            for (int turn = 0; turn < 3; turn++) {             // (50 bits a turn: down to 2^-136)
                qa_h8 pd[3];
                bool more = false;
                dn *= 0x1p-38f;
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    _Float16 a, b, c;
                    r[i] = qa_split(r[i] * 0x1p38f, a, b, c);
                    pd[0][i] = a;
                    pd[1][i] = b;
                    pd[2][i] = c;
                    more |= fabsf(r[i]) > 0.0f;
                }
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    const qa_h8 b = column(vv, t);
                    qa_f4 h = {0.f, 0.f, 0.f, 0.f}, u = h;
                    h = __builtin_amdgcn_mfma_f32_16x16x32_f16(pd[0], b, h, 0, 0, 0);
                    u = __builtin_amdgcn_mfma_f32_16x16x32_f16(pd[2], b, u, 0, 0, 0);
                    u = __builtin_amdgcn_mfma_f32_16x16x32_f16(pd[1], b, u, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        acc[t0 + t][e] = __builtin_fmaf(__builtin_fmaf(u[e], 0x1p-12f, h[e]), dn, acc[t0 + t][e]);
                }
                if (!__ballot(more)) break;
                dn *= 0x1p-12f;
            }
        };
        values(v0, 0);
        __builtin_amdgcn_sched_barrier(0);
        load_k();
        __builtin_amdgcn_sched_barrier(0);
        values(v1, 8);
    }
    // A key, value or query that is no finite number meets zeros and parts of
    // either sign above, where plain arithmetic has one product: the
    // workgroup does its share over as k_attn_masked does.  (Any of them
    // leaves an infinity or NaN in a sum.  A dead head's sums count too: the
    // same answer, later.)
    {
        float z = l * 0.0f;
#pragma unroll
        for (int t = 0; t < 16; t++)
#pragma unroll
            for (int e = 0; e < 4; e++) z = __builtin_fmaf(acc[t][e], 0.0f, z);
        if (__syncthreads_or(z != 0.0f)) {                     // (q is no longer read)
            qa_masked<G>(*reinterpret_cast<qa_masked_lds<G> *>(lds), out, gate, q, kc, vc, list, q_heads, kv_heads,
                         max_ctx, scale, cap, nsplit, part);
            return;
        }
    }
    // the waves' states meet
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (kg == 0) { wm[wave][ln] = m; wl[wave][ln] = l; }
    __syncthreads();                                           // (q is no longer read)
    float (*os)[QAM_HEADS][QAM_OST] = reinterpret_cast<float (*)[QAM_HEADS][QAM_OST]>(lds);
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int g = 4 * kg + e;
        const float M = fmaxf(fmaxf(wm[0][g], wm[1][g]), fmaxf(wm[2][g], wm[3][g]));
        const float f = qa_exp2(wm[wave][g] - M);
#pragma unroll
        for (int hf = 0; hf < 2; hf++)
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int t = 8 * hf + 4 * u;
                *reinterpret_cast<float4 *>(&os[wave][g][128 * hf + 8 * ln + 4 * u]) =
                    make_float4(acc[t][e] * f, acc[t + 1][e] * f, acc[t + 2][e] * f, acc[t + 3][e] * f);
            }
    }
    __syncthreads();
    float *pr = part ? part + (size_t)blockIdx.x * G * (QA_D + 2) : nullptr;
    for (int i = tid; i < G * (QA_D / 4); i += 256) {
        const int g = i / (QA_D / 4), d = 4 * (i % (QA_D / 4));
        const float M = fmaxf(fmaxf(wm[0][g], wm[1][g]), fmaxf(wm[2][g], wm[3][g]));
        const float L = (wl[0][g] * qa_exp2(wm[0][g] - M) + wl[1][g] * qa_exp2(wm[1][g] - M)) +
                        (wl[2][g] * qa_exp2(wm[2][g] - M) + wl[3][g] * qa_exp2(wm[3][g] - M));
        const float4 a = *reinterpret_cast<const float4 *>(&os[0][g][d]), b = *reinterpret_cast<const float4 *>(&os[1][g][d]);
        const float4 c = *reinterpret_cast<const float4 *>(&os[2][g][d]), e = *reinterpret_cast<const float4 *>(&os[3][g][d]);
        constexpr float dn = 1.0f / QAM_P_UNIT;
        float o[4] = {((a.x + b.x) + (c.x + e.x)) * dn, ((a.y + b.y) + (c.y + e.y)) * dn,
                      ((a.z + b.z) + (c.z + e.z)) * dn, ((a.w + b.w) + (c.w + e.w)) * dn};
        if (nsplit == 1) {
            const size_t ob = ((size_t)row * q_heads + (size_t)kvh * G + g) * QA_D + d;
            float4 gv = make_float4(0.f, 0.f, 0.f, 0.f);
            if (gate) gv = *reinterpret_cast<const float4 *>(gate + ob);
            const float gg[4] = {gv.x, gv.y, gv.z, gv.w};
#pragma unroll
            for (int u = 0; u < 4; u++) {
                o[u] = L > 0.0f ? o[u] / L : 0.0f;
                if (gate) o[u] *= 1.0f / (1.0f + expf(-gg[u]));
                out[ob + u] = o[u];
            }
        } else {
            if (d == 0) { pr[g] = M; pr[G + g] = L; }
#pragma unroll
            for (int u = 0; u < 4; u++) pr[2 * G + g * QA_D + d + u] = o[u];
        }
    }
}

// The splits of one (row, kv head, head): thread (p, t) of 4 x 256 adds dim t
// of the p-th quarter of the splits in split order, and the quarters meet in
// LDS.  Bound by its trips to memory, which is why a thread's loads (up to 32)
// all leave before the first use, eight at a time at clamped places: a thread
// for all splits of a dim, each load behind its own guard, took 7.2 us for 65
// splits of 24 heads where this takes 4.2 (a token's six layers 238 -> 219 us).
#define QA_MAX_SPLITS 128

template <int G>
__global__ void __launch_bounds__(1024) k_attn_merge(float *__restrict__ out, const float *__restrict__ gate,
                                                     const float *__restrict__ part, int q_heads, int kv_heads,
                                                     int nsplit)
{
    __shared__ float sf[QA_MAX_SPLITS], sA[4][QA_D];
    const int g = blockIdx.x % G, rk = blockIdx.x / G, row = rk / kv_heads, kvh = rk % kv_heads;
    const int tid = threadIdx.x, t = tid & 255, p = tid >> 8;
    const size_t stride = (size_t)G * (QA_D + 2);
    const float *pr = part + (size_t)rk * nsplit * stride;
    const size_t oi = ((size_t)row * q_heads + (size_t)kvh * G + g) * QA_D + t;
    // this quarter's splits [s0, s0 + cnt), requested with the maxima, sums
    // and gate (one round trip for the kernel's loads)
    const int per = (nsplit + 3) / 4, s0 = min(p * per, nsplit), cnt = min(per, nsplit - s0);
    constexpr int NQ = QA_MAX_SPLITS / 4;
    float a[NQ];
#pragma unroll
    for (int b = 0; b < NQ; b += 8)
        if (b < per)
#pragma unroll
            for (int i = b; i < b + 8; i++) a[i] = pr[min(s0 + i, nsplit - 1) * stride + 2 * G + (size_t)g * QA_D + t];
    const int sp = min(tid, nsplit - 1);
    const float m = pr[sp * stride + g], l = pr[sp * stride + G + g];
    const float gv = gate && p == 0 ? gate[oi] : 0.0f;
    // the maximum, each split's factor and the weighted sum of the splits'
    // sums, a lane a split (up to 128: two waves), the sum in a fixed tree
    // (each wave's xor tree, then wave 0's plus wave 1's)
    __shared__ float wmax[2], wsum[2];
    if (tid < 128) {
        const float v = qw_wave_max(tid < nsplit ? m : -FLT_MAX);
        if ((tid & 63) == 0) wmax[tid >> 6] = v;
    }
    __syncthreads();
    if (tid < 128) {
        float c = 0.0f;
        if (tid < nsplit) {
            const float f = qa_exp2(m - fmaxf(wmax[0], wmax[1]));
            sf[tid] = f;
            c = l * f;
        }
        c = qw_xor_sum<64>(c);
        if ((tid & 63) == 0) wsum[tid >> 6] = c;
    }
    __syncthreads();
    float A = 0.0f;
#pragma unroll
    for (int b = 0; b < NQ; b += 8)
        if (b < per)
#pragma unroll
            for (int i = b; i < b + 8; i++)
                if (i < cnt) A = __builtin_fmaf(a[i], sf[s0 + i], A);
    sA[p][t] = A;
    __syncthreads();
    if (p != 0) return;
    A = ((sA[0][t] + sA[1][t]) + sA[2][t]) + sA[3][t];
    const float L = wsum[0] + wsum[1];
    float o = L > 0.0f ? A / L : 0.0f;
    if (gate) o *= 1.0f / (1.0f + expf(-gv));
    out[oi] = o;
}

// ---- launchers ----------------------------------------------------------------------

static bool qs_shape_ok(int d, int rotary_dim) { return rotary_dim == QS_ROTARY && d >= 64 && d % 32 == 0 && d <= 256; }

template <bool POOLED>
static int qs_launch_scores(hipStream_t s, float *scores, const float *qn, const float *src, const uint16_t *kw,
                            const float *inv_freq, int rows, int nq, int d, int ratio, int base_pos,
                            int max_blocks, float eps)
{
    const int blocks = (base_pos + rows) / ratio;
    if (blocks == 0) return 0;
    const dim3 grid((blocks + QS_BLK - 1) / QS_BLK, (rows + QS_ROWS - 1) / QS_ROWS);
    const int D = d <= 64 ? 64 : d <= 128 ? 128 : d <= 192 ? 192 : 256;
    if (nq <= 16 && D <= 128) {
        // one row of stored keys: a wave a workgroup, so that 8192 blocks are
        // 512 workgroups.  More rows, stored keys: two tiles a wave share a
        // row's heads where workgroups of 32 rows fill the chip's 512 places,
        // else one, over the most rows that fill them.  Keys made here (half
        // of a short workgroup's time): the fewest rows that go in one round.
        // us, the K = 1 form / 32 rows and two tiles from 64 rows on / this:
        //   stored  64 rows,  512 blocks 35 / 54 / 12    made here 53 / 56 / 31
        //          256       2048        37 / 55 / 30              54 / 57 / 47
        //          512       4096       114 / 91 / 91             165 / 167 / 167
        const int gx1 = (blocks + 63) / 64, gx2 = (blocks + 127) / 128;
        auto fill = [&](int gx, int r) { return (long)gx * rows >= 512L * r; };
        auto fits = [&](int r) { return (long)gx1 * ((rows + r - 1) / r) <= 512; };
        const bool two = POOLED && (long)gx2 * ((rows + 31) / 32) >= 512;
        const int wr = POOLED ? two || fill(gx1, 32) ? QM_ROWS : fill(gx1, 16) ? 16 : QM_GROUP
                              : fits(8) ? QM_GROUP : fits(16) ? 16 : QM_ROWS;
        const unsigned gy = (unsigned)((rows + wr - 1) / wr);
#define QS_MX(DD, TB, NW, ONE)                                                                                         \
    hipLaunchKernelGGL((k_qsa_scores_mx<DD, POOLED, TB, NW, ONE>), dim3((blocks + 16 * TB * NW - 1) / (16 * TB * NW), gy), \
                       dim3(64 * NW), 0, s, scores, qn, src, kw, inv_freq, rows, nq, d, ratio, base_pos, max_blocks, eps, wr)
#define QS_MXD(DD)                                                                                                     \
    if constexpr (POOLED) {                                                                                            \
        if (rows == 1) QS_MX(DD, 1, 1, true);                                                                          \
        else if (two) QS_MX(DD, 2, 4, false);                                                                          \
        else QS_MX(DD, 1, 4, false);                                                                                   \
    } else {                                                                                                           \
        if (rows == 1) QS_MX(DD, 1, 4, true);                                                                          \
        else QS_MX(DD, 1, 4, false);                                                                                   \
    }
        if (D == 64) { QS_MXD(64) }
        else { QS_MXD(128) }
#undef QS_MXD
#undef QS_MX
        return (int)hipGetLastError();
    }
    const size_t lds = ((size_t)QS_BLK * (D + 4) + 4 * QS_BLK + (size_t)nq * D) * sizeof(float);
    if (lds > 160 * 1024) return hipErrorInvalidValue;
#define QS_GO(DD) hipLaunchKernelGGL((k_qsa_scores<DD, POOLED>), grid, dim3(QS_THREADS), lds, s, scores, qn, src, kw, \
                                     inv_freq, rows, nq, d, ratio, base_pos, max_blocks, eps)
    switch (D) {
    case 64: QS_GO(64); break;
    case 128: QS_GO(128); break;
    case 192: QS_GO(192); break;
    default: QS_GO(256); break;
    }
#undef QS_GO
    return (int)hipGetLastError();
}

extern "C" int qwk_qsa_scores(hipStream_t s, float *scores, const float *qn, const float *ikeys, const uint16_t *kw,
                              const float *inv_freq, int rows, int nq, int d, int ratio, int base_pos,
                              int rotary_dim, int max_blocks, float eps)
{
    if (!qs_shape_ok(d, rotary_dim) || rows < 0 || nq < 1 || ratio < 1 || base_pos < 0 ||
        (base_pos + rows) / ratio > max_blocks)
        return hipErrorInvalidValue;
    static bool attr = false;
    if (!attr) {
        attr = true;
        (void)hipFuncSetAttribute((const void *)k_qsa_scores<256, false>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipFuncSetAttribute((const void *)k_qsa_scores<192, false>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipFuncSetAttribute((const void *)k_qsa_scores<256, true>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipFuncSetAttribute((const void *)k_qsa_scores<192, true>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipFuncSetAttribute((const void *)k_qsa_scores<128, false>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipFuncSetAttribute((const void *)k_qsa_scores<128, true>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    }
    return qs_launch_scores<false>(s, scores, qn, ikeys, kw, inv_freq, rows, nq, d, ratio, base_pos, max_blocks, eps);
}

extern "C" int qwk_qsa_scores_pooled(hipStream_t s, float *scores, const float *qn, const float *pool, int rows,
                                     int nq, int d, int ratio, int base_pos, int max_blocks)
{
    if (!qs_shape_ok(d, QS_ROTARY) || rows < 0 || nq < 1 || ratio < 1 || base_pos < 0 ||
        (base_pos + rows) / ratio > max_blocks)
        return hipErrorInvalidValue;
    return qs_launch_scores<true>(s, scores, qn, pool, nullptr, nullptr, rows, nq, d, ratio, base_pos, max_blocks, 0.0f);
}

extern "C" int qwk_qsa_pool(hipStream_t s, float *pool, const float *ikeys, const uint16_t *kw, const float *inv_freq,
                            int d, int ratio, int b0, int b1, int rotary_dim, float eps)
{
    if (!qs_shape_ok(d, rotary_dim) || ratio < 1 || b0 < 0) return hipErrorInvalidValue;
    if (b1 <= b0) return 0;
    const int n = b1 - b0;
    const dim3 grid((n + 3) / 4);
    if (d <= 64) hipLaunchKernelGGL(k_qsa_pool<1>, grid, dim3(QS_THREADS), 0, s, pool, ikeys, kw, inv_freq, d, ratio, b0, n, eps);
    else if (d <= 128) hipLaunchKernelGGL(k_qsa_pool<2>, grid, dim3(QS_THREADS), 0, s, pool, ikeys, kw, inv_freq, d, ratio, b0, n, eps);
    else if (d <= 192) hipLaunchKernelGGL(k_qsa_pool<3>, grid, dim3(QS_THREADS), 0, s, pool, ikeys, kw, inv_freq, d, ratio, b0, n, eps);
    else hipLaunchKernelGGL(k_qsa_pool<4>, grid, dim3(QS_THREADS), 0, s, pool, ikeys, kw, inv_freq, d, ratio, b0, n, eps);
    return (int)hipGetLastError();
}

extern "C" int qwk_qsa_select(hipStream_t s, uint8_t *mask, uint32_t *list, const float *scores, int rows, int ratio,
                              int base_pos, int block_topk, int max_ctx, int max_blocks)
{
    if (rows < 0 || ratio < 1 || base_pos < 0 || block_topk < 0 || base_pos + rows > max_ctx ||
        (base_pos + rows) / ratio > max_blocks || max_blocks > QS_SEL_MAX_BLOCKS)
        return hipErrorInvalidValue;
    if (rows == 0) return 0;
    const int cap = block_topk * ratio + ratio;
    const size_t lds = ((size_t)((base_pos + rows) / ratio) + 16) & ~(size_t)15;
    static bool attr = false;
    if (!attr) {
        attr = true;
        (void)hipFuncSetAttribute((const void *)k_qsa_select, hipFuncAttributeMaxDynamicSharedMemorySize, QS_SEL_MAX_BLOCKS + 16);
    }
    hipLaunchKernelGGL(k_qsa_select, dim3(rows), dim3(QS_SEL_THREADS), lds, s, mask, list, scores, ratio, base_pos,
                       block_topk, max_ctx, max_blocks, cap);
    return (int)hipGetLastError();
}

// Splits of the position list per (row, kv head): enough workgroups to
// cover the chip when rows * kv_heads alone would not, each split at least
// one pass of QA_P positions.
static int qa_splits(int rows, int kv_heads, int cap)
{
    const int rk = rows * kv_heads, passes = (cap + QA_P - 1) / QA_P;
    if (rk >= 256 || passes <= 1) return 1;
    return max(1, min(min(passes, QA_MAX_SPLITS), (512 + rk - 1) / rk));
}

extern "C" size_t qwk_attn_masked_work_bytes(int rows, int q_heads, int kv_heads, int cap)
{
    if (kv_heads < 1 || rows < 1) return 0;
    const int ns = qa_splits(rows, kv_heads, cap);
    if (ns == 1) return 0;
    return (size_t)rows * kv_heads * ns * (q_heads / kv_heads) * (QA_D + 2) * sizeof(float);
}

template <int G>
static void qa_merge(hipStream_t s, float *out, const float *gate, const float *part, int rows, int q_heads,
                     int kv_heads, int ns)
{
    hipLaunchKernelGGL(k_attn_merge<G>, dim3(rows * kv_heads * G), dim3(1024), 0, s, out, gate, part, q_heads,
                       kv_heads, ns);
}

template <int G>
static void qa_launch(hipStream_t s, float *out, const float *gate, const float *q, const uint16_t *kc,
                      const uint16_t *vc, const uint32_t *list, int rows, int q_heads, int kv_heads, int max_ctx,
                      float scale, int cap, int ns, float *part)
{
    // the matrix cores from 8 heads a kv head on, where a split gives every
    // wave of a workgroup a pass of 32 positions (a decode step's splits are
    // one pass long: three waves would idle)
    const int per = ((cap + QA_P - 1) / QA_P + ns - 1) / ns;
    if constexpr (G >= 8) {
        if (per * QA_P >= 4 * QAM_STEP) {
            hipLaunchKernelGGL(k_attn_mx<G>, dim3(rows * kv_heads * ns), dim3(256), 0, s, out, gate, q, kc, vc, list,
                               q_heads, kv_heads, max_ctx, scale, cap, ns, part);
            if (ns > 1) qa_merge<G>(s, out, gate, part, rows, q_heads, kv_heads, ns);
            return;
        }
    }
    hipLaunchKernelGGL(k_attn_masked<G>, dim3(rows * kv_heads * ns), dim3(256), 0, s, out, gate, q, kc, vc, list,
                       q_heads, kv_heads, max_ctx, scale, cap, ns, part);
    if (ns > 1) qa_merge<G>(s, out, gate, part, rows, q_heads, kv_heads, ns);
}

extern "C" int qwk_attn_masked(hipStream_t s, float *out, const float *gate, const float *q, const uint16_t *kc,
                               const uint16_t *vc, const uint32_t *list, int rows, int q_heads, int kv_heads,
                               int head_dim, int max_ctx, float scale, int cap, void *work, size_t work_bytes)
{
    if (head_dim != QA_D || kv_heads < 1 || q_heads % kv_heads || rows < 0 || cap < 0) return hipErrorInvalidValue;
    if (rows == 0) return 0;
    int ns = qa_splits(rows, kv_heads, cap);
    if (ns > 1 && (!work || work_bytes < qwk_attn_masked_work_bytes(rows, q_heads, kv_heads, cap))) ns = 1;
    float *part = (float *)work;
    switch (q_heads / kv_heads) {
    case 1: qa_launch<1>(s, out, gate, q, kc, vc, list, rows, q_heads, kv_heads, max_ctx, scale, cap, ns, part); break;
    case 2: qa_launch<2>(s, out, gate, q, kc, vc, list, rows, q_heads, kv_heads, max_ctx, scale, cap, ns, part); break;
    case 4: qa_launch<4>(s, out, gate, q, kc, vc, list, rows, q_heads, kv_heads, max_ctx, scale, cap, ns, part); break;
    case 8: qa_launch<8>(s, out, gate, q, kc, vc, list, rows, q_heads, kv_heads, max_ctx, scale, cap, ns, part); break;
    case 12: qa_launch<12>(s, out, gate, q, kc, vc, list, rows, q_heads, kv_heads, max_ctx, scale, cap, ns, part); break;
    case 16: qa_launch<16>(s, out, gate, q, kc, vc, list, rows, q_heads, kv_heads, max_ctx, scale, cap, ns, part); break;
    default: return hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
}
