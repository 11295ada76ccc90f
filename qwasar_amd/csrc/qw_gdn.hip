// qw_gdn.hip -- the gated DeltaNet's three kernels (reference contract
// qwasar_gpu.h:318-358, CPU semantics qwasar_cpu.c:217-283):
//
//   k_conv1d_causal_silu  the causal depthwise conv over the mixed q/k/v
//                         channels with silu, its window carried in `state`
//   k_gdn_gates           g = exp(-exp(A_log) softplus(a + dt_bias)), beta = sigmoid(b)
//   k_gated_delta<PREP>   the delta-rule recurrence per value head,
//                             S *= g;  kv = S k;  S += k (v - kv) beta;  y = S q
//                         and, with PREP, q and k l2-normed and the gates
//                         computed inside the kernel; with CONV (one decode
//                         step) the conv too, for the channels it reads
//   k_gdn_chunk_pre, k_gdn_chunk   the same recurrence in chunks of 32 steps,
//                         for long calls
//
// The recurrence is serial in time but independent across the rows of each
// head's [dv, dk] state.  A wave owns four value rows: each 16-lane row of
// the wave one state row, each lane eight consecutive key columns held in
// registers for the whole call, so the state crosses HBM once per call, not
// once per step.  A workgroup (four waves) owns sixteen rows of one head; the
// timesteps' q, k, v and gates are staged 16 at a time into LDS, which the
// sixteen rows share (with PREP, q and k already scaled by their norms), so
// the serial loop reads only LDS.  Each dot product of a step is two fma
// chains of four columns in a lane, their sum, then the fixed xor tree over
// the 16 lanes (four DPP steps inside the row, no cross-row traffic).
#include "qw_device.h"
#include "qw_kernels.h"

#define QG_DK 128
#define QG_DV 128
#define QG_ROWS_PER_WG 16
#define QG_CHUNK 16
#define QG_PRE_MIN_ROWS 64      // prepared calls from this many steps on take k_gdn_pre
#define QG_THREADS 256

__device__ __forceinline__ float qg_softplus(float x) { return x > 20.0f ? x : log1pf(expf(x)); }

// ---- causal conv ------------------------------------------------------------

// Output t of a channel depends only on the inputs t - KS + 1 .. t (the
// carried window standing in for t < 0), never on an earlier output, so the
// launch runs over (channel, run of QG_CONV_T steps) in parallel: a thread
// a channel of one run, its window loaded once, each step one fma chain over
// the taps oldest first (from 0) and silu.  Snapshot t (t < n_snap) is the
// window after step t: inputs t - KS + 2 .. t.  The thread of a channel's
// first run is the only one that reads the carried window, and it also writes
// the window after the last step (the last KS - 1 inputs, older ones from the
// window it read), so the window is updated in place without a race between
// workgroups.
#define QG_CONV_T 16
template <int KS>
__global__ void __launch_bounds__(256) k_conv1d_causal_silu(float *__restrict__ y, const float *__restrict__ x,
                                                            float *__restrict__ state, const uint16_t *__restrict__ w,
                                                            int channels, int rows, float *__restrict__ snap,
                                                            int n_snap, int snap_stride)
{
    const int ch = blockIdx.x * 256 + threadIdx.x;
    if (ch >= channels) return;
    const int t0 = blockIdx.y * QG_CONV_T, t1 = min(t0 + QG_CONV_T, rows);
    float taps[KS], win[KS + QG_CONV_T], old[KS - 1];
#pragma unroll
    for (int j = 0; j < KS; j++) taps[j] = qw_bf16(w[(size_t)ch * KS + j]);
    // win[i] = input t0 - (KS - 1) + i
    if (t0 == 0) {
#pragma unroll
        for (int j = 0; j < KS - 1; j++) win[j] = old[j] = state[(size_t)j * channels + ch];
    } else {
#pragma unroll
        for (int j = 0; j < KS - 1; j++) win[j] = x[(size_t)(t0 - (KS - 1) + j) * channels + ch];
    }
#pragma unroll
    for (int u = 0; u < QG_CONV_T; u++) win[KS - 1 + u] = t0 + u < t1 ? x[(size_t)(t0 + u) * channels + ch] : 0.0f;
#pragma unroll
    for (int u = 0; u < QG_CONV_T; u++) {
        const int t = t0 + u;
        if (t < t1) {
            float acc = 0.0f;
#pragma unroll
            for (int j = 0; j < KS; j++) acc = __builtin_fmaf(win[u + j], taps[j], acc);
            y[(size_t)t * channels + ch] = acc / (1.0f + expf(-acc));
            if (t < n_snap) {
#pragma unroll
                for (int j = 0; j < KS - 1; j++) snap[(size_t)t * snap_stride + (size_t)j * channels + ch] = win[u + 1 + j];
            }
        }
    }
    if (t0 == 0) {
        // the window after the last step: inputs rows - KS + 1 .. rows - 1
#pragma unroll
        for (int j = 0; j < KS - 1; j++) {
            const int t = rows - (KS - 1) + j;
            float v = 0.0f;
#pragma unroll
            for (int m = 0; m < KS - 1; m++)
                if (m == KS - 1 + t) v = old[m];                       // rows < KS - 1: from the window read
            state[(size_t)j * channels + ch] = t >= 0 ? x[(size_t)t * channels + ch] : v;
        }
    }
}

// ---- gates ------------------------------------------------------------------

__device__ __forceinline__ void qg_gates(float a, float b, float A, float dt, float &g, float &beta)
{
    g = expf(-expf(A) * qg_softplus(a + dt));
    beta = 1.0f / (1.0f + expf(-b));
}

__global__ void __launch_bounds__(256) k_gdn_gates(float *__restrict__ g, float *__restrict__ beta,
                                                   const float *__restrict__ a, const float *__restrict__ b,
                                                   const uint16_t *__restrict__ A_log,
                                                   const uint16_t *__restrict__ dt_bias, int hv, int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int h = i % hv;
    qg_gates(a[i], b[i], qw_bf16(A_log[h]), qw_bf16(dt_bias[h]), g[i], beta[i]);
}

// ---- the recurrence -----------------------------------------------------------

struct qg_prep {
    const float *a, *b;
    const uint16_t *A_log, *dt_bias;
    float l2eps, q_scale, k_scale;
    // from k_gdn_pre (or null): each step's q and k norm factors
    // [rows][hk][2] and gates (g, beta) [rows][hv][2]
    const float *nrm, *gb;
};

// The l2 norm factor of one 128-value q or k vector, by a whole wave: lane
// l squares values l and l + 64 (an fma chain from 0), then the wave's xor
// tree.  Every lane gets the factor.
__device__ __forceinline__ float qg_norm(float a0, float a1, float l2eps, float scale)
{
    float ss = __builtin_fmaf(a0, a0, 0.0f);
    ss = __builtin_fmaf(a1, a1, ss);
    ss = qw_xor_sum<64>(ss);
    return 1.0f / sqrtf(ss / (float)QG_DK + l2eps) * scale;
}

// A long prepared call's norms and gates ahead of the recurrence, in
// parallel over every step: the first nvw / 4 workgroups a wave a vector
// (vector w: step w / (2 hk), key head (w / 2) % hk, k if w is odd), the
// rest a thread a (step, value head) gate; the recurrence's own functions,
// so the same bits as computed inside it.
__global__ void __launch_bounds__(256) k_gdn_pre(qg_prep pp, const float *__restrict__ q, const float *__restrict__ k,
                                                 int hk, int hv, int rows)
{
    const int nvw = rows * hk * 2, nbv = (nvw + 3) / 4;
    float *nrm = const_cast<float *>(pp.nrm), *gb = const_cast<float *>(pp.gb);
    if ((int)blockIdx.x < nbv) {
        const int w = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
        if (w >= nvw) return;
        const float *src = ((w & 1) ? k : q) + (size_t)(w >> 1) * QG_DK;
        const float f = qg_norm(src[lane], src[lane + 64], pp.l2eps, (w & 1) ? pp.k_scale : pp.q_scale);
        if (lane == 0) nrm[w] = f;
    } else {
        const int i = (blockIdx.x - nbv) * 256 + threadIdx.x;
        if (i >= rows * hv) return;
        const int h = i % hv;
        qg_gates(pp.a[i], pp.b[i], qw_bf16(pp.A_log[h]), qw_bf16(pp.dt_bias[h]), gb[2 * i], gb[2 * i + 1]);
    }
}

// The fused decode step's conv: the mixed channels before the conv, the
// window in and out (distinct buffers), the taps.
struct qg_conv {
    const float *x, *win;
    float *wout;
    const uint16_t *w;
    int channels;
};

// One channel of the causal conv with silu at one step, the arithmetic of
// k_conv1d_causal_silu (taps against the window oldest first, then the
// new sample, in one fma chain from 0); the window after the step goes to
// wout when `own`.
__device__ __forceinline__ float qg_conv1(const qg_conv &cv, int ch, bool own)
{
    const int C = cv.channels;
    float win[4], acc = 0.0f;
#pragma unroll
    for (int j = 0; j < 3; j++) win[j] = cv.win[(size_t)j * C + ch];
    win[3] = cv.x[ch];
#pragma unroll
    for (int j = 0; j < 4; j++) acc = __builtin_fmaf(win[j], qw_bf16(cv.w[(size_t)ch * 4 + j]), acc);
    if (own) {
#pragma unroll
        for (int j = 0; j < 3; j++) cv.wout[(size_t)j * C + ch] = win[j + 1];
    }
    return acc / (1.0f + expf(-acc));
}

// CONV (one step, PREP): q, k and v are the conv's outputs over the mixed
// channels [0, hk dk), [hk dk, 2 hk dk) and [2 hk dk, ...), computed here
// for the channels this workgroup reads; the first workgroup of each key
// head's group writes the window of its q and k channels, every workgroup
// that of its own v channels.
template <bool PREP, bool CONV = false>
__global__ void __launch_bounds__(QG_THREADS) k_gated_delta(float *__restrict__ y, const float *__restrict__ q,
                                                            const float *__restrict__ k, const float *__restrict__ v,
                                                            const float *__restrict__ g,
                                                            const float *__restrict__ beta, float *state, int hk,
                                                            int hv, int rows, float *__restrict__ snap, int n_snap,
                                                            int snap_stride, qg_prep pp, qg_conv cv = {})
{
    __shared__ float4 sq[QG_CHUNK][QG_DK / 4], sk[QG_CHUNK][QG_DK / 4];
    __shared__ float sv[QG_CHUNK][QG_ROWS_PER_WG];
    __shared__ float sg[QG_CHUNK][2];   // g, beta
    __shared__ float sn[QG_CHUNK][2];   // PREP: q and k norm factors

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int groups = QG_DV / QG_ROWS_PER_WG;
    const int h = blockIdx.x / groups, r0 = (blockIdx.x % groups) * QG_ROWS_PER_WG;
    const int hx = h / (hv / hk);
    const int rl = 4 * wave + (lane >> 4);        // row within the workgroup
    const int row = r0 + rl;
    const int c8 = lane & 15;                      // columns 8 c8 .. 8 c8 + 7

    float4 *sp = reinterpret_cast<float4 *>(state + ((size_t)h * QG_DV + row) * QG_DK) + 2 * c8;
    float4 st = sp[0], su = sp[1];
    const float A = PREP ? qw_bf16(pp.A_log[h]) : 0.0f;
    const float dt = PREP ? qw_bf16(pp.dt_bias[h]) : 0.0f;
    const size_t qstride = (size_t)hk * QG_DK, vstride = (size_t)hv * QG_DV;

    // Without CONV a chunk's q, k, v and gate inputs are fetched into
    // registers one chunk ahead, so their loads run under the previous
    // chunk's steps: thread tid holds float4s tid and tid + 256 of the
    // chunk's [16][32] q and k, value (tid / 16, tid % 16) and, for tid in
    // [128, 144), step tid - 128's gate inputs.
    static_assert(QG_CHUNK * (QG_DK / 4) == 2 * QG_THREADS && QG_CHUNK * QG_ROWS_PER_WG == QG_THREADS,
                  "one chunk's staging is two float4s of q and of k and one value a thread");
    float4 fq0 = {}, fq1 = {}, fk0 = {}, fk1 = {};
    float fv = 0.0f, fa = 0.0f, fb = 0.0f, fn = 0.0f;
    const bool pre = PREP && !CONV && pp.nrm;
    auto fetch = [&](int c) __attribute__((always_inline)) {
        const int nn = min(QG_CHUNK, rows - c);
        const int t0 = tid / (QG_DK / 4), t1 = t0 + QG_THREADS / (QG_DK / 4), cc = tid % (QG_DK / 4);
        const size_t o0 = (size_t)(c + t0) * qstride + (size_t)hx * QG_DK, o1 = o0 + (size_t)(t1 - t0) * qstride;
        if (t0 < nn) {
            fq0 = reinterpret_cast<const float4 *>(q + o0)[cc];
            fk0 = reinterpret_cast<const float4 *>(k + o0)[cc];
        }
        if (t1 < nn) {
            fq1 = reinterpret_cast<const float4 *>(q + o1)[cc];
            fk1 = reinterpret_cast<const float4 *>(k + o1)[cc];
        }
        if (tid / QG_ROWS_PER_WG < nn)
            fv = v[(size_t)(c + tid / QG_ROWS_PER_WG) * vstride + (size_t)h * QG_DV + r0 + tid % QG_ROWS_PER_WG];
        if (tid >= 128 && tid < 128 + nn) {
            const size_t gi = (size_t)(c + tid - 128) * hv + h;
            fa = pre ? pp.gb[2 * gi] : PREP ? pp.a[gi] : g[gi];
            fb = pre ? pp.gb[2 * gi + 1] : PREP ? pp.b[gi] : beta[gi];
        }
        if (pre && tid >= 160 && tid < 160 + 2 * nn)
            fn = pp.nrm[((size_t)(c + (tid - 160) / 2) * hk + hx) * 2 + (tid & 1)];
    };
    if (!CONV) fetch(0);

    for (int c0 = 0; c0 < rows; c0 += QG_CHUNK) {
        const int n = min(QG_CHUNK, rows - c0);
        __syncthreads();                           // the previous chunk is consumed
        if (CONV) {
            const int kd = hk * QG_DK;
            const bool own_qk = h % (hv / hk) == 0 && r0 == 0;
            float *fq = reinterpret_cast<float *>(&sq[0][0]), *fk = reinterpret_cast<float *>(&sk[0][0]);
            if (tid < QG_DK) fq[tid] = qg_conv1(cv, hx * QG_DK + tid, own_qk);
            else if (tid < 2 * QG_DK) fk[tid - QG_DK] = qg_conv1(cv, kd + hx * QG_DK + tid - QG_DK, own_qk);
            if (tid < QG_ROWS_PER_WG) sv[0][tid] = qg_conv1(cv, 2 * kd + h * QG_DV + r0 + tid, true);
            if (tid >= 128 && tid < 128 + n) {
                const size_t gi = (size_t)(c0 + tid - 128) * hv + h;
                qg_gates(pp.a[gi], pp.b[gi], A, dt, sg[tid - 128][0], sg[tid - 128][1]);
            }
        } else {
            const int t0 = tid / (QG_DK / 4), t1 = t0 + QG_THREADS / (QG_DK / 4), cc = tid % (QG_DK / 4);
            sq[t0][cc] = fq0;
            sk[t0][cc] = fk0;
            sq[t1][cc] = fq1;
            sk[t1][cc] = fk1;
            sv[tid / QG_ROWS_PER_WG][tid % QG_ROWS_PER_WG] = fv;
            if (tid >= 128 && tid < 128 + n) {
                if (PREP && !pre) qg_gates(fa, fb, A, dt, sg[tid - 128][0], sg[tid - 128][1]);
                else {
                    sg[tid - 128][0] = fa;
                    sg[tid - 128][1] = fb;
                }
            }
            if (pre && tid >= 160 && tid < 160 + 2 * n) sn[(tid - 160) / 2][tid & 1] = fn;
            if (c0 + QG_CHUNK < rows) fetch(c0 + QG_CHUNK);
        }
        if (PREP) {
            __syncthreads();
            // the l2 norms of the chunk's q and k vectors: a wave per (step,
            // vector), each lane two of the 128 values, then the wave's xor
            // tree; in a whole chunk a wave's eight vectors are loaded first
            // and their trees run side by side
            auto norm = [&](int p, float a0, float a1) __attribute__((always_inline)) {
                const float f = qg_norm(a0, a1, pp.l2eps, (p & 1) ? pp.k_scale : pp.q_scale);
                if (lane == 0) sn[p >> 1][p & 1] = f;
            };
            auto vec = [&](int p) __attribute__((always_inline)) {
                return reinterpret_cast<const float *>((p & 1) ? &sk[p >> 1][0] : &sq[p >> 1][0]);
            };
            if (pre) {
                // the factors came with the chunk
            } else if (n == QG_CHUNK) {
                static_assert(2 * QG_CHUNK == 8 * (QG_THREADS / 64), "eight vectors a wave");
                float a0[8], a1[8];
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    a0[j] = vec(wave + 4 * j)[lane];
                    a1[j] = vec(wave + 4 * j)[lane + 64];
                }
#pragma unroll
                for (int j = 0; j < 8; j++) norm(wave + 4 * j, a0[j], a1[j]);
            } else {
                for (int p = wave; p < 2 * n; p += QG_THREADS / 64) norm(p, vec(p)[lane], vec(p)[lane + 64]);
            }
            __syncthreads();
            for (int i = tid; i < n * (QG_DK / 4); i += QG_THREADS) {
                const int t = i / (QG_DK / 4), c = i % (QG_DK / 4);
                const float iq = sn[t][0], ik = sn[t][1];
                float4 a = sq[t][c], b = sk[t][c];
                a.x *= iq; a.y *= iq; a.z *= iq; a.w *= iq;
                b.x *= ik; b.y *= ik; b.z *= ik; b.w *= ik;
                sq[t][c] = a;
                sk[t][c] = b;
            }
        }
        __syncthreads();
        // a step; whole chunks unrolled, so that a step's output dot and
        // the next step's LDS reads overlap the state's serial chain
        auto step = [&](int t) __attribute__((always_inline)) {
            const float4 q0 = sq[t][2 * c8], q1 = sq[t][2 * c8 + 1], k0 = sk[t][2 * c8], k1 = sk[t][2 * c8 + 1];
            const float gt = sg[t][0], bt = sg[t][1];
            st.x *= gt; st.y *= gt; st.z *= gt; st.w *= gt;
            su.x *= gt; su.y *= gt; su.z *= gt; su.w *= gt;
            float ka = st.x * k0.x, kb = su.x * k1.x;
            ka = __builtin_fmaf(st.y, k0.y, ka);
            kb = __builtin_fmaf(su.y, k1.y, kb);
            ka = __builtin_fmaf(st.z, k0.z, ka);
            kb = __builtin_fmaf(su.z, k1.z, kb);
            ka = __builtin_fmaf(st.w, k0.w, ka);
            kb = __builtin_fmaf(su.w, k1.w, kb);
            const float kv = qw_xor_sum<16>(ka + kb);
            const float delta = (sv[t][rl] - kv) * bt;
            st.x = __builtin_fmaf(k0.x, delta, st.x);
            st.y = __builtin_fmaf(k0.y, delta, st.y);
            st.z = __builtin_fmaf(k0.z, delta, st.z);
            st.w = __builtin_fmaf(k0.w, delta, st.w);
            su.x = __builtin_fmaf(k1.x, delta, su.x);
            su.y = __builtin_fmaf(k1.y, delta, su.y);
            su.z = __builtin_fmaf(k1.z, delta, su.z);
            su.w = __builtin_fmaf(k1.w, delta, su.w);
            float oa = st.x * q0.x, ob = su.x * q1.x;
            oa = __builtin_fmaf(st.y, q0.y, oa);
            ob = __builtin_fmaf(su.y, q1.y, ob);
            oa = __builtin_fmaf(st.z, q0.z, oa);
            ob = __builtin_fmaf(su.z, q1.z, ob);
            oa = __builtin_fmaf(st.w, q0.w, oa);
            ob = __builtin_fmaf(su.w, q1.w, ob);
            const float o = qw_xor_sum<16>(oa + ob);
            const int tt = c0 + t;
            if (c8 == 0) y[(size_t)tt * vstride + (size_t)h * QG_DV + row] = o;
            if (tt < n_snap) {
                float4 *sn4 = reinterpret_cast<float4 *>(snap + (size_t)tt * snap_stride + ((size_t)h * QG_DV + row) * QG_DK) + 2 * c8;
                sn4[0] = st;
                sn4[1] = su;
            }
        };
        if (n == QG_CHUNK) {
#pragma unroll
            for (int t = 0; t < QG_CHUNK; t++) step(t);
        } else {
            for (int t = 0; t < n; t++) step(t);
        }
    }
    sp[0] = st;
    sp[1] = su;
}

// ---- the recurrence in chunks ---------------------------------------------------
//
// A long call (QG_LONG_MIN_ROWS steps on, no snapshots) takes QG_C steps at a
// time.  With P[t][i] the product of g over (i, t], G[t] the product of g up
// to t in the chunk, S0 the state before it and u_t = beta_t (v_t - g_t S_{t-1} k_t):
//   (I + L) U = beta (V - G K S0'),   L[t][i] = beta_t P[t][i] (k_t . k_i), i < t
//   Y = G Q S0' + (P o Q K') U,       S = G[C-1] S0 + sum_i P[C-1][i] u_i k_i'
// so the serial part is a few 16-wide products a chunk in place of QG_C
// dependent steps.  k_gdn_chunk_pre does everything that does not need the
// state, a workgroup a (key head, chunk): the norms, K K' and Q K', and for
// each of the key head's value heads the gates, P by running products (never
// a quotient or a difference of logarithms, which a strong decay would ruin)
// and T = (I + L)^-1 by forward substitution.  k_gdn_chunk walks the chunks,
// a workgroup 16 value rows of a head, every product on the fp32 matrix cores
// (v_mfma_f32_16x16x4_f32: fp32 inputs and sums, as the serial form).
// 2048 steps of 16 key and 48 value heads: 10 + 590 us serial (70 vector
// operations a step on the CUs that hold two workgroups), 39 + 264 here; the
// call with conv and output gate 690 -> 363.  Error against 64 bits over calls
// of 600 and 2048 steps: y 1.50 to 1.51e-7 serial, 1.48 to 1.51e-7 here, the
// state 1.19 to 1.33e-7 and 1.09 to 1.22e-7.  That takes short chains from zero
// met in trees, and the norms' factors and the gates' products in 64 bits
// (without: y 1.75e-7, 34 + 227 us).
// What bounds it now: k_gdn_chunk's chain a chunk (56 MFMAs of 35 cycles a
// wave and three hand-offs through LDS) on the CUs that hold two of the 384
// workgroups, and its operands' bytes (K and Q read by 8 workgroups a head: a
// build without the loads takes 165 us).
// A NaN or infinity must not reach the chunk's earlier steps through the zeros
// of T and Q K' above the diagonal, so a value row's first step with one is
// kept (`bad`): R and U are zero from there on as operands of those products,
// and the row's outputs from there on are NaN, its state what it comes to
// (34 us of the 264).
#define QG_C 32
#define QG_LONG_MIN_ROWS 256     // below, the serial kernel (and its bits) stay
#define QG_LONG_ROWS 4096        // steps a pair of launches takes: bounds the scratch
#define QG_CS (QG_DK + 4)        // floats an LDS row of 128 takes: 16-byte reads of 8 rows hit different banks
#define QG_TS (QG_C + 4)

typedef float qg_f4 __attribute__((ext_vector_type(4)));

// Scratch of one launch pair over `n` chunks.
struct qg_long {
    float *qn, *kn;          // [hk][n][2][8][64][4]: q and k, normed with PREP, in operand order
    float *T, *QK;           // [hv][n][2][2][64][4]: QG_C x QG_C, in operand order
    float4 *sc;              // [hv][n][QG_C]: beta, beta G, G, P[C-1]
};
static size_t qg_long_bytes(int hk, int hv, int rows, qg_long *w, char *base)
{
    const size_t n = (size_t)(rows + QG_C - 1) / QG_C;
    size_t off = 0;
    auto take = [&](size_t bytes) {
        char *p = base + off;
        off += (bytes + 255) & ~(size_t)255;
        return p;
    };
    qg_long l;
    l.qn = reinterpret_cast<float *>(take(n * QG_C * hk * QG_DK * 4));
    l.kn = reinterpret_cast<float *>(take(n * QG_C * hk * QG_DK * 4));
    l.T = reinterpret_cast<float *>(take((size_t)hv * n * QG_C * QG_C * 4));
    l.QK = reinterpret_cast<float *>(take((size_t)hv * n * QG_C * QG_C * 4));
    l.sc = reinterpret_cast<float4 *>(take((size_t)hv * n * QG_C * 16));
    if (w) *w = l;
    return off;
}

// D += A B over 16 k: lane (ln, kg) holds A[ln][4 kg ..] and B[4 kg ..][ln],
// and of D rows 4 kg .. 4 kg + 3 of column ln.  (Step s of the four takes
// element s of every lane: the same k of A and B.)
__device__ __forceinline__ qg_f4 qg_mm16(float4 a, float4 b, qg_f4 d)
{
    d = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, d, 0, 0, 0);
    d = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, d, 0, 0, 0);
    d = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, d, 0, 0, 0);
    d = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, d, 0, 0, 0);
    return d;
}

// Lane t's double in every lane.
__device__ __forceinline__ double qg_lane(double v, int t)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, t);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), t);
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// Steps past the call's last are g = 1, beta = 0, q = k = 0: they leave the
// state alone, and no output is written for them.  What k_gdn_chunk reads as
// MFMA operands is stored in its lanes' order, so that its loads are whole
// kilobytes (16 rows of 64 bytes a load were twice the lines).
template <bool PREP>
__global__ void __launch_bounds__(256) k_gdn_chunk_pre(qg_long w, const float *__restrict__ q,
                                                       const float *__restrict__ k, const float *__restrict__ g,
                                                       const float *__restrict__ beta, int hk, int hv, int rows,
                                                       qg_prep pp)
{
    // q and k, then (in their place) a wave's L and masked Q K'
    constexpr int NQ = 2 * QG_C * QG_CS, NL = 8 * QG_C * QG_TS;
    __shared__ __align__(16) float lds[NQ > NL ? NQ : NL];
    __shared__ __align__(16) float KK[QG_C][QG_TS], QK[QG_C][QG_TS];
    float (*Ks)[QG_CS] = reinterpret_cast<float (*)[QG_CS]>(lds), (*Qs)[QG_CS] = Ks + QG_C;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ln = lane & 15, kg = lane >> 4;
    const int c = blockIdx.x, hx = blockIdx.y, nch = gridDim.x, n = min(QG_C, rows - c * QG_C);

    // q and k: 8 lanes a step, 16 values each
    {
        const int t = tid >> 3, e = tid & 7, tt = c * QG_C + min(t, n - 1);
        const size_t o = ((size_t)tt * hk + hx) * QG_DK;
        float4 vq[4], vk[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            vq[i] = reinterpret_cast<const float4 *>(q + o)[e + 8 * i];
            vk[i] = reinterpret_cast<const float4 *>(k + o)[e + 8 * i];
        }
        float fq = t < n ? 1.0f : 0.0f, fk = fq;
        if (PREP) {
            // (a row's factor in 64 bits: its error is common to the row, where the sums' are not)
            double aq = 0.0, ak = 0.0;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float cq[4] = {vq[i].x, vq[i].y, vq[i].z, vq[i].w}, ck[4] = {vk[i].x, vk[i].y, vk[i].z, vk[i].w};
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    aq = __builtin_fma((double)cq[m], (double)cq[m], aq);
                    ak = __builtin_fma((double)ck[m], (double)ck[m], ak);
                }
            }
#pragma unroll
            for (int o = 1; o < 8; o <<= 1) {
                aq += __shfl_xor(aq, o, 64);
                ak += __shfl_xor(ak, o, 64);
            }
            fq *= (float)((double)pp.q_scale / sqrt(aq / QG_DK + (double)pp.l2eps));
            fk *= (float)((double)pp.k_scale / sqrt(ak / QG_DK + (double)pp.l2eps));
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // (a select, not the factor 0: what a step past the last reads may be anything)
            const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
            *reinterpret_cast<float4 *>(&Qs[t][4 * (e + 8 * i)]) =
                t < n ? make_float4(vq[i].x * fq, vq[i].y * fq, vq[i].z * fq, vq[i].w * fq) : z;
            *reinterpret_cast<float4 *>(&Ks[t][4 * (e + 8 * i)]) =
                t < n ? make_float4(vk[i].x * fk, vk[i].y * fk, vk[i].z * fk, vk[i].w * fk) : z;
        }
    }
    __syncthreads();
    // out in operand order: [tile of 16 steps][j][lane], lane (ln, kg) the four from 16 j + 4 kg of step ln
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int t0 = 16 * (i >> 1), j = 4 * (i & 1) + wave;
        const size_t o = (((size_t)hx * nch + c) * 16 + (t0 ? 8 : 0) + j) * 64 + lane;
        reinterpret_cast<float4 *>(w.qn)[o] = *reinterpret_cast<const float4 *>(&Qs[t0 + ln][16 * j + 4 * kg]);
        reinterpret_cast<float4 *>(w.kn)[o] = *reinterpret_cast<const float4 *>(&Ks[t0 + ln][16 * j + 4 * kg]);
    }
    // K K' and Q K', the tiles on and below the diagonal: (0, 0), (1, 0), (1, 1) of each
    for (int u = wave; u < 6; u += 4) {
        const int m = (u % 3) > 0 ? 16 : 0, i0 = (u % 3) > 1 ? 16 : 0;
        const float *A = u < 3 ? &Ks[m + ln][0] : &Qs[m + ln][0], *B = &Ks[i0 + ln][0];
        qg_f4 d[8];
#pragma unroll
        for (int i = 0; i < 8; i++)
            d[i] = qg_mm16(*reinterpret_cast<const float4 *>(A + 16 * i + 4 * kg),
                           *reinterpret_cast<const float4 *>(B + 16 * i + 4 * kg), qg_f4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int e = 0; e < 4; e++) (u < 3 ? KK : QK)[m + 4 * kg + e][i0 + ln] = ((d[0][e] + d[1][e]) + (d[2][e] + d[3][e])) +
                                                                                     ((d[4][e] + d[5][e]) + (d[6][e] + d[7][e]));
    }
    __syncthreads();                                              // q and k are consumed
    // a value head a wave: lane i has column i of P, L, the masked Q K' and T
    float (*Ls)[QG_TS] = reinterpret_cast<float (*)[QG_TS]>(lds) + wave * 2 * QG_C, (*Ms)[QG_TS] = Ls + QG_C;
    for (int r = wave; r < hv / hk; r += 4) {
        const int h = hx * (hv / hk) + r, i = lane & 31;
        const size_t hc = (size_t)h * nch + c;
        // step i's gate and beta; the gate and its running products in 64
        // bits (a product of 32 factors is off by 32 of their errors)
        double gi = 1.0;
        float bi = 0.0f;
        if (i < n) {
            const size_t at = (size_t)(c * QG_C + i) * hv + h;
            if (PREP) {
                const double u = (double)pp.a[at] + (double)qw_bf16(pp.dt_bias[h]);
                gi = exp(-exp((double)qw_bf16(pp.A_log[h])) * (u > 20.0 ? u : log1p(exp(u))));
                bi = (float)(1.0 / (1.0 + exp(-(double)pp.b[at])));
            } else { gi = (double)g[at]; bi = beta[at]; }
        }
        double p = 0.0, gam = 1.0;
#pragma unroll 4
        for (int t = 0; t < QG_C; t++) {
            const double gt = qg_lane(gi, t);
            const float bt = qw_lane(bi, t);
            if (t <= i) gam *= gt;
            p = t == i ? 1.0 : t > i ? p * gt : 0.0;
            if (lane < QG_C) {
                // (selects: what lies above the diagonal was never written)
                Ls[t][i] = t > i ? (float)(bt * p * KK[t][i]) : 0.0f;
                Ms[t][i] = t >= i ? (float)(p * QK[t][i]) : 0.0f;
            }
        }
        if (lane < QG_C) w.sc[hc * QG_C + i] = make_float4(bi, (float)(bi * gam), (float)gam, (float)p);
        __builtin_amdgcn_wave_barrier();
        float x[QG_C];
#pragma unroll
        for (int t = 0; t < QG_C; t++) {
            float a0 = t == i ? 1.0f : 0.0f, a1 = 0.0f;
#pragma unroll
            for (int j = 0; j < t; j += 4) {
                const float4 l = *reinterpret_cast<const float4 *>(&Ls[t][j]);
                a0 = __builtin_fmaf(-l.x, x[j], a0);
                if (j + 1 < t) a1 = __builtin_fmaf(-l.y, x[j + 1], a1);
                if (j + 2 < t) a0 = __builtin_fmaf(-l.z, x[j + 2], a0);
                if (j + 3 < t) a1 = __builtin_fmaf(-l.w, x[j + 3], a1);
            }
            x[t] = a0 + a1;
            if (lane < QG_C) Ls[t][i] = x[t];                     // T's row t takes L's place
            __builtin_amdgcn_wave_barrier();
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int f = 0; f < 4; f++) {                             // [tile][j][lane], as q and k
            const int t0 = 16 * (f >> 1), j = f & 1;
            const size_t o = (hc * 4 + f) * 64 + lane;
            reinterpret_cast<float4 *>(w.T)[o] = *reinterpret_cast<const float4 *>(&Ls[t0 + ln][16 * j + 4 * kg]);
            reinterpret_cast<float4 *>(w.QK)[o] = *reinterpret_cast<const float4 *>(&Ms[t0 + ln][16 * j + 4 * kg]);
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// A barrier for LDS that leaves the next chunk's loads in flight.
__device__ __forceinline__ void qg_sync()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Wave w of four: rows (w & 1) 16 .. of the chunk, of K for waves 0 and 1
// (which make U) and of Q for 2 and 3 (which make Y); and columns 32 w .. of
// the state, as D tiles of S' (k rows, v columns), so that a lane's four are
// a 16-byte piece of S[v][k].  16 value rows a workgroup, so that two share a
// CU and cover each other's barriers.  (32 rows, one a CU, before infinities
// were kept apart: 2048 steps 316 us against 243.)
__global__ void __launch_bounds__(256, 2) k_gdn_chunk(qg_long w, float *__restrict__ y, const float *__restrict__ v,
                                                      float *state, int hk, int hv, int rows)
{
    __shared__ __align__(16) float Ss[16][QG_CS], Ks[QG_C][QG_CS];
    __shared__ __align__(16) float Rt[16][QG_TS], Ut[16][QG_TS], Up[16][QG_TS];
    __shared__ int bad[2][16];       // by the chunk's parity
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), ln = lane & 15, kg = lane >> 4;
    // the workgroups of a key head (which read its q and k) on one XCD
    constexpr unsigned per = QG_DV / 16;
    const unsigned total = gridDim.x, b = blockIdx.x;
    const unsigned id = total % 8u == 0u ? (b % 8u) * (total / 8u) + b / 8u : b;
    const int h = (int)(id / per), v0 = 16 * (int)(id % per), hx = h / (hv / hk);
    const int nch = (rows + QG_C - 1) / QG_C, t0 = 16 * (wave & 1);
    const bool isq = wave >= 2;

    float *sp = state + ((size_t)h * QG_DV + v0 + ln) * QG_DK + 32 * wave + 4 * kg;
    qg_f4 S[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
        S[u] = *reinterpret_cast<const qg_f4 *>(sp + 16 * u);
        *reinterpret_cast<qg_f4 *>(&Ss[ln][32 * wave + 16 * u + 4 * kg]) = S[u];
    }
    // a chunk's operands, fetched a chunk ahead: 16 rows of K or Q, the rows'
    // scalars, T or the masked Q K' and (waves 0 and 1) V
    const float4 *kq = reinterpret_cast<const float4 *>(isq ? w.qn : w.kn) + ((size_t)hx * nch * 16 + t0 / 2) * 64 + lane;
    const float4 *tq = reinterpret_cast<const float4 *>(isq ? w.QK : w.T) + ((size_t)h * nch * 4 + t0 / 8) * 64 + lane;
    const float4 *sc = w.sc + (size_t)h * nch * QG_C + t0 + 4 * kg;
    float4 fa[8], ft[2], fs[4];
    float fv[4] = {}, fg;
    auto fetch = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 8; j++) fa[j] = kq[((size_t)c * 16 + j) * 64];
#pragma unroll
        for (int j = 0; j < 2; j++) ft[j] = tq[((size_t)c * 4 + j) * 64];
#pragma unroll
        for (int e = 0; e < 4; e++) fs[e] = sc[(size_t)c * QG_C + e];
        if (!isq) {
#pragma unroll
            for (int e = 0; e < 4; e++)
                fv[e] = v[((size_t)min(c * QG_C + t0 + 4 * kg + e, rows - 1) * hv + h) * QG_DV + v0 + ln];
        }
        fg = w.sc[((size_t)h * nch + c) * QG_C + QG_C - 1].z;     // G[C - 1]
    };
    if (tid < 32) (&bad[0][0])[tid] = QG_C;
    auto finite = [](float x) { return (__float_as_uint(x) & 0x7F800000u) != 0x7F800000u; };
    fetch(0);
    qg_sync();
    for (int c = 0; c < nch; c++) {
        float4 a[8], tm[2], s4[4];
        float vv[4];
#pragma unroll
        for (int j = 0; j < 8; j++) a[j] = fa[j];
#pragma unroll
        for (int j = 0; j < 2; j++) tm[j] = ft[j];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            s4[e] = fs[e];
            vv[e] = fv[e];
        }
        const float gc = fg;
        if (c + 1 < nch) fetch(c + 1);
        if (!isq) {
#pragma unroll
            for (int j = 0; j < 8; j++) *reinterpret_cast<float4 *>(&Ks[t0 + ln][16 * j + 4 * kg]) = a[j];
        }
        // K S0' or Q S0': eight chains a tile, met in a tree (here and below a
        // long chain, or one that starts on a large value, rounds more than the serial form)
        qg_f4 d;
        {
            qg_f4 dd[8];
            float4 sb[8];
#pragma unroll
            for (int j = 0; j < 8; j++) sb[j] = *reinterpret_cast<const float4 *>(&Ss[ln][16 * j + 4 * kg]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 8; j++) dd[j] = qg_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 8; j++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    dd[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(reinterpret_cast<const float *>(&a[j])[e],
                                                                 reinterpret_cast<const float *>(&sb[j])[e], dd[j], 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; e++)
                d[e] = ((dd[0][e] + dd[1][e]) + (dd[2][e] + dd[3][e])) +
                       ((dd[4][e] + dd[5][e]) + (dd[6][e] + dd[7][e]));
        }
        if (!isq) {
            qg_f4 r;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const bool in = c * QG_C + t0 + 4 * kg + e < rows;
                r[e] = in ? __builtin_fmaf(s4[e].x, vv[e], -(s4[e].y * d[e])) : 0.0f;
            }
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (!finite(r[e])) {
                    atomicMin(&bad[c & 1][ln], t0 + 4 * kg + e);
                    r[e] = 0.0f;
                }
            *reinterpret_cast<qg_f4 *>(&Rt[ln][t0 + 4 * kg]) = r;
        }
        qg_sync();
        // X over the chunk's 32 steps against T's or the masked Q K's 16 rows (upper right tile zero)
        auto over = [&](const float (*X)[QG_TS], qg_f4 &o) __attribute__((always_inline)) {
            const float4 x0 = *reinterpret_cast<const float4 *>(&X[ln][4 * kg]);
            const float4 x1 = *reinterpret_cast<const float4 *>(&X[ln][16 + 4 * kg]);
            qg_f4 p[4];
            p[0] = p[1] = p[2] = p[3] = qg_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                p[e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(reinterpret_cast<const float *>(&tm[0])[e],
                                                                reinterpret_cast<const float *>(&x0)[e], p[e & 1], 0, 0, 0);
                if (t0)
                    p[2 + (e & 1)] = __builtin_amdgcn_mfma_f32_16x16x4f32(reinterpret_cast<const float *>(&tm[1])[e],
                                                                          reinterpret_cast<const float *>(&x1)[e],
                                                                          p[2 + (e & 1)], 0, 0, 0);
            }
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] += (p[0][e] + p[1][e]) + (p[2][e] + p[3][e]);
        };
        if (tid >= 240) bad[(c + 1) & 1][tid - 240] = QG_C;   // the next chunk's
        if (!isq) {
            // U = T R
            qg_f4 u = {0.f, 0.f, 0.f, 0.f};
            over(Rt, u);
            qg_f4 up;
            const int fb = bad[c & 1][ln];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int t = t0 + 4 * kg + e;
                if (t >= fb) u[e] = __builtin_nanf("");
                up[e] = u[e] * s4[e].w;
                if (!finite(u[e])) {
                    atomicMin(&bad[c & 1][ln], t);
                    u[e] = 0.0f;
                }
            }
            *reinterpret_cast<qg_f4 *>(&Ut[ln][t0 + 4 * kg]) = u;
            *reinterpret_cast<qg_f4 *>(&Up[ln][t0 + 4 * kg]) = up;
        }
        qg_sync();
        // S' = G[C-1] S0' + K' (P U)
        {
            float4 bu[2], ka[2][2];
#pragma unroll
            for (int i = 0; i < 2; i++) bu[i] = *reinterpret_cast<const float4 *>(&Up[ln][16 * i + 4 * kg]);
#pragma unroll
            for (int u = 0; u < 2; u++)
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const int kc = 32 * wave + 16 * u + ln, r = 16 * i + 4 * kg;
                    ka[u][i] = make_float4(Ks[r][kc], Ks[r + 1][kc], Ks[r + 2][kc], Ks[r + 3][kc]);
                }
            qg_f4 ds[2];
            ds[0] = ds[1] = qg_f4{0.f, 0.f, 0.f, 0.f};
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int u = 0; u < 2; u++)
                        ds[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(reinterpret_cast<const float *>(&ka[u][i])[e],
                                                                     reinterpret_cast<const float *>(&bu[i])[e],
                                                                     ds[u], 0, 0, 0);
#pragma unroll
            for (int u = 0; u < 2; u++)
#pragma unroll
                for (int e = 0; e < 4; e++) S[u][e] = __builtin_fmaf(S[u][e], gc, ds[u][e]);
        }
        if (isq) {
            // Y = G Q S0' + (P o Q K') U
            qg_f4 o;
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = s4[e].z * d[e];
            over(Ut, o);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int t = c * QG_C + t0 + 4 * kg + e;
                const float yv = t0 + 4 * kg + e >= bad[c & 1][ln] ? __builtin_nanf("") : o[e];
                if (t < rows) y[((size_t)t * hv + h) * QG_DV + v0 + ln] = yv;
            }
        }
#pragma unroll
        for (int u = 0; u < 2; u++) *reinterpret_cast<qg_f4 *>(&Ss[ln][32 * wave + 16 * u + 4 * kg]) = S[u];
        qg_sync();
    }
#pragma unroll
    for (int u = 0; u < 2; u++) *reinterpret_cast<qg_f4 *>(sp + 16 * u) = S[u];
}

// ---- launchers ----------------------------------------------------------------

extern "C" int qwk_conv1d_causal_silu(hipStream_t s, float *y, const float *x, float *state, const uint16_t *w,
                                      int channels, int rows, int ksize, float *snap, int n_snap, int snap_stride)
{
    if (ksize != 4 || channels < 1 || rows < 0 || n_snap < 0 || (n_snap > 0 && (!snap || snap_stride < 3 * channels)))
        return hipErrorInvalidValue;
    if (rows == 0) return 0;
    hipLaunchKernelGGL(k_conv1d_causal_silu<4>, dim3((channels + 255) / 256, (rows + QG_CONV_T - 1) / QG_CONV_T),
                       dim3(256), 0, s, y, x, state, w,
                       channels, rows, snap, n_snap, snap_stride);
    return (int)hipGetLastError();
}

extern "C" int qwk_gdn_decode(hipStream_t s, float *y, const float *x, const float *win, float *wout,
                              const uint16_t *w, const qwk_gdn_prep *prep, float *state, int hk, int hv, int dk,
                              int dv)
{
    if (dk != QG_DK || dv != QG_DV || hk < 1 || hv < 1 || hv % hk || !prep || !x || !win || !wout || !w)
        return hipErrorInvalidValue;
    const int channels = 2 * hk * dk + hv * dv;
    const qg_prep pp = { prep->a, prep->b, prep->A_log, prep->dt_bias, prep->l2eps, prep->q_scale, prep->k_scale,
                         nullptr, nullptr };
    const qg_conv cv = { x, win, wout, w, channels };
    hipLaunchKernelGGL((k_gated_delta<true, true>), dim3(hv * (QG_DV / QG_ROWS_PER_WG)), dim3(QG_THREADS), 0, s, y,
                       nullptr, nullptr, nullptr, nullptr, nullptr, state, hk, hv, 1, nullptr, 0, 0, pp, cv);
    return (int)hipGetLastError();
}

extern "C" int qwk_gdn_gates(hipStream_t s, float *g, float *beta, const float *a, const float *b,
                             const uint16_t *A_log, const uint16_t *dt_bias, int hv, int rows)
{
    if (hv < 1 || rows < 0) return hipErrorInvalidValue;
    const int n = hv * rows;
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_gdn_gates, dim3((n + 255) / 256), dim3(256), 0, s, g, beta, a, b, A_log, dt_bias, hv, n);
    return (int)hipGetLastError();
}

// Whether a call takes the chunks, and its scratch: a function of the shape.
static bool qg_is_long(int hk, int hv, int rows, int n_snap)
{
    return rows >= QG_LONG_MIN_ROWS && n_snap == 0 && hk >= 1 && hv >= hk && hv % hk == 0;
}

extern "C" size_t qwk_gated_delta_work(int hk, int hv, int rows, int prep, int n_snap)
{
    if (qg_is_long(hk, hv, rows, n_snap))
        return qg_long_bytes(hk, hv, rows < QG_LONG_ROWS ? rows : QG_LONG_ROWS, nullptr, nullptr);
    if (!prep || rows < QG_PRE_MIN_ROWS || hk < 1 || hv < 1) return 0;
    return ((size_t)rows * hk * 2 + (size_t)rows * hv * 2) * sizeof(float);
}

extern "C" int qwk_gated_delta(hipStream_t s, float *y, const float *q, const float *k, const float *v,
                               const float *g, const float *beta, float *state, int hk, int hv, int dk, int dv,
                               int rows, float *snap, int n_snap, int snap_stride, const qwk_gdn_prep *prep,
                               void *work)
{
    if (dk != QG_DK || dv != QG_DV || hk < 1 || hv < 1 || hv % hk || rows < 0 || n_snap < 0 ||
        (n_snap > 0 && (!snap || snap_stride < hv * dv * dk || snap_stride % 4)))
        return hipErrorInvalidValue;
    if (rows == 0) return 0;
    const dim3 grid(hv * (QG_DV / QG_ROWS_PER_WG));
    if (work && qg_is_long(hk, hv, rows, n_snap)) {
        for (int r0 = 0; r0 < rows; r0 += QG_LONG_ROWS) {
            const int r = rows - r0 < QG_LONG_ROWS ? rows - r0 : QG_LONG_ROWS;
            const size_t oq = (size_t)r0 * hk * QG_DK, ov = (size_t)r0 * hv * QG_DV, og = (size_t)r0 * hv;
            qg_long w;
            qg_long_bytes(hk, hv, r, &w, static_cast<char *>(work));
            const dim3 pre((r + QG_C - 1) / QG_C, hk);
            if (prep) {
                const qg_prep pp = { prep->a + og, prep->b + og, prep->A_log, prep->dt_bias, prep->l2eps, prep->q_scale,
                                     prep->k_scale, nullptr, nullptr };
                hipLaunchKernelGGL(k_gdn_chunk_pre<true>, pre, dim3(256), 0, s, w, q + oq, k + oq, nullptr, nullptr, hk,
                                   hv, r, pp);
            } else {
                const qg_prep pp = {};
                hipLaunchKernelGGL(k_gdn_chunk_pre<false>, pre, dim3(256), 0, s, w, q + oq, k + oq, g + og, beta + og,
                                   hk, hv, r, pp);
            }
            hipLaunchKernelGGL(k_gdn_chunk, dim3(hv * (QG_DV / 16)), dim3(256), 0, s, w, y + ov, v + ov, state, hk, hv, r);
        }
        return (int)hipGetLastError();
    }
    if (prep) {
        qg_prep pp = { prep->a, prep->b, prep->A_log, prep->dt_bias, prep->l2eps, prep->q_scale, prep->k_scale,
                       nullptr, nullptr };
        if (work && rows >= QG_PRE_MIN_ROWS) {
            pp.nrm = static_cast<float *>(work);
            pp.gb = pp.nrm + (size_t)rows * hk * 2;
            const int nbv = (rows * hk * 2 + 3) / 4, nbg = (rows * hv + 255) / 256;
            hipLaunchKernelGGL(k_gdn_pre, dim3(nbv + nbg), dim3(256), 0, s, pp, q, k, hk, hv, rows);
        }
        hipLaunchKernelGGL(k_gated_delta<true>, grid, dim3(QG_THREADS), 0, s, y, q, k, v, nullptr, nullptr, state,
                           hk, hv, rows, snap, n_snap, snap_stride, pp);
    } else {
        const qg_prep pp = {};
        hipLaunchKernelGGL(k_gated_delta<false>, grid, dim3(QG_THREADS), 0, s, y, q, k, v, g, beta, state, hk, hv,
                           rows, snap, n_snap, snap_stride, pp);
    }
    return (int)hipGetLastError();
}
