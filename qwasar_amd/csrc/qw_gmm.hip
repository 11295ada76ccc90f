// qw_gmm.hip -- the 4-bit products over many rows, on gfx950 MFMA: the dense
// projection (qw_op_qmm_q4) and the grouped per-expert product of the
// reference's op sequence (qw_op_qmm_q4_gather).  One kernel, two steps:
//
//   k_xstage  the activation rows once as f16 (and each quantisation group's
//             sum), so that the product's many column blocks do not convert
//             them again
//   k_xgemm   the product
//
// Exactness of the weight operand.  A nibble q enters the MFMA as the f16
// denormal q 2^-24 (nibbles 0, 2, 4, 6 of a word) or q 2^-20 (nibbles 1, 3,
// 5, 7), which is the masked word itself: two ands, a shift, two ands a word
// and no rounding (gfx950's f16 MFMA multiplies denormals exactly).  The
// staged activations at the odd positions are 2^-4 of the others', so all
// products of a group carry one scale.  The group's scale is applied to the
// fp32 partial of its MFMAs:
//
//   y = sum_g s_g C_g + sum_g b_g X_g,   C_g = sum q x,   X_g = sum x,
//
// and the second sum is a product of its own: the biases (bf16, as stored)
// against X_g cut into three bf16 parts (24 bits: exactly), 16 groups' parts
// in two bf16 MFMAs.  So the weights enter with no rounding at all;
// activations are rounded to f16, the only approximation: a relative error of
// 2^-11 for elements down to 2^-29 of their row's largest (even positions) or
// 2^-25 (odd ones), and 2^-39 (2^-35) of that largest below.  (Unscaled f16,
// which small products still take, has 2^-11 from 2^-14 on, whatever the row:
// finer for odd elements of rows whose largest is above 2^11, and nothing
// above 65504.)
//
// k order within an MFMA.  The masks leave a word's nibbles in register order
// 0,4,1,5,2,6,3,7; the stage stores every 8-element block in that order.
//
// What bounds it.  Dense, many rows: the vector unit's work beside the matrix
// cores (per 64 k of a 16-column tile of a 64-row wave: 8 MFMAs of 16 cycles
// against 16 multiply-adds for the scale and 10 operations for the masks; the
// two units overlap by about half, as a loop of nothing else shows), so the
// product runs at about half of a matrix library's f16 rate.  1024 x 3072 x
// 10240: 96 us a call (670 TFLOP/s), where 64 x 64 tiles that converted the
// activations in every column block and put 1024 + q through the MFMA took
// 275.  Timing builds: without the loads of the stages 80 us, without their
// arithmetic 50.  Experts with few pairs: requests to L1.  A load of 64 lanes
// over 16 rows touches 16 lines, whatever it fetches, so the scales (and for
// narrow tiles the biases) come as one flat run of the block's columns, and
// the weights 128 bytes of a column a load where a tile is narrow: gate, up
// and down of 512 experts of 640 x 2560, 6 pairs each, 1650 -> 420 us.
// Both operands go straight to LDS (global_load_lds, 16-byte pieces, no
// registers), NST - 1 stages ahead, one barrier a stage, two workgroups a CU.
// Tried: every LDS read of a stage ahead of its MFMAs, and MFMAs interleaved
// with the vector work by hand: no faster (90 and 93 us the kernel).
#include "qw_device.h"
#include "qw_kernels.h"

#include <cfloat>
#include <climits>
#include <cmath>
#include <type_traits>

typedef _Float16 qw_h8 __attribute__((ext_vector_type(8)));
typedef __bf16 qw_b8 __attribute__((ext_vector_type(8)));
typedef float qw_f4 __attribute__((ext_vector_type(4)));

#define QX_KPAD 256              // staged rows are padded with zeros to a multiple of this
#define QX_SB 16                 // groups a block of the staged sums
#define QX_SLICE 8               // a slice of k is a multiple of this many groups
#define QX_SLOTS 512             // workgroups the chip holds at two a CU
#define QX_WIDE_K 1024           // rows of at least this many elements are staged by a workgroup each
#define QX_CHUNK_ROWS 8192       // rows a dense call stages at a time (bounds its scratch)

// ---- staging -------------------------------------------------------------------

// The power of two that puts a row's largest magnitude m in [2^14, 2^15).
__device__ __forceinline__ int qx_shift(float m)
{
    if (!(m > 0.0f && m <= FLT_MAX)) return 0;
    const int sh = 15 - __builtin_amdgcn_frexp_expf(m);
    return sh < -126 ? -126 : sh > 126 ? 126 : sh;
}

// W waves a row (one under QX_WIDE_K elements, else the workgroup's four: a
// lane's blocks of 8 stay in registers up to NI of them, so the row is read
// once).  The row is scaled by one power of two 2^sh that puts its largest
// magnitude in [2^14, 2^15), so no input overflows f16; ex gets 24 - sh, the
// exponent the product's sums are scaled back by (24 from the denormal
// nibbles).  xp holds a row's sums of the staged values 2^-24, 16 groups at a
// time: [block][part 0..2, zeros][16].  1021 rows of 12288: a wave a row and
// two reads took 24 us.
template <int G, int W, int NI>
__global__ __launch_bounds__(256) void k_xstage(_Float16 *__restrict__ ah, uint16_t *__restrict__ xp,
                                                int *__restrict__ ex, const float *__restrict__ x, int rows, int k,
                                                int kp, int nsb)
{
    constexpr int L = 64 * W;                                    // lanes a row
    __shared__ float wm[4];
    const int row = W == 1 ? blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x, lane = threadIdx.x & (L - 1);
    if (W == 1 && row >= rows) return;
    const int nb = k / 8, ng = k / G;
    const float4 *xr = reinterpret_cast<const float4 *>(x + (size_t)row * k);
    const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 v[NI][2];
    float m = 0.0f;
    auto top = [&](float4 lo, float4 hi) {
        m = fmaxf(m, fmaxf(fmaxf(fabsf(lo.x), fabsf(lo.y)), fmaxf(fabsf(lo.z), fabsf(lo.w))));
        m = fmaxf(m, fmaxf(fmaxf(fabsf(hi.x), fabsf(hi.y)), fmaxf(fabsf(hi.z), fabsf(hi.w))));
    };
#pragma unroll
    for (int i = 0; i < NI; i++) {
        // (every load issued, at a clamped place: a guarded one would be a branch and a wait)
        const int b = min(lane + i * L, nb - 1);
        v[i][0] = xr[2 * b];
        v[i][1] = xr[2 * b + 1];
    }
#pragma unroll
    for (int i = 0; i < NI; i++) {
        if (lane + i * L >= nb) v[i][0] = v[i][1] = z4;
        top(v[i][0], v[i][1]);
    }
    for (int b = lane + NI * L; b < nb; b += L) top(xr[2 * b], xr[2 * b + 1]);
    m = qw_wave_max(m);
    if (W > 1) {
        if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
        __syncthreads();
        m = fmaxf(fmaxf(wm[0], wm[1]), fmaxf(wm[2], wm[3]));
    }
    const int sh = qx_shift(m);
    if (lane == 0) ex[row] = 24 - sh;
    const float up = __builtin_ldexpf(1.0f, sh), up4 = __builtin_ldexpf(1.0f, sh - 4);
    qw_h8 *hr = reinterpret_cast<qw_h8 *>(ah + (size_t)row * kp);
    uint16_t *xr16 = xp + (size_t)row * nsb * 64;
    // (kp / 8 is a multiple of 32, so a group's G / 8 lanes are in or out together)
    auto block = [&](int b, float4 lo, float4 hi) {
        const float f[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        _Float16 q[8];
        float even = 0.0f, odd = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            q[j] = (_Float16)(f[j] * ((j & 1) ? up4 : up));
            if (j & 1) odd += (float)q[j];
            else even += (float)q[j];
        }
        hr[b] = qw_h8{q[0], q[4], q[1], q[5], q[2], q[6], q[3], q[7]};
        const float sum = qw_xor_sum<G / 8>(__builtin_fmaf(odd, 16.0f, even));
        const int g = b / (G / 8);
        if (b % (G / 8) == 0 && g < ng) {
            float r = sum * 0x1p-24f;
#pragma unroll
            for (int p = 0; p < 3; p++) {
                const uint32_t hi16 = __float_as_uint(r) & 0xFFFF0000u;
                xr16[(g / QX_SB) * 64 + p * QX_SB + g % QX_SB] = (uint16_t)(hi16 >> 16);
                r -= __uint_as_float(hi16);
            }
        }
    };
#pragma unroll
    for (int i = 0; i < NI; i++)
        if (lane + i * L < kp / 8) block(lane + i * L, v[i][0], v[i][1]);
    for (int b = lane + NI * L; b < kp / 8; b += L) block(b, b < nb ? xr[2 * b] : z4, b < nb ? xr[2 * b + 1] : z4);
    for (int i = lane; i < nsb * 64; i += L)
        if ((i & 63) >= 3 * QX_SB || (i >> 6) * QX_SB + (i & 15) >= ng) xr16[i] = 0;
}

// ---- the product ---------------------------------------------------------------------

struct QxArgs {
    float *y;
    const _Float16 *ah;      // [source rows, kp]
    const uint16_t *xp;      // [source rows, nsb * 64]
    const int *ex;           // [source rows]
    const int32_t *perm, *tiles;
    const uint32_t *w;
    const uint16_t *s, *b;
    int k, n, kp, nsb;
    int K, x_by_pair;        // grouped: the source row of pair p is x_by_pair ? p : p / K
    int rows;                // dense: rows
    int nblk, nbw;           // column blocks, and how many of them a workgroup runs back to back
    int kslice;              // k range of a blockIdx.y slice (whole stages, a multiple of QX_SLICE groups; k: no split)
    float *part;             // dense split-K: slice s writes part[s][rows][n]
};

// 16 bytes a lane from its own address straight into LDS at lds + 16 lane.
// Written as asm because the compiler, which cannot tell the ring's stages
// apart, waits for every such load before any LDS read; the waits on the
// vector memory counter in k_xgemm are this kernel's own.  (m0 is an operand, so
// the compiler knows of it; the instruction may not follow its write at once.)
__device__ __forceinline__ void qx_dma(uint32_t lds, const void *src)
{
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"{m0}"(lds), "v"(src) : "memory");
}

template <int N>
__device__ __forceinline__ void qx_wait()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// A workgroup: WM x WN waves, each MT x NT tiles of 16 x 16; k in stages of
// BK through a ring of NST in LDS.
//
// LDS layouts (a 16-byte piece is the unit a lane loads):
//   activations  [BM][BK]: piece p of row r at p ^ (r % 8), so the 8 lanes
//                that read one piece of 8 rows hit different banks
//   weights      [BN][BK / 8 words]: pieces of 4 words, swizzled by the
//                column for BK 128 and 256 alike
//   scales       [BN][groups] bf16, as in memory; [BN][SGL] at a time where
//                a row has more than SGL groups
// The swizzles are in the addresses a lane loads from, since the loads fill
// LDS in lane order.
template <int G, int MT, int NT, int WM, int WN, int BK, int NST, int SGL, bool GATHER>
__global__ __launch_bounds__(64 * WM * WN, 2) void k_xgemm(QxArgs a)
{
    constexpr int NW = WM * WN, BM = WM * MT * 16, BN = WN * NT * 16, THREADS = 64 * NW;
    constexpr int APR = BK / 8, WPR = BK / 32;                   // pieces a row / a column
    constexpr int ASZ = BM * BK * 2, WSZ = BN * BK / 2, STG = ASZ + WSZ;
    constexpr int AI = ASZ / 1024 / NW, WT = WSZ / 1024;         // loads a stage: a wave's of A, all of W
    constexpr int WI = (WT + NW - 1) / NW, WR = WT % NW;         // a wave's of W (waves from WR on one fewer)
    static_assert(ASZ % (1024 * NW) == 0 && WSZ % 1024 == 0 && BK % 64 == 0 && (SGL * G) % BK == 0 && SGL % 8 == 0,
                  "whole loads and whole stages");
    static_assert((AI + WI) * (NST - 2) < 64, "the wait's counter");
    __shared__ __align__(16) uint8_t ring[NST * STG];
    __shared__ __align__(16) uint16_t Sc[(BN * SGL + 511) / 512 * 512];
    __shared__ int rows_s[GATHER ? 2 * BM : 1];

    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
    const int ln = lane & 15, kg = lane >> 4;
    const int wm = wave / WN, wn = wave % WN;

    // Workgroup b runs on XCD b % 8: each XCD takes a contiguous run of the
    // items.  Grouped, an expert's column blocks are adjacent (they share its
    // activation rows); dense, a column block's row tiles are (they share its
    // weights).  The grouped grid is an upper bound: the run is cut from the
    // tiles there are.
    const int ntl = GATHER ? a.tiles[0] : (a.rows + BM - 1) / BM;
    const int ngr = (a.nblk + a.nbw - 1) / a.nbw, items = ntl * ngr, per = items >> 3, rem = items & 7;
    const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
    if (j >= per + (xcd < rem ? 1 : 0)) return;
    const int v = xcd * per + min(xcd, rem) + j;
    const int tile = GATHER ? v / ngr : v % ntl, nb0 = (GATHER ? v % ngr : v / ntl) * a.nbw;
    const int nb1 = min(nb0 + a.nbw, a.nblk);

    int expert = 0, first, len;
    if (GATHER) {
        expert = a.tiles[1 + 3 * tile];
        first = a.tiles[2 + 3 * tile];
        len = a.tiles[3 + 3 * tile];
        // source and destination of each tile row; rows past the tile's read its first again
        for (int m = t; m < BM; m += THREADS) {
            const int p = a.perm[first + (m < len ? m : 0)];
            rows_s[m] = a.x_by_pair ? p : p / a.K;
            rows_s[BM + m] = p;
        }
        __syncthreads();
    } else {
        first = tile * BM;
        len = min(BM, a.rows - first);
    }
    auto src_row = [&](int m) { return GATHER ? rows_s[m] : first + min(m, len - 1); };

    const int k = a.k, n = a.n, words = k / 8, groups = k / G;
    const int kb = (int)blockIdx.y * a.kslice, ke = min(k, kb + a.kslice), T = (ke - kb + BK - 1) / BK;
    // the slice's groups; it starts and ends at a multiple of 8 (or at the row's end), so a lane's 8 biases are in or out
    const int gb = GATHER ? 0 : kb / G, ge = GATHER ? groups : (ke + G - 1) / G;
    const uint32_t *wb = a.w + (size_t)expert * n * words;
    const uint16_t *sb = a.s + (size_t)expert * n * groups;
    const uint16_t *bb = a.b + (size_t)expert * n * groups;
    // how the scales come (uniform): a flat copy of the block's columns, 8
    // groups of a column a load, or one by one; the last two also the biases
    const bool wide = groups % 8 == 0 && (((uintptr_t)sb | (uintptr_t)bb) & 15) == 0;
    const bool flat = groups <= SGL && ((uintptr_t)sb & 15) == 0 && (n * (long)groups) % 8 == 0;
    // groups a column in Sc; one by one no more than a split product's slice has
    const int sld = GATHER || flat || wide ? min(groups, SGL) : min(min(groups, SGL), a.kslice / G);

    // ---- this lane's loads -----------------------------------------------------------
    const _Float16 *asrc[AI];
    const uint32_t *wrow[WI];
    int wpc[WI];
#pragma unroll
    for (int i = 0; i < AI; i++) {
        const int slot = (wave * AI + i) * 64 + lane, r = slot / APR, p = slot % APR;
        asrc[i] = a.ah + (size_t)src_row(r) * a.kp + kb + 8 * (p ^ (r & 7));
    }
#pragma unroll
    for (int i = 0; i < WI; i++) {
        const int slot = ((wave + NW * i) * 64 + lane) % (BN * WPR), c = slot / WPR, p = slot % WPR;
        wpc[i] = WPR == 2 ? p : WPR == 4 ? p ^ ((c >> 1) & 3) : p ^ (c & 7);
    }
    int n0;                                                      // the block's first column
    const uint32_t ring0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)&ring[0];
    const bool fewer = WR != 0 && wave >= WR;                    // this wave has one W load less
    auto issue = [&](int i) {
        const uint32_t st = ring0 + (uint32_t)(i % NST) * STG;
        const int k0 = kb + i * BK;
#pragma unroll
        for (int u = 0; u < AI; u++) qx_dma(st + (wave * AI + u) * 1024, asrc[u] + i * BK);
#pragma unroll
        for (int u = 0; u < WI; u++) {
            if (u == WI - 1 && fewer) break;
            // a piece past the row's end (k not a multiple of BK) meets zeros of A: any piece of the row will do
            const int pc = k0 / 32 + wpc[u];
            qx_dma(st + ASZ + (wave + NW * u) * 1024, wrow[u] + 4 * (pc < words / 4 ? pc : 0));
        }
    };
    auto landed = [&](int ahead) {       // all but the latest `ahead` stages' loads of this wave are in LDS
        if (ahead >= 2 && NST >= 4) {
            if (fewer) qx_wait<(NST >= 4 ? 2 : 0) * (AI + WI - 1)>();
            else qx_wait<(NST >= 4 ? 2 : 0) * (AI + WI)>();
        } else if (ahead == 1 && NST >= 3) {
            if (fewer) qx_wait<AI + WI - 1>();
            else qx_wait<AI + WI>();
        } else {
            qx_wait<0>();
        }
    };

    // the narrow tiles' biases come to LDS too (in place of a stage)
    static_assert(NST != 2 || STG >= (BN * SGL * 2 + 1023) / 1024 * 1024, "the biases' place");
    const bool lds_bias = NST == 2 && flat && ((uintptr_t)bb & 15) == 0;
    const uint32_t sc0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t *)&Sc[0];
    // the block's columns of the scales or biases as one run; pieces past the
    // bank's last column read its last 8 values again
    auto load_flat = [&](uint32_t to, const uint16_t *from) {
        const long end = (long)n * groups - 8;
        for (int i = wave; i * 512 < BN * groups; i += NW)
            qx_dma(to + i * 1024, from + min((long)n0 * groups + i * 512 + lane * 8, end));
    };
    auto load_bias = [&](uint32_t to) { load_flat(to, bb); };
    auto load_scales = [&](int g0) {
        if (flat) {
            load_flat(sc0, sb);
        } else if (wide) {
            for (int i = wave; i * 512 < BN * SGL; i += NW) {
                const int e = i * 512 + lane * 8, c = min(e / SGL, BN - 1), g = g0 + e % SGL;
                qx_dma(sc0 + i * 1024, sb + (size_t)min(n0 + c, n - 1) * groups + (g < groups ? g : 0));
            }
        } else {
            if constexpr (GATHER) {
                // (only a bank off a 16-byte boundary, or an odd one of more than SGL groups)
                for (int i = t; i < BN * sld; i += THREADS) {
                    const int c = i / sld, g = g0 + i % sld;
                    Sc[i] = g < groups ? sb[(size_t)min(n0 + c, n - 1) * groups + g] : 0;
                }
            } else {
                // LB in flight: one at a time, 128 columns of 96 groups were 48
                // trips to memory in a row (16 x 4160 x 6144, groups of 32: 42.8
                // -> 32.4 us a call).  Their places are stepped to: with a
                // division each, calls that never come here ran up to 7% longer
                constexpr int LB = MT * NT > 12 ? 4 : 8;
                const int dc = THREADS / sld, dg = THREADS % sld;
                int c = t / sld, g = t % sld;
                for (int i0 = t; i0 < BN * sld; i0 += LB * THREADS) {
                    uint16_t v[LB];
#pragma unroll
                    for (int u = 0; u < LB; u++) {
                        const uint16_t x = sb[(size_t)min(n0 + c, n - 1) * groups + min(g0 + g, groups - 1)];
                        v[u] = g0 + g < groups ? x : 0;
                        c += dc;
                        g += dg;
                        if (g >= sld) { g -= sld; c++; }
                    }
#pragma unroll
                    for (int u = 0; u < LB; u++)
                        if (i0 + u * THREADS < BN * sld) Sc[i0 + u * THREADS] = v[u];
                }
            }
        }
    };
    // a block's scales and first stages on their way
    auto begin = [&](int nb) {
        n0 = nb * BN;
#pragma unroll
        for (int i = 0; i < WI; i++) {
            const int slot = ((wave + NW * i) * 64 + lane) % (BN * WPR), c = slot / WPR;
            wrow[i] = wb + (size_t)min(n0 + c, n - 1) * words;
        }
        load_scales(kb / G);
        for (int i = 0; i < min(NST - 1, T); i++) issue(i);
    };
    begin(nb0);
    // the rows' exponents, all at once and before the stages (after them each was a trip to memory of its own)
    int ex[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int e = 0; e < 4; e++) ex[mt][e] = a.ex[src_row((wm * MT + mt) * 16 + 4 * kg + e)];

    // 16-row tiles of up to XS blocks of 16 groups keep their group sums for every block
    constexpr int XS = MT == 1 ? 5 : 1;
    const bool held = MT == 1 && a.nsb <= XS && kb == 0;
    uint4 xa[XS][MT][2] = {};
    if (lds_bias && held) {
#pragma unroll
        for (int u = 0; u < XS; u++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const uint4 *p = reinterpret_cast<const uint4 *>(
                    a.xp + (size_t)src_row((wm * MT + mt) * 16 + ln) * a.nsb * 64 + min(u, a.nsb - 1) * 64 + 8 * kg);
                xa[u][mt][0] = p[0];
                xa[u][mt][1] = p[4];
            }
    }

    for (int nb = nb0; nb < nb1; nb++) {
    qw_f4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[mt][nt] = qw_f4{0.f, 0.f, 0.f, 0.f};

    // ---- the biases' product, 16 groups at a time ------------------------------------
    // from memory, under the first stages' trip
    if (!lds_bias) {
        const uint16_t *xr[MT];
#pragma unroll
        for (int mt = 0; mt < MT; mt++) xr[mt] = a.xp + (size_t)src_row((wm * MT + mt) * 16 + ln) * a.nsb * 64 + 8 * kg;
        for (int sblk = gb / QX_SB; sblk * QX_SB < ge; sblk++) {
            uint4 bf[NT], af[MT][2];
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const int c = min(n0 + (wn * NT + nt) * 16 + ln, n - 1), g = sblk * QX_SB + 8 * (kg & 1);
                // (every load issued, at a clamped place; what is not of the slice's groups is zeroed after)
                const bool in = g >= gb && g < ge;
                const uint16_t *p = bb + (size_t)c * groups;
                if (wide) {
                    bf[nt] = *reinterpret_cast<const uint4 *>(p + (g < groups ? g : 0));
                    if (!in) bf[nt] = make_uint4(0, 0, 0, 0);
                } else if (groups % 4 == 0 && ((uintptr_t)bb & 7) == 0) {
                    const uint2 u = *reinterpret_cast<const uint2 *>(p + min(g, groups - 4));
                    const uint2 w = *reinterpret_cast<const uint2 *>(p + min(g + 4, groups - 4));
                    const bool hi = in && g + 4 < groups;
                    bf[nt] = make_uint4(in ? u.x : 0u, in ? u.y : 0u, hi ? w.x : 0u, hi ? w.y : 0u);
                } else {
                    uint32_t o[8];
#pragma unroll
                    for (int e = 0; e < 8; e++) o[e] = p[min(g + e, groups - 1)];
#pragma unroll
                    for (int e = 0; e < 8; e++) o[e] = in && g + e < groups ? o[e] : 0u;
                    bf[nt] = make_uint4(o[0] | o[1] << 16, o[2] | o[3] << 16, o[4] | o[5] << 16, o[6] | o[7] << 16);
                }
            }
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const uint4 *p = reinterpret_cast<const uint4 *>(xr[mt] + sblk * 64);
                af[mt][0] = p[0];
                af[mt][1] = p[4];
            }
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
#pragma unroll
                    for (int mt = 0; mt < MT; mt++)
                        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(qw_b8, af[mt][h]),
                                                                             __builtin_bit_cast(qw_b8, bf[nt]),
                                                                             acc[mt][nt], 0, 0, 0);
        }
    }

    // ---- the stages ----------------------------------------------------------------------
    // A MFMA step is 32 k of one group: with 64-wide groups lane group kg
    // holds k 16 kg .. 16 kg + 15 of the 64 (words and pieces 2 kg, 2 kg + 1,
    // one a step); with 32-wide ones k 8 kg .. of each 32 (word 4 s + kg).
    auto stage = [&](int i) {
        const uint8_t *As = ring + (size_t)(i % NST) * STG, *Ws = As + ASZ;
        const int gl = ((kb + i * BK) / G - (flat ? 0 : kb / G)) % SGL;   // the stage's first group in Sc
        // (past the row's last group, where A is zero: the last one's again)
        auto scale = [&](int c, int g) { return qw_bf16(Sc[c * sld + min(g, sld - 1)]); };
#pragma unroll
        for (int sub = 0; sub < BK / 64; sub++) {
            qw_h8 af[MT][2];
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const int p = sub * 8 + (G == 32 ? 4 * s + kg : 2 * kg + s);
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
                    const int r = (wm * MT + mt) * 16 + ln;
                    af[mt][s] = *reinterpret_cast<const qw_h8 *>(As + r * (BK * 2) + ((p ^ (r & 7)) * 16));
                }
            }
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const int c = (wn * NT + nt) * 16 + ln;
                const int sw = WPR == 2 ? 0 : WPR == 4 ? (c >> 1) & 3 : c & 7;
                const uint8_t *wr = Ws + c * (BK / 2);
                uint32_t w[2];
                if (G == 32) {
#pragma unroll
                    for (int s = 0; s < 2; s++)
                        w[s] = *reinterpret_cast<const uint32_t *>(wr + ((sub * 2 + s) ^ sw) * 16 + kg * 4);
                } else {
                    const uint2 u = *reinterpret_cast<const uint2 *>(wr + ((sub * 2 + (kg >> 1)) ^ sw) * 16 + (kg & 1) * 8);
                    w[0] = u.x;
                    w[1] = u.y;
                }
                qw_h8 bf[2];
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    const uint32_t w8 = w[s] >> 8;
                    const uint4 d = make_uint4(w[s] & 0x000F000Fu, w[s] & 0x00F000F0u, w8 & 0x000F000Fu, w8 & 0x00F000F0u);
                    bf[s] = __builtin_bit_cast(qw_h8, d);
                }
                const qw_f4 z = {0.f, 0.f, 0.f, 0.f};
                if (G == 32) {
#pragma unroll
                    for (int s = 0; s < 2; s++) {
                        const float sc = scale(c, gl + sub * 2 + s);
                        qw_f4 C[MT];
#pragma unroll
                        for (int mt = 0; mt < MT; mt++) C[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[mt][s], bf[s], z, 0, 0, 0);
#pragma unroll
                        for (int mt = 0; mt < MT; mt++)
#pragma unroll
                            for (int e = 0; e < 4; e++) acc[mt][nt][e] = __builtin_fmaf(sc, C[mt][e], acc[mt][nt][e]);
                    }
                } else {
                    const float sc = scale(c, gl + sub * 64 / G);
                    qw_f4 C[MT];
#pragma unroll
                    for (int mt = 0; mt < MT; mt++) C[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[mt][0], bf[0], z, 0, 0, 0);
#pragma unroll
                    for (int mt = 0; mt < MT; mt++) C[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[mt][1], bf[1], C[mt], 0, 0, 0);
#pragma unroll
                    for (int mt = 0; mt < MT; mt++)
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[mt][nt][e] = __builtin_fmaf(sc, C[mt][e], acc[mt][nt][e]);
                }
            }
        }
    };
    for (int i = 0; i < T; i++) {
        if (!flat && i > 0 && (i * BK) % (SGL * G) == 0) {       // every wave is done with the last SGL groups' scales
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            load_scales((kb + i * BK) / G);
            qx_wait<0>();
        }
        landed(min(NST - 2, T - 1 - i));
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        // stage i is in LDS, and every wave is done with stage i - 1, whose place stage i + NST - 1 takes
        if (i + NST - 1 < T) issue(i + NST - 1);
        else if (i + NST - 1 == T && lds_bias) load_bias(ring0 + (uint32_t)(T % NST) * STG);
        stage(i);
    }
    // narrow tiles: the biases came to LDS as stage T, in one flat copy (read
    // by every wave from memory they were as many requests as the weights)
    if (lds_bias) {
        qx_wait<0>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const uint16_t *Bs = reinterpret_cast<const uint16_t *>(ring + (size_t)(T % NST) * STG);
#pragma unroll 1
        for (int sblk = gb / QX_SB; sblk * QX_SB < ge; sblk++) {
            const int g = sblk * QX_SB + 8 * (kg & 1);
            uint4 xf[MT][2];
            if (held) {
#pragma unroll
                for (int q = 0; q < XS; q++)
                    if (q == sblk) {
#pragma unroll
                        for (int mt = 0; mt < MT; mt++) { xf[mt][0] = xa[q][mt][0]; xf[mt][1] = xa[q][mt][1]; }
                    }
            } else {
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
                    const uint4 *p = reinterpret_cast<const uint4 *>(
                        a.xp + (size_t)src_row((wm * MT + mt) * 16 + ln) * a.nsb * 64 + sblk * 64 + 8 * kg);
                    xf[mt][0] = p[0];
                    xf[mt][1] = p[4];
                }
            }
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const uint16_t *p = Bs + ((wn * NT + nt) * 16 + ln) * groups;
                uint32_t o[8];
#pragma unroll
                for (int e = 0; e < 8; e++) o[e] = p[min(g + e, groups - 1)];
#pragma unroll
                for (int e = 0; e < 8; e++) o[e] = g >= gb && g + e < ge ? o[e] : 0u;
                const uint4 bf = make_uint4(o[0] | o[1] << 16, o[2] | o[3] << 16, o[4] | o[5] << 16, o[6] | o[7] << 16);
#pragma unroll
                for (int h = 0; h < 2; h++)
#pragma unroll
                    for (int mt = 0; mt < MT; mt++)
                        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(qw_b8, xf[mt][h]),
                                                                             __builtin_bit_cast(qw_b8, bf),
                                                                             acc[mt][nt], 0, 0, 0);
            }
        }
    }

    // every wave is done with the ring and the scales: the next block's are
    // on their way while this one's results leave
    const int c0 = n0;
    if (nb + 1 < nb1) {
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        begin(nb + 1);
    }
    float *yo = !GATHER && a.part ? a.part + (size_t)blockIdx.y * a.rows * n : a.y;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int m = (wm * MT + mt) * 16 + 4 * kg + e;
            if (m >= len) continue;
            float *yr = yo + (size_t)(GATHER ? rows_s[BM + m] : first + m) * n;
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const int c = c0 + (wn * NT + nt) * 16 + ln;
                if (c < n) yr[c] = __builtin_ldexpf(acc[mt][nt][e], ex[mt][e]);
            }
        }
    }
}

// ---- small products ------------------------------------------------------------
//
// Where the whole product is a few microseconds, the stage's launch costs more
// than it saves (8 rows, 3072 x 512: 23.2 us a call against 25.7): one launch
// that converts the activations as it stages them, four waves a workgroup, a
// tile of BM rows against 64 columns.  A nibble enters as the f16 1024 + q
// (exact); the group's map is applied to the fp32 partial:
//   sum_i (s q_i + b) x_i = s C_g + (b - 1024 s) X_g,
//   C_g = sum_i (1024 + q_i) x_i,   X_g = sum_i x_i.
// Grouped, it takes short k (qwk_gather_gemm_small); and as it needs no
// scratch, the calls of either kind that would be staged but for scratch that
// cannot be had.
#define QW_GMM_BN 64
#define QW_GMM_BK 128
#define QW_GMM_THREADS 256
#define QW_GMM_APAD 8            // halves of padding per A row
#define QW_GMM_BSTRIDE 18        // words per B row in LDS (16 + 2: conflict-free b32 reads)

struct QwGmmArgs {
    float *y;
    const float *x;
    qwk_q4 m;
    int k, n, rows, nblk;
    int kslice;      // k range of a blockIdx.y slice (k: no split)
    float *part;     // split-K: slice s writes part[s][rows][n]
    const int32_t *perm, *tiles;
    int K, x_by_pair;        // grouped: as in QxArgs
};

union qw_h8u { qw_h8 h; uint32_t u[4]; uint4 v; };

template <int G, int BM, bool GATHER>
__global__ __launch_bounds__(QW_GMM_THREADS) void k_sgemm(QwGmmArgs a)
{
    constexpr int MT = BM / 16;
    constexpr int GPS = (QW_GMM_BK / G) > 0 ? QW_GMM_BK / G : 1;   // groups per stage
    __shared__ __align__(16) _Float16 As[BM][QW_GMM_BK + QW_GMM_APAD];
    __shared__ __align__(16) uint32_t Bw[QW_GMM_BN][QW_GMM_BSTRIDE];
    __shared__ float Xb[BM][QW_GMM_BK / 8];
    __shared__ float Xs[BM][GPS];
    __shared__ int sh_s[GATHER ? BM : 1], out_s[4];

    // XCD-aware order: consecutive virtual blocks (the n-blocks of one tile,
    // which share its activation rows) land on the same XCD and its L2.
    const unsigned total = gridDim.x, b = blockIdx.x;
    const unsigned v = (total % 8u == 0u) ? (b % 8u) * (total / 8u) + b / 8u : b;
    const int tile = (int)(v / (unsigned)a.nblk), nb = (int)(v % (unsigned)a.nblk);

    if (GATHER && tile >= a.tiles[0]) return;
    const int first = GATHER ? a.tiles[2 + 3 * tile] : tile * BM;
    const int len = GATHER ? a.tiles[3 + 3 * tile] : min(BM, a.rows - first);
    if (len <= 0) return;
    const int k = a.k, n = a.n, words = k / 8, groups = k / G;
    const int n0 = nb * QW_GMM_BN;
    const int kb = (int)blockIdx.y * a.kslice, ke = min(k, kb + a.kslice);
    const size_t bank = GATHER ? (size_t)a.tiles[1 + 3 * tile] * n : 0;      // the expert's first weight row
    const uint32_t *wb = a.m.w + bank * words;
    const uint16_t *sb = a.m.s + bank * groups, *bb = a.m.b + bank * groups;

    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const int ln = lane & 15, lg = lane >> 4;
    const int col = n0 + wave * 16 + ln;                 // this lane's weight row

    auto x_row = [&](int m) {
        const int p = GATHER ? a.perm[first + m] : first + m;
        return reinterpret_cast<const float4 *>(a.x + (size_t)(GATHER && !a.x_by_pair ? p / a.K : p) * k);
    };
    // Grouped rows as they are, which f16 holds well enough where their largest
    // is 2^-8 to 65504; a tile with one outside is done over with that row
    // scaled as k_xstage scales it, the others to the same bits.  (The maxima
    // first would be a trip to memory: 4 us of 20.)
    qw_f4 acc[MT], C[MT];
    float top[MT];                                       // of rows 16 i + t / 16, this thread's share
#pragma unroll
    for (int i = 0; i < MT; i++) top[i] = 0.0f;
    bool again = false;
    auto run = [&](auto scaled) __attribute__((always_inline)) {
    constexpr bool SCALED = decltype(scaled)::value, LOOK = GATHER && !SCALED;
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        acc[mt] = qw_f4{0.f, 0.f, 0.f, 0.f};
        C[mt] = acc[mt];
    }

    for (int k0 = kb; k0 < ke; k0 += QW_GMM_BK) {
        const int klen = min(QW_GMM_BK, ke - k0);
        // Activations: 8-element blocks, f16, written in nibble register order.
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const int m = 16 * i + t / 16, bk = t % 16;
            qw_h8u h;
            float bsum = 0.0f;
            if (m < len && bk * 8 < klen) {
                const float4 *xv = x_row(m) + (k0 + bk * 8) / 4;
                const float4 lo = xv[0], hi = xv[1];
                const float f[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
                const float up = SCALED ? __builtin_ldexpf(1.0f, sh_s[m]) : 1.0f;
                _Float16 q[8];
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    if (LOOK) top[i] = fmaxf(top[i], fabsf(f[j]));
                    q[j] = (_Float16)(SCALED ? f[j] * up : f[j]);
                    bsum += (float)q[j];
                }
                h.h = qw_h8{q[0], q[4], q[1], q[5], q[2], q[6], q[3], q[7]};
            } else {
                h.v = make_uint4(0, 0, 0, 0);
            }
            *reinterpret_cast<uint4 *>(&As[m][bk * 8]) = h.v;
            Xb[m][bk] = bsum;
        }
        if (LOOK && k0 + QW_GMM_BK >= ke) {            // (the barriers below hand it on)
            bool out = false;
#pragma unroll
            for (int i = 0; i < MT; i++) {
                uint64_t some = __ballot(top[i] > 0.0f), large = __ballot(top[i] >= 0x1p-8f);
                out |= __ballot(top[i] > 65504.0f && top[i] <= FLT_MAX) != 0;
#pragma unroll
                for (int r = 0; r < 4; r++) out |= (large >> 16 * r & 0xFFFF) == 0 && (some >> 16 * r & 0xFFFF) != 0;
            }
            if (lane == 0) out_s[wave] = out;
        }
        // Weights: 64 rows x 16 words, one 16-byte load per thread.
        {
            const int nn = t >> 2, q4 = t & 3;
            const int gn = n0 + nn, wk = k0 / 8 + q4 * 4;
            uint4 wv = make_uint4(0, 0, 0, 0);
            if (gn < n && q4 * 32 < klen)
                wv = *reinterpret_cast<const uint4 *>(wb + (size_t)gn * words + wk);
            uint2 *dst = reinterpret_cast<uint2 *>(&Bw[nn][q4 * 4]);
            dst[0] = make_uint2(wv.x, wv.y);
            dst[1] = make_uint2(wv.z, wv.w);
        }
        __syncthreads();
        for (int i = t; i < BM * GPS; i += QW_GMM_THREADS) {
            const int m = i / GPS, gi = i % GPS;
            float s = 0.0f;
            for (int j = 0; j < G / 8 && gi * (G / 8) + j < QW_GMM_BK / 8; j++) s += Xb[m][gi * (G / 8) + j];
            Xs[m][gi] = s;
        }
        __syncthreads();

        const int nsteps = klen / 32;
        for (int s = 0; s < nsteps; s++) {
            const int kk = k0 + 32 * s;
            if (kk % G == 0) {
#pragma unroll
                for (int mt = 0; mt < MT; mt++) C[mt] = qw_f4{0.f, 0.f, 0.f, 0.f};
            }
            const uint32_t wd = Bw[wave * 16 + ln][4 * s + lg];
            qw_h8u bf;
            bf.u[0] = (wd & 0x000F000Fu) | 0x64006400u;
            bf.u[1] = ((wd >> 4) & 0x000F000Fu) | 0x64006400u;
            bf.u[2] = ((wd >> 8) & 0x000F000Fu) | 0x64006400u;
            bf.u[3] = ((wd >> 12) & 0x000F000Fu) | 0x64006400u;
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const qw_h8 af = *reinterpret_cast<const qw_h8 *>(&As[mt * 16 + ln][32 * s + 8 * lg]);
                C[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, bf.h, C[mt], 0, 0, 0);
            }
            if ((kk + 32) % G == 0 || kk + 32 >= ke) {
                const int gabs = kk / G, gi = (kk - k0) / G;
                float sc = 0.0f, bp = 0.0f;
                if (col < n) {
                    sc = qw_bf16(sb[(size_t)col * groups + gabs]);
                    bp = qw_bf16(bb[(size_t)col * groups + gabs]) - 1024.0f * sc;
                }
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float xg = Xs[mt * 16 + 4 * lg + i][gi];
                        acc[mt][i] = __builtin_fmaf(sc, C[mt][i], __builtin_fmaf(bp, xg, acc[mt][i]));
                    }
                }
            }
        }
        __syncthreads();
    }

    };
    run(std::false_type{});
    if constexpr (GATHER) {
        again = (out_s[0] | out_s[1] | out_s[2] | out_s[3]) != 0;
        if (again) {
#pragma unroll
            for (int i = 0; i < MT; i++) {
#pragma unroll
                for (int o = 1; o < 16; o <<= 1) top[i] = fmaxf(top[i], __shfl_xor(top[i], o, 64));
                const bool in = top[i] >= 0x1p-8f && top[i] <= 65504.0f;
                if ((t & 15) == 0) sh_s[16 * i + t / 16] = in ? 0 : qx_shift(top[i]);
            }
            __syncthreads();
            run(std::true_type{});
        }
    }

    float *yo = a.part ? a.part + (size_t)blockIdx.y * a.rows * n : a.y;
    if (col < n) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int m = mt * 16 + 4 * lg + i;
                if (m < len) {
                    yo[(size_t)(GATHER ? a.perm[first + m] : first + m) * n + col] =
                        again ? __builtin_ldexpf(acc[mt][i], -sh_s[m]) : acc[mt][i];
                }
            }
        }
    }
}

// y[i] = part[0][i] + part[1][i] + ... in slice order
__global__ void k_qmm_reduce(float *__restrict__ y, const float *__restrict__ part, long total, int splits)
{
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
        float v = part[i];
        for (int sp = 1; sp < splits; sp++) v = v + part[(size_t)sp * total + i];
        y[i] = v;
    }
}

// ---- plans -------------------------------------------------------------------------------

static size_t qx_al(size_t b) { return (b + 255) & ~(size_t)255; }
static int qx_kp(int k) { return (k + QX_KPAD - 1) / QX_KPAD * QX_KPAD; }
static int qx_nsb(int k, int group) { return (k / group + QX_SB - 1) / QX_SB; }
static size_t qx_stage_bytes(int rows, int k, int group)
{
    return qx_al((size_t)rows * qx_kp(k) * 2) + qx_al((size_t)rows * qx_nsb(k, group) * 128) + qx_al((size_t)rows * 4);
}

static bool gmm_shape_ok(const float *x, qwk_q4 m, int k, int n, int group)
{
    return k >= 32 && k % 32 == 0 && n >= 1 && (group == 32 || group == 64 || group == 128) &&
           k % group == 0 && ((uintptr_t)x & 15u) == 0 && ((uintptr_t)m.w & 15u) == 0;
}

// Stages `rows` rows at `work` and points the arguments at them.
static void qx_stage(hipStream_t s, QxArgs &a, const float *x, int rows, int group, char *work)
{
    a.kp = qx_kp(a.k);
    a.nsb = qx_nsb(a.k, group);
    _Float16 *ah = reinterpret_cast<_Float16 *>(work);
    uint16_t *xp = reinterpret_cast<uint16_t *>(work + qx_al((size_t)rows * a.kp * 2));
    int *ex = reinterpret_cast<int *>(reinterpret_cast<char *>(xp) + qx_al((size_t)rows * a.nsb * 128));
    a.ah = ah;
    a.xp = xp;
    a.ex = ex;
    const bool wide = a.k >= QX_WIDE_K;
    const dim3 grid(wide ? rows : (rows + 3) / 4), blk(256);
#define QX_STAGE(GG)                                                                                                       \
    if (!wide) hipLaunchKernelGGL((k_xstage<GG, 1, 2>), grid, blk, 0, s, ah, xp, ex, x, rows, a.k, a.kp, a.nsb);            \
    else if (a.k <= 4096) hipLaunchKernelGGL((k_xstage<GG, 4, 2>), grid, blk, 0, s, ah, xp, ex, x, rows, a.k, a.kp, a.nsb); \
    else hipLaunchKernelGGL((k_xstage<GG, 4, 6>), grid, blk, 0, s, ah, xp, ex, x, rows, a.k, a.kp, a.nsb)
    if (group == 32) { QX_STAGE(32); }
    else if (group == 64) { QX_STAGE(64); }
    else { QX_STAGE(128); }
#undef QX_STAGE
}

// Column blocks a workgroup runs back to back: where k is short a block is
// over in a few stages, and a workgroup's start (its tile's rows, the first
// loads) would be most of it; kept to what still fills QX_SLOTS places.
static int qx_nbw(int k, int nblk, long tiles)
{
    int w = k >= 2048 ? 1 : 2048 / (k < 256 ? 256 : k);
    while (w > 1 && tiles * ((nblk + w - 1) / w) < QX_SLOTS) w--;
    return w < nblk ? w : nblk;
}

// The same for a grouped product, whose tiles the host can only estimate (the
// list's bound is half as many again): the number that ends first, in rounds
// of QX_SLOTS workgroups, each a start of about 2.5 stages of 256 k and its
// blocks' stages.  (Filling the places by the bound left 400 rows of 6 picks
// in 256 experts of 320 x 640 a second round of 30 workgroups, as long as the
// first: the layer op by op 178 us, now 161, 167 with 64 x 64 tiles.)
extern "C" int qwk_gather_gemm_blocks(int k, int n, int pairs, int E, int bm)
{
    E = E < 1 ? 1 : E;
    const int nblk = (n + 127) / 128;
    const double mean = (double)pairs / E, fill = mean / bm + 0.5;
    const double tiles = E * (1.0 - exp(-mean)) * (fill > 1.0 ? fill : 1.0);
    const int most = k >= 2048 ? 1 : 2048 / (k < 256 ? 256 : k), stages = (k + 255) / 256;
    int best = 1;
    double cost = 1e300;
    for (int w = 1; w <= most && w <= nblk; w++) {
        const double c = ceil(tiles * ((nblk + w - 1) / w) / QX_SLOTS) * (2.5 + w * stages);
        if (c < cost) { cost = c; best = w; }
    }
    return best;
}

// Whether a grouped product goes unstaged, to k_sgemm: where k is short and the
// touched experts' weights are few, the stage's launch and the blocks' starts
// cost more than they save.  us a call over cold banks, 64 x 64 tiles before /
// staged / this:
//   256 experts 320 x  640, 33 / 100 / 400 rows of 6  10 / 15 / 11, 19 / 21 / 20, 23 / 32 / 23
//   128         256 x 1664, 33 / 200 rows of 6        15 / 18 / 16, 19 / 26 / 20
//   512         256 x 1024,  9 rows of 10              8 / 12 /  9
// but 33 rows of the last (64 M weights) 23 / 19 / 24, and 640 x 320 of the
// first, 33 / 100 rows, 16 / 12, 19 / 19 staged.
extern "C" int qwk_gather_gemm_small(int k, int n, int pairs, int E, int bm)
{
    E = E < 1 ? 1 : E;
    return k <= 320 && bm == 16 && E * (1.0 - exp(-(double)pairs / E)) * n * k <= 58720256.0;
}

// Few rows a tile: four waves side by side over 128 columns.
template <int G, bool GATHER>
static void qx_narrow(hipStream_t s, QxArgs &a, int bm, int ntiles, int splits, int pairs = 0, int E = 0)
{
    a.nblk = (a.n + 127) / 128;
    a.nbw = GATHER ? qwk_gather_gemm_blocks(a.k, a.n, pairs, E, bm) : qx_nbw(a.k, a.nblk, (long)ntiles * splits);
    const long ngr = (a.nblk + a.nbw - 1) / a.nbw;
    const dim3 grid((unsigned)((ngr * ntiles + 7) / 8 * 8), (unsigned)splits), blk(256);
    if (bm == 16) hipLaunchKernelGGL((k_xgemm<G, 1, 2, 1, 4, 256, 2, 96, GATHER>), grid, blk, 0, s, a);
    else if (bm == 32) hipLaunchKernelGGL((k_xgemm<G, 2, 2, 1, 4, 256, 2, 48, GATHER>), grid, blk, 0, s, a);
    else hipLaunchKernelGGL((k_xgemm<G, 4, 2, 1, 4, 128, 2, 96, GATHER>), grid, blk, 0, s, a);
}

template <int G>
static void qx_wide(hipStream_t s, QxArgs &a, int nt, int splits)
{
    a.nblk = (a.n + 32 * nt - 1) / (32 * nt);
    const long ntiles = (a.rows + 127) / 128;
    a.nbw = qx_nbw(a.k, a.nblk, ntiles * splits);
    const long ngr = (a.nblk + a.nbw - 1) / a.nbw;
    const dim3 grid((unsigned)((ngr * ntiles + 7) / 8 * 8), (unsigned)splits), blk(256);
    switch (nt) {
    case 2: hipLaunchKernelGGL((k_xgemm<G, 4, 2, 2, 2, 64, 3, 48, false>), grid, blk, 0, s, a); break;
    case 3: hipLaunchKernelGGL((k_xgemm<G, 4, 3, 2, 2, 64, 3, 48, false>), grid, blk, 0, s, a); break;
    case 4: hipLaunchKernelGGL((k_xgemm<G, 4, 4, 2, 2, 64, 3, 48, false>), grid, blk, 0, s, a); break;
    default: hipLaunchKernelGGL((k_xgemm<G, 4, 5, 2, 2, 64, 3, 48, false>), grid, blk, 0, s, a); break;
    }
}

template <int G, bool GATHER>
static void qs_launch_g(hipStream_t s, const QwGmmArgs &a, int bm, int ntiles, int splits)
{
    const dim3 grid((unsigned)(a.nblk * ntiles), (unsigned)splits), blk(QW_GMM_THREADS);
    if (bm == 16) hipLaunchKernelGGL((k_sgemm<G, 16, GATHER>), grid, blk, 0, s, a);
    else if (bm == 32) hipLaunchKernelGGL((k_sgemm<G, 32, GATHER>), grid, blk, 0, s, a);
    else hipLaunchKernelGGL((k_sgemm<G, 64, GATHER>), grid, blk, 0, s, a);
}

template <bool GATHER>
static void qs_launch(hipStream_t s, const QwGmmArgs &a, int group, int bm, int ntiles, int splits)
{
    if (group == 32) qs_launch_g<32, GATHER>(s, a, bm, ntiles, splits);
    else if (group == 64) qs_launch_g<64, GATHER>(s, a, bm, ntiles, splits);
    else qs_launch_g<128, GATHER>(s, a, bm, ntiles, splits);
}

extern "C" size_t qwk_gather_gemm_work_bytes(int k, int pairs, int K, int x_by_pair, int group)
{
    if (k < 1 || pairs < 1 || K < 1 || group < 1) return 0;
    return qx_stage_bytes(x_by_pair ? pairs : (pairs + K - 1) / K, k, group);
}

extern "C" int qwk_gather_gemm(hipStream_t s, float *y, const float *x, const int32_t *perm,
                               const int32_t *tiles, qwk_q4 m, int k, int n, int pairs, int E, int K, int x_by_pair,
                               int group, int bm, int max_tiles, void *work, size_t work_bytes)
{
    if (!gmm_shape_ok(x, m, k, n, group) || K < 1 || (bm != 16 && bm != 32 && bm != 64)) return (int)hipErrorInvalidValue;
    if (max_tiles <= 0 || pairs <= 0) return 0;
    if (qwk_gather_gemm_small(k, n, pairs, E, bm) || !work || ((uintptr_t)work & 15u) ||
        work_bytes < qwk_gather_gemm_work_bytes(k, pairs, K, x_by_pair, group)) {
        const QwGmmArgs a = {y, x, m, k, n, 0, (n + QW_GMM_BN - 1) / QW_GMM_BN, k, nullptr, perm, tiles, K, x_by_pair};
        qs_launch<true>(s, a, group, bm, max_tiles, 1);
        return (int)hipGetLastError();
    }
    QxArgs a = {};
    a.y = y; a.perm = perm; a.tiles = tiles; a.w = m.w; a.s = m.s; a.b = m.b;
    a.k = k; a.n = n; a.K = K; a.x_by_pair = x_by_pair; a.kslice = k;
    qx_stage(s, a, x, x_by_pair ? pairs : (pairs + K - 1) / K, group, static_cast<char *>(work));
    if (group == 32) qx_narrow<32, true>(s, a, bm, max_tiles, 1, pairs, E);
    else if (group == 64) qx_narrow<64, true>(s, a, bm, max_tiles, 1, pairs, E);
    else qx_narrow<128, true>(s, a, bm, max_tiles, 1, pairs, E);
    return (int)hipGetLastError();
}

// Small products' plan: split-K when the tiles alone would leave the chip
// under two workgroups a CU: enough k slices for ~QW_QMM_SPLIT_WG workgroups,
// each a whole number of QW_GMM_BK steps (so of quantisation groups) and no
// shorter than QW_QMM_SPLIT_MIN_K.
#define QW_QMM_SPLIT_BELOW 512
#define QW_QMM_SPLIT_WG 1024
#define QW_QMM_SPLIT_MIN_K 512

// Which products are small: under 2^27 multiply-adds, or a short k, which
// gives the stages little to overlap.  us a call, this against the staged
// form: 9 x 3072 x 3072 24.9 / 27.2, 20 x 1024 x 1024 23.0 / 24.9, 56 x 320 x
// 12288 20.3 / 22.6, but 112 x 3072 x 1024 30.8 / 28.9, 512 x 320 x 12288 38.2
// / 32.5.  (16 x 3072 x 3072 would be 25.4 / 26.7 still; but the staged form
// scales a row, so that no input overflows f16, and keeps what it has.)
static bool qmm_small(int k, int n, int rows)
{
    const double macs = (double)rows * n * k;
    return macs < 134217728.0 || (k <= 512 && macs < 2147483648.0);
}

static int qmm_bm(int rows) { return rows >= 64 ? 64 : (rows >= 32 ? 32 : 16); }

static int qmm_splits(int k, int n, int rows, int *kslice)
{
    const int bm = qmm_bm(rows);
    const long tiles = (long)((n + QW_GMM_BN - 1) / QW_GMM_BN) * ((rows + bm - 1) / bm);
    *kslice = k;
    if (tiles >= QW_QMM_SPLIT_BELOW) return 1;
    long sp = (QW_QMM_SPLIT_WG + tiles - 1) / tiles;
    if (sp > k / QW_QMM_SPLIT_MIN_K) sp = k / QW_QMM_SPLIT_MIN_K;
    if (sp < 2) return 1;
    const int ks = (int)(((k + sp - 1) / sp + QW_GMM_BK - 1) / QW_GMM_BK * QW_GMM_BK);
    *kslice = ks;
    return (k + ks - 1) / ks;
}

static void qmm_reduce(hipStream_t s, float *y, const float *part, long total, int splits)
{
    const long want = (total + 255) / 256;
    hipLaunchKernelGGL(k_qmm_reduce, dim3((unsigned)(want < 4096 ? want : 4096)), dim3(256), 0, s, y, part, total, splits);
}

// The staged plan, a function of the shape only: tiles of 16, 32 or 64 rows
// against 128 columns, or of 128 rows against 32 nt, and where that leaves the
// chip's QX_SLOTS workgroup places empty k cut into slices (of whole stages
// and QX_SLICE groups), whose partial sums are added in slice order.  The plan
// is the one that ends first by the times below: what 64 k cost a workgroup
// with a CU of its own and with another on it, its start, the scales where
// they do not come as one flat copy, and the partials.  The times are a fit
// to 16400 timed (shape, plan) pairs: 844 shapes of 8 to 2048 rows, k 320 to
// 12288, n 320 to 12288.  The plan chosen is 1.2% slower than the best of them
// on average (20% at worst); up to 32 rows of 2^27 to 2^28 multiply-adds, and
// there only, it is up to 7% (2 us) slower than k_sgemm.
// us a call: k_sgemm / 128-row tiles from 65 rows on, slices of 16 groups and
// a split priced four times too dear / this:
//   17 x 5888 x 3456 31 / 34 / 28      192 x 3456 x  5888  55 / 66 / 44
//   65 x 3072 x 8192 50 / 38 / 34      256 x 3072 x  8192 114 / 52 / 45
//  129 x 3456 x 5888 51 / 64 / 44      400 x 5888 x  3456  96 / 68 / 59
//  512 x 3072 x 3072 65 / 54 / 45      129 x 6144 x 10240 156 / 96 / 60
//  groups of 32: 38 x 4160 x 6144 42 / 48 / 38, 63 x 5504 x 1536 34 / 42 / 32
struct QxPlan { int bm, nt, splits, kslice; };
struct QxTile {
    int bm, nt, lo, hi;          // for calls of lo to hi rows
    double alone, paired;        // us for 64 k
    int setup, sgl;              // a workgroup's start in 64-k stages; k_xgemm's SGL
};
static const QxTile QX_TILES[] = {
    {16, 2, 1, 64, 0.29, 0.335, 6, 96},         {32, 2, 17, 128, 0.29, 0.38, 6, 48},
    {64, 2, 33, 512, 0.53, 0.64, 6, 96},        {128, 2, 65, INT_MAX, 0.64, 0.76, 8, 48},
    {128, 3, 65, INT_MAX, 0.80, 0.92, 8, 48},   {128, 4, 65, INT_MAX, 0.96, 1.08, 8, 48},
    {128, 5, 65, INT_MAX, 1.13, 1.24, 8, 48},
};

static QxPlan qx_plan(int k, int n, int rows, int group)
{
    QxPlan best = {};
    double cost = 1e300;
    const int unit = QX_SLICE * group, units = (k + unit - 1) / unit, groups = k / group;
    const double mb = (double)rows * n * 4e-6;
    for (const QxTile &t : QX_TILES) {
        if (rows < t.lo || rows > t.hi) continue;
        const bool wide = t.bm == 128, flat = groups <= t.sgl && (long)n * groups % 8 == 0;
        const int bn = wide ? 32 * t.nt : 128;
        const long tiles = (long)((rows + t.bm - 1) / t.bm) * ((n + bn - 1) / bn);
        // groups of 32 have half the k a scale; in stages: a group's scales that
        // do not come flat, and the stop for each further window of them
        const double per = group != 32 ? 1.0 : wide ? 1.65 : 1.5;
        const double scales = flat ? 0.0 : wide ? 0.07 : group == 32 ? 0.33 : 0.2, window = flat ? 0.0 : wide ? 1.0 : 3.0;
        for (int sp = 1; sp <= units && (sp == 1 || tiles * sp <= 2 * QX_SLOTS); sp++) {
            const int ks = sp == 1 ? k : (units + sp - 1) / sp * unit, gs = ks / group;
            if ((k + ks - 1) / ks != sp) continue;
            const long wgs = tiles * sp, full = wgs / QX_SLOTS, rem = wgs % QX_SLOTS;
            const double stages = (ks + 63) / 64 + t.setup + scales * gs + window * ((gs - 1) / t.sgl);
            double c = per * stages * (full * t.paired + (rem > QX_SLOTS / 2 ? t.paired : rem ? t.alone : 0.0));
            if (sp > 1) c += 1.3 + 0.65 * sp + 0.21 * mb * (sp + 1);
            if (c < cost) {
                cost = c;
                best = QxPlan{t.bm, t.nt, sp, ks};
            }
        }
    }
    return best;
}

// The plan of a call's first rows, for tests: rows a tile (0: k_sgemm),
// 32-column steps of its width, slices of k, k a slice.
extern "C" void qwk_qmm_plan(int k, int n, int rows, int group, int out[4])
{
    QxPlan p = {};
    if (qmm_small(k, n, rows)) p.splits = qmm_splits(k, n, rows, &p.kslice);
    else p = qx_plan(k, n, rows < QX_CHUNK_ROWS ? rows : QX_CHUNK_ROWS, group);
    out[0] = p.bm;
    out[1] = p.bm == 128 ? p.nt : p.bm ? 4 : 2;
    out[2] = p.splits;
    out[3] = p.kslice;
}

extern "C" size_t qwk_qmm_work_bytes(int k, int n, int rows, int group)
{
    if (k < 1 || n < 1 || rows < 1 || group < 1) return 0;
    if (qmm_small(k, n, rows)) {
        int ks;
        const int sp = qmm_splits(k, n, rows, &ks);
        return sp > 1 ? (size_t)sp * rows * n * sizeof(float) : 0;
    }
    const int r = rows < QX_CHUNK_ROWS ? rows : QX_CHUNK_ROWS;
    const QxPlan p = qx_plan(k, n, r, group);
    // (a last, shorter chunk may be split where whole ones are not)
    const int tail = rows % QX_CHUNK_ROWS;
    const QxPlan pt = tail && tail != r ? qx_plan(k, n, tail, group) : p;
    const size_t pb = p.splits > 1 ? (size_t)p.splits * r * n * 4 : 0;
    const size_t tb = tail && tail != r && pt.splits > 1 ? (size_t)pt.splits * tail * n * 4 : 0;
    return qx_stage_bytes(r, k, group) + (pb > tb ? pb : tb);
}

extern "C" int qwk_qmm(hipStream_t s, float *y, const float *x, qwk_q4 m, int k, int n, int rows, int group,
                       void *work, size_t work_bytes)
{
    if (!gmm_shape_ok(x, m, k, n, group) || rows < 1) return (int)hipErrorInvalidValue;
    const size_t need = qwk_qmm_work_bytes(k, n, rows, group);
    const bool lacks = need > 0 && (!work || ((uintptr_t)work & 15u) || work_bytes < need);
    if (lacks || qmm_small(k, n, rows)) {
        int ks = k;
        const int sp = lacks ? 1 : qmm_splits(k, n, rows, &ks), bm = qmm_bm(rows);
        const QwGmmArgs a = {y, x, m, k, n, rows, (n + QW_GMM_BN - 1) / QW_GMM_BN, ks,
                             sp > 1 ? static_cast<float *>(work) : nullptr, nullptr, nullptr, 1, 1};
        qs_launch<false>(s, a, group, bm, (rows + bm - 1) / bm, sp);
        if (sp > 1) qmm_reduce(s, y, a.part, (long)rows * n, sp);
        return (int)hipGetLastError();
    }
    for (int r0 = 0; r0 < rows; r0 += QX_CHUNK_ROWS) {
        const int r = rows - r0 < QX_CHUNK_ROWS ? rows - r0 : QX_CHUNK_ROWS;
        const QxPlan p = qx_plan(k, n, r, group);
        QxArgs a = {};
        a.y = y + (size_t)r0 * n;
        a.w = m.w; a.s = m.s; a.b = m.b;
        a.k = k; a.n = n; a.K = 1; a.x_by_pair = 1; a.rows = r; a.kslice = p.kslice;
        char *part = static_cast<char *>(work) + qx_stage_bytes(r, k, group);
        a.part = p.splits > 1 ? reinterpret_cast<float *>(part) : nullptr;
        qx_stage(s, a, x + (size_t)r0 * k, r, group, static_cast<char *>(work));
        if (p.bm == 128) {
            if (group == 32) qx_wide<32>(s, a, p.nt, p.splits);
            else if (group == 64) qx_wide<64>(s, a, p.nt, p.splits);
            else qx_wide<128>(s, a, p.nt, p.splits);
        } else {
            const int nt = (r + p.bm - 1) / p.bm;
            if (group == 32) qx_narrow<32, false>(s, a, p.bm, nt, p.splits);
            else if (group == 64) qx_narrow<64, false>(s, a, p.bm, nt, p.splits);
            else qx_narrow<128, false>(s, a, p.bm, nt, p.splits);
        }
        if (p.splits > 1) qmm_reduce(s, a.y, a.part, (long)r * n, p.splits);
        const int rc = (int)hipGetLastError();
        if (rc) return rc;
    }
    return 0;
}
