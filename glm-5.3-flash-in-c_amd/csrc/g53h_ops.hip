/* g53h_ops.hip - the expert path's building blocks on gfx950, bit-exact with the reference:
 *
 *   k_mm_f8_generic   FP8 block-scaled (or int4) matvec for any shape (ragged blocks, any
 *                     br/bc), one thread per (token, row): the unit-level glm53f_mm. The
 *                     layer paths use the kernels of g53h_moe.hip, g53h_rows.hip and the
 *                     decode files.
 *   k_swiglu          clamped SwiGLU.
 *   k_router_scores   sigmoid(W x) and sigmoid + bias for T tokens, one wave per expert.
 *   k_router_select_w top-k by repeated argmax (strict >, lowest index), renormalise, scale.
 *   k_route_topn      next-layer prediction.
 */
#include <hip/hip_runtime.h>
#include <math.h>

#include "g53h.h"
#include "g53h_core.h"
#include "g53h_kern.h"
#include "g53h_runtime.h"

/* ------------------------------------------------------------- FP8 matvec ---- */
#include "g53h_rowdot.h"

typedef float g53_f2 __attribute__((ext_vector_type(2)));
typedef uint32_t g53_u4 __attribute__((ext_vector_type(4)));

__global__ void k_mm_f8_generic(float *__restrict__ y, const float *__restrict__ x, int T, G53hMat m)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)T * m.rows) return;
    const int t = (int)(i / m.rows), o = (int)(i % m.rows);
    y[(size_t)t * m.rows + o] = g53_row_dot(m, o, x + (size_t)t * m.cols);
}

/* The same product for FP8 matrices with 128-column blocks (row-major codes, any rows, columns,
 * alignment and scale rows), TG tokens at a time. A workgroup owns 64 rows x TG tokens; wave w
 * takes column blocks w, w + NW, ... and lane r row r, so a weight is decoded once for TG tokens
 * and x is the same for every lane: scalar loads, two groups a request and asked for one group's
 * products ahead (they return in any order, so a wait is for all of them), and no LDS traffic in
 * the inner loop. A wave loads its block's 64 x 128 codes as whole 128-byte runs (8
 * lanes a row), a round ahead, and turns them through 4 KB of LDS, 32 rows at a time; 16-byte
 * pieces are swizzled by row pairs, so that 16 lanes meet no bank twice. Each block's scaled
 * double sum goes to LDS, and the thread that owns (row, token) adds a round's NW sums in block
 * order, as the reference does.
 * Bound by the fp32 chains, one FMA per weight and token: the reference rounds each product into
 * one of eight chains, so matrix cores do not apply. 4096 x 2048, 24 tokens: 73 us with a
 * thread per (row, token), 19 us here. AL: codes and columns in multiples of 16 bytes. */
template <int TG, int NW, bool AL>
__global__ void __launch_bounds__(64 * NW, 4) k_mm_f8_rows(float *__restrict__ y, const float *__restrict__ x, int T,
                                                           G53hMat m)
{
    static_assert(TG <= NW, "one owner thread per (row, token)");
    __shared__ __attribute__((aligned(16))) g53_u4 stage[NW][256];
    __shared__ double pb[2][NW][TG][64];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned ng = (unsigned)(T + TG - 1) / TG;         /* the token groups of a row tile are neighbours */
    const int r0 = (int)(blockIdx.x / ng) * 64, t0 = (int)(blockIdx.x % ng) * TG;
    const int cols = m.cols, nb = (cols + 127) >> 7, rounds = (nb + NW - 1) / NW;
    const int row = min(r0 + lane, m.rows - 1);              /* past the end: computed, not stored */
    const float *srow = m.s + (size_t)(row / m.br) * m.scols;
    g53_u4 *st = stage[w];
    const int key = (lane >> 1) & 7;
    const int lr = lane >> 3, lp = lane & 7;                 /* this lane's piece of a load: row, 16 bytes */
    g53_u4 q[8];
    auto load = [&](int b) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int rr = min(r0 + 8 * j + lr, m.rows - 1), c0 = b * 128 + lp * 16;
            if constexpr (AL) {                              /* past the last column: its last piece again */
                q[j] = *(const g53_u4 *)(m.w + (size_t)rr * cols + min(c0, cols - 16));
            } else {                                         /* the words that hold the piece's bytes */
                q[j] = g53_u4{0, 0, 0, 0};
                if (c0 >= cols) continue;
                const uint8_t *src = m.w + (size_t)rr * cols + c0;
                const int sh = (int)((uintptr_t)src & 3), left = min(cols - c0, 16);
                const uint32_t *p = (const uint32_t *)(src - sh);
                uint32_t v[5];
#pragma unroll
                for (int k = 0; k < 5; k++) v[k] = 4 * k < left + sh ? p[k] : 0u;
                q[j].x = __builtin_amdgcn_alignbyte(v[1], v[0], sh);
                q[j].y = __builtin_amdgcn_alignbyte(v[2], v[1], sh);
                q[j].z = __builtin_amdgcn_alignbyte(v[3], v[2], sh);
                q[j].w = __builtin_amdgcn_alignbyte(v[4], v[3], sh);
            }
        }
    };
    const float *xt[TG];
#pragma unroll
    for (int t = 0; t < TG; t++) xt[t] = x + (size_t)min(t0 + t, T - 1) * cols;
    double acc = 0.0;
    if (w < nb) load(w);
    for (int rd = 0; rd < rounds; rd++) {
        const int b = rd * NW + w;
        if (b < nb) {
            float a[TG][8] = {};
            float xv[2][TG][8];                              /* x of two neighbouring groups */
            auto xload = [&](float (&d)[TG][8], int c) {     /* columns c .. c + 7, scalar loads */
#pragma unroll
                for (int t = 0; t < TG; t++)
#pragma unroll
                    for (int l = 0; l < 8; l++) d[t][l] = xt[t][c + l];
            };
            auto group = [&](uint32_t lo, uint32_t hi, const float (&d)[TG][8]) {
                const g53_f2 f01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)lo, false);
                const g53_f2 f23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)lo, true);
                const g53_f2 f45 = __builtin_amdgcn_cvt_pk_f32_fp8((int)hi, false);
                const g53_f2 f67 = __builtin_amdgcn_cvt_pk_f32_fp8((int)hi, true);
                const float f[8] = {f01.x, f01.y, f23.x, f23.y, f45.x, f45.y, f67.x, f67.y};
#pragma unroll
                for (int t = 0; t < TG; t++)
#pragma unroll
                    for (int l = 0; l < 8; l++) a[t][l] = __builtin_fmaf(f[l], d[t][l], a[t][l]);
            };
            const int W = min(cols - b * 128, 128);
            g53_u4 v[8];                                      /* this lane's row of the block */
#pragma unroll
            for (int j = 0; j < 8; j++) {                    /* 32 rows at a time */
                const int rr = 8 * (j & 3) + lr;
                st[rr * 8 + (lp ^ ((rr >> 1) & 7))] = q[j];
                if ((j & 3) == 3) {
#pragma unroll
                    for (int p = 0; p < 8; p++) {
                        const g53_u4 u = st[(lane & 31) * 8 + (p ^ key)];
                        v[p] = j == 3 || lane >= 32 ? u : v[p];
                    }
                }
            }
            if (b + NW < nb) load(b + NW);
            if (W == 128) {
                /* a group's x is requested while the group before it is multiplied (the compiler asks for two
                 * groups at once, every other time) */
                xload(xv[0], b * 128);
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    if (i < 15) xload(xv[(i + 1) & 1], b * 128 + 8 * (i + 1));
                    __builtin_amdgcn_sched_barrier(0);
                    group((i & 1) ? v[i >> 1].z : v[i >> 1].x, (i & 1) ? v[i >> 1].w : v[i >> 1].y, xv[i & 1]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll
                for (int i = 0; i < 16; i++)
                    if (i * 8 + 8 <= W) {
                        xload(xv[0], b * 128 + 8 * i);
                        group((i & 1) ? v[i >> 1].z : v[i >> 1].x, (i & 1) ? v[i >> 1].w : v[i >> 1].y, xv[0]);
                    }
            }
            const int nt = W & 7;                            /* the block's last columns, one by one */
            uint32_t tw[2] = {0, 0};
            if (nt)
#pragma unroll
                for (int p = 0; p < 8; p++) {
                    if ((W >> 3) == 2 * p) { tw[0] = v[p].x; tw[1] = v[p].y; }
                    if ((W >> 3) == 2 * p + 1) { tw[0] = v[p].z; tw[1] = v[p].w; }
                }
            const float sc = srow[b];
#pragma unroll
            for (int t = 0; t < TG; t++) {
                double s = (((double)a[t][0] + a[t][4]) + ((double)a[t][2] + a[t][6])) +
                           (((double)a[t][1] + a[t][5]) + ((double)a[t][3] + a[t][7]));
                for (int j = 0; j < nt; j++)
                    s += (double)g53_e4m3_hw((uint8_t)(tw[j >> 2] >> (8 * (j & 3)))) * (double)xt[t][b * 128 + W - nt + j];
                pb[rd & 1][w][t][lane] = s * (double)sc;
            }
        }
        __syncthreads();
        if (tid < 64 * TG) {
#pragma unroll
            for (int k = 0; k < NW; k++)
                if (rd * NW + k < nb) acc = acc + pb[rd & 1][k][tid >> 6][lane];
        }
    }
    if (tid < 64 * TG && r0 + lane < m.rows && t0 + (tid >> 6) < T)
        y[(size_t)(t0 + (tid >> 6)) * m.rows + r0 + lane] = (float)acc;
}

extern "C" int g53h_mm_f8(float *y, const float *x, int T, const G53hMat *m)
{
    if (g53h_ready()) return -1;
    if (T <= 0) return 0;
    if (!m || !m->w || !m->s) return g53h_fail("g53h_mm_f8: unbound matrix");
    if (m->rows <= 0 || m->cols <= 0 || m->br <= 0 || m->bc <= 0 ||
        m->scols != (m->cols + m->bc - 1) / m->bc || ((m->flags & G53H_MAT_I4) && (m->cols & 1)))
        return g53h_fail("g53h_mm_f8: bad geometry %dx%d block %dx%d scols %d", m->rows, m->cols,
                         m->br, m->bc, m->scols);
    if (m->flags & (G53H_MAT_TILED | G53H_MAT_MTILED | G53H_MAT_I4T))
        return g53h_fail("g53h_mm_f8: tiled codes are read by the layer kernels only (flags %d)", m->flags);
    /* FP8 with 128-column blocks: a row tile. Two tokens a workgroup share each weight's decode; while single
     * tokens leave every CU at most one workgroup the call is a chain of latencies instead, and 16 waves, each
     * with its block's codes in flight, shorten it. Measured, (1 token, 16 waves) against (2, 8): 4096 x 4096 1
     * token 10.5 against 14.8 us, 2048 x 4096 4 tokens 12.6 against 15.4; 4096 x 2048 24 tokens 28.6 against
     * 19.1, 4096 x 4096 64 tokens 123 against 64. (3 and 4 tokens: 20 and 31 us at 24, the chains' registers
     * spill.) Codes and columns that are not in multiples of 16 bytes load by words: 4096 x 1030, 24 tokens
     * 36.5 us with a thread per (row, token), 19.0 here; 333 x 2047, 5: 55.0, 12.1.
     * A thread per (row, token) is the faster one where the only block, or the second of two, is partial and
     * its columns, taken 8 at a time, are most of the work: below 128 columns (us, thread / tile: 4096 x 100, 1
     * token 3.8 / 4.9, 24 tokens 4.3 / 10.3; 4096 x 17, 300: 8.2 / 62.4; 2048 x 112, 64: 4.7 / 7.3; aligned and
     * one workgroup a CU, 4096 x 112, 1: 3.7 / 3.6), and unaligned rows of 136 to 207 in whole tiles (4096 x 136,
     * 24: 5.0 / 8.2; 4096 x 200, 64: 13.8 / 16.6; 129 columns, 64: 20.3 / 16.3; 250, 64: 23.8 / 20.6). */
    const long tiles = ((long)m->rows + 63) / 64;
    const int al = m->cols % 16 == 0 && ((uintptr_t)m->w & 15) == 0, one = tiles * T <= g53h_num_cus();
    const int narrow = m->cols < 128 ? !(al && one)
                                     : !al && !one && m->rows % 64 == 0 && m->cols >= 136 && m->cols < 208;
    const long per_tile = 0xffffffffL / (one ? 1024 : 512) / tiles * (one ? 1 : 2);
    const int tile = m->flags == 0 && m->bc == 128 && !narrow && per_tile > 0;
    /* a launch holds fewer than 2^32 threads (more are cut off without an error): tokens in slices */
    const long per = tile ? per_tile : 0xffffff00L / m->rows;
    hipStream_t st = g53h_stream();
    for (long t0 = 0; t0 < T; t0 += per) {
        const int n = (int)(T - t0 < per ? T - t0 : per);
        float *ys = y + (size_t)t0 * m->rows;
        const float *xs = x + (size_t)t0 * m->cols;
        if (!tile) {
            hipLaunchKernelGGL(k_mm_f8_generic, dim3((unsigned)(((long)n * m->rows + 127) / 128)), dim3(128), 0, st, ys, xs,
                               n, *m);
            G53_LAUNCHED("k_mm_f8_generic");
            continue;
        }
        const dim3 g((unsigned)(tiles * (one ? n : (n + 1) / 2)));
#define G53_MM(TG, NW, AL) hipLaunchKernelGGL((k_mm_f8_rows<TG, NW, AL>), g, dim3(64 * NW), 0, st, ys, xs, n, *m)
        if (one && al) G53_MM(1, 16, true);
        else if (one) G53_MM(1, 16, false);
        else if (al) G53_MM(2, 8, true);
        else G53_MM(2, 8, false);
#undef G53_MM
        G53_LAUNCHED("k_mm_f8_rows");
    }
    return 0;
}

/* ----------------------------------------------------------------- SwiGLU ---- */
__global__ void k_swiglu(float *__restrict__ y, const float *__restrict__ gu, int n, int T, float limit)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)n * T) return;
    const int t = (int)(i / n), k = (int)(i % n);
    const float *g = gu + (size_t)t * 2 * n;
    y[i] = g53_swiglu1(g[k], g[n + k], limit);
}

extern "C" int g53h_swiglu(float *y, const float *gu, int n, int T, float limit)
{
    if (g53h_ready()) return -1;
    const long m = (long)n * T;
    if (m <= 0) return 0;
    hipLaunchKernelGGL(k_swiglu, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, g53h_stream(), y,
                       gu, n, T, limit);
    G53_LAUNCHED("k_swiglu");
    return 0;
}

/* Swiglu over separate gate/up slot outputs: g, u [rows_total][n] -> y. */
__global__ void k_swiglu_split(float *__restrict__ y, const float *__restrict__ g,
                               const float *__restrict__ u, long m, float limit)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m) y[i] = g53_swiglu1(g[i], u[i], limit);
}

int g53h_swiglu_split(float *y, const float *g, const float *u, long m, float limit)
{
    if (m <= 0) return 0;
    hipLaunchKernelGGL(k_swiglu_split, dim3((unsigned)((m + 255) / 256)), dim3(256), 0,
                       g53h_stream(), y, g, u, m, limit);
    G53_LAUNCHED("k_swiglu_split");
    return 0;
}

#include "g53h_gemv.h"

/* scores[t][e] = sigmoid(dot); choice[t][e] = score + bias[e]. One wave per (token, expert),
 * one wave per workgroup so the experts spread over every CU. */
__global__ void __launch_bounds__(64) k_router_scores(float *__restrict__ score, float *__restrict__ choice,
                                                      const float *__restrict__ x, int T,
                                                      const void *__restrict__ gate, int dt,
                                                      const float *__restrict__ bias, int NE, int E)
{
    const int lane = threadIdx.x;
    const int e = blockIdx.x, t = blockIdx.y;
    const float d = g53_router_dot(gate, dt, e, E, x + (size_t)t * E, lane);
    if (lane == 0) {
        const float s = g53_sigmoidf(d);
        score[(size_t)t * NE + e] = s;
        if (choice) choice[(size_t)t * NE + e] = s + bias[e];
    }
}

/* The same scores for many tokens on the FP64 matrix cores (v_mfma_f64_16x16x4f64). Every
 * product (double)bf16 * (double)x is exact in double, as in k_router_scores; the instruction
 * adds them with double FMAs, in an order of its own. A workgroup computes the 16 x 16 tile (bx, by) of
 * experts e0 = 16 * bx .. +15 and tokens t0 = 16 * by .. +15 over column range bz; its four waves
 * split the columns (wave w takes columns 64w .. 64w+63 of every 256-column chunk) and their
 * partial sums are added in LDS at the end. Operands: lane l gives A[l % 16][l / 16] (an
 * expert's weight) and B[l / 16][l % 16] (a token's x); step s uses column 64w + 16(l/16) + s
 * of the chunk, so a lane reads 32 consecutive router bytes per chunk. Result: lane l, register
 * r holds C[4r + l/16][l % 16]. x chunks are staged in LDS. bf16 router rows, E a multiple of
 * 256. The double instruction's rate bounds it from some hundred tokens on, below that the wait for
 * a chunk, so the next chunk's operands are requested before this one is multiplied (288 experts x
 * 4096 with the selection, us: 150 tokens 26.3 -> 20.2, 384: 47.3 -> 32.7, 2048: 109.8 -> 103.5, where a
 * 32 x 32 tile per wave over eight column ranges had been faster than the unpipelined loop).
 * The grid is (bx, by, bz), or flat (S column ranges) with a contiguous run of tiles, experts fastest, on
 * each of the 8 XCDs that workgroups are dealt to in turn, so that a token tile is fetched into one L2
 * instead of into as many as it meets experts. */
typedef double g53_v4d __attribute__((ext_vector_type(4)));
typedef float g53_v4f __attribute__((ext_vector_type(4)));
#define G53_RM_XST 260                                  /* LDS floats per token row       */
__global__ void __launch_bounds__(256) k_router_mfma(float *__restrict__ score, float *__restrict__ choice,
                                                     const float *__restrict__ x, int T,
                                                     const uint16_t *__restrict__ gate,
                                                     const float *__restrict__ bias, int NE, int E, int klen, int S,
                                                     double *__restrict__ psum)
{
    int bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
    if (S) {                                                 /* flat */
        const int ET = (NE + 15) >> 4, TT = (T + 15) >> 4;
        const int j = (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
        if (j >= ET * TT * S) return;
        bx = j % ET; by = (j / ET) % TT; bz = j / (ET * TT);
    }
    __shared__ __attribute__((aligned(16))) float xs[16 * G53_RM_XST];
    __shared__ g53_v4d part[3][64];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int t0 = by * 16, e0 = bx * 16;
    const int i = lane & 15, g = lane >> 4;
    const int er = e0 + i < NE ? e0 + i : NE - 1;          /* rows past NE: discarded       */
    const uint16_t *wrow = gate + (size_t)er * E + w * 64 + g * 16;
    const float *xl = xs + i * G53_RM_XST + w * 64 + g * 16;
    g53_v4d acc = {0.0, 0.0, 0.0, 0.0};
    const int kb = bz * klen;                                /* this workgroup's column range */
    /* the next chunk's operands come to registers while this one's are multiplied */
    g53_u4 wv[2];
    g53_v4f xv[4];
    const int xc = (threadIdx.x & 63) * 4;
    auto load = [&](int k0) {
        wv[0] = *(const g53_u4 *)(wrow + k0);
        wv[1] = *(const g53_u4 *)(wrow + k0 + 8);
#pragma unroll
        for (int q = 0; q < 4; q++) xv[q] = *(const g53_v4f *)(x + (size_t)min(t0 + w + 4 * q, T - 1) * E + k0 + xc);
    };
    load(kb);
    for (int k0 = kb; k0 < kb + klen; k0 += 256) {
        const g53_u4 d[2] = {wv[0], wv[1]};
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; q++) *(g53_v4f *)(xs + (w + 4 * q) * G53_RM_XST + xc) = xv[q];
        __syncthreads();
        if (k0 + 256 < kb + klen) load(k0 + 256);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)g53_bitsf(d[k >> 2][k & 3] << 16), (double)xl[2 * k], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)g53_bitsf(d[k >> 2][k & 3] & 0xffff0000u), (double)xl[2 * k + 1],
                                                       acc, 0, 0, 0);
        }
    }
    if (w > 0) part[w - 1][lane] = acc;
    __syncthreads();
    if (w > 0) return;
    acc = acc + part[0][lane] + part[1][lane] + part[2][lane];
    const int t = t0 + i;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int e = e0 + 4 * r + g;
        if (t < T && e < NE && psum) {                        /* a column range: its sum */
            psum[((size_t)bz * T + t) * NE + e] = acc[r];
        } else if (t < T && e < NE) {
            const float s = g53_sigmoidf((float)acc[r]);
            score[(size_t)t * NE + e] = s;
            if (choice) choice[(size_t)t * NE + e] = s + bias[e];
        }
    }
}

extern "C" __device__ unsigned __ockl_wfred_max_u32(unsigned);

/* Top-k and weights of each token: one wave per token, four per workgroup, and the top-k as K
 * rounds of arg-max over keys each lane holds sorted (the reference's rounds of "first
 * strictly greater", src/core/glm53f_ops.c:957-969: the larger choice first, the lower index
 * among equal ones, NaN and -inf never). With part != NULL the logits are first summed from
 * the S column ranges in column order and the scores and choices written. A token with fewer
 * than K selectable experts gets index 0 with expert 0's score in the missing slots and sets
 * *nan_flag (the reference aborts there). Then the weights: the unbiased scores of the chosen
 * experts, renormalised in double if norm_topk (:970-975), times routed_scale. When experts !=
 * NULL the chosen experts' descriptors (and the shared expert's) are copied to slots[t][*], so
 * the expert kernels find their matrices with one load. NE <= 64 * NV. */
template <int NV>
__device__ __forceinline__ void g53_select_token(int t, int lane, int *__restrict__ idx, float *__restrict__ w,
                                                 float *__restrict__ score, float *__restrict__ choice,
                                                 const double *__restrict__ part, int S,
                                                 const float *__restrict__ bias, int T, int NE, int K,
                                                 int norm_topk, float routed_scale, int *__restrict__ nan_flag,
                                                 int set_flag, const G53hExpert *__restrict__ experts,
                                                 const G53hExpert *__restrict__ shared,
                                                 G53hExpert *__restrict__ slots)
{
    uint32_t key[NV];
    int vid[NV];
    float vsc[NV];
    double d[NV];
    if (part) {
        const int ec = NE - 1;
        if constexpr (NV <= 8) {                              /* every range's loads in flight at once */
            double pv[8][NV];
#pragma unroll
            for (int q = 0; q < 8; q++)
#pragma unroll
                for (int v = 0; v < NV; v++)
                    pv[q][v] = part[((size_t)min(q, S - 1) * T + t) * NE + min(lane + 64 * v, ec)];
#pragma unroll
            for (int v = 0; v < NV; v++) {
                d[v] = pv[0][v];
#pragma unroll
                for (int q = 1; q < 8; q++)
                    if (q < S) d[v] = d[v] + pv[q][v];
            }
        } else {                                              /* range by range: NV loads in flight */
#pragma unroll
            for (int v = 0; v < NV; v++) d[v] = part[(size_t)t * NE + min(lane + 64 * v, ec)];
            for (int q = 1; q < S; q++)
#pragma unroll
                for (int v = 0; v < NV; v++) d[v] = d[v] + part[((size_t)q * T + t) * NE + min(lane + 64 * v, ec)];
        }
    }
#pragma unroll
    for (int v = 0; v < NV; v++) {
        const int e = lane + 64 * v;
        float sc = 0.0f, ch = -INFINITY;
        if (e < NE) {
            const size_t o = (size_t)t * NE + e;
            if (part) {
                sc = g53_sigmoidf((float)d[v]);
                ch = sc + bias[e];
                score[o] = sc;
                choice[o] = ch;
            } else {
                sc = score[o];
                ch = choice[o];
            }
        }
        key[v] = (ch > -INFINITY) ? g53_fkey(ch) : 0u;        /* 0: never chosen */
        vid[v] = e;
        vsc[v] = sc;
    }
    const float sc0 = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(vsc[0]), 0));   /* expert 0's */
    /* each lane sorts its keys, largest first, the lower index first among equal keys */
#pragma unroll
    for (int pass = 0; pass < NV; pass++)
#pragma unroll
        for (int q = pass & 1; q + 1 < NV; q += 2) {
            const bool sw_ = key[q + 1] > key[q];
            const uint32_t k0 = key[q], k1 = key[q + 1];
            const int i0 = vid[q], i1 = vid[q + 1];
            const float s0 = vsc[q], s1 = vsc[q + 1];
            key[q] = sw_ ? k1 : k0; key[q + 1] = sw_ ? k0 : k1;
            vid[q] = sw_ ? i1 : i0; vid[q + 1] = sw_ ? i0 : i1;
            vsc[q] = sw_ ? s1 : s0; vsc[q + 1] = sw_ ? s0 : s1;
        }
    int pos = 0, my_e = 0;                                    /* lane j keeps round j's winner */
    float my_s = sc0;
    for (int j = 0; j < K; j++) {
        const uint32_t m = __ockl_wfred_max_u32(key[0]);
        if (m == 0) break;                                    /* fewer than K selectable */
        const uint64_t cand = __ballot(key[0] == m);
        int win;
        if (__popcll(cand) == 1) win = (int)__builtin_ctzll(cand);
        else win = (int)(__ockl_wfred_min_u32(key[0] == m ? (uint32_t)vid[0] : 0xffffffffu) & 63);
        const int e = __builtin_amdgcn_readlane(vid[0], win);
        const float ws = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(vsc[0]), win));
        if (lane == j) { my_e = e; my_s = ws; }
        const bool me = lane == win;                          /* the winner shifts its list */
#pragma unroll
        for (int q = 0; q + 1 < NV; q++) {
            key[q] = me ? key[q + 1] : key[q];
            vid[q] = me ? vid[q + 1] : vid[q];
            vsc[q] = me ? vsc[q + 1] : vsc[q];
        }
        key[NV - 1] = me ? 0u : key[NV - 1];
        pos++;
    }
    if (lane == 0 && nan_flag) {
        if (set_flag) *nan_flag = pos < K;                    /* one token: the flag's only writer */
        else if (pos < K) atomicOr(nan_flag, 1);
    }
    float wj = my_s;
    if (norm_topk) {
        double sum = 0.0;
        for (int j = 0; j < K; j++) sum += (double)__uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(my_s), j));
        wj = (float)((double)my_s / (sum + 1e-20));
    }
    if (lane < K) {
        idx[(size_t)t * K + lane] = my_e;
        w[(size_t)t * K + lane] = wj * routed_scale;
    }
    if (experts) {
        const int nslots = K + (shared ? 1 : 0);
        const int words = (int)(sizeof(G53hExpert) / 4);
        for (int q = lane; q < nslots * words; q += 64) {
            const int j = q / words, k = q % words;
            const int ej = __shfl(my_e, j < K ? j : 0);
            const G53hExpert *src = j < K ? &experts[ej] : shared;
            ((int *)&slots[(size_t)t * nslots + j])[k] = ((const int *)src)[k];
        }
    }
}

template <int NV>
__global__ void __launch_bounds__(256) k_router_select_w(int *__restrict__ idx, float *__restrict__ w,
                                                         float *__restrict__ score, float *__restrict__ choice,
                                                         const double *__restrict__ part, int S,
                                                         const float *__restrict__ bias, int T, int NE, int K,
                                                         int norm_topk, float routed_scale,
                                                         int *__restrict__ nan_flag,
                                                         const G53hExpert *__restrict__ experts,
                                                         const G53hExpert *__restrict__ shared,
                                                         G53hExpert *__restrict__ slots)
{
    const int lane = threadIdx.x & 63;
    const int t = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (t >= T) return;
    g53_select_token<NV>(t, lane, idx, w, score, choice, part, S, bias, T, NE, K, norm_topk, routed_scale, nan_flag,
                         0, experts, shared, slots);
}

/* Scores and selection of a small bf16 router in one launch, a workgroup per token. 16 lanes take an
 * expert (lane l of them columns 8 l + 128 i .. + 7, its products added in order, then across the
 * lanes: exact as in k_router_scores); then the first wave selects. E a multiple of 128. */
template <int NV>
__global__ void __launch_bounds__(1024) k_router_small(int *__restrict__ idx, float *__restrict__ w,
                                                      const float *__restrict__ x, const uint16_t *__restrict__ gate,
                                                      const float *__restrict__ bias, int NE, int E, int K,
                                                      int norm_topk, float routed_scale, int *__restrict__ nan_flag,
                                                      const G53hExpert *__restrict__ experts,
                                                      const G53hExpert *__restrict__ shared,
                                                      G53hExpert *__restrict__ slots)
{
    __shared__ float score[64 * NV], choice[64 * NV];
    const int t = blockIdx.x, lane = threadIdx.x & 63, l = threadIdx.x & 15;
    const float *xt = x + (size_t)t * E + 8 * l;
    for (int e0 = 0; e0 < NE; e0 += (int)blockDim.x >> 4) {
        const int e = e0 + (int)(threadIdx.x >> 4);
        const uint16_t *row = gate + (size_t)(e < NE ? e : NE - 1) * E + 8 * l;
        double acc = 0.0;
#pragma unroll 4
        for (int i = 0; i < E; i += 128) {
            const uint4 q = *(const uint4 *)(row + i);
            const float4 x0 = *(const float4 *)(xt + i), x1 = *(const float4 *)(xt + i + 4);
            const uint32_t d[4] = {q.x, q.y, q.z, q.w};
            const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
            for (int k = 0; k < 4; k++) {
                acc += (double)g53_bitsf(d[k] << 16) * (double)xv[2 * k];
                acc += (double)g53_bitsf(d[k] & 0xffff0000u) * (double)xv[2 * k + 1];
            }
        }
        for (int o = 8; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
        if (l == 0 && e < NE) {
            const float s = g53_sigmoidf((float)acc);
            score[e] = s;
            choice[e] = s + bias[e];
        }
    }
    __syncthreads();
    if (threadIdx.x >= 64) return;
    g53_select_token<NV>(0, lane, idx + (size_t)t * K, w + (size_t)t * K, score, choice, nullptr, 1, bias, 1, NE, K,
                         norm_topk, routed_scale, nan_flag, 0, experts, shared,
                         slots ? slots + (size_t)t * (K + (shared ? 1 : 0)) : nullptr);
}

/* slots[t][j] = experts[idx[t][j]] (j < K), slots[t][K] = *shared: the descriptor table of
 * the expert kernels, for callers that route elsewhere. */
__global__ void k_resolve_slots(G53hExpert *__restrict__ slots, const G53hExpert *__restrict__ experts,
                                const int *__restrict__ idx, const G53hExpert *__restrict__ shared, int T,
                                int K, int nslots)
{
    const int words = (int)(sizeof(G53hExpert) / 4);
    const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (long)T * nslots * words) return;
    const int k = (int)(q % words), j = (int)((q / words) % nslots), t = (int)(q / ((long)words * nslots));
    const G53hExpert *src = j < K ? &experts[idx[(size_t)t * K + j]] : shared;
    ((int *)&slots[(size_t)t * nslots + j])[k] = ((const int *)src)[k];
}

int g53h_resolve_slots(G53hExpert *slots, const G53hExpert *experts, const int *idx, const G53hExpert *shared,
                       int T, int K)
{
    const int nslots = K + (shared ? 1 : 0);
    const long n = (long)T * nslots * (long)(sizeof(G53hExpert) / 4);
    hipLaunchKernelGGL(k_resolve_slots, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, g53h_stream(), slots,
                       experts, idx, shared, T, K, nslots);
    G53_LAUNCHED("k_resolve_slots");
    return 0;
}

/* Library-owned buffer of the split router's partial sums (grown as needed, kept). */
static void *g_router_part = nullptr;
static size_t g_router_part_bytes = 0;
static void *g53_router_part(size_t bytes)
{
    if (bytes <= g_router_part_bytes) return g_router_part;
    if (g_router_part) {
        if (hipStreamSynchronize(g53h_stream()) != hipSuccess || hipFree(g_router_part) != hipSuccess) {
            g53h_fail("g53h_router: cannot release the partial-sum buffer");
            return nullptr;
        }
        g_router_part = nullptr;
        g_router_part_bytes = 0;
    }
    if (hipMalloc(&g_router_part, bytes) != hipSuccess) {
        (void)hipGetLastError();
        g53h_fail("g53h_router: cannot allocate %zu bytes of partial sums", bytes);
        return nullptr;
    }
    g_router_part_bytes = bytes;
    return g_router_part;
}

/* A router of at most 128 KB, a workgroup per token: one launch where there were two (us; 16 experts x
 * 256: 1 token 6.6 -> 5.5, 8 tokens 8.3 -> 5.2; 64 x 1024: 8 tokens 9.0 -> 7.9; 128 x 512, 256 tokens:
 * 9.8 -> 8.8). One token of a larger one is faster over all its experts' workgroups (64 x 1024: 6.6,
 * here 7.4), more than 256 tokens and more experts over the matrix cores (64 x 1024, 320 tokens: 10.2,
 * here 11.7; 256 x 256, 64 tokens: 9.3, here 9.9). */
static bool g53_router_small(int T, int gate_dt, int NE, int E)
{
    return gate_dt == 1 && E % 128 == 0 && (long)NE * E <= (T == 1 ? 8192 : 65536) &&
           NE <= (T == 1 ? 32 : 128) && T <= 256;
}

/* Workgroups up to which a batch with few tiles splits its columns: 10 a CU where the selection takes every
 * range's sums in one flight of loads (288 experts x 4096, both launches, us: 150 tokens 22.7 at 640
 * workgroups, 20.2 at 2560; 256: 28.4, 24.4; 5120 is no faster), 2.5 a CU above 320 experts, where it takes
 * them range by range (1024 x 2048: 64 tokens 37.7 at 640, 66.5 at 2560; 512 x 4096, 150: 45.0, 59.0). */
static int g53_router_split_wgs(int NE) { return NE <= 320 ? 2560 : 640; }

/* Partial sums that a batch of at most T tokens may need over the column ranges (S T <= 16 workgroups /
 * et): a smaller batch after a larger one, a captured one for instance, allocates nothing. */
static size_t g53_router_part_need(int T, int NE, int E)
{
    const size_t et = (NE + 15) / 16, rows = min((size_t)8 * T, (size_t)16 * g53_router_split_wgs(NE) / et);
    return E % 512 == 0 ? rows * NE * sizeof(double) : 0;
}
size_t g53h_router_growth(int T, int gate_dt, int NE, int E)
{
    if (T < 2 || gate_dt != 1 || g53_router_small(T, gate_dt, NE, E)) return 0;
    const size_t n = g53_router_part_need(T, NE, E);
    return n <= g_router_part_bytes ? 0 : n;
}

int g53h_router_into(int *idx, float *w, const float *x, int T, const void *gate, int gate_dt,
                     const float *bias, int NE, int E, int K, int norm_topk, float routed_scale,
                     int *nan_flag, float *scratch, const G53hExpert *experts, const G53hExpert *shared,
                     G53hExpert *slots)
{
    if (NE < 1 || NE > 1024) return g53h_fail("g53h_router: %d experts (max 1024)", NE);
    if (K < 1 || K > NE || K > GLM53F_MAX_TOPK_DEV) return g53h_fail("g53h_router: topk %d", K);
    if (g53_router_small(T, gate_dt, NE, E) && (((uintptr_t)x | (uintptr_t)gate) & 15) == 0) {
        hipLaunchKernelGGL(k_router_small<2>, dim3(T), dim3(NE > 32 ? 1024 : 512), 0, g53h_stream(), idx, w, x,
                           (const uint16_t *)gate, bias, NE, E, K, norm_topk, routed_scale, nan_flag, experts, shared, slots);
        G53_LAUNCHED("k_router_small");
        return 0;
    }
    float *score = scratch, *choice = scratch + (size_t)T * NE;
    const double *psum = nullptr;                            /* split logits, summed by the selection */
    int nsum = 1;
    if (T >= 2 && gate_dt == 1 && E % 256 == 0) {           /* batches: the matrix-core form */
        /* few tiles (small T): the columns are split over up to 8 workgroups per tile; the partial sums are
         * added in column order after */
        const int tiles = ((NE + 15) / 16) * ((T + 15) / 16);
        int S = 1;
        while (S < 8 && tiles * S * 2 <= g53_router_split_wgs(NE) && (E / (S * 2)) % 256 == 0) S *= 2;
        double *part = nullptr;
        if (E % 512 == 0) {
            part = (double *)g53_router_part(g53_router_part_need(T, NE, E));
            if (!part) return -1;
            if (S == 1) part = nullptr;
        }
        /* The flat order with few expert tiles and activations that fill the 32 MB of L2 (experts x hidden, both
         * launches, us, grid / flat: 64 x 4096, 4096 tokens 64.0 / 56.8; 128 x 4096, 2048: 58.7 / 54.0; 24 x 2048,
         * 8192: 47.9 / 43.9; the 32 x 32 kernel before: 54.8, 52.1, 43.8), and where a grid has too few rows for
         * the tokens. More expert tiles gain nothing (288 x 4096, 2048: 102.3 / 102.7; 192 x 4096, 8192: 255.1 /
         * 254.9), smaller batches lose the index arithmetic's time (288 x 4096, 5: 11.7 / 12.0). */
        const int tt = (T + 15) / 16, fits = (long)tiles * S < (1 << 24) - 8;        /* 2^32 threads a launch */
        const int flat = fits && ((NE <= 160 && (long)T * E >= (8 << 20)) || tt > 65535);
        const dim3 grid = flat ? dim3((unsigned)(tiles * S + 7) / 8 * 8) : dim3((NE + 15) / 16, tt, S);
        hipLaunchKernelGGL(k_router_mfma, grid, dim3(256), 0, g53h_stream(), score, choice, x, T,
                           (const uint16_t *)gate, bias, NE, E, E / S, flat ? S : 0, part);
        G53_LAUNCHED("k_router_mfma");
        if (S > 1) { psum = part; nsum = S; }
    } else {
        hipLaunchKernelGGL(k_router_scores, dim3(NE, T), dim3(64), 0, g53h_stream(), score, choice, x, T, gate,
                           gate_dt, bias, NE, E);
        G53_LAUNCHED("k_router_scores");
    }
    /* the selection, after the sum of the column ranges when the logits were split */
    const dim3 gs((unsigned)((T + 3) / 4));
    if (NE <= 320)
        hipLaunchKernelGGL(k_router_select_w<5>, gs, dim3(256), 0, g53h_stream(), idx, w, score, choice, psum, nsum,
                           bias, T, NE, K, norm_topk, routed_scale, nan_flag, experts, shared, slots);
    else
        hipLaunchKernelGGL(k_router_select_w<16>, gs, dim3(256), 0, g53h_stream(), idx, w, score, choice, psum, nsum,
                           bias, T, NE, K, norm_topk, routed_scale, nan_flag, experts, shared, slots);
    G53_LAUNCHED("k_router_select_w");
    return 0;
}

extern "C" int g53h_router(int *idx, float *w, const float *x, int T, const void *gate, int gate_dt,
                           const float *bias, int NE, int E, int K, int norm_topk,
                           float routed_scale, int *nan_flag)
{
    if (g53h_ready()) return -1;
    if (T <= 0) return 0;
    float *ws = (float *)g53h_workspace((size_t)2 * T * (NE > 0 ? NE : 1) * sizeof(float));
    if (!ws) return -1;
    return g53h_router_into(idx, w, x, T, gate, gate_dt, bias, NE, E, K, norm_topk, routed_scale,
                            nan_flag, ws, nullptr, nullptr, nullptr);
}


/* Wave-wide argmax with the reference's rule: strictly greater wins, so the lowest index among
 * equal maxima; an empty candidate (index < 0) never wins. */
__device__ inline void g53_argmax_merge(float &bv, int &bi, float ov, int oi)
{
    if (oi < 0) return;
    if (bi < 0 || ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
}

__global__ void __launch_bounds__(64) k_route_topn(int *__restrict__ idx, int n,
                                                   const float *__restrict__ choice, int NE,
                                                   const float *__restrict__ score, float *__restrict__ score_out)
{
    g53_topn_token((int)blockIdx.x, (int)threadIdx.x, idx, n, choice, NE, score, score_out);
}

/* One decode token's routing and next-layer prediction in two launches: the scores of both
 * routers (blockIdx.y 0: this layer's, 1: the next layer's), then workgroup 0 selects the top-k
 * with weights and writes the NaN flag (0 or 1), workgroup 1 the next layer's top-n. */
__global__ void __launch_bounds__(64) k_router_scores2(float *__restrict__ sc0, float *__restrict__ ch0,
                                                       const void *__restrict__ g0, int dt0,
                                                       const float *__restrict__ b0,
                                                       float *__restrict__ sc1, float *__restrict__ ch1,
                                                       const void *__restrict__ g1, int dt1,
                                                       const float *__restrict__ b1, const float *__restrict__ x,
                                                       int NE, int E)
{
    const int lane = threadIdx.x, e = blockIdx.x, which = blockIdx.y;
    const float d = g53_router_dot(which ? g1 : g0, which ? dt1 : dt0, e, E, x, lane);
    if (lane == 0) {
        const float s = g53_sigmoidf(d);
        (which ? sc1 : sc0)[e] = s;
        (which ? ch1 : ch0)[e] = s + (which ? b1 : b0)[e];
    }
}

template <int NV>
__global__ void __launch_bounds__(128) k_route_decode(int *__restrict__ idx, float *__restrict__ w,
                                                      int *__restrict__ nan_flag, float *__restrict__ score,
                                                      float *__restrict__ choice, const float *__restrict__ bias,
                                                      int NE, int K, int norm_topk, float routed_scale,
                                                      int *__restrict__ pred, int n, const float *__restrict__ nscore,
                                                      const float *__restrict__ nchoice, unsigned *__restrict__ mb,
                                                      int mb_slot, int mb_off_w, unsigned seq)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (wave == 0)
        g53_select_token<NV>(0, lane, idx, w, score, choice, nullptr, 1, bias, 1, NE, K, norm_topk, routed_scale,
                             nan_flag, 1, nullptr, nullptr, nullptr);
    else if (n > 0)
        g53_topn_token(0, lane, pred, n, nchoice, NE, nscore, nullptr);
    if (!mb) return;
    /* the host's copy: idx [K], the flag, pred [n], then the sequence word */
    __threadfence_block();
    __syncthreads();
    unsigned *d = mb + mb_off_w;
    for (int i = threadIdx.x; i < K + 1 + n; i += 128)
        d[i] = (unsigned)(i < K ? idx[i] : i == K ? nan_flag[0] : pred[i - K - 1]);
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(mb + mb_slot, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

/* The prefill prediction's vote (src/core/glm53f_ops.c:1206-1225): the experts named in ids
 * [T][n] ordered by how many tokens named them, most first, ties in the order of their first
 * appearance (t, then j). out[0] = the number of distinct experts, out[1 + r] = the expert of
 * rank r. One workgroup: counts and first positions in LDS, then each expert's rank counted
 * against every other. */
__global__ void __launch_bounds__(1024) k_vote(int *__restrict__ out, const int *__restrict__ ids, int T, int n,
                                               int NE)
{
    __shared__ int votes[1024], first[1024];
    for (int e = threadIdx.x; e < NE; e += 1024) { votes[e] = 0; first[e] = 0x7fffffff; }
    __syncthreads();
    for (int q = threadIdx.x; q < T * n; q += 1024) {
        const int e = ids[q];
        if (e < 0 || e >= NE) continue;
        atomicAdd(&votes[e], 1);
        atomicMin(&first[e], q);
    }
    __syncthreads();
    int distinct = 0;
    for (int e = threadIdx.x; e < NE; e += 1024) {                   /* NE <= 1024 */
        const int v = votes[e];
        if (!v) continue;
        const int f = first[e];
        int r = 0;
        for (int o = 0; o < NE; o++) {
            const int vo = votes[o];
            r += vo > v || (vo == v && vo && first[o] < f);
        }
        out[1 + r] = e;
    }
    if (threadIdx.x < NE) distinct = votes[threadIdx.x] != 0;        /* NE <= 1024: one each */
    const int total = __syncthreads_count(distinct);
    if (threadIdx.x == 0) out[0] = total;
}

extern "C" int g53h_route_topn(int *idx, int n, const float *x, const void *gate, int gate_dt,
                               const float *bias, int NE, int E)
{
    if (g53h_ready()) return -1;
    if (n <= 0) return 0;
    if (NE < 1 || NE > 64 * G53_SEL_PER_LANE) return g53h_fail("g53h_route_topn: %d experts", NE);
    float *ws = (float *)g53h_workspace((size_t)2 * NE * sizeof(float));
    if (!ws) return -1;
    hipLaunchKernelGGL(k_router_scores, dim3(NE, 1), dim3(64), 0, g53h_stream(), ws + NE, ws, x, 1, gate,
                       gate_dt, bias, NE, E);
    G53_LAUNCHED("k_router_scores");
    hipLaunchKernelGGL(k_route_topn, dim3(1), dim3(64), 0, g53h_stream(), idx, n, ws, NE, ws + NE, nullptr);
    G53_LAUNCHED("k_route_topn");
    return 0;
}

extern "C" int g53h_route_topn_batch(int *idx, float *score_out, int n, const float *x, int T, const void *gate,
                                     int gate_dt, const float *bias, int NE, int E)
{
    if (g53h_ready()) return -1;
    if (n <= 0 || T <= 0) return 0;
    if (NE < 1 || NE > 64 * G53_SEL_PER_LANE) return g53h_fail("g53h_route_topn_batch: %d experts", NE);
    if (n > NE) return g53h_fail("g53h_route_topn_batch: %d of %d experts", n, NE);
    float *ws = (float *)g53h_workspace((size_t)2 * T * NE * sizeof(float));
    if (!ws) return -1;
    float *choice = ws, *score = ws + (size_t)T * NE;
    hipLaunchKernelGGL(k_router_scores, dim3(NE, T), dim3(64), 0, g53h_stream(), score, choice, x, T, gate,
                       gate_dt, bias, NE, E);
    G53_LAUNCHED("k_router_scores");
    hipLaunchKernelGGL(k_route_topn, dim3(T), dim3(64), 0, g53h_stream(), idx, n, choice, NE, score, score_out);
    G53_LAUNCHED("k_route_topn");
    return 0;
}

extern "C" int g53h_vote(int *out, const int *ids, int T, int n, int NE)
{
    if (g53h_ready()) return -1;
    if (NE < 1 || NE > 1024) return g53h_fail("g53h_vote: %d experts", NE);
    if (T < 0 || n < 0) return g53h_fail("g53h_vote: %d x %d ids", T, n);
    hipLaunchKernelGGL(k_vote, dim3(1), dim3(1024), 0, g53h_stream(), out, ids, T, n, NE);
    G53_LAUNCHED("k_vote");
    return 0;
}

extern "C" int g53h_route_decode(int *idx, float *w, int *nan_flag, int *pred, int n, const float *x, const void *gate,
                                 int gate_dt, const float *bias, const void *next_gate, int next_dt,
                                 const float *next_bias, int NE, int E, int K, int norm_topk, float routed_scale,
                                 int mb_slot, unsigned seq, size_t mb_off)
{
    if (g53h_ready()) return -1;
    if (NE < 1 || NE > 1024) return g53h_fail("g53h_route_decode: %d experts (max 1024)", NE);
    if (K < 1 || K > NE || K > GLM53F_MAX_TOPK_DEV) return g53h_fail("g53h_route_decode: topk %d", K);
    const int pn = next_gate && n > 0;
    if (pn && n > NE) return g53h_fail("g53h_route_decode: %d of %d experts", n, NE);
    if (!pn) n = 0;
    if (mb_slot >= 0 && (mb_slot >= G53H_MBOX_SLOTS || mb_off % 4 || mb_off < G53H_MBOX_SLOTS * 4 ||
                         mb_off + 4 * (size_t)(K + 1 + n) > G53H_MBOX_BYTES))
        return g53h_fail("g53h_route_decode: mailbox slot %d offset %zu", mb_slot, mb_off);
    float *ws = (float *)g53h_workspace((size_t)4 * NE * sizeof(float));
    if (!ws) return -1;
    float *sc0 = ws, *ch0 = ws + NE, *sc1 = ws + 2 * NE, *ch1 = ws + 3 * NE;
    hipLaunchKernelGGL(k_router_scores2, dim3(NE, pn ? 2 : 1), dim3(64), 0, g53h_stream(), sc0, ch0, gate, gate_dt,
                       bias, sc1, ch1, pn ? next_gate : gate, next_dt, pn ? next_bias : bias, x, NE, E);
    G53_LAUNCHED("k_router_scores2");
    unsigned *mb = mb_slot >= 0 ? g53h_mailbox_dev() : nullptr;
    const int off_w = (int)(mb_off / 4);
    if (NE <= 320)
        hipLaunchKernelGGL(k_route_decode<5>, dim3(1), dim3(128), 0, g53h_stream(), idx, w, nan_flag, sc0, ch0, bias,
                           NE, K, norm_topk, routed_scale, pred, n, sc1, ch1, mb, mb_slot, off_w, seq);
    else
        hipLaunchKernelGGL(k_route_decode<16>, dim3(1), dim3(128), 0, g53h_stream(), idx, w, nan_flag, sc0, ch0, bias,
                           NE, K, norm_topk, routed_scale, pred, n, sc1, ch1, mb, mb_slot, off_w, seq);
    G53_LAUNCHED("k_route_decode");
    if (mb) g53h_note_publish(mb_slot, seq);
    return 0;
}

/* ------------------------------------------------- speculative decode: next scores, publish ---- */
static float *g_next = nullptr;          /* [2][1024]: choice (score + bias), then score */
static G53NextReq g_next_req;

float *g53h_next_buf(void)
{
    if (!g_next) g_next = (float *)g53h_alloc(2 * 1024 * sizeof(float));
    return g_next;
}
G53NextReq *g53h_next_req(void) { return &g_next_req; }


extern "C" int g53h_decode_next(const float *x, const void *next_gate, int next_dt, const float *next_bias, int NE,
                                int E)
{
    if (g53h_ready()) return -1;
    if (NE < 1 || NE > 1024 || !x || !next_gate || !next_bias)
        return g53h_fail("g53h_decode_next: %d experts (max 1024)", NE);
    if (!g53h_next_buf()) return -1;
    g_next_req = G53NextReq{1, x, next_gate, next_dt, next_bias, NE, E};
    return 0;
}

extern "C" int g53h_route_next(const float *x, const void *next_gate, int next_dt, const float *next_bias, int NE,
                               int E)
{
    if (g53h_ready()) return -1;
    if (NE < 1 || NE > 1024) return g53h_fail("g53h_route_next: %d experts (max 1024)", NE);
    if (!g53h_next_buf()) return -1;
    hipLaunchKernelGGL(k_router_scores, dim3(NE, 1), dim3(64), 0, g53h_stream(), g_next + 1024, g_next, x, 1,
                       next_gate, next_dt, next_bias, NE, E);
    G53_LAUNCHED("k_router_scores");
    return 0;
}

/* Wave 0 takes the next layer's top-n (the selection of k_route_decode, src/core/glm53f_ops.c:
 * 1021-1042), then the workgroup writes the host's copy: idx [K], the NaN flag, pred [n] at
 * route_off_w; the error words and the output at out_off_w; then the sequence word. */
__global__ void __launch_bounds__(256) k_dec_publish(unsigned *__restrict__ mb, int slot, unsigned seq,
                                                     int route_off_w, const int *__restrict__ idx, int K,
                                                     int *__restrict__ pred, int n, const float *__restrict__ choice,
                                                     const float *__restrict__ score, int NE, int out_off_w,
                                                     const uint32_t *__restrict__ out, int nw,
                                                     const int *__restrict__ errs)
{
    /* wave 0 the top-n while the other waves copy the error words and the output */
    if (threadIdx.x < 64) {
        if (n > 0) g53_topn_token(0, (int)threadIdx.x, pred, n, choice, NE, score, nullptr);
    } else {
        uint32_t *d = mb + out_off_w;
        for (int i = threadIdx.x - 64; i < G53H_NERR; i += 192) d[i] = (uint32_t)errs[i];
        g53_copy_words(d + G53H_NERR, out, nw, (int)threadIdx.x - 64, 192);
    }
    __threadfence_block();
    __syncthreads();
    unsigned *r = mb + route_off_w;
    const int nan = ((errs[0] | errs[1]) & 2) ? 1 : 0;
    for (int i = threadIdx.x; i < K + 1 + n; i += 256)
        r[i] = (unsigned)(i < K ? idx[i] : i == K ? nan : pred[i - K - 1]);
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(mb + slot, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

/* The mailbox areas of a publication: in range, word-aligned, not overlapping. */
static int pub_areas_bad(int slot, size_t route_off, int K, int n, size_t out_off, size_t out_bytes)
{
    return slot < 0 || slot >= G53H_MBOX_SLOTS || route_off % 4 || out_off % 4 || out_bytes % 4 ||
           route_off < G53H_MBOX_SLOTS * 4 || out_off < G53H_MBOX_SLOTS * 4 ||
           route_off + 4 * (size_t)(K + 1 + n) > G53H_MBOX_BYTES || out_off + 4 * G53H_NERR + out_bytes > G53H_MBOX_BYTES ||
           (route_off < out_off + 4 * G53H_NERR + out_bytes && out_off < route_off + 4 * (size_t)(K + 1 + n));
}

extern "C" int g53h_decode_publish(int slot, unsigned seq, size_t route_off, const int *idx_d, int K, int *pred_d,
                                   int n, int NE, size_t out_off, const void *out_d, size_t out_bytes)
{
    if (g53h_ready()) return -1;
    if (K < 1 || K > GLM53F_MAX_TOPK_DEV || n < 0 || n > NE || NE < 1 || NE > 1024 || (n > 0 && (!g_next || !pred_d)))
        return g53h_fail("g53h_decode_publish: topk %d, n %d of %d experts (g53h_route_next first)", K, n, NE);
    if (g_next_req.armed) {          /* requested, and no decode launch computed them */
        g_next_req.armed = 0;
        if (g_next_req.NE != NE ||
            g53h_route_next(g_next_req.x, g_next_req.gate, g_next_req.dt, g_next_req.bias, g_next_req.NE, g_next_req.E))
            return g53h_fail("g53h_decode_publish: the next layer's scores (%d experts) cannot be computed", NE);
    }
    if (pub_areas_bad(slot, route_off, K, n, out_off, out_bytes))
        return g53h_fail("g53h_decode_publish: slot %d, routing at %zu, %zu bytes at %zu", slot, route_off, out_bytes,
                         out_off);
    hipLaunchKernelGGL(k_dec_publish, dim3(1), dim3(256), 0, g53h_stream(), g53h_mailbox_dev(), slot, seq,
                       (int)(route_off / 4), idx_d, K, pred_d, n, g_next, g_next + 1024, NE, (int)(out_off / 4),
                       (const uint32_t *)out_d, (int)(out_bytes / 4), g53h_errblock());
    G53_LAUNCHED("k_dec_publish");
    g53h_note_publish(slot, seq);
    return 0;
}
