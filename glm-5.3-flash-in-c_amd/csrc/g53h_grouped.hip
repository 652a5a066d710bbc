/* g53h_grouped.hip - batched decode and prefill of the routed-expert MoE layer on gfx950:
 * token-sorted grouped GEMMs on the CDNA4 FP8 matrix cores.
 *
 * The reference runs a chunk of tokens expert by expert (src/core/glm53f_ops.c:1144-1342,
 * moe_chunk): route every token, gather the tokens of each chosen expert, apply gate/up,
 * the clamped SwiGLU and down to that group (matmul_f8_batch, :376-444), then combine each
 * token's slots in double in top-k order and add the shared expert (:1329-1340). This file
 * does the same with every expert's weights read from HBM once per call:
 *
 *   1. router             the exact router kernels of g53h_ops.hip (top-k bit-exact).
 *   2. k_grp_prep         counting sort of the (token, slot) pairs by expert, stable in token
 *                         order; segment e holds expert e's tokens, segment NE the shared
 *                         expert's (every token); a tile is <= 64 consecutive positions of one
 *                         segment.
 *   3. (same launch)      each token's activations as NPX E4M3 planes with a power-of-two
 *                         token scale: x = 2^-k (q0 + q1 / 16 + q2 / 256 ...). For bf16-valued
 *                         inputs two planes hold x exactly (8 significant bits = 4 + 4).
 *   4. k_grp_gemm<true>   per (tile, 128-row block): gate and up rows of the expert times the
 *                         tile's tokens on v_mfma_scale_f32_32x32x64_f8f6f4, one 128x128 scale
 *                         block per step, the block scale applied to each block's fp32 sum;
 *                         SwiGLU in the epilogue; the activation leaves as NPA E4M3 planes with
 *                         a fixed power-of-two scale (|act| <= max(limit, 0.28) * limit).
 *   5. k_grp_gemm<false>  per (tile, 256-row block): down rows times the activation planes;
 *                         contributions to contrib[position][hidden] (zeros for an absent
 *                         expert, the reference's drop path).
 *   6. k_grp_combine      out[t] = (float)(sum_j (double)w[t][j] * contrib[pos(t, j)]) in slot
 *                         order, then + shared contribution (float), as :1329-1340.
 *
 * Arithmetic: E4M3 x E4M3 products are exact in fp32; the matrix core sums them in fp32 in
 * its own order. So results differ from the reference's (fp32 FMA lanes, double block sums)
 * by fp32 summation order and by the activation planes' rounding, inside the tolerance the
 * path is held to (2e-3 relative + 1e-2 absolute per output). Routing is bit-exact.
 *
 * Operand layout of the 32x32x64 FP8 matrix instruction (one wave): lane l supplies row
 * l % 32 of A and column l % 32 of B, 32 K-bytes each, from K group l / 32; both operands use
 * the same K assignment, so any fixed map of K bytes to (group, byte) gives the same dot
 * product. Here group g of step s covers bytes g*64 + s*32 .. +32 of a 128-byte scale block,
 * so a lane reads 64 consecutive bytes of its weight row per block. Result: lane l, register
 * r holds C[8*(r/4) + 4*(l/32) + r%4][l % 32].
 *
 * Octet-tiled layers (G53H_MAT_TILED, the HBM cache's slots): a row's 128 bytes of a block are
 * the tiled unit's row, whose byte b holds column sigma(b / 16) + 8 (b % 16) of the block
 * (include/g53h.h). The activation planes are then written in that same order within every
 * 128-column block, so weight byte b meets activation byte b as before, and a wave's 32 rows of
 * a block are four whole 1 KB units instead of 32 rows 4 KB apart.
 */
#include <hip/hip_runtime.h>
#include <math.h>

#include "g53h.h"
#include "g53h_core.h"
#include "g53h_kern.h"
#include "g53h_runtime.h"

typedef int g53_v8i __attribute__((ext_vector_type(8)));
typedef float g53_v16f __attribute__((ext_vector_type(16)));
typedef int g53_v4i __attribute__((ext_vector_type(4)));

#define G53_GRP_NT    64      /* positions per tile                                        */
#define G53_GRP_MAXT  2048    /* tokens per planning pass                                   */
#define G53_GRP_NPX   2       /* E4M3 planes of the input activations                       */
#define G53_GRP_NPA   2       /* E4M3 planes of the SwiGLU activations                      */
#define G53_GRP_MASKS 12288   /* LDS 64-token masks of the planner (chunks x experts)       */
#define G53_GRP_NW    8       /* waves of a GEMM workgroup                                   */
/* error flags (meta[1]) */
#define G53_GRP_EIDX  1       /* a routed index outside [0, n_experts)                      */
#define G53_GRP_EDESC 8       /* an expert descriptor without the expected 128x128 layout   */

/* ------------------------------------------------------------------ planning ---- */
/* meta[]: [0] tiles, [1] error flags, then the first item of each XCD's range (9 entries: XCD x
 * takes items [b[x], b[x+1])) for gate/up and for down */
#define G53_GRP_BGU   2
#define G53_GRP_BDN   11

/* Estimated cost of one row of a segment's items (one item per tile) with n positions, in
 * tenths of the time of a tile of at most 32 positions (37 us; up to 64 positions 44 us). */
__device__ __forceinline__ int g53_grp_tile_cost(int n) { return n <= 32 ? 10 : 12; }
__device__ __forceinline__ int g53_grp_seg_cost(int n)
{
    const int full = n / G53_GRP_NT, rem = n % G53_GRP_NT;
    return full * g53_grp_tile_cost(G53_GRP_NT) + (rem ? g53_grp_tile_cost(rem) : 0);
}

/* Counting sort of the T*K (token, slot) pairs by expert, stable in token order. For each
 * chunk c of 64 tokens and expert e, mask[c][e] has bit t%64 set when token t chose e; the
 * position of (t, e) is off[e] + (tokens of e in earlier chunks) + popcount(mask bits below
 * t). One workgroup of 1024 threads; dynamic LDS sized by the host. */
__device__ void g53_grp_plan(uint64_t *pl_lds, const int *__restrict__ idx, int T, int K, int NE, int has_sh,
                             int *__restrict__ tok_of, int *__restrict__ pos_of, int4 *__restrict__ tiles,
                             int *__restrict__ meta, int mb_gu, int mb_dn)
{
    const int nch = (T + 63) >> 6, nm = nch * NE, tid = threadIdx.x;
    uint64_t *mask = pl_lds;
    int *pre = (int *)(mask + nm);                 /* [nch][NE]                              */
    int *off = pre + nm;                           /* [NE + 2]: segment offsets              */
    int *tb = off + NE + 2;                        /* [NE + 2]: first tile of each segment   */
    int *pc = tb + NE + 2;                         /* [NE + 2]: cost of the segments before  */
    const int nseg = NE + (has_sh ? 1 : 0);
    for (int i = tid; i < nm; i += 1024) mask[i] = 0;
    __syncthreads();
    int bad = 0;
    for (int f = tid; f < T * K; f += 1024) {
        const int t = f / K, e = idx[f];
        if (e < 0 || e >= NE) { bad = 1; continue; }
        atomicOr((unsigned long long *)&mask[(t >> 6) * NE + e], 1ull << (t & 63));
    }
    if (bad) atomicOr(&meta[1], G53_GRP_EIDX);
    __syncthreads();
    /* per expert: tokens in earlier chunks, and the count (into off[] for the scan below) */
    for (int e = tid; e < NE; e += 1024) {
        int run = 0;
        for (int c = 0; c < nch; c++) {
            pre[c * NE + e] = run;
            run += __popcll(mask[c * NE + e]);
        }
        off[e] = run;
    }
    if (tid == 0) off[NE] = has_sh ? T : 0;
    __syncthreads();
    /* exclusive scans of counts and tile counts by the first wave, 64 segments per round */
    if (tid < 64) {
        int cp = 0, ct = 0, cc = 0;
        for (int b = 0; b < nseg; b += 64) {
            const int s = b + tid;
            const int n = s < nseg ? off[s] : 0;
            const int c = g53_grp_seg_cost(n);
            int ip = n, it = (n + G53_GRP_NT - 1) / G53_GRP_NT, ic = c;
            for (int d = 1; d < 64; d <<= 1) {
                const int up = __shfl_up(ip, d), ut = __shfl_up(it, d), uc = __shfl_up(ic, d);
                if (tid >= d) { ip += up; it += ut; ic += uc; }
            }
            if (s < nseg) {
                off[s] = cp + ip - n;
                tb[s] = ct + it - (n + G53_GRP_NT - 1) / G53_GRP_NT;
                pc[s] = cc + ic - c;
            }
            cp += __shfl(ip, 63);
            ct += __shfl(it, 63);
            cc += __shfl(ic, 63);
        }
        if (tid == 0) { off[nseg] = cp; tb[nseg] = ct; pc[nseg] = cc; meta[0] = ct; }
    }
    __syncthreads();
    /* each XCD's item range, of equal estimated cost: lanes 0-8 for gate/up, 16-24 for down */
    if (tid < 32 && (tid & 15) <= 8) {
        const int x = tid & 15, MB = tid < 16 ? mb_gu : mb_dn;
        int item;
        if (x == 0) item = 0;
        else if (x == 8) item = tb[nseg] * MB;
        else {
            const long long tau = (long long)pc[nseg] * x / 8;   /* target, in units of one row of items */
            int lo = 0, hi = nseg;                                /* the last segment with pc <= tau */
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (pc[mid] <= tau) lo = mid; else hi = mid - 1;
            }
            item = tb[lo] * MB;
            if (lo < nseg) {
                const int rc = pc[lo + 1] - pc[lo], nts = tb[lo + 1] - tb[lo];
                const long long j = rc > 0 ? ((tau - pc[lo]) * MB) / rc : 0;   /* whole rows of items */
                item += (int)(j < MB ? j : MB) * nts;
            }
        }
        meta[(tid < 16 ? G53_GRP_BGU : G53_GRP_BDN) + x] = item;
    }
    __syncthreads();
    const int ps = K + 1;
    for (int f = tid; f < T * K; f += 1024) {
        const int t = f / K, j = f % K, e = idx[f];
        if (e < 0 || e >= NE) { pos_of[t * ps + j] = -1; continue; }
        const int c = t >> 6;
        const uint64_t m = mask[c * NE + e];
        const int pos = off[e] + pre[c * NE + e] + __popcll(m & ((1ull << (t & 63)) - 1ull));
        pos_of[t * ps + j] = pos;
        tok_of[pos] = t;
    }
    if (has_sh)
        for (int t = tid; t < T; t += 1024) {
            const int pos = off[NE] + t;
            pos_of[t * ps + K] = pos;
            tok_of[pos] = t;
        }
    for (int s = tid; s < nseg; s += 1024) {
        const int n = off[s + 1] - off[s];
        const int nt = (n + G53_GRP_NT - 1) / G53_GRP_NT;
        for (int i = 0; i < nt; i++) {
            const int m = n - i * G53_GRP_NT;
            tiles[tb[s] + i] = make_int4(s, off[s] + i * G53_GRP_NT, m < G53_GRP_NT ? m : G53_GRP_NT, tb[s] | nt << 16);
        }
    }
}

/* ------------------------------------------------------------ E4M3 planes ---- */
/* Four values v[0..3] (already scaled into E4M3 range) as NP planes of packed E4M3 bytes:
 * plane p holds round(r_p * 16^p), r_0 = v, r_{p+1} = r_p - plane p's value / 16^p. */
template <int NP>
__device__ __forceinline__ void g53_split_planes(const float (&v)[4], uint32_t (&out)[NP])
{
    float r[4] = {v[0], v[1], v[2], v[3]};
#pragma unroll
    for (int p = 0; p < NP; p++) {
        int w = __builtin_amdgcn_cvt_pk_fp8_f32(r[0], r[1], 0, false);
        w = __builtin_amdgcn_cvt_pk_fp8_f32(r[2], r[3], w, true);
        out[p] = (uint32_t)w;
        if (p + 1 < NP) {
            r[0] = (r[0] - __builtin_amdgcn_cvt_f32_fp8(w, 0)) * 16.0f;
            r[1] = (r[1] - __builtin_amdgcn_cvt_f32_fp8(w, 1)) * 16.0f;
            r[2] = (r[2] - __builtin_amdgcn_cvt_f32_fp8(w, 2)) * 16.0f;
            r[3] = (r[3] - __builtin_amdgcn_cvt_f32_fp8(w, 3)) * 16.0f;
        }
    }
}

/* Byte position of column c of a 128-column block in the octet-tiled order: run sigma(c % 8)
 * (sigma is its own inverse), element c / 8 of the run. */
__device__ __forceinline__ int g53_grp_tpos(int c)
{
    const int a = c & 7;
    return 16 * (((a & 1) << 2) | (a & 2) | (a >> 2)) + (c >> 3);
}

/* Four consecutive E4M3 codes (one word, column c0 .. c0 + 3 of a row) stored at dst: as they
 * are, or (tiled) each at its octet-tiled position within its 128-column block. */
__device__ __forceinline__ void g53_grp_st4(uint8_t *row, int c0, uint32_t q, int tiled)
{
    if (!tiled) {
        *(uint32_t *)(row + c0) = q;
        return;
    }
    uint8_t *blk = row + (c0 & ~127);
#pragma unroll
    for (int k = 0; k < 4; k++) blk[g53_grp_tpos((c0 + k) & 127)] = (uint8_t)(q >> (8 * k));
}

typedef float g53_v4f __attribute__((ext_vector_type(4)));

/* A token's row of x as NPX planes xq[p][t][E] with scale 2^k, k = 8 - exponent(absmax), so
 * every |x| * 2^k < 256; xinv[t] = 2^-k. 256 threads a token, tg of them this one; the workgroup's
 * four tokens share its barrier. E at most 4096, a multiple of 16: the row stays in registers. */
template <int NP>
__device__ __forceinline__ void g53_grp_xq(float *red, const float *__restrict__ x, int E, int T, int t, int tg,
                                           uint8_t *__restrict__ xq, float *__restrict__ xinv, int tiled)
{
    const float *xr = x + (size_t)min(t, T - 1) * E;
    g53_v4f v[4];
    float m = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int i = tg * 4 + q * 1024;
        v[q] = i < E ? *(const g53_v4f *)(xr + i) : g53_v4f{0.f, 0.f, 0.f, 0.f};
        m = fmaxf(m, fmaxf(fmaxf(fabsf(v[q][0]), fabsf(v[q][1])), fmaxf(fabsf(v[q][2]), fabsf(v[q][3]))));
    }
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    float *rt = red + (threadIdx.x >> 8) * 4;
    if ((tg & 63) == 0) rt[tg >> 6] = m;
    __syncthreads();
    if (t >= T) return;
    m = fmaxf(fmaxf(rt[0], rt[1]), fmaxf(rt[2], rt[3]));
    int ex = 0;
    if (m > 0.0f && m <= 3.0e38f) (void)frexpf(m, &ex);          /* m < 2^ex */
    const int k = 8 - ex;
    const float sc = ldexpf(1.0f, k);
    if (tg == 0) xinv[t] = ldexpf(1.0f, -k);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int i = tg * 4 + q * 1024;
        if (i >= E) break;
        const float s[4] = {v[q][0] * sc, v[q][1] * sc, v[q][2] * sc, v[q][3] * sc};
        uint32_t pq[NP];
        g53_split_planes<NP>(s, pq);
#pragma unroll
        for (int p = 0; p < NP; p++) g53_grp_st4(xq + ((size_t)p * T + t) * E, i, pq[p], tiled);
    }
}

/* Workgroup 0 plans, the others take four tokens' planes each, in one launch: neither needs the
 * other's result. Both are short chains of latencies (with 5 tokens 6.0 and 4.7 us, with 2048 25 and
 * 17.5, one after the other before). Grid 1 + ceil(T / 4). */
__global__ void __launch_bounds__(1024)
k_grp_prep(const int *__restrict__ idx, int T, int K, int NE, int has_sh, int *__restrict__ tok_of,
           int *__restrict__ pos_of, int4 *__restrict__ tiles, int *__restrict__ meta, int mb_gu, int mb_dn,
           const float *__restrict__ x, int E, uint8_t *__restrict__ xq, float *__restrict__ xinv, int tiled)
{
    extern __shared__ __attribute__((aligned(16))) uint64_t pl_lds[];
    if (blockIdx.x == 0)
        g53_grp_plan(pl_lds, idx, T, K, NE, has_sh, tok_of, pos_of, tiles, meta, mb_gu, mb_dn);
    else
        g53_grp_xq<G53_GRP_NPX>((float *)pl_lds, x, E, T, ((int)blockIdx.x - 1) * 4 + (int)(threadIdx.x >> 8),
                                threadIdx.x & 255, xq, xinv, tiled);
}

/* ------------------------------------------------------------- grouped GEMM ---- */
/* Both GEMMs share one pipeline. A workgroup is 8 waves and stays for the whole launch, one per
 * CU; it walks its items (256 weight rows x one tile) as one stream of steps of 128 weight columns.
 * A step's operands - 256 rows x 128 codes, and the tile's positions x 128 codes x 2 planes - go
 * straight to LDS (global_load_lds, 1 KB a wave instruction), into a ring of three slots, three steps
 * ahead, across item boundaries: no registers hold loads in flight, every code is fetched as part
 * of a whole 128-byte run, and one barrier per step hands a slot over. The waits count loads by
 * hand, so the loads are inline assembly: the compiler would wait for every LDS load before any
 * LDS read. Everything else a step needs comes by scalar loads, which have a counter of their own.
 *
 * LDS rows are 128 bytes, 16-byte piece c of row r at piece c ^ ((r / 2) % 8): the 16 lanes of one
 * LDS access read piece c of 16 consecutive rows and meet no bank twice.
 *
 * Wave w multiplies 64 of the 256 rows (row group w % 4: two matrix-core tiles) by the 32 positions
 * of half w / 4, so a tile of up to 32 positions occupies one wave of each SIMD.
 */
#define G53_GRP_SA   (256 * 128)                      /* a slot's weight rows                     */
#define G53_GRP_PL   (G53_GRP_NT * 128)               /* one plane of the slot's positions        */
#define G53_GRP_SLOT (G53_GRP_SA + 2 * G53_GRP_PL)
#define G53_GRP_NS   3
static_assert(G53_GRP_NT == 64 && G53_GRP_NPX == 2 && G53_GRP_NPA == 2 && G53_GRP_NW == 8, "slot and wave layout");

/* A value every lane reads alike from memory that no kernel of this launch writes: a scalar load. */
template <class V>
__device__ __forceinline__ V g53_sld(const V *p)
{
    return *(const __attribute__((address_space(4))) V *)(uintptr_t)p;
}

/* A wave's four octets of weight rows (1 KB each, 16 bytes per lane at base + v0 .. v3) to LDS bytes
 * lds, lds + 1024, ...; nt: streamed once. M0 holds the LDS address and must be written ahead of the
 * load that uses it. */
#define G53_DMA_ROWS(NT)                                                                                       \
    asm volatile("s_mov_b32 m0, %5\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %0, %4" NT                            \
                 "\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 1\n\tglobal_load_lds_dwordx4 %1, %4" NT                 \
                 "\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 1\n\tglobal_load_lds_dwordx4 %2, %4" NT                 \
                 "\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 1\n\tglobal_load_lds_dwordx4 %3, %4" NT                 \
                 :: "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "s"(base), "s"(lds) : "memory", "m0", "scc")
__device__ __forceinline__ void g53_dma_rows(const uint32_t (&v)[4], const uint8_t *base, uint32_t lds)
{
    G53_DMA_ROWS("");
}
__device__ __forceinline__ void g53_dma_rows_nt(const uint32_t (&v)[4], const uint8_t *base, uint32_t lds)
{
    G53_DMA_ROWS(" nt");
}
#undef G53_DMA_ROWS
/* 16 bytes per lane from base + off to LDS byte lds + 16 * lane. */
__device__ __forceinline__ void g53_dma16(uint32_t off, const uint8_t *base, uint32_t lds)
{
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %0, %1"
                 :: "v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
/* 4 bytes per lane from p to LDS byte lds + 4 * lane. */
__device__ __forceinline__ void g53_dma4(const float *p, uint32_t lds)
{
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 4\n\tglobal_load_lds_dword %0, off"
                 :: "v"(p), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void g53_grp_bar()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

/* A descriptor with the layout the grouped kernels assume: exactly the pass's. */
__device__ __forceinline__ bool g53_grp_mat_ok(const G53hMat *m, int rows, int cols, int tiled)
{
    const int fl = g53_sld(&m->flags);
    const int want = tiled == 2 ? G53H_MAT_MTILED : tiled ? G53H_MAT_TILED : 0;
    return (fl & (G53H_MAT_I4 | G53H_MAT_I4T | G53H_MAT_TILED | G53H_MAT_MTILED)) == want && g53_sld(&m->br) == 128 &&
           g53_sld(&m->bc) == 128 && g53_sld(&m->rows) == rows && g53_sld(&m->cols) == cols &&
           g53_sld(&m->scols) >= cols / 128;
}
__device__ __forceinline__ bool g53_grp_desc_ok(const G53hExpert *x, int E, int I, int tiled)
{
    return g53_grp_mat_ok(&x->gate, I, E, tiled) && g53_grp_mat_ok(&x->up, I, E, tiled) &&
           g53_grp_mat_ok(&x->down, E, I, tiled);
}

template <int N>
struct G53Int {
    static constexpr int value = N;
};

struct G53GrpArgs {
    const G53hExpert *experts;     /* [NE]                                               */
    const G53hExpert *shared;      /* or NULL                                            */
    const int4 *tiles;             /* {segment, first position, count, first tile of the
                                      segment | tiles of the segment << 16}                */
    const int *meta;               /* [0] tile count, [1] error flags                    */
    int *meta_w;
    const int *tok_of;             /* [P]: position -> token                             */
    const uint8_t *xq;             /* [NPX][T][E]                                        */
    const float *xinv;             /* [T]: the tokens' scales                            */
    uint8_t *aq;                   /* [NPA][P][I]                                        */
    float *contrib;                /* [P][E]                                             */
    int T, P, E, I, NE;
    float limit, aq_scale, aq_inv;
    int tiled;                     /* 1: experts octet-tiled, planes in the tiled column order;
                                      2: experts MFMA-tiled, planes in column order        */
    int partial;                   /* 1: experts without weights are outside this batch and
                                      left alone, unless marked dropped (gate.flags & G53H_MAT_DROPPED)    */
    uint64_t *trace;               /* optional: [items][8] timestamps of each gate/up item   */
};

/* The clamped SwiGLU of src/core/glm53f_ops.c:486-494 (gate clamped from above, up both ways)
 * with the hardware exponential: the result is rounded to two E4M3 planes (about 8 significant
 * bits) right after, so the reference's expf to the last bit buys nothing here. Infinities and
 * NaN follow the reference: sigmoid(-inf) = 0. */
__device__ __forceinline__ float g53_grp_swiglu(float g, float u, float limit)
{
    const float gi = g > limit ? limit : g;
    const float ui = u > limit ? limit : (u < -limit ? -limit : u);
    return gi * __frcp_rn(1.0f + __expf(-gi)) * ui;
}

/* A wave's operands of one step: up to two matrix-core tiles of 32 weight rows, and 32 positions
 * in two planes, two K steps each. */
struct G53GrpOps {
    g53_v8i a[2][2], x[2][2];                                /* [tile][K step], [plane][K step] */
    float c0, c1;                                            /* block scales of C registers 0-7, 8-15 */
};
/* Fragment k (0-3 positions, 4-7 weights) of a step's operands from the slot at sl: a4 and x4 are
 * the lane's four 16-byte pieces (two K steps of two) of its weight row and of its position, the
 * second tile's rows DA bytes further. */
template <int DA, int k>
__device__ __forceinline__ void g53_grp_fetch(G53GrpOps &o, const uint8_t *sl, const int (&a4)[4], const int (&x4)[4])
{
    constexpr int s = k & 1, m = (k >> 1) & 1;
    const uint8_t *b0 = sl + (k < 4 ? x4[2 * s] + m * G53_GRP_PL : a4[2 * s] + m * DA);
    const uint8_t *b1 = sl + (k < 4 ? x4[2 * s + 1] + m * G53_GRP_PL : a4[2 * s + 1] + m * DA);
    const g53_v4i lo = *(const g53_v4i *)b0, hi = *(const g53_v4i *)b1;
    (k < 4 ? o.x[m][s] : o.a[m][s]) = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}
/* The two tiles' products in turn (two independent chains); between<m>() goes in after matrix
 * instruction m (0-7): a wave issues in order, and 64 cycles of matrix work hide the LDS reads and
 * loads that would otherwise be issued before it. */
template <class F>
__device__ __forceinline__ void g53_grp_mul(g53_v16f (&acc)[2], const G53GrpOps &o, F &&between)
{
    g53_v16f b[2] = {};
#define G53_MUL(m)                                                                                             \
    b[m & 1] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(o.a[m & 1][(m >> 1) & 1], o.x[m >> 2][(m >> 1) & 1], \
                                                               b[m & 1], 0, 0, 0, 127, 0, 127 - 4 * (m >> 2)); \
    __builtin_amdgcn_sched_barrier(0);                                                                         \
    between(G53Int<m>{});                                                                                      \
    __builtin_amdgcn_sched_barrier(0)
    G53_MUL(0); G53_MUL(1); G53_MUL(2); G53_MUL(3); G53_MUL(4); G53_MUL(5); G53_MUL(6); G53_MUL(7);
#undef G53_MUL
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[f][r] = fmaf(b[f][r], r < 8 ? o.c0 : o.c1, acc[f][r]);
}

/* The items of a launch. The dispatcher deals workgroups round-robin over the 8 XCDs, so the
 * workgroups of XCD x (blockIdx.x % 8 == x) share the items [blo, bhi) (a range of equal estimated
 * cost, from the planner) and take them in turn. Items are numbered segment by segment, and inside
 * a segment row block by row block, all tiles of a block in a row: the tiles of one expert that
 * re-read the same weight rows run side by side on one XCD and find them in its L2. */
struct G53GrpItem {
    int4 tl;                       /* the tile; tl.z == 0: no item                       */
    int mb, many;                  /* row block; whether other tiles share its rows      */
    int num;
    const G53hExpert *ex;
};

/* GATEUP: gate/up rows and SwiGLU for (tile, 128 intermediate rows): LDS rows 0-127 are the gate
 * rows, 128-255 the up rows of the same indices, and a wave's 32 rows are 16 gate rows and the same
 * 16 up rows, so C registers r and r + 8 of a lane are gate and up of one row and position; the
 * activations leave as E4M3 planes. Otherwise: 256 down rows times the activation planes into the
 * contributions.
 *
 * Bound by HBM while tiles hold at most 32 positions: 32 KB of codes a step and CU. Hidden 4096,
 * inter 2048, 288 experts, gate/up: 150 tokens over 202 experts 613 -> 540 us (6.3 TB/s; a stream of
 * the same bytes and nothing else reaches 6.2, non-temporal 6.6), 64 tokens 436 -> 410 us. (Weights in
 * registers, fetched in 16-byte pieces of 32 rows, two blocks in flight behind the positions' loads,
 * gave the first figures.) 2048 tokens: 1124 -> 1100 us: 453 tiles, of which most hold 33 - 64
 * positions; a step then takes about 1900 cycles (1024 of matrix instructions a SIMD, which the LDS
 * reads, the scaling and the barrier do not overlap whole) at the 1.6 GHz that the card's power
 * allows, and no wave waits for memory. */
template <bool GATEUP>
__global__ void __launch_bounds__(64 * G53_GRP_NW, 1) k_grp_gemm(G53GrpArgs a)
{
    __shared__ __attribute__((aligned(1024))) uint8_t ring[G53_GRP_NS * G53_GRP_SLOT];
    /* the items' token scales (of position 32 h + 8 v + q at [2 v + h][8 q]) and block scales: two rows */
    __shared__ float xil[2][8][64];
    __shared__ float scl[2][64];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 31, g = lane >> 5;
    const int K = GATEUP ? a.E : a.I, MB = GATEUP ? a.I / 128 : a.E / 256, nkb = K / 128;
    const int nper = (int)(gridDim.x >> 3), bnd = (GATEUP ? G53_GRP_BGU : G53_GRP_BDN) + (int)(blockIdx.x & 7);
    const int bhi = g53_sld(a.meta + bnd + 1);
    int loc = g53_sld(a.meta + bnd) + (int)(blockIdx.x >> 3);
    const uint32_t lring = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)ring;
    const uint32_t lxil = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float *)&xil[0][0][0];
    const uint32_t lscl = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float *)&scl[0][0];

    /* this lane's part of a load instruction: row lane / 8 of eight, piece lane % 8 of LDS */
    const int lr = lane >> 3, lp = lane & 7;
    uint32_t voa[4];                                         /* the wave's four octets of weight rows */
#pragma unroll
    for (int o = 0; o < 4; o++) {
        const int c = lp ^ ((4 * (o & 1) + (lane >> 4)) & 7);
        /* piece c of row lr: of a row's 128 bytes, or of an MFMA-tiled unit its columns 16 c .. */
        voa[o] = (uint32_t)(8 * o * K + (a.tiled == 2 ? (c & 1) * 512 + (c >> 1) * 128 + lr * 16
                                         : a.tiled ? lr * 128 + c * 16 : lr * K + c * 16));
    }
    const uint32_t vox = (uint32_t)((lp ^ ((4 * (w & 1) + (lane >> 4)) & 7)) * 16);
    const int kst = a.tiled ? 1024 : 128, ksh = __builtin_ctz(K);    /* K: a power of two */
    const size_t xps = GATEUP ? (size_t)a.T * a.E : (size_t)a.P * a.I;
    auto item_at = [&](int n) {
        G53GrpItem it;
        const int w0 = g53_sld(&a.tiles[n / MB].w);          /* a tile of the item's segment */
        const int ts0 = w0 & 0xffff, nts = w0 >> 16, q = n - ts0 * MB;
        it.mb = q / nts;
        it.many = nts > 1;
        const int *t = (const int *)(a.tiles + ts0 + q % nts);
        it.tl = make_int4(g53_sld(t), g53_sld(t + 1), g53_sld(t + 2), 0);
        it.num = n;
        it.ex = it.tl.x < a.NE ? a.experts + it.tl.x : a.shared;
        return it;
    };
    /* the workgroup's next item whose expert can be multiplied; the others are dealt with here */
    auto next_item = [&]() {
        for (;; loc += nper) {
            if (loc >= bhi) return G53GrpItem{make_int4(0, 0, 0, 0), 0, 0, 0, nullptr};
            G53GrpItem it = item_at(loc);
            const G53hExpert *ex = it.ex;
            const bool present = ex && g53_sld(&ex->gate.w) != nullptr;
            if (present && g53_grp_desc_ok(ex, a.E, a.I, a.tiled)) {
                loc += nper;
                return it;
            }
            if (GATEUP) {                                    /* the down launch writes its zeros */
                if (present && tid == 0) atomicOr(&a.meta_w[1], G53_GRP_EDESC);
            } else if (present || !a.partial || (ex && (g53_sld(&ex->gate.flags) & G53H_MAT_DROPPED))) {
                for (int q = tid; q < it.tl.z * 64; q += 64 * G53_GRP_NW)
                    *(float4 *)(a.contrib + (size_t)(it.tl.y + (q >> 6)) * a.E + it.mb * 256 + (q & 63) * 4) =
                        make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
    };

    /* an item as requests need it: its bases, and this lane's positions in the planes */
    struct Bound {
        const uint8_t *pa, *px;
        uint32_t vx[2];
        int mode;                                            /* 0 streamed, 1 shared by tiles, 2 unaligned */
    };
    auto bind = [&](const G53GrpItem &it) {
        Bound r;
        const int n = it.tl.z, row = (w & 3) * 8;
        const uint8_t *m;
        if (GATEUP) {
            m = w < 4 ? g53_sld(&it.ex->gate.w) : g53_sld(&it.ex->up.w);
            r.pa = m + (size_t)(it.mb * 128 + (w & 3) * 32) * K;
            r.px = a.xq;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                int tk = 0;
#pragma unroll
                for (int q = 0; q < 8; q++) {                /* past the tile's end: its first position */
                    const int rr = row + 32 * h + q, v = g53_sld(a.tok_of + it.tl.y + (rr < n ? rr : 0));
                    tk = lr == q ? v : tk;
                }
                r.vx[h] = (uint32_t)((w >> 2) * xps + (size_t)tk * K) + vox;
            }
        } else {
            m = g53_sld(&it.ex->down.w);
            r.pa = m + (size_t)(it.mb * 256 + w * 32) * K;
            r.px = a.aq + (size_t)it.tl.y * K;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int rr = row + 32 * h + lr;
                r.vx[h] = (uint32_t)((w >> 2) * xps + (size_t)(rr < n ? rr : 0) * K) + vox;
            }
        }
        r.mode = ((uintptr_t)m & 15) ? 2 : it.many;
        return r;
    };
    /* request the block at r.pa / r.px into a slot (LDS byte so) and step to the next block */
    auto request = [&](Bound &r, uint32_t so) {
        const uint32_t ls = lring + so + w * 4096, lx = lring + so + G53_GRP_SA + (w >> 2) * G53_GRP_PL + (w & 3) * 1024;
        /* rows that one tile reads are streamed past the caches: 540 against 567 us at 150 tokens
         * (gate/up); rows that several tiles read come from L2 for all but the first */
        if (r.mode == 0) g53_dma_rows_nt(voa, r.pa, ls);
        else if (r.mode == 1) g53_dma_rows(voa, r.pa, ls);
        else {                                               /* codes that are not 16-byte aligned: by registers */
#pragma unroll
            for (int o = 0; o < 4; o++) {
                g53_v4i v;
                __builtin_memcpy(&v, r.pa + voa[o], 16);
                *(g53_v4i *)(ring + so + w * 4096 + o * 1024 + lane * 16) = v;
            }
        }
        g53_dma16(r.vx[0], r.px, lx);
        g53_dma16(r.vx[1], r.px, lx + 4096);
        /* with fewer than six loads the steps' waits would not count right: this wave's all land here */
        if (r.mode == 2) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        r.pa += kst;
        r.px += 128;
    };
    auto scales = [&](const G53GrpItem &it, const Bound &r, int par) {   /* the item's scales */
        if (GATEUP && w < 4) {                               /* of the tokens whose first plane the wave requests */
            g53_dma4(a.xinv + (r.vx[0] >> ksh), lxil + par * 2048 + w * 512);
            g53_dma4(a.xinv + (r.vx[1] >> ksh), lxil + par * 2048 + w * 512 + 256);
        }
        if (w == 1) {                                        /* rows: gate and up, or the item's two of down */
            const G53hExpert *ex = it.ex;
            const float *r0, *r1;
            if (GATEUP) {
                r0 = g53_sld(&ex->gate.s) + (size_t)it.mb * g53_sld(&ex->gate.scols);
                r1 = g53_sld(&ex->up.s) + (size_t)it.mb * g53_sld(&ex->up.scols);
            } else {
                r0 = g53_sld(&ex->down.s) + (size_t)(2 * it.mb) * g53_sld(&ex->down.scols);
                r1 = r0 + g53_sld(&ex->down.scols);
            }
            g53_dma4((g ? r1 : r0) + min(i, nkb - 1), lscl + par * 256);
        }
    };
    /* this wave's first row in an item (gate/up: intermediate row) and its half of the positions;
     * its lanes' operand pieces in a slot */
    const int rw = (w & 3) * (GATEUP ? 32 : 64), half = w >> 2;
    int a4[4], x4[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int po = ((4 * g + q) ^ ((i >> 1) & 7)) * 16;
        a4[q] = (GATEUP ? rw + (i & 15) + (i & 16) * 8 : rw + i) * 128 + po;
        x4[q] = G53_GRP_SA + (half * 32 + i) * 128 + po;
    }
    /* fragment k of the operands of block kb of the item of parity pr from a slot (8: its scales) */
    auto fetch = [&](auto k, G53GrpOps &o, int kb, int pr, uint32_t so) {
        if constexpr (decltype(k)::value == 8) {
            o.c0 = scl[pr][GATEUP ? kb : (w & 2) * 16 + kb];
            o.c1 = GATEUP ? scl[pr][32 + kb] : o.c0;
        } else {
            g53_grp_fetch<(GATEUP ? 16 : 32) * 128, decltype(k)::value>(o, ring + so, a4, x4);
        }
    };
    auto fetch_all = [&](G53GrpOps &o, int kb, int pr, uint32_t so) {
        fetch(G53Int<0>{}, o, kb, pr, so); fetch(G53Int<1>{}, o, kb, pr, so); fetch(G53Int<2>{}, o, kb, pr, so);
        fetch(G53Int<3>{}, o, kb, pr, so); fetch(G53Int<4>{}, o, kb, pr, so); fetch(G53Int<5>{}, o, kb, pr, so);
        fetch(G53Int<6>{}, o, kb, pr, so); fetch(G53Int<7>{}, o, kb, pr, so); fetch(G53Int<8>{}, o, kb, pr, so);
    };

    G53GrpItem cur = next_item();
    if (cur.tl.z == 0) return;
    Bound bd = bind(cur);
    G53GrpOps ops[2];
    int par = 0;
    uint32_t so = 0;                                         /* slot of the step being multiplied */
    scales(cur, bd, 0);
    request(bd, 0);
    request(bd, G53_GRP_SLOT);
    request(bd, 2 * G53_GRP_SLOT);
    asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
    g53_grp_bar();
    fetch_all(ops[0], 0, 0, 0);
    for (;;) {
        const int n = cur.tl.z, pos0 = cur.tl.y;
        if (GATEUP && a.trace && tid == 0) {
            uint64_t *tr = a.trace + (size_t)cur.num * 8;
            tr[0] = __builtin_amdgcn_s_memrealtime();
            tr[4] = (uint64_t)__smid() << 32 | (uint32_t)(pos0 << 8 | n);
            tr[5] = (uint64_t)blockIdx.x << 32 | (uint32_t)(cur.tl.x << 8 | cur.mb);
        }
        const G53GrpItem nx = next_item();
        /* past the last item, its own blocks are requested again, so that every step is alike */
        const Bound nb = bind(nx.tl.z ? nx : cur);
        const bool act = half * 32 < n, actn = half * 32 < nx.tl.z;
        g53_v16f acc[2] = {};
        /* A step: the next step's six loads have landed - this wave's by the wait, every wave's by
         * the barrier, which also ends every wave's reads of the step being multiplied, so its slot
         * is requested again, three steps ahead; the next step's operands leave LDS while this
         * step's, read a step ago, are multiplied. Waves without positions only load. */
        auto step = [&](int kb, G53GrpOps &o, G53GrpOps &on) {
            asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
            g53_grp_bar();
            if (kb == nkb - 3) {
                bd = nb;
                if (nx.tl.z) scales(nx, bd, par ^ 1);
            }
            const uint32_t rs = so;
            so = so == 2 * G53_GRP_SLOT ? 0u : so + G53_GRP_SLOT;
            const bool last = kb + 1 == nkb;
            const int kn = last ? 0 : kb + 1, pn = last ? par ^ 1 : par;
            if (act)
                g53_grp_mul(acc, o, [&](auto m) {
                    fetch(m, on, kn, pn, so);
                    if constexpr (decltype(m)::value == 0) request(bd, rs);
                    if constexpr (decltype(m)::value == 7) fetch(G53Int<8>{}, on, kn, pn, so);
                });
            else {
                request(bd, rs);
                if (last && actn) fetch_all(on, kn, pn, so);
            }
        };
        for (int kb = 0; kb < nkb; kb += 2) {
            step(kb, ops[0], ops[1]);
            step(kb + 1, ops[1], ops[0]);
        }
        if (GATEUP && a.trace && tid == 0) a.trace[(size_t)cur.num * 8 + 2] = __builtin_amdgcn_s_memrealtime();
        const int j = half * 32 + i;                         /* this lane's position */
        if (GATEUP) {
            /* SwiGLU; the activation planes of the item's 128 rows are put together in the slot
             * whose operands have been read, in their final byte order (the tiled order within the 128-column
             * block when the pass is tiled), and leave as whole 16-byte pieces */
            uint8_t *ao = ring + so;
            const float xi = xil[par][2 * (i >> 3) + half][8 * (i & 7)];
            g53_grp_bar();                                   /* every wave is done with the slot */
#pragma unroll
            for (int f = 0; f < 2; f++) {
                if (j >= n) continue;
                uint32_t pk[2][G53_GRP_NPA];
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    float v[4];
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const int r = q * 4 + k;
                        v[k] = g53_grp_swiglu(acc[f][r] * xi, acc[f][r + 8] * xi, a.limit) * a.aq_scale;
                    }
                    g53_split_planes<G53_GRP_NPA>(v, pk[q]);
                }
                /* C register q * 4 + k holds row rb + q * 8 + g * 4 + k of the block */
                const int rb = rw + f * 16;
#pragma unroll
                for (int p = 0; p < G53_GRP_NPA; p++) {
                    uint8_t *d = ao + (p * G53_GRP_NT + j) * 128;
                    if (a.tiled == 1) {     /* rows of q = 0 and 1 are neighbouring bytes of one run */
#pragma unroll
                        for (int k = 0; k < 4; k++)
                            *(uint16_t *)(d + (g53_grp_tpos(g * 4 + k) & ~15) + (rb >> 3)) =
                                (uint16_t)(((pk[0][p] >> (8 * k)) & 0xffu) | (((pk[1][p] >> (8 * k)) & 0xffu) << 8));
                    } else {
                        *(uint32_t *)(d + rb + g * 4) = pk[0][p];
                        *(uint32_t *)(d + rb + 8 + g * 4) = pk[1][p];
                    }
                }
            }
            g53_grp_bar();
            for (int c = tid; c < n * G53_GRP_NPA * 8; c += 64 * G53_GRP_NW) {
                const int p = c / (n * 8), jq = c - p * n * 8, jj = jq >> 3, piece = jq & 7;
                *(g53_v4i *)(a.aq + ((size_t)p * a.P + pos0 + jj) * a.I + cur.mb * 128 + piece * 16) =
                    *(const g53_v4i *)(ao + (p * G53_GRP_NT + jj) * 128 + piece * 16);
            }
            if (a.trace && tid == 0) a.trace[(size_t)cur.num * 8 + 3] = __builtin_amdgcn_s_memrealtime();
        } else {
#pragma unroll
            for (int f = 0; f < 2; f++) {
                if (j >= n) continue;
                float *dst = a.contrib + (size_t)(pos0 + j) * a.E + cur.mb * 256 + rw + f * 32 + g * 4;
#pragma unroll
                for (int q = 0; q < 4; q++)
                    *(float4 *)(dst + q * 8) = make_float4(acc[f][q * 4] * a.aq_inv, acc[f][q * 4 + 1] * a.aq_inv,
                                                           acc[f][q * 4 + 2] * a.aq_inv, acc[f][q * 4 + 3] * a.aq_inv);
            }
        }
        if (nx.tl.z == 0) break;
        cur = nx;
        par ^= 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         /* no load may outlive the workgroup's LDS */
}

/* out[t][d] = (float)(sum_j (double)w[t][j] * (double)contrib[pos(t,j)][d]) (+ shared, float):
 * src/core/glm53f_ops.c:1329-1340. Four consecutive d per thread. */
__global__ void __launch_bounds__(256)
k_grp_combine(float *__restrict__ out, const float *__restrict__ contrib, const float *__restrict__ wts,
              const int *__restrict__ pos_of, int T, int E, int K, int has_sh, int *__restrict__ err,
              int *__restrict__ meta)
{
    /* the pass's error flags into the library's, and the tile count and flags cleared for the
     * next pass (every kernel that reads or sets them has finished) */
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (meta[1]) atomicOr(err, meta[1]);
        meta[0] = 0;
        meta[1] = 0;
    }
    const long q = (long)blockIdx.x * 256 + threadIdx.x;
    if (q * 4 >= (long)T * E) return;
    const int t = (int)(q * 4 / E), d = (int)(q * 4 % E);
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    for (int j = 0; j < K; j++) {
        const int p = pos_of[t * (K + 1) + j];
        const double wj = (double)wts[(size_t)t * K + j];
        float4 c = make_float4(0.f, 0.f, 0.f, 0.f);
        if (p >= 0) c = *(const float4 *)(contrib + (size_t)p * E + d);
        s0 = s0 + wj * (double)c.x; s1 = s1 + wj * (double)c.y;
        s2 = s2 + wj * (double)c.z; s3 = s3 + wj * (double)c.w;
    }
    float4 o = make_float4((float)s0, (float)s1, (float)s2, (float)s3);
    if (has_sh) {
        const float4 c = *(const float4 *)(contrib + (size_t)pos_of[t * (K + 1) + K] * E + d);
        o.x = o.x + c.x; o.y = o.y + c.y; o.z = o.z + c.z; o.w = o.w + c.w;
    }
    *(float4 *)(out + (size_t)t * E + d) = o;
}

/* ------------------------------------------------------------------ dispatch ---- */
static int g_grp_mode = 1;           /* 1: T >= 2 takes this path when the shapes fit */
static uint64_t *g_grp_trace = nullptr;

/* Diagnostics: with dev_buf != NULL (device, >= gate/up items x 8 uint64), the gate/up kernel
 * records timestamps (100 MHz) of each item's phases, its CU and workgroup; NULL turns it off. */
extern "C" int g53h_set_grouped_trace(void *dev_buf)
{
    g_grp_trace = (uint64_t *)dev_buf;
    return 0;
}
static int *g_grp_err = nullptr;     /* device: accumulated error flags               */

static size_t al256(size_t v) { return (v + 255) & ~(size_t)255; }

extern "C" int g53h_set_grouped(int mode)
{
    const int prev = g_grp_mode;
    g_grp_mode = mode ? 1 : 0;
    return prev;
}

/* The layer shapes this path serves (routing aside). */
static int g53_grp_shapes_ok(const G53hMoeLayer *L)
{
    if (!L) return 0;
    const float lim = L->swiglu_limit;
    const int nbe = L->hidden / 128, nbi = L->inter / 128;
    const int pow2 = (nbe & (nbe - 1)) == 0 && (nbi & (nbi - 1)) == 0;
    return L->block_c == 128 && L->hidden % 512 == 0 && L->inter % 512 == 0 && pow2 && nbe <= 32 && nbi <= 32 &&
           L->topk >= 1 && L->topk <= 16 && L->n_experts >= L->topk && L->n_experts <= 1024 && lim > 0.0f &&
           lim < 1.0e4f;
}

extern "C" int g53h_grouped_ok(const G53hMoeLayer *L)
{
    /* MFMA-tiled experts are taken through g53h_grouped_begin_layout only */
    return L && L->router && L->bias && (L->tiled == 0 || L->tiled == 1) && g53_grp_shapes_ok(L);
}

int g53h_grouped_use(const G53hMoeLayer *L, int T) { return g_grp_mode && T >= 2 && g53h_grouped_ok(L); }



extern "C" int g53h_grouped_errors(void)
{
    if (g53h_ready()) return 0;
    int v = 0;
    if (g53h_check(hipStreamSynchronize(g53h_stream()), "sync", __FILE__, __LINE__)) return -1;
    if (g53h_check(hipMemcpy(&v, g53h_errblock() + 2, 4, hipMemcpyDeviceToHost), "d2h", __FILE__, __LINE__)) return -1;
    if (v && g53h_check(hipMemset(g53h_errblock() + 2, 0, 4), "memset", __FILE__, __LINE__)) return -1;
    return v;
}

/* One planning pass of tc <= G53_GRP_MAXT tokens, in three phases: plan (sort, tiles, input
 * planes), run (the expert GEMMs for the experts present in L->experts / L->shared), combine. */
struct G53GrpPass {
    int active, tc, K, hs, maxtiles;
    int *pos_of, *meta;
    float *contrib;
    G53GrpArgs a;
};
static G53GrpPass g_pass;

/* layout: 0 row-major, 1 octet-tiled, 2 MFMA-tiled experts. */
static int g53_grp_plan_pass(const float *x, int tc, const G53hMoeLayer *L, const int *idx, char *ws, int *meta, int layout)
{
    const int E = L->hidden, I = L->inter, K = L->topk, NE = L->n_experts, hs = L->shared ? 1 : 0;
    const int P = tc * K + hs * tc;
    const int maxtiles = (tc * K + G53_GRP_NT - 1) / G53_GRP_NT + NE + hs * ((tc + G53_GRP_NT - 1) / G53_GRP_NT);
    hipStream_t st = g53h_stream();
    char *p = ws;
    int *tok_of = (int *)p;   p += al256((size_t)P * 4);
    int *pos_of = (int *)p;   p += al256((size_t)tc * (K + 1) * 4);
    int4 *tiles = (int4 *)p;  p += al256((size_t)maxtiles * 16);
    uint8_t *xq = (uint8_t *)p; p += al256((size_t)G53_GRP_NPX * tc * E);
    float *xinv = (float *)p; p += al256((size_t)tc * 4);
    uint8_t *aq = (uint8_t *)p; p += al256((size_t)G53_GRP_NPA * P * I);
    float *contrib = (float *)p;
    const int nch = (tc + 63) / 64;
    const size_t lds = (size_t)nch * NE * 12 + (size_t)(NE + 2) * 12 + 64;   /* planes: 16 words */
    if (lds > 160 * 1024) return g53h_fail("g53h_moe_grouped: %zu bytes of planner LDS", lds);
    if (lds > 65536) G53_TRY(hipFuncSetAttribute((const void *)k_grp_prep, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k_grp_prep, dim3(1 + (tc + 3) / 4), dim3(1024), lds, st, idx, tc, K, NE, hs, tok_of, pos_of, tiles,
                       meta, I / 128, E / 256, x, E, xq, xinv, layout == 1);
    G53_LAUNCHED("k_grp_prep");
    g53h_prof_mark(G53_PROF_GROUPED);
    float bound = L->swiglu_limit > 0.28f ? L->swiglu_limit : 0.28f;
    bound *= L->swiglu_limit;
    int ex = 0;
    (void)frexpf(bound, &ex);                      /* |act| <= bound < 2^ex */
    G53GrpArgs &a = g_pass.a;
    a.experts = L->experts; a.shared = L->shared; a.tiles = tiles; a.meta = meta; a.meta_w = meta;
    a.tok_of = tok_of; a.xq = xq; a.xinv = xinv; a.aq = aq; a.contrib = contrib;
    a.T = tc; a.P = P; a.E = E; a.I = I; a.NE = NE;
    a.limit = L->swiglu_limit; a.aq_scale = ldexpf(1.0f, 8 - ex); a.aq_inv = ldexpf(1.0f, ex - 8);
    a.partial = 0;
    a.tiled = layout;
    a.trace = g_grp_trace;
    g_pass.active = 1; g_pass.tc = tc; g_pass.K = K; g_pass.hs = hs; g_pass.maxtiles = maxtiles;
    g_pass.pos_of = pos_of; g_pass.meta = meta; g_pass.contrib = contrib;
    return 0;
}

static int g53_grp_run_pass(const G53hExpert *experts, const G53hExpert *shared, int partial)
{
    G53GrpArgs &a = g_pass.a;
    a.experts = experts; a.shared = shared; a.partial = partial;
    const int E = a.E, I = a.I, maxtiles = g_pass.maxtiles;
    hipStream_t st = g53h_stream();
    const unsigned cap = (unsigned)g53h_num_cus() / 8 * 8;
    unsigned g1 = (unsigned)(maxtiles * (I / 128) + 7) / 8 * 8, g2 = (unsigned)(maxtiles * (E / 256) + 7) / 8 * 8;
    if (cap >= 8) { g1 = g1 < cap ? g1 : cap; g2 = g2 < cap ? g2 : cap; }
    hipLaunchKernelGGL((k_grp_gemm<true>), dim3(g1), dim3(64 * G53_GRP_NW), 0, st, a);
    G53_LAUNCHED("k_grp_gateup");
    g53h_prof_mark(G53_PROF_GATEUP);
    hipLaunchKernelGGL((k_grp_gemm<false>), dim3(g2), dim3(64 * G53_GRP_NW), 0, st, a);
    G53_LAUNCHED("k_grp_down");
    g53h_prof_mark(G53_PROF_DOWN);
    return 0;
}

static int g53_grp_combine_pass(float *out, const float *wts)
{
    hipStream_t st = g53h_stream();
    const int tc = g_pass.tc, E = g_pass.a.E;
    const long nq = (long)tc * E / 4;
    hipLaunchKernelGGL(k_grp_combine, dim3((unsigned)((nq + 255) / 256)), dim3(256), 0, st, out, g_pass.contrib, wts,
                       g_pass.pos_of, tc, E, g_pass.K, g_pass.hs, g53h_errblock() + 2, g_pass.meta);
    G53_LAUNCHED("k_grp_combine");
    g53h_prof_mark(G53_PROF_COMBINE);
    g_pass.active = 0;
    return 0;
}

static int g53_grp_chunk(float *out, const float *x, int tc, const G53hMoeLayer *L, const int *idx,
                         const float *wts, char *ws, int *meta)
{
    if (g53_grp_plan_pass(x, tc, L, idx, ws, meta, L->tiled ? 1 : 0) || g53_grp_run_pass(L->experts, L->shared, 0)) return -1;
    return g53_grp_combine_pass(out, wts);
}

/* Workspace of one planning pass of tc tokens. */
static size_t g53_grp_ws(const G53hMoeLayer *L, int tc)
{
    const int E = L->hidden, I = L->inter, K = L->topk, NE = L->n_experts, hs = L->shared ? 1 : 0;
    const size_t P = (size_t)tc * K + (size_t)hs * tc;
    const int maxtiles = (tc * K + G53_GRP_NT - 1) / G53_GRP_NT + NE + hs * ((tc + G53_GRP_NT - 1) / G53_GRP_NT);
    return al256(P * 4) + al256((size_t)tc * (K + 1) * 4) + al256((size_t)maxtiles * 16) +
           al256((size_t)G53_GRP_NPX * tc * E) + al256((size_t)tc * 4) + al256((size_t)G53_GRP_NPA * P * I) +
           al256(P * E * 4);
}

/* The grouped layer: router (exact), then planning passes of at most G53_GRP_MAXT tokens whose
 * 64-token masks fit the planner's LDS. idx_out / w_out receive the routing when non-NULL. */
extern "C" int g53h_moe_grouped(float *out, const float *x, int T, const G53hMoeLayer *L, int *idx_out,
                                float *w_out)
{
    if (g53h_ready()) return -1;
    if (!g53h_grouped_ok(L)) return g53h_fail("g53h_moe_grouped: layer shapes not supported");
    if (T < 0) return g53h_fail("g53h_moe_grouped: T %d", T);
    if (T == 0) return 0;
    const int K = L->topk, NE = L->n_experts;
    int tcmax = G53_GRP_MASKS / NE * 64;
    if (tcmax > G53_GRP_MAXT) tcmax = G53_GRP_MAXT;
    const int tc0 = T < tcmax ? T : tcmax;
    if (!g_grp_err) {
        G53_TRY(hipMalloc((void **)&g_grp_err, 256));
        G53_TRY(hipMemset(g_grp_err, 0, 256));
    }
    const size_t rsz = al256((size_t)2 * T * NE * 4), isz = al256((size_t)T * K * 4);
    char *ws = (char *)g53h_workspace(rsz + 2 * isz + g53_grp_ws(L, tc0));
    if (!ws) return -1;
    int *idx = idx_out ? idx_out : (int *)(ws + rsz);
    float *w = w_out ? w_out : (float *)(ws + rsz + isz);
    g53h_prof_mark(G53_PROF_START);
    if (g53h_router_into(idx, w, x, T, L->router, L->router_dt, L->bias, NE, L->hidden, K, L->norm_topk,
                         L->routed_scale, nullptr, (float *)ws, nullptr, nullptr, nullptr))
        return -1;
    g53h_prof_mark(G53_PROF_ROUTER);
    int *meta = g_grp_err + 16;                    /* [0] tiles, [1] flags; zero between calls */
    for (int t0 = 0; t0 < T; t0 += tc0) {
        const int tc = T - t0 < tc0 ? T - t0 : tc0;
        if (g53_grp_chunk(out + (size_t)t0 * L->hidden, x + (size_t)t0 * L->hidden, tc, L, idx + (size_t)t0 * K,
                          w + (size_t)t0 * K, ws + rsz + 2 * isz, meta))
            return -1;
    }
    return 0;
}

/* ------------------------------------------------------------- phased entry ---- */
static int g53_grp_tcmax(int NE)
{
    int tcmax = G53_GRP_MASKS / NE * 64;
    return tcmax > G53_GRP_MAXT ? G53_GRP_MAXT : tcmax;
}

/* HBM that g53h_router and one planning pass of T tokens would allocate now (each uses the workspace in
 * turn): 0 when the library holds enough already. */
extern "C" size_t g53h_grouped_growth(const G53hMoeLayer *L, int T)
{
    const size_t ws = g53_grp_ws(L, T), scores = (size_t)2 * T * L->n_experts * sizeof(float);
    return g53h_workspace_growth(ws > scores ? ws : scores) + g53h_router_growth(T, L->router_dt, L->n_experts, L->hidden);
}

extern "C" int g53h_grouped_max_tokens(const G53hMoeLayer *L)
{
    if (!g_grp_mode || !g53_grp_shapes_ok(L)) return 0;
    return g53_grp_tcmax(L->n_experts);
}

/* g53h_grouped_begin for experts of a given layout: also MFMA-tiled ones (2), which the drop-in's
 * cache may hold. */
extern "C" int g53h_grouped_begin_layout(const float *x, int T, const G53hMoeLayer *L, const int *idx, int layout)
{
    if (g53h_ready()) return -1;
    if (!g53_grp_shapes_ok(L)) return g53h_fail("g53h_grouped_begin: layer shapes not supported");
    if (T < 1 || T > g53_grp_tcmax(L->n_experts)) return g53h_fail("g53h_grouped_begin: T %d", T);
    if (!g_grp_err) {
        G53_TRY(hipMalloc((void **)&g_grp_err, 256));
        G53_TRY(hipMemset(g_grp_err, 0, 256));
    }
    char *ws = (char *)g53h_workspace(g53_grp_ws(L, T));
    if (!ws) return -1;
    return g53_grp_plan_pass(x, T, L, idx, ws, g_grp_err + 16, layout);
}

extern "C" int g53h_grouped_begin(const float *x, int T, const G53hMoeLayer *L, const int *idx)
{
    return g53h_grouped_begin_layout(x, T, L, idx, L && L->tiled ? 1 : 0);
}

extern "C" int g53h_grouped_batch(const G53hMoeLayer *L)
{
    if (!g_pass.active) return g53h_fail("g53h_grouped_batch: no pass begun");
    if (L && (g_pass.a.tiled == 2 ? L->tiled : L->tiled ? 1 : 0) != g_pass.a.tiled)
        return g53h_fail("g53h_grouped_batch: the pass was planned for %s experts", g_pass.a.tiled == 2 ? "MFMA-tiled" : g_pass.a.tiled ? "octet-tiled" : "row-major");
    if (!L || L->n_experts != g_pass.a.NE || L->hidden != g_pass.a.E || L->inter != g_pass.a.I)
        return g53h_fail("g53h_grouped_batch: another layer than the pass's");
    if (L->shared && !g_pass.hs) return g53h_fail("g53h_grouped_batch: the pass was planned without a shared expert");
    return g53_grp_run_pass(L->experts, L->shared, 1);
}

extern "C" int g53h_grouped_end(float *out, const float *wts)
{
    if (!g_pass.active) return g53h_fail("g53h_grouped_end: no pass begun");
    return g53_grp_combine_pass(out, wts);
}
