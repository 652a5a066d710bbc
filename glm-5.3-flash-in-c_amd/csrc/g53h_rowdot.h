/* g53h_rowdot.h - the reference's per-block sums, shared by the kernels that compute one
 * column block (FP8) or group (int4) of a row at a time. */
#ifndef G53H_ROWDOT_H
#define G53H_ROWDOT_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "g53h.h"
#include "g53h_core.h"

/* E4M3FN code -> float by the gfx950 conversion instruction (exact; 0x7f / 0xff give NaN, as
 * g53_e4m3_to_f32 and the reference's table). */
__device__ __forceinline__ static float g53_e4m3_hw(uint8_t b) { return __builtin_amdgcn_cvt_f32_fp8((int)b, 0); }

/* The reference's per-block arithmetic (src/core/glm53f_ops.c:195-227): eight fp32 lanes of
 * fused products stepping by 8 columns, reduced in double by a fixed tree, the block tail
 * added in double, the block sum scaled in double and accumulated over blocks in order. */
__device__ __forceinline__ static double g53_block_dot(const uint8_t *row, const float *x, int j0, int j1)
{
    float a[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    int j = j0;
    for (; j + 8 <= j1; j += 8)
        for (int l = 0; l < 8; l++) a[l] = __builtin_fmaf(g53_e4m3_hw(row[j + l]), x[j + l], a[l]);
    double bsum = (((double)a[0] + a[4]) + ((double)a[2] + a[6]))
                + (((double)a[1] + a[5]) + ((double)a[3] + a[7]));
    for (; j < j1; j++) bsum += (double)g53_e4m3_hw(row[j]) * (double)x[j];
    return bsum;
}

/* The int4 format's group sum (src/core/glm53f_ops.c:247-287): the same eight fp32 lanes over
 * levels (nibble - 8, the even column in the low nibble), the double tree, the tail in double. */
__device__ __forceinline__ static double g53_group_dot_i4(const uint8_t *row, const float *x, int j0, int j1)
{
    float a[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    int j = j0;
    for (; j + 8 <= j1; j += 8)
        for (int l = 0; l < 8; l++) {
            const uint8_t b = row[(j + l) >> 1];
            const int lv = (int)(((j + l) & 1) ? (b >> 4) : (b & 15)) - 8;
            a[l] = __builtin_fmaf((float)lv, x[j + l], a[l]);
        }
    double bsum = (((double)a[0] + a[4]) + ((double)a[2] + a[6]))
                + (((double)a[1] + a[5]) + ((double)a[3] + a[7]));
    for (; j < j1; j++) {
        const uint8_t b = row[j >> 1];
        const int lv = (int)((j & 1) ? (b >> 4) : (b & 15)) - 8;
        bsum += (double)lv * (double)x[j];
    }
    return bsum;
}

/* One row's product, one lane: int4 (any even group), and FP8 of any blocks. */
__device__ inline float g53_row_dot_i4(const G53hMat &m, int o, const float *x)
{
    const uint8_t *row = m.w + (size_t)o * (m.cols / 2);
    const float *srow = m.s + (size_t)o * m.scols;
    double acc = 0.0;
    for (int g = 0, j0 = 0; j0 < m.cols; g++, j0 += m.bc) {
        const int j1 = (j0 + m.bc < m.cols) ? j0 + m.bc : m.cols;
        const double p = g53_group_dot_i4(row, x, j0, j1) * (double)srow[g];
        acc = acc + p;
    }
    return (float)acc;
}

__device__ inline float g53_row_dot(const G53hMat &m, int o, const float *x)
{
    if (m.flags & G53H_MAT_I4) return g53_row_dot_i4(m, o, x);
    const uint8_t *row = m.w + (size_t)o * m.cols;
    const float *srow = m.s + (size_t)(o / m.br) * m.scols;
    double acc = 0.0;
    for (int b = 0, j0 = 0; j0 < m.cols; b++, j0 += m.bc) {
        const int j1 = (j0 + m.bc < m.cols) ? j0 + m.bc : m.cols;
        const double bsum = g53_block_dot(row, x, j0, j1);
        const double p = bsum * (double)srow[b];
        acc = acc + p;
    }
    return (float)acc;
}

/* The same for an octet-tiled FP8 row (128-column blocks): accumulator l of a block is the 16 bytes
 * of run g53h_tile_acc(l) (its own inverse) of the unit's row. */
__device__ inline float g53_row_dot_tiled(const G53hMat &m, int o, const float *x)
{
    const float *srow = m.s + (size_t)(o / m.br) * m.scols;
    double acc = 0.0;
    for (int b = 0; b < m.scols; b++) {
        const uint8_t *u = m.w + ((size_t)(o >> 3) * m.scols + b) * 1024 + (o & 7) * 128;
        float a[8];
        for (int l = 0; l < 8; l++) {
            const uint8_t *run = u + 16 * (((l & 1) << 2) | (l & 2) | (l >> 2));
            a[l] = 0.0f;
            for (int j = 0; j < 16; j++) a[l] = __builtin_fmaf(g53_e4m3_hw(run[j]), x[b * 128 + 8 * j + l], a[l]);
        }
        const double s = (((double)a[0] + a[4]) + ((double)a[2] + a[6])) +
                         (((double)a[1] + a[5]) + ((double)a[3] + a[7]));
        acc = acc + s * (double)srow[b];
    }
    return (float)acc;
}

/* A matrix the row kernels read: row-major FP8 or int4, or a usable octet-tiled one, of 128-column
 * blocks and whole row octets (the tiled format's definition). The matrix-core layouts and int4-tiled
 * levels are not read. */
__device__ __forceinline__ bool g53_rows_ok(const G53hMat &m)
{
    if (m.flags & (G53H_MAT_MTILED | G53H_MAT_I4T)) return false;
    if (!(m.flags & G53H_MAT_TILED) || (m.flags & G53H_MAT_I4)) return true;
    return m.bc == 128 && m.cols == 128 * m.scols && (m.rows & 7) == 0 && ((uintptr_t)m.w & 15) == 0;
}

#endif /* G53H_ROWDOT_H */
