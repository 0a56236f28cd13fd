/* Device plan of a tile low-rank product (shared by the C host code that
 * builds it and the HIP kernels of csrc/hip/tlr.hip). */
#ifndef STARSH_HIP_TLR_H
#define STARSH_HIP_TLR_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* 32 columns (nc <= 32) of one factor, len rows each (ld len) at f_off of
 * the factor buffer: their products with rows x_off.. of the vectors are
 * coefficients out_off .. out_off+nc-1 (nrhs values each). */
typedef struct
{
    int64_t f_off, x_off, out_off;
    int len, nc;
} tlr_unit;

/* One contribution to a block row: kind 0 = F T with F (rows x cols, ld) at
 * f_off of the factor buffer and T the cols coefficients from src_off on;
 * kind 1 = D X[src_off..] with D (rows x cols, ld); kind 2 = D^T X[src_off..]
 * with D (cols x rows, ld).  Wide contributions are split into several
 * entries of at most TLR_ENTRY_COLS columns, which the four waves of a strip
 * share. */
#define TLR_ENTRY_COLS 64
typedef struct
{
    int64_t f_off, src_off;
    int ld, cols, kind, pad;
} tlr_entry;

/* A strip of rows of one block row: rows rofs.. of the block, which are rows
 * row0.. of the vectors, and the block row's entries first..last-1. */
typedef struct
{
    int64_t row0;
    int rofs, nrows, first, last;
} tlr_chunk;

/* The product's plan in device memory; strip: rows per strip, 16, 32 or
 * 64. */
typedef struct
{
    int nunits, nchunks, strip;
    tlr_unit *d_units;
    tlr_chunk *d_chunks;
    tlr_entry *d_entries;
    double *d_fac;
} tlr_plan;

/* Static device scratch of the allocation-free product: its size in
 * doubles, the devices it is set up for, the per-device set-up (called by
 * starsh_hip_init with the device current) and the lookup of its device
 * address on a set-up device. */
#define TLR_SCRATCH_DOUBLES ((int64_t)1 << 22)
#define TLR_MAX_DEVICES 64
int tlr_scratch_setup(int device);
int tlr_scratch(int device, double **ptr);

/* Y = alpha * M * X + beta * Y; d_tmp holds the coefficients, 2 x the sum of
 * the far-field ranks x nrhs doubles. */
int starsh_hip_tlr_apply(const tlr_plan *pl, double *d_tmp, int nrhs,
        double alpha, const double *d_x, int ldx, double beta, double *d_y,
        int ldy);

/* Seconds per starsh_hip_tlr_apply with alpha 1, beta 0 (mean over reps
 * launches after one warm-up; events on the library stream). */
int starsh_hip_tlr_time(const tlr_plan *pl, double *d_tmp, int nrhs,
        const double *d_x, int ldx, double *d_y, int ldy, int reps,
        double *seconds);

/* Conjugate gradients on the library stream, nrhs columns of n (n apart).
 * State of a column: |r|^2, the value |r| is checked against, and the
 * iteration that met it (-1: none yet; -2: the value is negative, and as in
 * cg.c the column is left alone and never meets it). */
typedef struct
{
    double rsold, rscheck;
    int done, pad;
} tlr_cg_state;
/* Doubles of d_part and states of d_st. */
#define TLR_CG_PART(nrhs) ((size_t)(nrhs)*512)
#define TLR_CG_STATES(nrhs) ((size_t)(nrhs)*2)
/* The state before iteration 0. */
int starsh_hip_cg_start(int64_t n, int nrhs, double tol, const double *d_r,
        double *d_part, tlr_cg_state *d_st);
/* Iteration it with q = M p; the state after it is d_st + ((it+1) & 1)
 * nrhs. */
int starsh_hip_cg_iteration(int64_t n, int nrhs, int it, double *d_p,
        const double *d_q, double *d_x, double *d_r, double *d_part,
        tlr_cg_state *d_st);
/* y += a x, y = x. */
int starsh_hip_vaxpy(int64_t n, double a, const double *d_x, double *d_y);
int starsh_hip_vcopy(int64_t n, const double *d_x, double *d_y);

#ifdef __cplusplus
}
#endif

#endif
