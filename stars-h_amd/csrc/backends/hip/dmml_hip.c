/* Products with a compressed matrix and conjugate gradients on the GPU.
 *
 * starsh_blrm__dmml_hip follows src/backends/sequential/blrm/dmml.c:16-145
 * of ecrc/stars-h 0.3.1 (B = alpha*M*A + beta*B with host arrays, the
 * vectors in cluster order): far-field tile (i, j) adds U (V^T A_j) to B_i
 * and, in a symmetric format with i != j, V (U^T A_i) to B_j; near-field
 * tiles add D A_j (and D^T A_i), D taken from near_D when onfly == 0 and
 * generated by the problem's kernel when onfly == 1.
 *
 * starsh_itersolvers__dcg_hip follows src/itersolvers/cg.c:24-95 (the
 * iteration, the per-column stopping rule |r| < tol |r_0| and the return
 * value: the iteration index at which every column converged, or -1).
 *
 * The device-resident operator starsh_hip_tlr (no reference counterpart)
 * uploads the factors once for repeated products. */
#include <string.h>
#include "common.h"
#include "starsh-hip.h"
#include "rsdd.h"
#include "tlr.h"

struct starsh_hip_tlr
{
    STARSH_int nrows, ncols;
    tlr_plan plan;
    size_t fac_doubles;
    int64_t tmp_units;       /* sum over far tiles of 2 r */
    int64_t noalloc_units;   /* the same plus n per twin tile: what the fixed
                                limit of the allocation-free product counts
                                (its kernels no longer store the n) */
    double *d_tmp;
    int tmp_nrhs;            /* right-hand sides d_tmp has room for */
};

void starsh_hip_tlr_free(starsh_hip_tlr *T)
{
    if(T == NULL)
        return;
    starsh_hip_free(T->plan.d_units);
    starsh_hip_free(T->plan.d_chunks);
    starsh_hip_free(T->plan.d_entries);
    starsh_hip_free(T->plan.d_fac);
    starsh_hip_free(T->d_tmp);
    free(T);
}

static int upload(void **d, const void *h, size_t bytes)
{
    *d = NULL;
    if(bytes == 0)
        return STARSH_SUCCESS;
    int info = starsh_hip_malloc(d, bytes);
    if(info != STARSH_SUCCESS)
        return info;
    return starsh_hip_memcpy_h2d(*d, h, bytes);
}

/* Offsets of a far-field tile's factors and coefficients. */
typedef struct
{
    int64_t u_off, v_off, tmp_off;
} tlr_far;

/* Entries a contribution of `cols` columns takes. */
static int64_t pieces(int64_t cols)
{
    return (cols+TLR_ENTRY_COLS-1)/TLR_ENTRY_COLS;
}

static int64_t add_units(tlr_unit *u, int64_t f_off, int len, int r,
        int64_t x_off, int64_t out_off)
{
    int64_t n = 0;
    for(int c = 0; c < r; c += 32, n++)
    {
        u[n].f_off = f_off+(int64_t)c*len;
        u[n].x_off = x_off;
        u[n].out_off = out_off+c;
        u[n].len = len;
        u[n].nc = r-c < 32 ? r-c : 32;
    }
    return n;
}

static int64_t add_entries(tlr_entry *e, int kind, int64_t f_off, int ld,
        int64_t cols, int64_t src_off)
{
    int64_t n = 0;
    for(int64_t c = 0; c < cols; c += TLR_ENTRY_COLS, n++)
    {
        memset(e+n, 0, sizeof(*e));
        e[n].kind = kind;
        e[n].f_off = f_off+(kind == 2 ? c : c*ld);
        e[n].src_off = src_off+c;
        e[n].ld = ld;
        e[n].cols = (int)(cols-c < TLR_ENTRY_COLS ? cols-c : TLR_ENTRY_COLS);
    }
    return n;
}

int starsh_hip_tlr_new(starsh_hip_tlr **out, STARSH_blrm *M)
{
    if(out == NULL || M == NULL || M->format == NULL)
        return STARSH_WRONG_PARAMETER;
    *out = NULL;
    STARSH_blrf *F = M->format;
    STARSH_problem *P = F->problem;
    STARSH_cluster *R = F->row_cluster, *C = F->col_cluster;
    STARSH_int nfar = F->nblocks_far, nnear = F->nblocks_near;
    const int symm = F->symm == 'S';
    if(M->onfly == 0 && nnear > 0 && M->near_D == NULL)
        return STARSH_WRONG_PARAMETER;
    STARSH_int nbr = R->nblocks;
    /* factor buffer: U, V of every far tile, then D of every near tile */
    size_t nfac = 0;
    for(STARSH_int bi = 0; bi < nfar; bi++)
    {
        STARSH_int i = F->block_far[2*bi], j = F->block_far[2*bi+1];
        int r = M->far_rank[bi];
        if(r < 0)
            return STARSH_WRONG_PARAMETER;
        nfac += (size_t)(R->size[i]+C->size[j])*r;
    }
    for(STARSH_int bi = 0; bi < nnear; bi++)
    {
        STARSH_int i = F->block_near[2*bi], j = F->block_near[2*bi+1];
        nfac += (size_t)R->size[i]*C->size[j];
    }
    /* entries per block row: far i == b, far twin j == b, near i == b,
     * near twin j == b, each of at most TLR_ENTRY_COLS columns; units: 32
     * columns of a factor whose coefficients are needed (V, and U of a
     * tile with a twin) */
    int64_t nunits = 0;
    for(STARSH_int bi = 0; bi < nfar; bi++)
        nunits += (int64_t)((M->far_rank[bi]+31)/32)*
            (symm && F->block_far[2*bi] != F->block_far[2*bi+1] ? 2 : 1);
    int64_t *count = calloc(nbr+1, sizeof(int64_t));
    int64_t *first = calloc(nbr+1, sizeof(int64_t));
    /* the host arrays that make up the factor buffer, in order; dense tiles
     * on the fly are generated into hnear first */
    const STARSH_int nseg = 2*nfar+nnear;
    const double **seg = malloc(sizeof(*seg)*(nseg > 0 ? nseg : 1));
    int64_t *seglen = malloc(sizeof(int64_t)*(nseg > 0 ? nseg : 1));
    double *hnear = M->onfly == 0 ? NULL : malloc(sizeof(double)*(nfac > 0 ?
                nfac : 1));
    tlr_unit *hunits = malloc(sizeof(tlr_unit)*(nunits > 0 ? nunits : 1));
    tlr_far *hfar = malloc(sizeof(tlr_far)*(nfar > 0 ? nfar : 1));
    int64_t *nearoff = malloc(sizeof(int64_t)*(nnear > 0 ? nnear : 1));
    starsh_hip_tlr *T = calloc(1, sizeof(*T));
    tlr_entry *hent = NULL;
    tlr_chunk *hch = NULL;
    int info = STARSH_MALLOC_ERROR;
    if(!count || !first || !seg || !seglen || (M->onfly != 0 && !hnear) ||
            !hunits || !hfar || !nearoff || !T)
        goto fail;
    T->nrows = P->shape[0];
    T->ncols = P->shape[P->ndim-1];
    size_t off = 0;
    int64_t tmp = 0, twins = 0;
    for(STARSH_int bi = 0; bi < nfar; bi++)
    {
        STARSH_int i = F->block_far[2*bi], j = F->block_far[2*bi+1];
        int m = (int)R->size[i], n = (int)C->size[j], r = M->far_rank[bi];
        const int twin = symm && i != j;
        tlr_far *t = &hfar[bi];
        t->u_off = (int64_t)off;
        seg[2*bi] = r > 0 ? M->far_U[bi]->data : NULL;
        seglen[2*bi] = (int64_t)m*r;
        off += (size_t)m*r;
        t->v_off = (int64_t)off;
        seg[2*bi+1] = r > 0 ? M->far_V[bi]->data : NULL;
        seglen[2*bi+1] = (int64_t)n*r;
        off += (size_t)n*r;
        t->tmp_off = tmp;
        tmp += 2*(int64_t)r;
        if(twin && r > 0)
            twins += n;
        /* first[b+1]: units of block row b, see below */
        first[(twin ? j : i)+1] += (r+31)/32;
        if(twin)
            first[i+1] += (r+31)/32;
        count[i] += pieces(r);
        if(twin)
            count[j] += pieces(r);
    }
    /* Units go by the block row whose strips read the same factor again (V of
     * a tile with a twin: j), and the strips in the opposite order: what the
     * first launch read last is read first by the second, and again first by
     * the next product, while it is in the 256 MB cache in front of the
     * memory.  N=64000, tile 1600, one vector, with both in one direction
     * and so: 358 MB 117.3 and 116.3 us, 431 MB 142.4 and 141.0, 700 MB
     * 229.0 and 228.4; two vectors, 359 MB 159.0 and 152.5, 16, 716 MB 310
     * and 300.  It costs up to 2% where the cache holds the operator anyway
     * (126 MB 46.0 and 47.0) and without twins, whose factors it is about
     * (four vectors, 686 MB 166.6 and 169.5) */
    for(STARSH_int b = 0; b < nbr; b++)
        first[b+1] += first[b];
    for(STARSH_int bi = 0; bi < nfar; bi++)
    {
        STARSH_int i = F->block_far[2*bi], j = F->block_far[2*bi+1];
        int m = (int)R->size[i], n = (int)C->size[j], r = M->far_rank[bi];
        const int twin = symm && i != j;
        const tlr_far *t = &hfar[bi];
        int64_t *u = &first[twin ? j : i];
        *u += add_units(hunits+*u, t->v_off, n, r, C->start[j], t->tmp_off);
        if(twin)
            first[i] += add_units(hunits+first[i], t->u_off, m, r,
                    R->start[i], t->tmp_off+r);
    }
    for(STARSH_int bi = 0; bi < nnear; bi++)
    {
        STARSH_int i = F->block_near[2*bi], j = F->block_near[2*bi+1];
        int m = (int)R->size[i], n = (int)C->size[j];
        nearoff[bi] = (int64_t)off;
        seg[2*nfar+bi] = M->onfly == 0 ? M->near_D[bi]->data : hnear+off;
        seglen[2*nfar+bi] = (int64_t)m*n;
        if(M->onfly != 0)
            P->kernel(m, n, R->pivot+R->start[i], C->pivot+C->start[j],
                    R->data, C->data, hnear+off, m);
        off += (size_t)m*n;
        count[i] += pieces(n);
        if(symm && i != j)
            count[j] += pieces(m);
    }
    /* CSR of entries by block row */
    int64_t nent = 0;
    for(STARSH_int b = 0; b < nbr; b++)
    {
        int64_t c = count[b];
        count[b] = nent;
        nent += c;
    }
    count[nbr] = nent;
    hent = malloc(sizeof(tlr_entry)*(nent > 0 ? nent : 1));
    int64_t *fill = malloc(sizeof(int64_t)*(nbr > 0 ? nbr : 1));
    if(!hent || !fill)
    {
        free(fill);
        goto fail;
    }
    memcpy(fill, count, sizeof(int64_t)*nbr);
    for(STARSH_int bi = 0; bi < nfar; bi++)
    {
        const tlr_far *t = &hfar[bi];
        STARSH_int i = F->block_far[2*bi], j = F->block_far[2*bi+1];
        int m = (int)R->size[i], n = (int)C->size[j], r = M->far_rank[bi];
        fill[i] += add_entries(hent+fill[i], 0, t->u_off, m, r, t->tmp_off);
        if(symm && i != j)
            fill[j] += add_entries(hent+fill[j], 0, t->v_off, n, r,
                    t->tmp_off+r);
    }
    for(STARSH_int bi = 0; bi < nnear; bi++)
    {
        STARSH_int i = F->block_near[2*bi], j = F->block_near[2*bi+1];
        int m = (int)R->size[i], n = (int)C->size[j];
        fill[i] += add_entries(hent+fill[i], 1, nearoff[bi], m, n,
                C->start[j]);
        if(symm && i != j)
            fill[j] += add_entries(hent+fill[j], 2, nearoff[bi], m, m,
                    R->start[i]);
    }
    free(fill);
    /* strips of every block row: 64 rows, fewer where that would leave the
     * chip without two workgroups per CU */
    int strip = 64;
    while(strip > 16 && T->nrows/strip < 512)
        strip /= 2;
    int64_t nch = 0;
    for(STARSH_int b = 0; b < nbr; b++)
        nch += (R->size[b]+strip-1)/strip;
    hch = malloc(sizeof(tlr_chunk)*(nch > 0 ? nch : 1));
    if(!hch)
        goto fail;
    int64_t at = nch;       /* last block row first */
    for(STARSH_int b = 0; b < nbr; b++)
        for(STARSH_int r0 = 0; r0 < R->size[b]; r0 += strip)
        {
            tlr_chunk *c = &hch[--at];
            c->row0 = R->start[b]+r0;
            c->rofs = (int)r0;
            c->nrows = (int)(R->size[b]-r0 < strip ? R->size[b]-r0 : strip);
            c->first = (int)count[b];
            c->last = (int)count[b+1];
        }
    T->plan.nunits = (int)nunits;
    T->plan.nchunks = (int)nch;
    T->plan.strip = strip;
    T->fac_doubles = off;
    T->tmp_units = tmp;
    T->noalloc_units = tmp+twins;
    info = off == 0 ? STARSH_SUCCESS :
        starsh_hip_malloc((void **)&T->plan.d_fac, sizeof(double)*off);
    if(info == STARSH_SUCCESS)
        info = hip_upload_segments(T->plan.d_fac, nseg, seg, seglen);
    if(info == STARSH_SUCCESS)
        info = upload((void **)&T->plan.d_units, hunits,
                sizeof(tlr_unit)*nunits);
    if(info == STARSH_SUCCESS)
        info = upload((void **)&T->plan.d_entries, hent,
                sizeof(tlr_entry)*nent);
    if(info == STARSH_SUCCESS)
        info = upload((void **)&T->plan.d_chunks, hch, sizeof(tlr_chunk)*nch);
    if(info != STARSH_SUCCESS)
        goto fail;
    free(count);
    free(first);
    free(seg);
    free(seglen);
    free(hnear);
    free(hunits);
    free(hfar);
    free(nearoff);
    free(hent);
    free(hch);
    *out = T;
    return STARSH_SUCCESS;
fail:
    free(count);
    free(first);
    free(seg);
    free(seglen);
    free(hnear);
    free(hunits);
    free(hfar);
    free(nearoff);
    free(hent);
    free(hch);
    starsh_hip_tlr_free(T);
    return info;
}

static int tmp_reserve(starsh_hip_tlr *T, int nrhs)
{
    if(nrhs <= T->tmp_nrhs)
        return STARSH_SUCCESS;
    starsh_hip_free(T->d_tmp);
    T->d_tmp = NULL;
    T->tmp_nrhs = 0;
    size_t bytes = sizeof(double)*(size_t)(T->tmp_units > 0 ? T->tmp_units :
            1)*nrhs;
    int info = starsh_hip_malloc((void **)&T->d_tmp, bytes);
    if(info == STARSH_SUCCESS)
        T->tmp_nrhs = nrhs;
    return info;
}

int starsh_hip_tlr_dmml(starsh_hip_tlr *T, int nrhs, double alpha,
        const double *d_A, int lda, double beta, double *d_B, int ldb)
{
    if(T == NULL || nrhs < 0 || (nrhs > 0 && (d_A == NULL || d_B == NULL ||
                    lda < T->ncols || ldb < T->nrows)))
        return STARSH_WRONG_PARAMETER;
    if(nrhs == 0)
        return STARSH_SUCCESS;
    int info = tmp_reserve(T, nrhs);
    if(info != STARSH_SUCCESS)
        return info;
    return starsh_hip_tlr_apply(&T->plan, T->d_tmp, nrhs, alpha, d_A, lda,
            beta, d_B, ldb);
}

int starsh_hip_current_device(void);

int starsh_hip_tlr_dmml_noalloc(starsh_hip_tlr *T, int nrhs, double alpha,
        const double *d_A, int lda, double beta, double *d_B, int ldb)
{
    if(T == NULL || nrhs < 0 || (nrhs > 0 && (d_A == NULL || d_B == NULL ||
                    lda < T->ncols || ldb < T->nrows)))
        return STARSH_WRONG_PARAMETER;
    if(nrhs == 0)
        return STARSH_SUCCESS;
    const int64_t need = (T->noalloc_units > 0 ? T->noalloc_units : 1)*
        (int64_t)nrhs;
    if(need > TLR_SCRATCH_DOUBLES)
    {
        STARSH_ERROR("the size of this product, %lld ((2 x sum of far-field "
                "ranks + rows of the transposed tiles) x nrhs), is above the "
                "limit of the allocation-free product, %lld (use "
                "starsh_hip_tlr_dmml)",
                (long long)need, (long long)TLR_SCRATCH_DOUBLES);
        return STARSH_WRONG_PARAMETER;
    }
    /* the device address of the static scratch, looked up when the
     * library set up this device (starsh_hip_tlr_new did) */
    double *ptr = NULL;
    if(tlr_scratch(starsh_hip_current_device(), &ptr) != STARSH_SUCCESS)
    {
        STARSH_ERROR("the product scratch is not set up on this device");
        return STARSH_UNKNOWN_ERROR;
    }
    return starsh_hip_tlr_apply(&T->plan, ptr, nrhs, alpha, d_A, lda, beta,
            d_B, ldb);
}

int starsh_hip_tlr_bench(starsh_hip_tlr *T, int nrhs, int reps,
        double *seconds, double *bytes)
{
    if(T == NULL || nrhs <= 0 || reps <= 0 || seconds == NULL)
        return STARSH_WRONG_PARAMETER;
    double *dx = NULL, *dy = NULL;
    size_t nx = (size_t)T->ncols*nrhs, ny = (size_t)T->nrows*nrhs;
    int info = tmp_reserve(T, nrhs);
    if(info == STARSH_SUCCESS)
        info = starsh_hip_malloc((void **)&dx, sizeof(double)*nx);
    if(info == STARSH_SUCCESS)
        info = starsh_hip_malloc((void **)&dy, sizeof(double)*ny);
    double *hx = info == STARSH_SUCCESS ? malloc(sizeof(double)*nx) : NULL;
    if(info == STARSH_SUCCESS && hx == NULL)
        info = STARSH_MALLOC_ERROR;
    if(info == STARSH_SUCCESS)
    {
        for(size_t i = 0; i < nx; i++)
            hx[i] = 1.0/(1.0+(double)(i % 97));
        info = starsh_hip_memcpy_h2d(dx, hx, sizeof(double)*nx);
    }
    if(info == STARSH_SUCCESS)
        info = starsh_hip_tlr_time(&T->plan, T->d_tmp, nrhs, dx,
                (int)T->ncols, dy, (int)T->nrows, reps, seconds);
    /* algorithmic bytes: every factor and near tile read once, X read,
     * Y written */
    if(bytes)
        *bytes = sizeof(double)*((double)T->fac_doubles+(double)nx+
                (double)ny);
    free(hx);
    starsh_hip_free(dx);
    starsh_hip_free(dy);
    return info;
}

int starsh_blrm__dmml_hip(STARSH_blrm *matrix, int nrhs, double alpha,
        double *A, int lda, double beta, double *B, int ldb)
{
    if(matrix == NULL || nrhs < 0)
        return STARSH_WRONG_PARAMETER;
    if(nrhs == 0)
        return STARSH_SUCCESS;
    starsh_hip_tlr *T = NULL;
    int info = starsh_hip_tlr_new(&T, matrix);
    if(info != STARSH_SUCCESS)
        return info;
    if(lda < T->ncols || ldb < T->nrows)
    {
        starsh_hip_tlr_free(T);
        return STARSH_WRONG_PARAMETER;
    }
    double *dA = NULL, *dB = NULL;
    size_t na = (size_t)lda*(nrhs-1)+T->ncols;
    size_t nb = (size_t)ldb*(nrhs-1)+T->nrows;
    info = starsh_hip_malloc((void **)&dA, sizeof(double)*na);
    if(info == STARSH_SUCCESS)
        info = starsh_hip_malloc((void **)&dB, sizeof(double)*nb);
    if(info == STARSH_SUCCESS)
        info = starsh_hip_memcpy_h2d(dA, A, sizeof(double)*na);
    if(info == STARSH_SUCCESS && beta != 0.0)
        info = starsh_hip_memcpy_h2d(dB, B, sizeof(double)*nb);
    if(info == STARSH_SUCCESS)
        info = starsh_hip_tlr_dmml(T, nrhs, alpha, dA, lda, beta, dB, ldb);
    if(info == STARSH_SUCCESS)
    {
        /* only the nrows entries of each column belong to B */
        if(ldb == T->nrows)
            info = starsh_hip_memcpy_d2h(B, dB, sizeof(double)*nb);
        else
            for(int q = 0; q < nrhs && info == STARSH_SUCCESS; q++)
                info = starsh_hip_memcpy_d2h(B+(size_t)q*ldb,
                        dB+(size_t)q*ldb, sizeof(double)*T->nrows);
    }
    starsh_hip_free(dA);
    starsh_hip_free(dB);
    starsh_hip_tlr_free(T);
    return info;
}

int starsh_itersolvers__dcg_hip(STARSH_blrm *matrix, int nrhs, double *B,
        int ldb, double *X, int ldx, double tol, double *work)
{
    (void)work;     /* device buffers are used instead */
    if(matrix == NULL || nrhs <= 0 || B == NULL || X == NULL)
        return STARSH_WRONG_PARAMETER;
    starsh_hip_tlr *T = NULL;
    int info = starsh_hip_tlr_new(&T, matrix);
    if(info != STARSH_SUCCESS)
        return info;
    const int n = (int)T->nrows;
    if(T->ncols != n || ldb < n || ldx < n)
    {
        starsh_hip_tlr_free(T);
        return STARSH_WRONG_PARAMETER;
    }
    const size_t nn = (size_t)n*nrhs;
    double *dB = NULL, *dX = NULL, *dR = NULL, *dP = NULL, *dQ = NULL;
    double *dpart = NULL;
    tlr_cg_state *dst = NULL, *hst = malloc(sizeof(tlr_cg_state)*nrhs);
    int result = -1;
    if(hst == NULL)
        info = STARSH_MALLOC_ERROR;
    double **bufs[] = {&dB, &dX, &dR, &dP, &dQ};
    for(int b = 0; b < 5 && info == STARSH_SUCCESS; b++)
        info = starsh_hip_malloc((void **)bufs[b], sizeof(double)*nn);
    if(info == STARSH_SUCCESS)
        info = starsh_hip_malloc((void **)&dpart, sizeof(double)*
                TLR_CG_PART(nrhs));
    if(info == STARSH_SUCCESS)
        info = starsh_hip_malloc((void **)&dst, sizeof(tlr_cg_state)*
                TLR_CG_STATES(nrhs));
    for(int q = 0; q < nrhs && info == STARSH_SUCCESS; q++)
    {
        info = starsh_hip_memcpy_h2d(dB+(size_t)q*n, B+(size_t)q*ldb,
                sizeof(double)*n);
        if(info == STARSH_SUCCESS)
            info = starsh_hip_memcpy_h2d(dX+(size_t)q*n, X+(size_t)q*ldx,
                    sizeof(double)*n);
    }
    /* R = B - M X, P = R (cg.c:39-43) */
    if(info == STARSH_SUCCESS)
        info = starsh_hip_tlr_dmml(T, nrhs, -1.0, dX, n, 0.0, dR, n);
    if(info == STARSH_SUCCESS)
        info = starsh_hip_vaxpy((int64_t)nn, 1.0, dB, dR);
    if(info == STARSH_SUCCESS)
        info = starsh_hip_vcopy((int64_t)nn, dR, dP);
    if(info == STARSH_SUCCESS)
        info = starsh_hip_cg_start(n, nrhs, tol, dR, dpart, dst);
    /* The iterations are queued without waiting: a column that has met its
     * stopping rule is left alone by the kernels, and the states are read
     * back after 4, 12 and then every 16 iterations (two dot products read
     * back per iteration took as long as its kernels). */
    int look = 4, batch = 4;
    for(int it = 0; it < n && info == STARSH_SUCCESS; it++)
    {
        info = starsh_hip_tlr_dmml(T, nrhs, 1.0, dP, n, 0.0, dQ, n);
        if(info == STARSH_SUCCESS)
            info = starsh_hip_cg_iteration(n, nrhs, it, dP, dQ, dX, dR,
                    dpart, dst);
        if(info != STARSH_SUCCESS || (it+1 < look && it+1 < n))
            continue;
        batch = batch < 16 ? 2*batch : 16;
        look += batch;
        info = starsh_hip_memcpy_d2h(hst, dst+(size_t)((it+1) & 1)*nrhs,
                sizeof(tlr_cg_state)*nrhs);
        int last = -1, finished = 0, running = 0;
        for(int q = 0; info == STARSH_SUCCESS && q < nrhs; q++)
        {
            finished += hst[q].done >= 0;
            running += hst[q].done == -1;
            last = hst[q].done > last ? hst[q].done : last;
        }
        if(info == STARSH_SUCCESS && running == 0)
        {
            result = finished == nrhs ? last : -1;
            break;
        }
    }
    for(int q = 0; q < nrhs && info == STARSH_SUCCESS; q++)
        info = starsh_hip_memcpy_d2h(X+(size_t)q*ldx, dX+(size_t)q*n,
                sizeof(double)*n);
    for(int b = 0; b < 5; b++)
        starsh_hip_free(*bufs[b]);
    starsh_hip_free(dpart);
    starsh_hip_free(dst);
    free(hst);
    starsh_hip_tlr_free(T);
    if(info != STARSH_SUCCESS)
        return -1;
    return result;
}

/* The reference's names (include/starsh.h:601-604, 671-672). */
int starsh_blrm__dmml(STARSH_blrm *matrix, int nrhs, double alpha,
        double *A, int lda, double beta, double *B, int ldb)
{
    return starsh_blrm__dmml_hip(matrix, nrhs, alpha, A, lda, beta, B, ldb);
}

int starsh_blrm__dmml_omp(STARSH_blrm *matrix, int nrhs, double alpha,
        double *A, int lda, double beta, double *B, int ldb)
{
    return starsh_blrm__dmml_hip(matrix, nrhs, alpha, A, lda, beta, B, ldb);
}

int starsh_itersolvers__dcg_omp(STARSH_blrm *matrix, int nrhs, double *B,
        int ldb, double *X, int ldx, double tol, double *work)
{
    return starsh_itersolvers__dcg_hip(matrix, nrhs, B, ldb, X, ldx, tol,
            work);
}
