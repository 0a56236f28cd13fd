/* Global relative Frobenius error of a compressed matrix on the GPU.
 * Follows src/backends/openmp/blrm/dfe.c:16-148 of ecrc/stars-h 0.3.1:
 * every far-field tile is regenerated and |A|, |A - U V^T| are measured;
 * near-field tiles contribute |A|; off-diagonal tiles of a symmetric format
 * count twice (factor sqrt(2) on both norms).  The result is
 * |far differences|_2 / |all tile norms|_2.  Near-field tiles are
 * regenerated on the GPU rather than read from near_D: near_D holds the
 * same kernel values (generated by the same device code). */
#include "common.h"
#include "kernels_host.h"
#include "rsdd.h"
#include "hip_driver.h"

double starsh_blrm__dfe_hip_tiles(STARSH_blrm *matrix, double *far_err,
        double *far_norm)
{
    STARSH_blrm *M = matrix;
    if(M == NULL || M->format == NULL)
        return -1;
    STARSH_blrf *F = M->format;
    hip_problem hp;
    if(hip_driver_prepare(F, 1, 0.0, 0, &hp) != STARSH_SUCCESS)
        return -1;
    STARSH_cluster *RC = F->row_cluster, *CC = F->col_cluster;
    STARSH_int nfar = F->nblocks_far, nnear = F->nblocks_near;
    STARSH_int nt = nfar+nnear;
    double result = -1;
    int *m = malloc(sizeof(int)*(nt+1)), *n = malloc(sizeof(int)*(nt+1));
    int *rk = malloc(sizeof(int)*(nt+1));
    int64_t *r0 = malloc(sizeof(int64_t)*(nt+1));
    int64_t *c0 = malloc(sizeof(int64_t)*(nt+1));
    int64_t *uo = malloc(sizeof(int64_t)*(nt+1));
    int64_t *vo = malloc(sizeof(int64_t)*(nt+1));
    double *a2 = malloc(sizeof(double)*(nt+1));
    double *d2 = malloc(sizeof(double)*(nt+1));
    const double **seg = malloc(sizeof(*seg)*(2*nfar+1));
    int64_t *seglen = malloc(sizeof(int64_t)*(2*nfar+1));
    double *dU = NULL, *dV = NULL;
    if(!m || !n || !rk || !r0 || !c0 || !uo || !vo || !a2 || !d2 || !seg ||
            !seglen)
        goto done;
    int64_t su = 0, sv = 0;
    for(STARSH_int bi = 0; bi < nt; bi++)
    {
        int far = bi < nfar;
        STARSH_int i = far ? F->block_far[2*bi] : F->block_near[2*(bi-nfar)];
        STARSH_int j = far ? F->block_far[2*bi+1] :
            F->block_near[2*(bi-nfar)+1];
        m[bi] = (int)RC->size[i];
        n[bi] = (int)CC->size[j];
        r0[bi] = RC->start[i];
        c0[bi] = CC->start[j];
        rk[bi] = far ? M->far_rank[bi] : 0;
        if(rk[bi] < 0)
            goto done;
        uo[bi] = su;
        vo[bi] = sv;
        su += (int64_t)m[bi]*rk[bi];
        sv += (int64_t)n[bi]*rk[bi];
    }
    /* U of every far-field tile, then V */
    for(STARSH_int bi = 0; bi < nfar; bi++)
    {
        seg[bi] = rk[bi] > 0 ? M->far_U[bi]->data : NULL;
        seglen[bi] = (int64_t)m[bi]*rk[bi];
        seg[nfar+bi] = rk[bi] > 0 ? M->far_V[bi]->data : NULL;
        seglen[nfar+bi] = (int64_t)n[bi]*rk[bi];
    }
    if(starsh_hip_malloc((void **)&dU, sizeof(double)*su) != 0 ||
            starsh_hip_malloc((void **)&dV, sizeof(double)*sv) != 0 ||
            hip_upload_segments(dU, nfar, seg, seglen) != 0 ||
            hip_upload_segments(dV, nfar, seg+nfar, seglen+nfar) != 0)
        goto done;
    if(starsh_hip_tile_errors(&hp.kd, hp.d_xr, hp.nr, hp.d_xc, hp.nc,
                (int)nt, r0, c0, m, n, rk, dU, uo, dV, vo, a2, d2) != 0)
        goto done;
    {
        double diff = 0, norm = 0, sq2 = sqrt(2.);
        for(STARSH_int bi = 0; bi < nt; bi++)
        {
            int far = bi < nfar;
            STARSH_int i = far ? F->block_far[2*bi] :
                F->block_near[2*(bi-nfar)];
            STARSH_int j = far ? F->block_far[2*bi+1] :
                F->block_near[2*(bi-nfar)+1];
            double tn = sqrt(a2[bi]), td = sqrt(d2[bi]);
            if(far)
            {
                if(far_err)
                    far_err[bi] = tn > 0 ? td/tn : 0.0;
                if(far_norm)
                    far_norm[bi] = tn;
            }
            if(i != j && F->symm == 'S')
            {
                tn *= sq2;
                td *= sq2;
            }
            norm += tn*tn;
            if(far)
                diff += td*td;
        }
        result = sqrt(diff)/sqrt(norm);
    }
done:
    starsh_hip_free(dU);
    starsh_hip_free(dV);
    free(seg); free(seglen); free(m); free(n); free(rk); free(r0); free(c0);
    free(uo); free(vo); free(a2); free(d2);
    hip_driver_release(&hp);
    return result;
}

double starsh_blrm__dfe_hip(STARSH_blrm *matrix)
{
    return starsh_blrm__dfe_hip_tiles(matrix, NULL, NULL);
}

/* The reference's names (include/starsh.h:622-623). */
double starsh_blrm__dfe(STARSH_blrm *matrix)
{
    return starsh_blrm__dfe_hip(matrix);
}

double starsh_blrm__dfe_omp(STARSH_blrm *matrix)
{
    return starsh_blrm__dfe_hip(matrix);
}
