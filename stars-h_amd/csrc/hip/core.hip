// Core of the randomized SVD: singular values and vectors of the small
// matrix R2 (p x p, with B[:p, :]^T = Q2 R2), the rank by the reference rule
// (src/backends/sequential/dense/dsvfr.c:16-47) and the matrix X from which
// U and V are formed.
//
// One-sided (Hestenes) Jacobi on the columns of R2^T gives R2^T J = W with
// orthogonal columns; the column norms of W are the singular values of B
// and X = W diag(sigma)^-1 holds B's left singular vectors.  Hence, with
// B = Us S Vs^T,
//   U = Q[:, :p] X[:, :r],   V = Vs S = B^T Us = Bt[:, :p] X[:, :r]
// (V = S Vs^T rows as in drsdd.c:83-87), and no rotation is accumulated.
// R2 comes from a QR of B's leading rows, which are graded like the
// singular values; Jacobi on R2^T converges in fewer sweeps than on R2.
#include <float.h>
#include "pipeline.h"
#include "jacobi_rotation.h"

namespace {

constexpr int JACOBI_SWEEPS_DEFAULT = 60;

// Four waves per tile keep a group of 8 or more lanes per column pair up to 64
// rows and leave room for other tiles on the CU; above, W takes the room and
// sixteen waves shorten its chain.  With cores on both sides, few tiles go in
// one launch of sixteen waves, as those of a second one would wait for the
// first; many go in one launch for each.  Device time of whole compressions
// (2D exp and sqexp), all with four waves, all with sixteen, in two launches:
//   55 tiles, largest core at most 50 rows      1.35   1.46      - ms
//   55, 107                                     5.28   3.62   4.10
//   210, 96 (tiles of 1600)                    14.6   13.4   13.9
//   276, 86                                     4.71   3.95   4.12
//   465, 96                                     6.20   4.03   4.18
//   820, 50                                     2.45   3.28      -
//   820, 96 (tiles of 250)                      6.90   5.32   4.87
//   820, 110                                    9.65   7.50   7.30
//   820, 96, most below 64 (tiles of 1600)     33.6   34.4   33.7
//   1035, 86                                    7.87   8.27   7.89
constexpr int CORE_SMALL_PMAX = 64, CORE_SPLIT_TILES = 512;

__device__ inline double group_sum(double v, int g)
{
    return group_sum_lanes(v, g);
}

// One-sided Jacobi step on the column pair (wa, wb) of length p by a group
// of g threads (gl = index in the group): returns true if it rotated.
__device__ inline bool rotate_pair(double *wa, double *wb, int p, int g,
        int gl, double ctol)
{
    double al = 0.0, be = 0.0, ga = 0.0;
    for(int i = gl; i < p; i += g)
    {
        double u = wa[i], v = wb[i];
        al += u*u;
        be += v*v;
        ga += u*v;
    }
    al = group_sum(al, g);
    be = group_sum(be, g);
    ga = group_sum(ga, g);
    if(!jr_rotates(al, be, ga, ctol))
        return false;
    double c, s;
    jacobi_rotation(al, be, ga, c, s);
    for(int i = gl; i < p; i += g)
    {
        double u = wa[i], v = wb[i];
        wa[i] = c*u-s*v;
        wb[i] = s*u+c*v;
    }
    return true;
}

// rotate_pair with both columns read into registers once (E rows per
// thread, p <= E g): the loads of a rotation are issued together and the
// update reads no memory.  The same sums in the same order (rows past p
// hold zeros, which leave every sum unchanged), so the same rotation.
template <int E>
__device__ inline bool rotate_pair_reg(double *wa, double *wb, int p, int g,
        int gl, double ctol)
{
    double u[E], v[E];
    double al = 0.0, be = 0.0, ga = 0.0;
#pragma unroll
    for(int t = 0; t < E; t++)
    {
        const int i = gl+t*g;
        u[t] = i < p ? wa[i] : 0.0;
        v[t] = i < p ? wb[i] : 0.0;
    }
#pragma unroll
    for(int t = 0; t < E; t++)
    {
        al += u[t]*u[t];
        be += v[t]*v[t];
        ga += u[t]*v[t];
    }
    al = group_sum(al, g);
    be = group_sum(be, g);
    ga = group_sum(ga, g);
    if(!jr_rotates(al, be, ga, ctol))
        return false;
    double c, s;
    jacobi_rotation(al, be, ga, c, s);
#pragma unroll
    for(int q = 0; q < E; q++)
    {
        const int i = gl+q*g;
        if(i < p)
        {
            wa[i] = c*u[q]-s*v[q];
            wb[i] = s*u[q]+c*v[q];
        }
    }
    return true;
}

// W: p x p working matrix in LDS (ld p).  A group of g threads handles one
// column pair, g consecutive rows at a time; the groups are as large as
// the threads allow with a group for every pair of a round.
template <int NT>
__device__ void jacobi(double *W, int p, int max_sweeps, int *sweeps_out)
{
    __shared__ int rotations;
    const int pe = p+(p & 1);
    const int npairs = pe/2;
    int g = 64;
    while(g > 1 && g*npairs > NT)
        g >>= 1;
    const int ngroups = NT/g;
    const int grp = threadIdx.x/g, gl = threadIdx.x % g;
    const double ctol = (double)p*DBL_EPSILON;
    int sweep;
    for(sweep = 0; sweep < max_sweeps; sweep++)
    {
        if(threadIdx.x == 0)
            rotations = 0;
        __syncthreads();
        for(int round = 0; round < pe-1; round++)
        {
            for(int pi = grp; pi < npairs; pi += ngroups)
            {
                // Circle method: position 0 fixed, others rotate.
                int a = pi+round, b = pe-1-pi+round;
                a = a > pe-1 ? a-(pe-1) : a;
                b = b > pe-1 ? b-(pe-1) : b;
                a = pi == 0 ? 0 : a;
                if(a > b)
                {
                    int tmp = a;
                    a = b;
                    b = tmp;
                }
                if(b >= p)
                    continue;
                double *wa = W+(int64_t)a*p, *wb = W+(int64_t)b*p;
                const bool rot = p <= 4*g ?
                    rotate_pair_reg<4>(wa, wb, p, g, gl, ctol) :
                    p <= 8*g ? rotate_pair_reg<8>(wa, wb, p, g, gl, ctol) :
                    rotate_pair(wa, wb, p, g, gl, ctol);
                if(rot && gl == 0)
                    atomicAdd(&rotations, 1);
            }
            __syncthreads();
        }
        if(rotations == 0)
            break;
        __syncthreads();
    }
    *sweeps_out = sweep;
}

// Singular values of a tile of which nothing is left (zero sketch): all
// vanish and the rank is 0.
__device__ inline void zero_core(TileDesc &td, double *ws)
{
    for(int j = threadIdx.x; j < td.k; j += blockDim.x)
        ws[td.s_off+j] = 0.0;
    if(threadIdx.x == 0)
        td.rank = 0;
}

// From W with orthogonal columns (p x p, ld ldw, scaled by 1/wunscale): the
// singular values (its column norms) in descending order, the rank and X,
// the r leading columns of W scaled to unit length.  above: the rank is
// known to exceed its limit (the sweeps ended early).  sig: 2 (p+1) doubles
// and perm: p ints of LDS.
__device__ void finish_core(TileDesc &td, double *ws, const double *W,
        int ldw, double wunscale, double *sig, int *perm, int sweeps,
        bool unconverged, bool above)
{
    __shared__ int s_rank;
    const int p = td.p, k = td.k;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double *sorted = sig+p+1;
    for(int j = wave; j < p; j += blockDim.x >> 6)
    {
        double s = 0.0;
        for(int i = lane; i < p; i += 64)
        {
            const double w = W[(int64_t)j*ldw+i];
            s += w*w;
        }
        s = group_sum(s, 64);
        if(lane == 0)
            sig[j] = sqrt(s);
    }
    __syncthreads();
    // Descending order, ties by index.
    for(int j = threadIdx.x; j < p; j += blockDim.x)
    {
        int pos = 0;
        double v = sig[j];
        for(int l = 0; l < p; l++)
            pos += sig[l] > v || (sig[l] == v && l < j);
        perm[pos] = j;
        sorted[pos] = v*wunscale;
    }
    if(threadIdx.x == 0)
        sorted[p] = sqrt(td.tail2);
    __syncthreads();
    double *S = ws+td.s_off;
    for(int j = threadIdx.x; j < k; j += blockDim.x)
        S[j] = j <= p ? sorted[j] : 0.0;
    if(threadIdx.x == 0)
    {
        // dsvfr over the k values, in the reference's order; the zeros past
        // the first p+1 values leave every sum and the loop's condition
        // unchanged, so the loops start after them
        const double tol = td.tol;
        const int nz = p < k ? p+1 : k;
        int i;
        double err_tol = 0;
        for(i = 0; i < nz; i++)
            err_tol += sorted[i]*sorted[i];
        int r;
        if(err_tol == 0)
            r = 0;
        else
        {
            i = nz;
            err_tol *= tol*tol;
            double tmp = sorted[nz-1]*sorted[nz-1];
            while(i > 1 && err_tol >= tmp)
            {
                i--;
                tmp += sorted[i-1]*sorted[i-1];
            }
            r = i;
        }
        if(r > p)
            r = p;
        // a rank above maxrank, or a core SVD that did not converge within
        // the sweep limit (the counterpart of info != 0 from dgesdd), marks
        // a false far-field tile (drsdd.c:78,89-92); the exact engines also
        // require rank < min(m, n)/2 (dsdd.c:53, dqp3.c:84)
        const int mn = td.m < td.n ? td.m : td.n;
        if(r > td.maxrank || unconverged || above ||
                ((td.rule & RSDD_RULE_HALF) && r >= mn/2))
            r = -1;
        s_rank = r;
        td.rank = r;
        // bit 2: not converged; 4: ended with the verdict alone, the
        // singular values have not converged; bits 8-15: sweeps, 16-26: p
        // (diagnostics)
        td.flags |= (unconverged ? 4 : 0) | (above ? 16 : 0) |
            (min(sweeps, 255) << 8) | (p << 16);
    }
    __syncthreads();
    const int r = s_rank;
    if(r <= 0)
        return;
    double *X = ws+td.w_off;
    for(int c = wave; c < r; c += blockDim.x >> 6)
    {
        const int j = perm[c];
        const double sj = sig[j];
        for(int i = lane; i < p; i += 64)
            X[(int64_t)c*p+i] = W[(int64_t)j*ldw+i]/sj;
    }
}

// The tiles with above < p <= lds_p: W in LDS, one workgroup per tile.
// Dynamic LDS: 2 (lds_p+1) doubles of singular values, W (lds_p^2 doubles),
// then lds_p ints.
template <int NT>
__global__ __launch_bounds__(NT) void core_kernel(TileDesc *tiles,
        double *ws, int above, int lds_p, int max_sweeps)
{
    extern __shared__ double dyn[];
    double *sig = dyn, *W = dyn+2*(lds_p+1);
    int *perm = (int *)(W+(int64_t)lds_p*lds_p);
    __shared__ unsigned long long s_wmax;
    TileDesc &td = tiles[blockIdx.x];
    const int p = td.p, k = td.k;
    if(p > lds_p || p <= above)
        return;
    if(p <= 0)
    {
        zero_core(td, ws);
        return;
    }
    const double *R2 = ws+td.r_off;
    // W = R2^T, scaled by the power of two 2^-e that brings its largest
    // entry into [1/2, 1).  The scaling is exact, so the rotations are
    // those of R2^T itself, but squared norms and their squares inside the
    // rotation stay far from the bottom of the FP64 range for tiles whose
    // entries are tiny (far tiles of fast-decaying kernels).
    if(threadIdx.x == 0)
        s_wmax = 0;
    __syncthreads();
    double wmax = 0.0;
    for(int e = threadIdx.x; e < p*p; e += blockDim.x)
    {
        int i = e % p, j = e / p;
        const double v = R2[(int64_t)i*k+j];
        W[(int64_t)j*p+i] = v;
        wmax = fmax(wmax, fabs(v));
    }
    // non-negative doubles order like their bit patterns
    atomicMax(&s_wmax, (unsigned long long)__double_as_longlong(wmax));
    __syncthreads();
    int wexp = 0;
    const double wm = __longlong_as_double((long long)s_wmax);
    if(wm > 0.0 && wm < INFINITY)
        frexp(wm, &wexp);
    const double wscale = ldexp(1.0, -wexp), wunscale = ldexp(1.0, wexp);
    if(wexp != 0)
        for(int e = threadIdx.x; e < p*p; e += blockDim.x)
            W[e] *= wscale;
    __syncthreads();
    int sweeps = 0;
    jacobi<NT>(W, p, max_sweeps, &sweeps);
    __syncthreads();
    finish_core(td, ws, W, p, wunscale, sig, perm, sweeps,
            sweeps >= max_sweeps, false);
}

// The tiles with p > lds_p after pipeline_jacobi_block.  Dynamic LDS: 2
// (pmax+1) doubles, then pmax ints.
__global__ __launch_bounds__(1024) void core_finish_kernel(TileDesc *tiles,
        double *ws, int lds_p, int pmax)
{
    extern __shared__ double dyn[];
    int *perm = (int *)(dyn+2*(pmax+1));
    TileDesc &td = tiles[blockIdx.x];
    if(td.p <= lds_p)
        return;
    finish_core(td, ws, ws+td.j_off, (td.p+15)/16*16, ldexp(1.0, td.wexp),
            dyn, perm, td.sweeps, td.jdone == 0, td.jdone == 2);
}

template <int NT>
int launch_core(TileDesc *d_tiles, int ntiles, double *ws, int above,
        int lds_p, int max_sweeps, hipStream_t s)
{
    const size_t bytes = sizeof(double)*(2*((size_t)lds_p+1)+
            (size_t)lds_p*lds_p)+sizeof(int)*(size_t)lds_p;
    HIP_TRY(hipFuncSetAttribute((const void *)core_kernel<NT>,
                hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
    hipLaunchKernelGGL(core_kernel<NT>, dim3(ntiles), dim3(NT), bytes, s,
            d_tiles, ws, above, lds_p, max_sweeps);
    HIP_TRY(hipGetLastError());
    return STARSH_SUCCESS;
}

} // namespace

// Sweep limit of the Jacobi core: a tile whose core has not converged
// after this many sweeps is reported as a false far-field tile.
static int jacobi_max_sweeps = JACOBI_SWEEPS_DEFAULT;

extern "C" int starsh_hip_jacobi_sweeps(int sweeps)
{
    if(sweeps < 0 || sweeps > JACOBI_SWEEPS_DEFAULT)
        return STARSH_WRONG_PARAMETER;
    jacobi_max_sweeps = sweeps == 0 ? JACOBI_SWEEPS_DEFAULT : sweeps;
    return STARSH_SUCCESS;
}

int pipeline_core(TileDesc *d_tiles, int ntiles, double *ws, int pmax,
        bool certify, int *d_list, int count, int *d_out, int *h_out,
        hipStream_t s)
{
    if(ntiles <= 0)
        return STARSH_SUCCESS;
    if(pmax > 1024)
        return STARSH_WRONG_PARAMETER;
    const int pm = pmax > 0 ? pmax : 1;
    const int lds_p = pm <= CORE_LDS_PMAX ? pm : CORE_LDS_PMAX;
    // up to which size the tiles take four waves
    const int small = lds_p <= CORE_SMALL_PMAX ? lds_p :
        ntiles > CORE_SPLIT_TILES ? CORE_SMALL_PMAX : -1;
    int info = STARSH_SUCCESS;
    if(small > 0)
        info = launch_core<256>(d_tiles, ntiles, ws, -1, small,
                jacobi_max_sweeps, s);
    if(info == STARSH_SUCCESS && lds_p > small)
        info = launch_core<1024>(d_tiles, ntiles, ws, small, lds_p,
                jacobi_max_sweeps, s);
    if(info != STARSH_SUCCESS)
        return info;
    if(pm > lds_p)
    {
        info = pipeline_jacobi_block(d_tiles, d_list, count, ws,
                pm, jacobi_max_sweeps, certify, d_out, h_out, s);
        if(info != STARSH_SUCCESS)
            return info;
        const size_t bytes = sizeof(double)*2*((size_t)pm+1)+
            sizeof(int)*(size_t)pm;
        hipLaunchKernelGGL(core_finish_kernel, dim3(ntiles), dim3(1024),
                bytes, s, d_tiles, ws, lds_p, pm);
        HIP_TRY(hipGetLastError());
    }
    return STARSH_SUCCESS;
}
