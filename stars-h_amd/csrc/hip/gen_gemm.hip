// FP64 MFMA GEMMs whose left operand is a kernel tile generated on the fly:
//   SKETCH  Y[m x k]  = A[m x n] Omega[n x k]
//   PROJ    Bt[n x kc] = A^T[n x m] Q[m x kc]
// A never exists in memory.  Each wave owns 16 rows of the block and all BN
// columns, so every generated entry is produced exactly once per block and
// feeds BN/16 MFMAs; lane l generates A[row = l%16][k = l/16] directly in
// the A-operand layout of v_mfma_f64_16x16x4f64.  The right operand is
// staged through LDS, double buffered, one barrier per K step of 16.
#include "pipeline.h"

typedef double double4_t __attribute__((ext_vector_type(4)));

namespace {

constexpr int BM = 64;
constexpr int BK = 16;

// Column block width and 16-row groups per wave (1 or 2), 0 for the
// choice by size below; set by starsh_hip_set_option.
int gen_gemm_bn = 0;
int gen_gemm_rw = 0;
// The same, chosen by the autotuner for the current call, per operation
// ([0] sketch, [1] projection; 0 = by size); the options above win.
int gen_gemm_tuned_bn[2] = {0, 0};
int gen_gemm_tuned_rw[2] = {0, 0};

// PROJ=false: rows are row points, K runs over column points.
// PROJ=true : rows are column points, K runs over row points (A^T).
// gnbm x gnbn is the block grid of the largest tile of the launch.  SKETCH:
// columns cbeg..cend-1 only, and no tile whose range the columns before them
// have exhausted already.
template <int NDIM, int FAM, int BN, int RW, bool PROJ>
__global__ __launch_bounds__(256) void gen_gemm_kernel(const TileDesc *tiles,
        GemmArgs g, int ntiles, int gnbm, int gnbn, int cbeg, int cend)
{
    constexpr int NF = BN/16;
    constexpr int BMR = BM*RW;      // rows per block: RW 16-row groups/wave
    int tile, bm, bn;
    if(!map_block(blockIdx.x, ntiles, gnbm, gnbn, !PROJ, tile, bm, bn))
        return;
    const TileDesc t = tiles[tile];
    int M, N, K, ldb, ldc;
    const double *B;
    double *C;
    int64_t rbase, kbase;
    const double *xrow, *xk;
    int64_t nrow, nk;
    if(!PROJ)
    {
        if(t.flags & 1)
            return;
        M = t.m; N = t.k < cend ? t.k : cend; K = t.n;
        B = g.ws+t.om_off; ldb = t.n;
        C = g.ws+t.q_off; ldc = t.m;
        rbase = t.r0; kbase = t.c0;
        xrow = t.xr; nrow = t.nr;
        xk = t.xc; nk = t.nc;
    }
    else
    {
        M = t.n; N = t.kc; K = t.m;
        B = g.ws+t.q_off; ldb = t.m;
        C = g.ws+t.bt_off; ldc = t.n;
        rbase = t.c0; kbase = t.r0;
        xrow = t.xc; nrow = t.nc;
        xk = t.xr; nk = t.nr;
    }
    if(M <= 0 || N <= 0)
        return;
    const int row0 = bm*BMR, col0 = cbeg+bn*BN;
    if(row0 >= M || col0 >= N)
        return;
    // 16-column fragments that hold columns of this tile (wave-uniform)
    const int nf_live = (N-col0+15)/16 < NF ? (N-col0+15)/16 : NF;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    __shared__ double Bs[2][BK][BN+2];

    // this lane's generated rows (fixed) and its K offset inside a 4-step
    const int grow0 = row0+wave*16*RW+(lane & 15);
    unsigned okmask = 0;      // bit r: row grow0 + 16 r is inside the tile
    double xi[RW][NDIM];
#pragma unroll
    for(int r = 0; r < RW; r++)
    {
        const bool ok = grow0+16*r < M;
        okmask |= ok ? 1u << r : 0u;
#pragma unroll
        for(int d = 0; d < NDIM; d++)
            xi[r][d] = ok ? xrow[d*nrow+rbase+grow0+16*r] : 0.0;
    }
    const int kl = lane >> 4;

    double4_t acc[RW][NF];
#pragma unroll
    for(int r = 0; r < RW; r++)
#pragma unroll
        for(int f = 0; f < NF; f++)
            acc[r][f] = double4_t{0.0, 0.0, 0.0, 0.0};

    // B staging: thread loads (kk = tid%16, j = tid/16 + 16 s)
    const int bk = tid & 15, bj = tid >> 4;
    double breg[NF];
    double areg[RW][4];

    auto load_b = [&](int k0) {
#pragma unroll
        for(int s = 0; s < NF; s++)
        {
            const int j = col0+bj+16*s, k = k0+bk;
            breg[s] = (j < N && k < K) ? B[(int64_t)j*ldb+k] : 0.0;
        }
    };
    auto store_b = [&](int buf) {
#pragma unroll
        for(int s = 0; s < NF; s++)
            Bs[buf][bk][bj+16*s] = breg[s];
    };
    auto gen_a = [&](int k0) {
        if constexpr(BN*RW <= 128)
        {
            // few MFMAs per entry: issue the point loads together
            double yv[4][NDIM];
#pragma unroll
            for(int q = 0; q < 4; q++)
            {
                const int k = k0+4*q+kl;
                const int64_t j = kbase+(k < K ? k : K-1);
#pragma unroll
                for(int d = 0; d < NDIM; d++)
                    yv[q][d] = xk[d*nk+j];
            }
#pragma unroll
            for(int r = 0; r < RW; r++)
#pragma unroll
                for(int q = 0; q < 4; q++)
                {
                    const int k = k0+4*q+kl;
                    const double v = kval_pt<NDIM, FAM>(t.kp, xi[r], yv[q]);
                    areg[r][q] = ((okmask >> r & 1u) && k < K) ? v : 0.0;
                }
        }
        else
        {
            // MFMA-bound: keep registers for the accumulators
#pragma unroll
            for(int q = 0; q < 4; q++)
            {
                const int k = k0+4*q+kl;
#pragma unroll
                for(int r = 0; r < RW; r++)
                {
                    const double v = kval<NDIM, FAM>(t.kp, xi[r], xk, nk,
                            kbase+(k < K ? k : K-1));
                    areg[r][q] = ((okmask >> r & 1u) && k < K) ? v : 0.0;
                }
            }
        }
    };

    load_b(0);
    store_b(0);
    gen_a(0);
    __syncthreads();
    int buf = 0;
    for(int k0 = 0; k0 < K; k0 += BK)
    {
        double acur[RW][4];
#pragma unroll
        for(int r = 0; r < RW; r++)
#pragma unroll
            for(int q = 0; q < 4; q++)
                acur[r][q] = areg[r][q];
        const bool more = k0+BK < K;
        if(more)
        {
            load_b(k0+BK);
            gen_a(k0+BK);
        }
        if constexpr(BN*RW <= 128)
        {
            // fragments past the tile's own width are skipped (uniform)
#pragma unroll
            for(int f = 0; f < NF; f++)
                if(f < nf_live)
                {
#pragma unroll
                    for(int q = 0; q < 4; q++)
                    {
                        const double b = Bs[buf][4*q+kl][f*16+(lane & 15)];
#pragma unroll
                        for(int r = 0; r < RW; r++)
                            acc[r][f] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                                    acur[r][q], b, acc[r][f], 0, 0, 0);
                    }
                }
        }
        else
        {
#pragma unroll
            for(int q = 0; q < 4; q++)
            {
#pragma unroll
                for(int f = 0; f < NF; f++)
                {
                    // fragments past the tile's own width are skipped
                    // (uniform); each B value feeds RW MFMAs
                    if(!PROJ || f < nf_live)
                    {
                        const double b = Bs[buf][4*q+kl][f*16+(lane & 15)];
#pragma unroll
                        for(int r = 0; r < RW; r++)
                            acc[r][f] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                                    acur[r][q], b, acc[r][f], 0, 0, 0);
                    }
                }
            }
        }
        if(more)
            store_b(buf ^ 1);
        __syncthreads();
        buf ^= 1;
    }
    // epilogue: lane holds rows lane/16 + 4 v, column lane%16 of each frag
#pragma unroll
    for(int r = 0; r < RW; r++)
#pragma unroll
        for(int f = 0; f < NF; f++)
        {
            const int gj = col0+f*16+(lane & 15);
            if(gj >= N)
                continue;
#pragma unroll
            for(int v = 0; v < 4; v++)
            {
                const int gi = row0+wave*16*RW+r*16+(lane >> 4)+4*v;
                if(gi < M)
                    C[(int64_t)gj*ldc+gi] = acc[r][f][v];
            }
        }
}

template <int NDIM, int FAM, int BN, int RW, bool PROJ>
int launch_one(const TileDesc *d_tiles, int ntiles, int mmax, int cbeg,
        int cend, const GemmArgs &g, hipStream_t s)
{
    const int nbm = (mmax+BM*RW-1)/(BM*RW);
    const int nbn = (cend-cbeg+BN-1)/BN;
    const int64_t grid = mapped_grid(ntiles, nbm, nbn, !PROJ);
    if(grid > 0x7fffffff)
        return STARSH_WRONG_PARAMETER;
    hipLaunchKernelGGL((gen_gemm_kernel<NDIM, FAM, BN, RW, PROJ>),
            dim3((unsigned)grid), dim3(256), 0, s, d_tiles, g, ntiles, nbm,
            nbn, cbeg, cend);
    HIP_TRY(hipGetLastError());
    return STARSH_SUCCESS;
}

template <bool PROJ>
struct GenLaunch
{
    const TileDesc *tiles;
    int ntiles, mmax, cbeg, cend, bn, rw;
    const GemmArgs &g;
    hipStream_t s;
    template <int NDIM, int FAM> int operator()() const
    {
#define ONE(BN, RW) return launch_one<NDIM, FAM, BN, RW, PROJ>(tiles, \
        ntiles, mmax, cbeg, cend, g, s)
        if(bn == 256)
        {
            if(rw == 2)
                ONE(256, 2);
            ONE(256, 1);
        }
        if(bn == 128)
        {
            if(rw == 2)
                ONE(128, 2);
            ONE(128, 1);
        }
        if(rw == 2)
            ONE(64, 2);
        ONE(64, 1);
#undef ONE
    }
};

// Column block and row groups forced by the options or the autotuner (0:
// not).
int forced_bn(int proj)
{
    return gen_gemm_bn > 0 ? gen_gemm_bn : gen_gemm_tuned_bn[proj];
}

int forced_rw(int proj)
{
    return gen_gemm_rw > 0 ? gen_gemm_rw : gen_gemm_tuned_rw[proj];
}

} // namespace

extern "C" int starsh_hip_gen_gemm_rw(int rw)
{
    if(rw != 0 && rw != 1 && rw != 2)
        return STARSH_WRONG_PARAMETER;
    gen_gemm_rw = rw;
    return STARSH_SUCCESS;
}

extern "C" int hip_set_tuned_gemm(int proj, int bn, int rw)
{
    if((proj != 0 && proj != 1) || (bn != 0 && bn != 64 && bn != 128 &&
                bn != 256) || (rw != 0 && rw != 1 && rw != 2))
        return STARSH_WRONG_PARAMETER;
    gen_gemm_tuned_bn[proj] = bn;
    gen_gemm_tuned_rw[proj] = rw;
    return STARSH_SUCCESS;
}

extern "C" int starsh_hip_gen_gemm_bn(int bn)
{
    if(bn != 0 && bn != 64 && bn != 128 && bn != 256)
        return STARSH_WRONG_PARAMETER;
    gen_gemm_bn = bn;
    return STARSH_SUCCESS;
}

// The sketch's columns go in chunks, computed as the Gram-Schmidt reaches
// them: a tile whose range is exhausted by then has no use for the rest (the
// random columns after that point are dropped unread).  A chunk is one column
// block.  Wide blocks reuse each generated entry most, so the first chunk is
// narrow only where tiles that need every column lose nothing by it: with
// more than 256 columns, when the padding that the narrow blocks save pays
// for them (417-448 and 513-640 columns, say, but not 449-512).  The costs of
// 64, 128 and 256 columns measured, scaled to 22.6 for 256: 2D sqexp 820
// tiles of 1600 8.2, 14.4 (23.7 ms for 256); 2D exp the same 8.6, 14.6, 820
// of 500 7.8, 14.0; 3D Matern 136 of 2048 8.4, 12.3; sin(kr)/r 153 of 1536
// 7.3, 11.8; Coulomb 6.9, 12.4.  The highest are taken: with the lowest,
// 449-512 columns would go narrow as well, 5% slower for the 2D kernels.  2D
// sqexp
// N=64000, 416 columns, all tiles exhausted within 96: sketch 45.3 -> 15.3
// ms; sin(kr)/r N=25000, 400 columns, 17 of 153 tiles needing all: 11.7 ->
// 9.4 ms.
int pipeline_sketch_chunks(int k, SketchChunk *c)
{
    const int fb = forced_bn(0), rw = forced_rw(0) > 0 ? forced_rw(0) : 1;
    int n = 0;
    auto add = [&](int beg, int bn) {
        const int end = beg+bn < k ? beg+bn : k;
        c[n++] = SketchChunk{beg, end, bn, rw};
        return end;
    };
    // block for the last r columns, and its cost
    auto block = [](int r) { return r <= 64 ? 64 : r <= 128 ? 128 : 256; };
    auto cost = [](int bn) {
        return bn == 64 ? 8.6 : bn == 128 ? 14.6 : 22.6; };
    int beg = 0;
    if(fb > 0)
        while(beg < k)
            beg = add(beg, fb);
    else if(k <= 256)
        add(0, block(k));
    else
    {
        const int rest = k-128;
        const double wide = (k+255)/256*cost(256);
        const double narrow = cost(128)+rest/256*cost(256)+
            (rest % 256 ? cost(block(rest % 256)) : 0.0);
        beg = add(0, narrow <= 1.03*wide ? 128 : 256);
        while(beg < k)
            beg = add(beg, k-beg > 256 ? 256 : block(k-beg));
    }
    return n;
}

int pipeline_sketch_gen(const TileDesc *d_tiles, int ntiles, int mmax,
        const SketchChunk &c, const GemmArgs &g, hipStream_t s)
{
    if(ntiles <= 0 || mmax <= 0 || c.end <= c.beg)
        return STARSH_SUCCESS;
    return dispatch_kernel(g.ndim, g.family, GenLaunch<false>{d_tiles,
            ntiles, mmax, c.beg, c.end, c.bn, c.rw, g, s});
}

int pipeline_proj_gen(const TileDesc *d_tiles, int ntiles, int mmax,
        int nmax, const GemmArgs &g, hipStream_t s)
{
    if(ntiles <= 0 || mmax <= 0 || nmax <= 0)
        return STARSH_SUCCESS;
    // By size (measured at tile 1600): N = kept columns, often just under a
    // multiple of 256, wastes less on 128-column blocks with two 16-row
    // groups per wave.
    int bn = nmax > 64 ? 128 : 64, rw = nmax > 64 ? 2 : 1;
    if(forced_bn(1) > 0)
        bn = forced_bn(1);
    if(forced_rw(1) > 0)
        rw = forced_rw(1);
    return dispatch_kernel(g.ndim, g.family, GenLaunch<true>{d_tiles, ntiles,
            mmax, 0, nmax, bn, rw, g, s});
}
