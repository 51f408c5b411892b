// cholesky_big.hip — FP64 Cholesky solve for normal matrices too large for one workgroup's LDS.
//
// Solver::solve (solver.h:70-105: cusolverDnDpotrf + Dpotrs on the FP64 copy of the FP32 normal
// matrix, copyMatsFloatToDouble / copyVectorDoubleToFloatNegated, solver.cu:11-81) for the
// joint identity-stage system (K up to a few thousand: 199 + 199 + 94 per frame).  Blocked
// right-looking factorisation in place on an FP64 copy in HBM, 32-column panels:
//   k_chol_first   the first 32x32 diagonal block, factored by one wavefront per matrix, and -g put
//                  into the matrix's unused upper triangle as one more row below the last;
//   k_chol_offdiag a grid of 64-row blocks per matrix: the panel below the diagonal block, L21 =
//                  A21 L11^-T (one row per thread in registers, L11 and its reciprocal diagonal in
//                  LDS); the row of -g with it, which leaves L^-1 (-g) behind;
//   k_chol_update  a grid of 32x32 tiles of the trailing lower triangle per matrix:
//                  A22 -= L21 L21^T, both 32-row slices of the panel staged in LDS; the workgroup
//                  of the next diagonal block factors it at once;
//   k_chol_back    one workgroup per matrix: L^T delta = L^-1 (-g) by 32-row panels, right-looking.
// The chain of K dependent columns bounds it, at two launches a panel: one matrix of 1338 unknowns
// took 2976 us with the diagonal block in a launch of its own (15 us each), rows solved entry by
// entry (29 us), and the forward solve after the factorisation (about half of 747 us); now 1386 us.
// A non-positive (or NaN) pivot marks the matrix TDI_NOT_PD; its later launches do nothing.
#include "chol.h"
#include "common.h"

namespace tdi {

namespace {

constexpr int CB = 32;   // panel width

__global__ void __launch_bounds__(256) k_f32_to_f64(size_t n, const float* __restrict__ in, double* __restrict__ out)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        out[i] = in[i];
}

// Where entry j of the row of -g (then of L^-1 (-g)) is kept: the strict upper triangle of row 0, and for
// the last entry of row 1 (K >= CHOL_BIG_MINK).
__device__ __forceinline__ size_t rhs_at(int K, int j) { return j < K - 1 ? (size_t)j + 1 : (size_t)2 * K - 1; }

// The diagonal block of the panel at k0, in r (lane i: row i, entries j <= i; rows and columns past nb
// the identity's), factored by one wavefront and written.  In a step the root and the division of a
// column are independent of the update by the column before, which fills their gaps.
__device__ __forceinline__ void chol_diag(int K, int k0, int nb, double* __restrict__ M, double (&r)[CB],
                                          int* __restrict__ status)
{
    const int lane = threadIdx.x & 63;
    bool bad = false;
    double dg = 0.0;
#pragma unroll
    for (int k = 0; k < CB; ++k) {
        const double d = lane_read(r[k], k);
        bad = bad || !(d > 0.0);
        const double dk = sqrt(d), inv = 1.0 / dk;
        dg = lane == k ? dk : dg;
        r[k] *= inv;
        if (k > 0) {
#pragma unroll
            for (int j = k + 1; j < CB; ++j) r[j] = fma(-r[k - 1], lane_read(r[k - 1], j), r[j]);
        }
        if (k + 1 < CB) r[k + 1] = fma(-r[k], lane_read(r[k], k + 1), r[k + 1]);
        __builtin_amdgcn_sched_barrier(0);
    }
    if (bad) {
        if (lane == 0) *status = TDI_NOT_PD;
        return;
    }
    if (lane < nb) {
        double* Mw = M + (size_t)(k0 + lane) * K + k0;
#pragma unroll
        for (int j = 0; j < CB; ++j)
            if (j < lane) Mw[j] = r[j];
        Mw[lane] = dg;
    }
}

template <typename TG>
__global__ void __launch_bounds__(64) k_chol_first(int K, double* __restrict__ A, const TG* __restrict__ g,
                                                    int* __restrict__ status)
{
    const int mtx = blockIdx.x, lane = threadIdx.x, nb = min(CB, K);
    if (status[mtx] != TDI_OK) return;
    double* M = A + (size_t)mtx * K * K;
    const double* Mr = M + (size_t)min(lane, nb - 1) * K;
    double r[CB];
#pragma unroll
    for (int j = 0; j < CB; ++j) {
        const double x = Mr[min(j, nb - 1)];
        r[j] = (lane < nb && j < nb && j <= lane) ? x : (lane == j ? 1.0 : 0.0);
    }
    for (int j = lane; j < K; j += 64) M[rhs_at(K, j)] = -(double)g[(size_t)mtx * K + j];
    chol_diag(K, 0, nb, M, r, status + mtx);
}

// The panel below the diagonal block: row r of A21 (row K: -g) solves x L11^T = a, 64 rows per workgroup
// (a grid over the rows), each row in its thread's registers, L11 by columns and the reciprocals of its
// diagonal in LDS (read as broadcasts).  An entry that is done leaves every later one at once (the same
// products in the same order as entry by entry, but a chain of 64 operations instead of 528).
__global__ void __launch_bounds__(64) k_chol_offdiag(int K, int k0, double* __restrict__ A,
                                                      const int* __restrict__ status)
{
    const int mtx = blockIdx.y;
    if (status[mtx] != TDI_OK) return;
    double* M = A + (size_t)mtx * K * K;
    const int nb = min(CB, K - k0), tid = threadIdx.x;
    const int r0 = k0 + nb + blockIdx.x * 64;
    __shared__ double2 D2[CB][CB / 2];      // D[j][i] = L11[i][j]
    __shared__ double sinv[CB];
    double* D = reinterpret_cast<double*>(D2);
    const int gr = r0 + tid;
    const bool in = gr <= K, last = gr >= K;
    double* Mr = M + (size_t)min(gr, K - 1) * K + k0;
    double p[CB];
    {
        // every load issued before the LDS stores (64 threads, 16 entries of L11 each)
        double v[CB * CB / 64];
#pragma unroll
        for (int q = 0; q < CB * CB / 64; ++q) {
            const int e = tid + 64 * q, i = e / CB, j = e - i * CB;
            const double x = M[(size_t)(k0 + min(i, nb - 1)) * K + k0 + min(j, nb - 1)];
            v[q] = (i < nb && j < nb && j <= i) ? x : (i == j ? 1.0 : 0.0);
        }
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            const int c = min(j, nb - 1);
            const double x = last ? M[rhs_at(K, k0 + c)] : Mr[c];
            p[j] = j < nb ? x : 0.0;
        }
#pragma unroll
        for (int q = 0; q < CB * CB / 64; ++q) {
            const int e = tid + 64 * q, i = e / CB, j = e - i * CB;
            D[j * CB + i] = v[q];
            if (i == j) sinv[j] = 1.0 / v[q];
        }
    }
    __syncthreads();
    double2 l[CB / 2], ln[CB / 2];
#pragma unroll
    for (int q = 0; q < CB / 2; ++q) l[q] = D2[0][q];
#pragma unroll
    for (int j = 0; j < CB; ++j) {
#pragma unroll
        for (int q = (j + 2) / 2; q < CB / 2; ++q) ln[q] = D2[min(j + 1, CB - 1)][q];
        p[j] *= sinv[j];
#pragma unroll
        for (int q = j + 1; q < CB; ++q) p[q] = fma(-p[j], (q & 1) ? l[q / 2].y : l[q / 2].x, p[q]);
        // the updates stay here: put off, they would keep every column's entries in registers
#pragma unroll
        for (int q = j + 1; q < CB; ++q) asm volatile("" : "+v"(p[q]) :: "memory");
#pragma unroll
        for (int q = 0; q < CB / 2; ++q) l[q] = ln[q];
    }
    if (!in) return;
#pragma unroll
    for (int j = 0; j < CB; ++j)
        if (j < nb) {
            if (last) M[rhs_at(K, k0 + j)] = p[j];
            else Mr[j] = p[j];
        }
}

// Tile (ti, tj), ti >= tj, of the trailing matrix below/right of the panel at k0.
__global__ void __launch_bounds__(256) k_chol_update(int K, int k0, double* __restrict__ A,
                                                      int* __restrict__ status)
{
    const int mtx = blockIdx.y;
    const int r0 = k0 + CB;                        // first trailing row
    const int T = (K - r0 + CB - 1) / CB;
    int t = blockIdx.x, ti = 0;
    while (ti < T && t > ti) { t -= ti + 1; ++ti; }   // tile t of row ti: tj = t, 0 <= tj <= ti
    if (ti >= T) return;
    const int tj = t;
    double* M = A + (size_t)mtx * K * K;
    __shared__ double Li[CB][CB + 1], Lj[CB][CB + 1];
    __shared__ int sok;
    const int tid = threadIdx.x;
    const int nb = min(CB, K - k0);
    // one read for the whole workgroup: the one that factors the next diagonal block may write it meanwhile
    if (tid == 0) sok = status[mtx] == TDI_OK;
    {
        // every load of both slices issued before the LDS stores (256 threads, 4 entries each)
        double vi[CB * CB / 256], vj[CB * CB / 256];
#pragma unroll
        for (int q = 0; q < CB * CB / 256; ++q) {
            const int e = tid + 256 * q, r = e / CB, c = e - r * CB;
            const int ri = r0 + ti * CB + r, rj = r0 + tj * CB + r;
            const double xi = M[(size_t)min(ri, K - 1) * K + k0 + min(c, nb - 1)];
            const double xj = M[(size_t)min(rj, K - 1) * K + k0 + min(c, nb - 1)];
            vi[q] = (ri < K && c < nb) ? xi : 0.0;
            vj[q] = (rj < K && c < nb) ? xj : 0.0;
        }
#pragma unroll
        for (int q = 0; q < CB * CB / 256; ++q) {
            const int e = tid + 256 * q, r = e / CB, c = e - r * CB;
            Li[r][c] = vi[q];
            Lj[r][c] = vj[q];
        }
    }
    __syncthreads();
    if (!sok) return;
    // 256 threads x 4 entries: thread (a, b4) computes row a, columns b4..b4+3 of the tile
    const int a = tid >> 3, b4 = (tid & 7) * 4;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int c = 0; c < CB; ++c) {
        const double li = Li[a][c];
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = fma(li, Lj[b4 + q][c], acc[q]);
    }
    const int gi = r0 + ti * CB + a;
    if (ti != 0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int gj = r0 + tj * CB + b4 + q;
            if (gi < K && gj < K && gj <= gi) M[(size_t)gi * K + gj] -= acc[q];
        }
    }
    if (ti == tj && tid < CB && r0 + tj * CB + tid < K) {       // the row of -g, at the tile's columns
        double* y = M + rhs_at(K, r0 + tj * CB + tid);
        double s[CB / 4];                    // sums of four in order, then by pairs
#pragma unroll
        for (int c = 0; c < CB; ++c)         // L is 0 past nb
            s[c / 4] = fma(Lj[tid][c], M[rhs_at(K, k0 + min(c, nb - 1))], c % 4 ? s[c / 4] : 0.0);
        *y -= ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    }
    if (ti != 0) return;
    // the next panel's diagonal block
    double v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = M[(size_t)min(gi, K - 1) * K + min(r0 + b4 + q, K - 1)] - acc[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q)
        Li[a][b4 + q] = (gi < K && r0 + b4 + q <= gi) ? v[q] : (a == b4 + q ? 1.0 : 0.0);
    __syncthreads();
    if (tid >= 64) return;
    double r[CB];
#pragma unroll
    for (int j = 0; j < CB; ++j) r[j] = tid < CB ? Li[tid & (CB - 1)][j] : 0.0;
    chol_diag(K, r0, min(CB, K - r0), M, r, status + mtx);
}

// L^T delta = y (left by the factorisation), one workgroup per matrix, by 32-row panels from the last,
// with the solution in LDS (K <= CHOL_BIG_MAXK), right-looking.  The panels' serial parts bound it, so
// wavefront 0 solves a panel's triangle (lane i holding column i, the solved entries passed by lane
// reads) while the others already load the panel's rows, a column each, and all the next panel's
// diagonal block.
constexpr int BACK_THREADS = 768, BACK_COLS = BACK_THREADS - 64;   // three wavefronts a SIMD: 32 rows fit in registers

template <typename TD>
__global__ void __launch_bounds__(BACK_THREADS) k_chol_back(int K, const double* __restrict__ A, TD* __restrict__ delta,
                                                             const int* __restrict__ status)
{
    const int mtx = blockIdx.x;
    if (status[mtx] != TDI_OK) return;
    const double* L = A + (size_t)mtx * K * K;
    __shared__ double sy[CHOL_BIG_MAXK];
    __shared__ double sD[CB][CB + 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int i = tid; i < K; i += blockDim.x) sy[i] = L[rhs_at(K, i)];
    // entry e of the diagonal block at p0 (the identity past the matrix); a thread has two at most
    auto entry = [&](int p0, int e) {
        const int nb = min(CB, K - p0), di = (e >> 5) & (CB - 1), dj = e & (CB - 1);
        const double x = L[(size_t)(p0 + min(di, nb - 1)) * K + p0 + min(dj, nb - 1)];
        return di < nb && dj < nb ? x : di == dj ? 1.0 : 0.0;
    };
    const int last = ((K - 1) / CB) * CB;
    auto store = [&](double a, double b) {
        sD[tid >> 5][tid & (CB - 1)] = a;
        if (tid + BACK_THREADS < CB * CB) sD[(tid + BACK_THREADS) >> 5][tid & (CB - 1)] = b;
    };
    store(entry(last, tid), entry(last, tid + BACK_THREADS));
    __syncthreads();
    for (int p0 = last; p0 >= 0; p0 -= CB) {
        const int nb = min(CB, K - p0), col = tid - 64;
        const int pn = max(p0 - CB, 0);
        const double na = entry(pn, tid), nc = entry(pn, tid + BACK_THREADS);
        double lv[CB];
        if (wave == 0) {
            int c = lane & (CB - 1);
            asm volatile("" : "+v"(c));        // the comparisons are made here, not kept over the panels
            double lc[CB];
#pragma unroll
            for (int j = 0; j < CB; ++j) lc[j] = j > c ? sD[j][c] : 0.0;
            const double dd = ch_finite(sD[c][c]), rinv = 1.0 / dd;
            double r = c < nb ? sy[p0 + c] : 0.0;
#pragma unroll
            for (int j = CB - 1; j >= 0; --j) r = fma(-lc[j], lane_read(ch_div(r, dd, rinv), j), r);
            if (lane < nb) sy[p0 + lane] = ch_div(r, dd, rinv);
        } else {
            const double* Lc = L + (size_t)p0 * K + min(col, max(p0 - 1, 0));
#pragma unroll
            for (int j = 0; j < CB; ++j) lv[j] = Lc[(size_t)min(j, nb - 1) * K];
        }
        __syncthreads();
        if (wave > 0 && col < p0) {
            double acc = 0.0;
#pragma unroll
            for (int j = 0; j < CB; ++j)
                if (j < nb) acc = fma(lv[j], sy[p0 + j], acc);
            sy[col] -= acc;
            for (int i = col + BACK_COLS; i < p0; i += BACK_COLS) {
                const double* Lc = L + (size_t)p0 * K + i;
                acc = 0.0;
#pragma unroll
                for (int j = 0; j < CB; ++j) {
                    const double l = Lc[(size_t)min(j, nb - 1) * K];
                    acc = fma(j < nb ? l : 0.0, sy[p0 + min(j, nb - 1)], acc);
                }
                sy[i] -= acc;
            }
        }
        store(na, nc);
        __syncthreads();
    }
    for (int i = tid; i < K; i += blockDim.x) delta[(size_t)mtx * K + i] = (TD)sy[i];
}

} // namespace

// Factorisation and solve on the FP64 matrices A (overwritten by the factor); g FP32 or FP64.
template <typename TG, typename TD>
static int chol_big_run(int n, int K, double* A, const TG* g, TD* delta, int* status, hipStream_t s)
{
    hipLaunchKernelGGL(k_chol_first<TG>, dim3(n), dim3(64), 0, s, K, A, g, status);
    for (int k0 = 0; k0 < K; k0 += CB) {
        const int below = std::max(0, K - k0 - CB);
        hipLaunchKernelGGL(k_chol_offdiag, dim3((below + 64) / 64, n), dim3(64), 0, s, K, k0, A, status);
        const int T = (below + CB - 1) / CB;
        if (T > 0) hipLaunchKernelGGL(k_chol_update, dim3(T * (T + 1) / 2, n), dim3(256), 0, s, K, k0, A, status);
        if (hipGetLastError() != hipSuccess) return TDI_ERR_HIP;
    }
    hipLaunchKernelGGL(k_chol_back<TD>, dim3(n), dim3(BACK_THREADS), 0, s, K, A, delta, status);
    return hipGetLastError() != hipSuccess ? TDI_ERR_HIP : TDI_OK;
}

static int chol_big_args(int K)
{
    if (K > CHOL_BIG_MAXK) {
        set_error("cholesky: K=%d > %d", K, CHOL_BIG_MAXK);
        return TDI_ERR_ARG;
    }
    if (K < CHOL_BIG_MINK) {                 // rhs_at
        set_error("cholesky (large K): K=%d < %d", K, CHOL_BIG_MINK);
        return TDI_ERR_ARG;
    }
    return TDI_OK;
}

int launch_cholesky_big(int n, int K, const float* H, const float* g, float* delta, int* status, hipStream_t s)
{
    if (int rc = chol_big_args(K)) return rc;
    double* A = nullptr;
    const size_t nkk = (size_t)n * K * K;
    if (hipMalloc((void**)&A, sizeof(double) * nkk) != hipSuccess) {
        set_error("cholesky: %zu bytes of FP64 scratch not available", sizeof(double) * nkk);
        return TDI_ERR_NOMEM;
    }
    int rc = TDI_OK;
    std::vector<int> ok(n, TDI_OK);
    if (hipMemcpyAsync(status, ok.data(), sizeof(int) * n, hipMemcpyHostToDevice, s) != hipSuccess) rc = TDI_ERR_HIP;
    if (!rc) {
        hipLaunchKernelGGL(k_f32_to_f64, dim3((unsigned)std::min<size_t>((nkk + 255) / 256, 65536)), dim3(256), 0, s, nkk,
                           H, A);
        rc = chol_big_run(n, K, A, g, delta, status, s);
    }
    const hipError_t e = hipStreamSynchronize(s);
    if (!rc && e != hipSuccess) rc = TDI_ERR_HIP;
    if (rc) set_error("cholesky (large K): %s", hipGetErrorString(e));
    (void)hipFree(A);
    return rc;
}

template <typename TD>
static int cholesky_big_f64(int n, int K, double* A, const double* g, TD* delta, int* status, hipStream_t s)
{
    if (int rc = chol_big_args(K)) return rc;
    std::vector<int> ok(n, TDI_OK);
    TDI_HIP(hipMemcpyAsync(status, ok.data(), sizeof(int) * n, hipMemcpyHostToDevice, s));
    const int rc = chol_big_run(n, K, A, g, delta, status, s);
    // the status upload reads the host vector: it must finish before the vector goes
    TDI_HIP(hipStreamSynchronize(s));
    if (rc) set_error("cholesky (large K): launch failed");
    return rc;
}

int launch_cholesky_big_f64(int n, int K, double* A, const double* g, float* delta, int* status, hipStream_t s)
{
    return cholesky_big_f64(n, K, A, g, delta, status, s);
}

int launch_cholesky_big_f64(int n, int K, double* A, const double* g, double* delta, int* status, hipStream_t s)
{
    return cholesky_big_f64(n, K, A, g, delta, status, s);
}

} // namespace tdi
