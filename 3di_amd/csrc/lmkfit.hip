// lmkfit.hip — the landmark-only log-barrier fit with slack, one workgroup per frame, FP64.
//
// Logbarrier_Initializer::set_minimal_slack (logbarrier_initializer.cu:1041-1090) and fit_model
// with use_slack (1095-1267), for T = 1 and no identity unknowns (li_init, video_fitter.cu:30).
// The reference drives each Newton step from the host: ~40 small launches for the terms
// (compute_gradient_and_hessian, 1272-1842), a cuSOLVER factorisation, and one host round trip
// per line-search trial.  Here a workgroup runs the whole fit of its frame — every round,
// Newton step, factorisation and trial — in one launch, with the frame's state in LDS:
//   unknowns z = (eps[0..Kl), tau_x, tau_y, tau_z, u1, u2, u3, s), n = Kl + 7, np = n - 1;
//   J: the projected-landmark derivatives (rows x_i, y_i) of half the landmarks at a time, the
//      columns padded with zeros to whole 16 x 16 blocks; the Hessian's lower blocks, padded with
//      the identity, and their factor then take the same LDS;
//   the Gauss-Newton block sum_i wx_i dx_i dx_i^T + wy_i dy_i dy_i^T is formed from J scaled by
//      sqrt(w) on the FP64 MFMA, its blocks staying in registers over the halves;
//   the landmarks move by a multiple of E d along a step, so a trial is one wavefront's work, and
//      the four wavefronts try four step lengths at once.
// Dependent steps bound a frame (the factorisation's columns, the rotation's and the logarithms'
// operations), the worst frames most: 512 frames, the worst of 8 steps and 61 trials, took 2688 us
// with column-by-column elimination and a thread per landmark, now 663 us.
// Objective, gradient and Hessian follow the reference term by term (see tdi_api.h); log, sqrt
// and division are FP64.
#include <cmath>

#include "chol.h"
#include "common.h"

namespace tdi {

namespace {

constexpr int LF_THREADS = 256;
constexpr int LF_NMAX = 96;                     // n = Kl + 7 <= 96
constexpr int LF_HALF = (NLMK + 1) / 2;         // landmarks whose rows are in LDS at once
constexpr int LF_ROWS = (2 * LF_HALF + 3) & ~3; // J rows in LDS
constexpr int LF_TMAX = LF_NMAX / CHB;
constexpr int LF_TILES_PER_WAVE = (LF_TMAX * (LF_TMAX + 1) / 2 + 3) / 4;

// Row stride of J for nT blocks of columns: two rows fall on disjoint halves of the banks.
__host__ __device__ constexpr int lf_stride(int nT) { return CHB * (nT | 1); }

struct LmkRep {
    int status, iterations, rounds, accepted;
    float slack0, slack;
};

struct LfShared {
    double z[LF_NMAX], d[LF_NMAX], g[LF_NMAX];
    double p[NLMK][3], q[NLMK][3];   // landmarks at z, and their move along d (model frame)
    double c[NLMK][4];               // camera frame at z, and 1 / depth^2
    double R[9], dR[27];
    double cx[NLMK], cy[NLMK], hx[NLMK], hy[NLMK], qg[NLMK], qh[NLMK], gmin[NLMK];
    double sw[2 * LF_HALF + LF_ROWS];   // sqrt of the weights of rows x_i, y_i, then zeros
    double ot[LF_THREADS / 64];
    int flag;
};

struct LfFrame {
    const int* ids;    // the landmarks' vertices
    const float* E;    // expression basis rows
    int ld;
    const float *lb, *ub;   // bounds of the expression unknowns
    float phix, phiy, cx, cy, face_size;
    const float* lm;   // [6][51]: x, y, box lx, ux, ly, uy
    int Kl, n, np, nT;
};

// The derivative of u's rotation R in u_i (rodrigues_f64_d's, i differing by lane).
__device__ __forceinline__ void lf_rotation_d(const double* u, int i, const double* R, double* dR)
{
    const double th = sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]), inv = 1.0 / (th * th);
    const double U[9] = {0, u[2], -u[1], -u[2], 0, u[0], u[1], -u[0], 0};
    const double ui = i == 0 ? u[0] : i == 1 ? u[1] : u[2];
    double e[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) e[k] = -(i == 0 ? R[k] : i == 1 ? R[3 + k] : R[6 + k]) + (i == k ? 1.0 : 0.0);
    const double w[3] = {u[1] * e[2] - u[2] * e[1], u[2] * e[0] - u[0] * e[2], u[0] * e[1] - u[1] * e[0]};
    const double A[9] = {ui * U[0], ui * U[1] + w[2], ui * U[2] - w[1], ui * U[3] - w[2], ui * U[4], ui * U[5] + w[0],
                         ui * U[6] + w[1], ui * U[7] - w[0], ui * U[8]};
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            double acc = 0.0;
#pragma unroll
            for (int k = 0; k < 3; ++k) acc += A[k * 3 + r] * R[c * 3 + k];
            dR[c * 3 + r] = acc * inv;
        }
}

// out = E v for the landmarks' rows, 16 lanes to a row so that a row is read in whole sectors.
__device__ __forceinline__ void lf_vertices(const LfFrame& F, const double* v, double (*out)[3])
{
    const int tid = threadIdx.x, l16 = tid & 15;
    double vk[LF_TMAX];
#pragma unroll
    for (int c = 0; c < LF_TMAX; ++c) vk[c] = l16 + 16 * c < F.Kl ? v[l16 + 16 * c] : 0.0;
#pragma unroll 5
    for (int r0 = 0; r0 < 3 * NLMK; r0 += LF_THREADS / 16) {
        const int r = r0 + (tid >> 4), rc = min(r, 3 * NLMK - 1), i = rc / 3, a = rc - 3 * i;
        const float* e = F.E + (size_t)(3 * F.ids[i] + a) * F.ld;
        double x = 0.0;
#pragma unroll
        for (int c = 0; c < LF_TMAX; ++c)
            if (16 * c < F.Kl) x = fma((double)e[min(l16 + 16 * c, F.Kl - 1)], vk[c], x);
        for (int o = 8; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
        if (l16 == 0 && r < 3 * NLMK) out[i][a] = x;
    }
}

// The objective at z + t d (barrier weight tau_b on the slack) by one wavefront, a landmark to a lane.
__device__ __forceinline__ double lf_objective(const LfFrame& F, double t, double tau_b, const LfShared& S)
{
    const int lane = threadIdx.x & 63, Kl = F.Kl;
    const bool here = t == 0.0;      // d may hold the step of a round that ended
    auto at = [&](int k) { return here ? S.z[k] : fma(t, S.d[k], S.z[k]); };
    double u[3], R[9], acc = 0.0;
    for (int k = 0; k < 3; ++k) u[k] = at(Kl + 3 + k);
    rodrigues_f64(u, R);
    if (lane < NLMK) {
        const double s = at(F.np), fs = F.face_size;
        double p[3], c[3];
        for (int a = 0; a < 3; ++a) p[a] = here ? S.p[lane][a] : fma(t, S.q[lane][a], S.p[lane][a]);
        for (int a = 0; a < 3; ++a) c[a] = R[a] * p[0] + R[3 + a] * p[1] + R[6 + a] * p[2] + at(Kl + a);
        const double xp = F.phix * c[0] / c[2] + F.cx, yp = F.phiy * c[1] / c[2] + F.cy;
        const double lx = F.lm[lane], ly = F.lm[NLMK + lane];
        const double Gxm = s + xp - (lx + (double)F.lm[2 * NLMK + lane] * fs);
        const double Gxp = s + (lx + (double)F.lm[3 * NLMK + lane] * fs) - xp;
        const double Gym = s + yp - (ly + (double)F.lm[4 * NLMK + lane] * fs);
        const double Gyp = s + (ly + (double)F.lm[5 * NLMK + lane] * fs) - yp;
        acc = -log(Gxm) - log(Gym) - log(Gxp) - log(Gyp);
        if (lane == 0) acc += tau_b * s;
    }
    for (int k = lane; k < Kl; k += 64) {
        const float lbf = F.lb[k], ubf = F.ub[k];
        if (ubf < INFINITY && lbf > -INFINITY) {
            const double x = at(k), fub = x - (double)ubf, flb = (double)lbf - x;
            acc += -log(-fub) - log(-flb);
        }
    }
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    return acc;
}

// The per-landmark coefficients of the gradient and Hessian at z, and R, dR and c, in S: the last three
// threads have the derivatives of the rotation, thread 4 i + q constraint q of landmark i (x below, x
// above, y below, y above).
__device__ __forceinline__ void lf_coefficients(const LfFrame& F, LfShared& S)
{
    const int tid = threadIdx.x, Kl = F.Kl;
    double R[9];
    rodrigues_f64(S.z + Kl + 3, R);
    if (tid >= LF_THREADS - 3) {
        double dR[9];
        const int i = LF_THREADS - 1 - tid;
        lf_rotation_d(S.z + Kl + 3, i, R, dR);
#pragma unroll
        for (int k = 0; k < 9; ++k) S.dR[9 * i + k] = dR[k];
        if (i == 0) {
#pragma unroll
            for (int k = 0; k < 9; ++k) S.R[k] = R[k];
        }
    }
    if (tid < 4 * NLMK) {
        const int i = tid >> 2, q = tid & 3, ax = q >> 1;
        const double s = S.z[F.np];
        double c[3];
        for (int a = 0; a < 3; ++a)
            c[a] = R[a] * S.p[i][0] + R[3 + a] * S.p[i][1] + R[6 + a] * S.p[i][2] + S.z[Kl + a];
        S.c[i][q] = q == 0 ? c[0] : q == 1 ? c[1] : q == 2 ? c[2] : 1.0 / (c[2] * c[2]);
        const double pr = (double)(ax ? F.phiy : F.phix) * (ax ? c[1] : c[0]) / c[2] + (double)(ax ? F.cy : F.cx);
        const double fs = F.face_size, l = F.lm[ax * NLMK + i], box = F.lm[(2 + q) * NLMK + i];
        const double G = (q & 1) ? s + (l + box * fs) - pr : s + pr - (l + box * fs);
        // the least constraint of the landmark, NaN if one is
        const double G1 = __shfl_xor(G, 1, 64);
        double lo = (G != G || G1 != G1) ? NAN : fmin(G, G1);
        const double lo1 = __shfl_xor(lo, 2, 64);
        lo = (lo != lo || lo1 != lo1) ? NAN : fmin(lo, lo1);
        const double iG = 1.0 / G, iG2 = 1.0 / (G * G), qe = 1.0 / (1e-6 + G);
        const double iH = __shfl_xor(iG, 1, 64), iH2 = __shfl_xor(iG2, 1, 64);   // the constraint above, for even q
        double sq = qe + __shfl_xor(qe, 2, 64), sq2 = qe * qe + __shfl_xor(qe * qe, 2, 64);
        sq += __shfl_xor(sq, 1, 64);
        sq2 += __shfl_xor(sq2, 1, 64);
        if (!(q & 1)) {
            (ax ? S.cy : S.cx)[i] = -iG + iH;
            (ax ? S.hy : S.hx)[i] = iG2 - iH2;
            S.sw[2 * i + ax] = sqrt(iG2 + iH2);
        }
        if (q == 0) {
            S.gmin[i] = lo;
            S.qg[i] = sq;
            S.qh[i] = sq2;
        }
    }
    __syncthreads();
}

// Gradient and Gauss-Newton Hessian at z, from the last lf_coefficients; the lower
// blocks of H are written over J in `dyn`.
__device__ __forceinline__ void lf_terms(const LfFrame& F, double tau_b, double* dyn, LfShared& S)
{
    const double* zv = S.z;
    const int tid = threadIdx.x, Kl = F.Kl, n = F.n, np = F.np, nT = F.nT, ldj = lf_stride(nT), nc = CHB * nT;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, kq = lane >> 4;
    double* J = dyn;
    ch_v4d acc[LF_TILES_PER_WAVE];
#pragma unroll
    for (int q = 0; q < LF_TILES_PER_WAVE; ++q) acc[q] = ch_v4d{0.0, 0.0, 0.0, 0.0};
    double gs = 0.0, hs = 0.0;
#pragma unroll 1
    for (int i0 = 0; i0 < NLMK; i0 += LF_HALF) {
        const int ni = min(LF_HALF, NLMK - i0);
        // four landmark rows of a thread at a time, their loads first
        for (int e0 = tid; e0 < LF_ROWS / 2 * nc; e0 += 4 * LF_THREADS) {
            float ev[4][3];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int e = e0 + u * LF_THREADS, ii = e / nc, j = e - ii * nc;
                const int v = F.ids[min(i0 + ii, NLMK - 1)];
#pragma unroll
                for (int a = 0; a < 3; ++a) ev[u][a] = F.E[(size_t)(3 * v + a) * F.ld + min(j, Kl - 1)];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int e = e0 + u * LF_THREADS, ii = e / nc, j = e - ii * nc, i = min(i0 + ii, NLMK - 1);
                if (ii >= LF_ROWS / 2) break;
                // the camera-frame derivative is M (v0, v1, v2): the basis by R, the mean vertex by dR
                const double* M = j < Kl + 3 ? S.R : S.dR + 9 * min(j - Kl - 3, 2);
                const double v0 = j < Kl ? (double)ev[u][0] : S.p[i][0], v1 = j < Kl ? (double)ev[u][1] : S.p[i][1],
                             v2 = j < Kl ? (double)ev[u][2] : S.p[i][2];
                double dv[3];
#pragma unroll
                for (int a = 0; a < 3; ++a) dv[a] = M[a] * v0 + M[3 + a] * v1 + M[6 + a] * v2;
                if (j >= Kl && j < Kl + 3) {
#pragma unroll
                    for (int a = 0; a < 3; ++a) dv[a] = j - Kl == a ? 1.0 : 0.0;
                }
                const double cx = S.c[i][0], cy = S.c[i][1], cz = S.c[i][2], iz2 = S.c[i][3];
                const bool in = j < np && ii < ni;
                J[(size_t)(2 * ii) * ldj + j] = in ? ch_div(F.phix * (dv[0] * cz - dv[2] * cx), cz * cz, iz2) : 0.0;
                J[(size_t)(2 * ii + 1) * ldj + j] = in ? ch_div(F.phiy * (dv[1] * cz - dv[2] * cy), cz * cz, iz2) : 0.0;
            }
        }
        __syncthreads();
        // gradient and the slack column from the raw derivatives
        if (tid < np) {
#pragma unroll 13
            for (int ii = 0; ii < ni; ++ii) {
                const double dx = J[(size_t)(2 * ii) * ldj + tid], dy = J[(size_t)(2 * ii + 1) * ldj + tid];
                gs += S.cx[i0 + ii] * dx + S.cy[i0 + ii] * dy;
                hs += S.hx[i0 + ii] * dx + S.hy[i0 + ii] * dy;
            }
        }
        // block t of the lower triangle to wavefront t % 4; the rows past the landmarks are zero
#pragma unroll
        for (int q = 0; q < LF_TILES_PER_WAVE; ++q) {
            int I = 0, C = wave + 4 * q;
            while (C > I) { ++I; C -= I; }
            if (I >= nT) continue;
            const double* ja = J + kq * ldj + CHB * I + l16;
            const double* jb = J + kq * ldj + CHB * C + l16;
#pragma unroll
            for (int k = 0; k < LF_ROWS / 4; ++k) {
                const double w = S.sw[2 * i0 + 4 * k + kq];
                acc[q] = ch_mma(ja[(size_t)(4 * k) * ldj] * w, jb[(size_t)(4 * k) * ldj] * w, acc[q]);
            }
        }
        __syncthreads();
    }
    double* H = dyn;
#pragma unroll
    for (int q = 0; q < LF_TILES_PER_WAVE; ++q) {
        int I = 0, C = wave + 4 * q;
        while (C > I) { ++I; C -= I; }
        if (I >= nT) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) H[ch_block(I, C) + ch_row(0.0, lane, r) * CHP + l16] = acc[q][r];
    }
    __syncthreads();
    // the bounds, the slack's row and the padding
    if (tid < np) {
        const int r = tid & 15, B = tid >> 4;
        if (tid < Kl) {
            const float lbf = F.lb[tid], ubf = F.ub[tid];
            if (ubf < INFINITY && lbf > -INFINITY) {
                const double x = zv[tid], fub = x - (double)ubf, flb = (double)lbf - x;
                gs += -1.0 / fub + 1.0 / flb;
                const double a = -1.0 / (fub + 1e-12), b = 1.0 / (flb + 1e-12);
                H[ch_block(B, B) + r * CHP + r] += a * a + b * b;
            }
        }
        S.g[tid] = gs;
        H[ch_block(np >> 4, B) + (np & 15) * CHP + r] = hs;
    } else if (tid >= n && tid < nc) {
        H[ch_block(nT - 1, nT - 1) + (tid & 15) * (CHP + 1)] = 1.0;
    } else if (tid == LF_THREADS - 1) {
        double qs = 0.0, hss = 0.0;
#pragma unroll 17
        for (int i = 0; i < NLMK; ++i) { qs += S.qg[i]; hss += S.qh[i]; }
        S.g[np] = tau_b - qs;
        H[ch_block(np >> 4, np >> 4) + (np & 15) * (CHP + 1)] = hss;
        S.flag = 0;
    }
    __syncthreads();
}

// Cholesky factorisation of H (lower blocks in LDS) and the solve H d = -g.  Returns false (in
// every thread) on a pivot that is not positive.
__device__ __forceinline__ bool lf_solve(int n, int nT, double* H, LfShared& S)
{
    const int lane = threadIdx.x & 63;
    if (!ch_factor<double>(H, nT, &S.flag)) return false;
    if (threadIdx.x < 64) {
        double x0 = lane < n ? -S.g[lane] : 0.0, x1 = lane + 64 < n ? -S.g[lane + 64] : 0.0;
        ch_solve<double, double>(H, nT, x0, x1);
        if (lane < n) S.d[lane] = x0;
        if (lane + 64 < n) S.d[lane + 64] = x1;
    }
    __syncthreads();
    return true;
}

// mode 0: the fit (theta in/out, rep); mode 1: terms at zin (Hout, gout, objout).
__global__ void __launch_bounds__(LF_THREADS, 2) k_lmk_slack(ModelGPU m, Layout L, const FrameGPU* __restrict__ frames,
                                                          const float* __restrict__ lmk, float* __restrict__ theta,
                                                          int Kl, int mode, const double* __restrict__ zin,
                                                          double tau_in, double* __restrict__ Hout,
                                                          double* __restrict__ gout, double* __restrict__ objout,
                                                          LmkRep* __restrict__ rep)
{
    extern __shared__ __align__(16) double dyn[];
    __shared__ LfShared S;
    const int f = blockIdx.x, tid = threadIdx.x;
    LfFrame F;
    F.ids = m.lmk_ids;
    F.E = m.exp_basis;
    F.ld = m.exp_ld;
    F.lb = m.lb + L.off_exp;
    F.ub = m.ub + L.off_exp;
    F.phix = frames[f].phix;
    F.phiy = frames[f].phiy;
    F.cx = frames[f].cx;
    F.cy = frames[f].cy;
    F.face_size = frames[f].face_size;
    F.lm = lmk + (size_t)f * 6 * NLMK;
    F.Kl = Kl;
    F.n = Kl + 7;
    F.np = Kl + 6;
    F.nT = (F.n + CHB - 1) / CHB;
    const int n = F.n, np = F.np;
    float* th = theta + (size_t)f * L.K;
    // the start (mode 1: the point asked for), and the landmarks there: mean + identity terms + E z
    for (int j = tid; j < n; j += LF_THREADS)
        S.z[j] = mode == 1 ? zin[(size_t)f * n + j] : j >= Kl && j < Kl + 6 ? (double)th[L.off_pose + j - Kl] : 0.0;
    for (int r = 2 * NLMK + tid; r < 2 * LF_HALF + LF_ROWS; r += LF_THREADS) S.sw[r] = 0.0;
    for (int r = tid; r < 3 * NLMK; r += LF_THREADS) {
        const int i = r / 3, a = r - 3 * i;
        const size_t row = (size_t)(3 * m.lmk_ids[i] + a);
        double x = m.mean[row];
#pragma unroll 16
        for (int k = 0; k < L.nid; ++k) x += (double)m.id_basis[row * m.id_ld + k] * (double)th[L.off_id + k];
        S.p[i][a] = x;
    }
    __syncthreads();
    if (mode == 1) {
        lf_vertices(F, S.z, S.q);
        __syncthreads();
        for (int r = tid; r < 3 * NLMK; r += LF_THREADS) S.p[r / 3][r % 3] += S.q[r / 3][r % 3];
        __syncthreads();
        const double obj = lf_objective(F, 0.0, tau_in, S);
        lf_coefficients(F, S);
        lf_terms(F, tau_in, dyn, S);
        if (objout && tid == 0) objout[f] = obj;
        if (gout)
            for (int j = tid; j < n; j += LF_THREADS) gout[(size_t)f * n + j] = S.g[j];
        if (Hout)
            for (int e = tid; e < n * n; e += LF_THREADS) {
                const int a = max(e / n, e % n), b = min(e / n, e % n);
                Hout[(size_t)f * n * n + e] = dyn[ch_block(a >> 4, b >> 4) + (a & 15) * CHP + (b & 15)];
            }
        return;
    }
    // set_minimal_slack: s = 5 - min G at s = 0
    lf_coefficients(F, S);
    if (tid == 0) {
        double lo = S.gmin[0];
#pragma unroll 10
        for (int i = 1; i < NLMK; ++i) lo = (S.gmin[i] != S.gmin[i] || lo != lo) ? NAN : fmin(lo, S.gmin[i]);
        S.z[np] = 5.0 - lo;
    }
    __syncthreads();
    const double slack0 = S.z[np];
    int iterations = 0, rounds = 0, accepted = 0;
    bool success = false;
    double tau_b = 10.0;
    for (int round = 0; round < 5 && !success; ++round) {
        tau_b *= 10.0;
        ++rounds;
        bool have = false;        // obj is the objective at z, with this round's tau_b
        double obj = 0.0;
        for (int it = 0; it < 100; ++it) {
            if (S.z[np] < -0.01) { success = true; break; }
            if (!have) obj = lf_objective(F, 0.0, tau_b, S);
            lf_coefficients(F, S);
            lf_terms(F, tau_b, dyn, S);
            ++iterations;
            if (!lf_solve(n, F.nT, dyn, S)) break;
            lf_vertices(F, S.d, S.q);
            __syncthreads();
            // the first step length of 1, 1/2, .. down to 0.01 that lowers the objective, a wavefront to each
            have = false;
            double t = 0.0;
            for (double t0 = 1.0; t0 >= 0.01 && !have; t0 *= 0.0625) {
                const double tw = ldexp(t0, -(tid >> 6));
                if (tw >= 0.01) {
                    const double ot = lf_objective(F, tw, tau_b, S);
                    if ((tid & 63) == 0) S.ot[tid >> 6] = ot;
                }
                __syncthreads();
                t = t0;
                for (int w = 0; w < LF_THREADS / 64 && t >= 0.01; ++w, t *= 0.5)
                    if (S.ot[w] < obj) {
                        obj = S.ot[w];
                        have = true;
                        break;
                    }
                __syncthreads();
            }
            if (!have) break;
            for (int j = tid; j < n; j += LF_THREADS) S.z[j] = fma(t, S.d[j], S.z[j]);
            for (int r = tid; r < 3 * NLMK; r += LF_THREADS)
                S.p[r / 3][r % 3] = fma(t, S.q[r / 3][r % 3], S.p[r / 3][r % 3]);
            __syncthreads();
            ++accepted;
        }
    }
    if (success) {
        for (int k = tid; k < Kl; k += LF_THREADS) th[L.off_exp + k] = (float)S.z[k];
        if (tid < 6) th[L.off_pose + tid] = (float)S.z[Kl + tid];
    }
    if (tid == 0) {
        LmkRep r;
        r.status = success ? TDI_OK : TDI_LMK_INFEASIBLE;
        r.iterations = iterations;
        r.rounds = rounds;
        r.accepted = accepted;
        r.slack0 = (float)slack0;
        r.slack = (float)S.z[np];
        rep[f] = r;
    }
}

} // namespace

int launch_lmk_slack(const ModelGPU& m, const Layout& L, const FrameGPU* frames, const float* lmk, int n,
                     float* theta, int Kl, int mode, const double* zin, double tau, double* H, double* g,
                     double* obj, void* rep, hipStream_t s)
{
    if (Kl < 1 || Kl > L.nexp || Kl + 7 > LF_NMAX) {
        set_error("landmark slack fit: k_exp = %d, expected 1..min(%d, %d)", Kl, L.nexp, LF_NMAX - 7);
        return TDI_ERR_ARG;
    }
    if (n <= 0) return TDI_OK;
    const int nT = (Kl + 7 + CHB - 1) / CHB;
    const size_t lds = sizeof(double) * std::max(LF_ROWS * lf_stride(nT), nT * (nT + 1) / 2 * CHN);
    hipLaunchKernelGGL(k_lmk_slack, dim3(n), dim3(LF_THREADS), lds, s, m, L, frames, lmk, theta, Kl, mode, zin, tau,
                       H, g, obj, reinterpret_cast<LmkRep*>(rep));
    TDI_HIP(hipGetLastError());
    return TDI_OK;
}

} // namespace tdi
