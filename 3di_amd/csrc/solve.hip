// solve.hip — log barrier, batched Cholesky and the Gauss-Newton/line-search state machine.
//
// Reference:
//   Logbarrier_Initializer::compute_gradient_and_hessian (logbarrier_initializer.cu:1272-1842)
//   with compute_Gs (458-518), fill_optimization_dc_landmark/_dI_depsilon_landmark/
//   _dI_dalpha_landmark (587-910), update_gradient/update_diagonal_of_hessian_wbounds
//   (915-948) and evaluate_objective_function (1921-2081): landmark-box constraints
//   G = box edge distance of the projected landmark, objective -sum log G, gradient
//   sum -dG/G, Gauss-Newton Hessian sum (dG/G)(dG/G)^T; coefficient bounds
//   -log(ub-x) - log(x-lb) with exact gradient and diagonal Hessian.
//   Solver::solve (solver.h:70-105): cusolverDnDpotrf + Dpotrs in FP64, delta = -H^-1 g.
//   fit_3DMM_shape_rigid (model_fitter.cu:121-375): Armijo backtracking with ALPHA 0.4,
//   BETA 0.8, stop when -delta.g < 3e-4 or t < t_min, reject steps with tau_z < 0, shrink
//   on "face too large" or a NaN barrier.
//
// The batched state machine keeps every per-frame decision of the reference but runs it
// for all frames of a batch with masks: frames that have accepted a step or stopped sit out later
// rounds.  The fit is a sequence of captured pieces; k_ls_status tells the host how many frames
// still search and whether any is active, and the host launches the pieces that some frame needs.
#include "chol.h"
#include "common.h"

namespace tdi {

namespace {

constexpr int BMAXK = 112;

// The log barrier of one frame per workgroup, FP64 throughout (rotation and its derivatives, landmark
// positions, constraint values, weights, projected-landmark derivatives, sums, H); the FP32 g receives
// one rounding per term.  It is a few thousand operations, so latency bounds it: the rotation and the
// landmark vertices are the synthesis's (rt, P0) instead of a serial sin/cos and 79-term sums, every
// logarithm has a thread, and gathers are issued in batches.  One frame of 94 unknowns: 129
// objectives and 24 derivative launches took 4552 us, now 592 and 1002 us.

struct LmkBox {              // constraint values of one landmark (compute_Gs)
    double vx, vy, vz, Gxm, Gym, Gxp, Gyp;
};

__device__ __forceinline__ LmkBox landmark_box(const FrameGPU& fr, const double* rt, const double* p, const float* L6,
                                               int i)
{
    LmkBox o;
    o.vx = rt[0] * p[0] + rt[3] * p[1] + rt[6] * p[2] + rt[9];
    o.vy = rt[1] * p[0] + rt[4] * p[1] + rt[7] * p[2] + rt[10];
    o.vz = rt[2] * p[0] + rt[5] * p[1] + rt[8] * p[2] + rt[11];
    const double xproj = fr.phix * o.vx / o.vz + fr.cx;
    const double yproj = fr.phiy * o.vy / o.vz + fr.cy;
    const double lx = L6[i], ly = L6[NLMK + i];
    const double blx = L6[2 * NLMK + i], bux = L6[3 * NLMK + i];
    const double bly = L6[4 * NLMK + i], buy = L6[5 * NLMK + i];
    const double fs = fr.face_size;
    o.Gxm = xproj - (lx + blx * fs);
    o.Gym = yproj - (ly + bly * fs);
    o.Gxp = (lx + bux * fs) - xproj;
    o.Gyp = (ly + buy * fs) - yproj;
    return o;
}

// Objective: obj[f] = objb[f] = the barrier's value; face_ok (when given): the "face too large" test
// of compute_nonrigid_shape2 (renderer.cu:836-857) on projected landmark vertices 0, 9 and 40.
__global__ void __launch_bounds__(256) k_barrier_obj(ModelGPU m, Layout L, const FrameGPU* __restrict__ frames,
                                                      const int* __restrict__ act, int n,
                                                      const float* __restrict__ theta, const double* __restrict__ rt,
                                                      const double* __restrict__ P0, const float4* __restrict__ vproj,
                                                      LmkArrays lm, int use_lmk, float ref_face_size,
                                                      double* __restrict__ obj, double* __restrict__ objb,
                                                      int* __restrict__ face_ok)
{
    if ((int)blockIdx.x >= fl_count(act, n)) return;
    const int f = fl_frame(act, blockIdx.x);
    const FrameGPU fr = frames[f];
    const float* tf = theta + (size_t)f * L.K;
    __shared__ double sred[4];
    const int tid = threadIdx.x;
    if (face_ok && tid == 255) {
        int ok = 1;
        if (ref_face_size > 0.f) {
            const float4* vp = vproj + (size_t)f * m.V;
            const float4 a = vp[m.lmk_ids[0]], b = vp[m.lmk_ids[9]], c = vp[m.lmk_ids[40]];
            const float iod = fabsf(b.x - a.x), lem = fabsf(a.y - c.y), rem = fabsf(b.y - c.y);
            const float lim = 2.f * ref_face_size;
            ok = !(iod > lim || lem > lim || rem > lim);
        }
        face_ok[f] = ok;
    }
    double acc = 0.0;
    if (use_lmk && tid < 4 * NLMK) {              // one side of one landmark's box per thread
        const int i = tid >> 2, side = tid & 3;
        double R[12], p[3];
        const double* pl = P0 + ((size_t)f * m.V + m.lmk_ids[i]) * 3;
        for (int q = 0; q < 12; ++q) R[q] = rt[(size_t)f * 12 + q];
        for (int a = 0; a < 3; ++a) p[a] = pl[a];
        const LmkBox o = landmark_box(fr, R, p, lm.base + (size_t)f * 6 * NLMK, i);
        acc = -log(side == 0 ? o.Gxm : side == 1 ? o.Gym : side == 2 ? o.Gxp : o.Gyp);
    }
    for (int e = 255 - tid; e < 2 * L.K; e += blockDim.x) {   // coefficient bounds (only finite ones)
        const int j = e >> 1;
        const float lb = m.lb[j], ub = m.ub[j];
        if (!(ub < INFINITY) || !(lb > -INFINITY)) continue;
        const double x = tf[j];
        acc += -log(e & 1 ? x - (double)lb : (double)ub - x);
    }
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
    if ((tid & 63) == 0) sred[tid >> 6] = acc;
    __syncthreads();
    if (tid == 0) {
        const double s = sred[0] + sred[1] + sred[2] + sred[3];
        obj[f] = s;
        objb[f] = s;
    }
}

// What the derivative terms of one frame start from, in LDS.
struct BarrierFrame {
    double rt[12], dR[27];
    double p[NLMK][3], v[NLMK][3];
    double zz[NLMK], izz[NLMK];                      // depth squared and its reciprocal
    double rx[NLMK], ry[NLMK], gx[NLMK], gy[NLMK];   // square roots of the Gauss-Newton weights, gradient weights
    int id[NLMK];
};

// Fills it (every thread of the workgroup; ends with a barrier).
__device__ __forceinline__ void barrier_frame(const ModelGPU& m, const Layout& L, const FrameGPU& fr, int f,
                                              const float* __restrict__ tf, const double* __restrict__ rt,
                                              const double* __restrict__ P0, const float* __restrict__ L6, BarrierFrame& B)
{
    const int tid = threadIdx.x;
    if (tid < 12) B.rt[tid] = rt[(size_t)f * 12 + tid];
    if (tid >= 64 && tid < 64 + 3 * NLMK) {
        const int e = tid - 64, i = e / 3, a = e - 3 * i, id = m.lmk_ids[i];
        if (a == 0) B.id[i] = id;
        B.p[i][a] = P0[((size_t)f * m.V + id) * 3 + a];
    }
    __syncthreads();
    if (tid < 27) {
        // entry (row r, column c) of dR/du_i, as rodrigues_f64_d forms it
        const int i = tid / 9, c = (tid % 9) / 3, r = tid % 3;
        double u[3], e[3], w[3], Rc[3];
        for (int a = 0; a < 3; ++a) {
            u[a] = tf[L.off_pose + 3 + a];
            e[a] = -B.rt[i * 3 + a] + (i == a);
            Rc[a] = B.rt[c * 3 + a];
        }
        const double th = sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
        const double inv = 1.0 / (th * th);
        w[0] = u[1] * e[2] - u[2] * e[1];
        w[1] = u[2] * e[0] - u[0] * e[2];
        w[2] = u[0] * e[1] - u[1] * e[0];
        // row r of u_i [u]x + [w]x: zero at column r, -x2 or +x1 ... around it
        const double ui = i == 0 ? u[0] : i == 1 ? u[1] : u[2];
        double acc = 0.0;
        for (int k = 0; k < 3; ++k) {
            if (k == r) continue;
            const int o = 3 - r - k;                              // the third axis
            const double sg = (k - r == 1 || k - r == -2) ? -1.0 : 1.0;
            const double uo = o == 0 ? u[0] : o == 1 ? u[1] : u[2], wo = o == 0 ? w[0] : o == 1 ? w[1] : w[2];
            acc += (ui * (sg * uo) + sg * wo) * Rc[k];
        }
        B.dR[tid] = acc * inv;
    }
    if (tid >= 64 && tid < 64 + NLMK) {
        const int i = tid - 64;
        const LmkBox o = landmark_box(fr, B.rt, B.p[i], L6, i);
        B.v[i][0] = o.vx; B.v[i][1] = o.vy; B.v[i][2] = o.vz;
        B.zz[i] = o.vz * o.vz;
        B.izz[i] = 1.0 / B.zz[i];
        B.rx[i] = sqrt(1.0 / (o.Gxm * o.Gxm) + 1.0 / (o.Gxp * o.Gxp));
        B.ry[i] = sqrt(1.0 / (o.Gym * o.Gym) + 1.0 / (o.Gyp * o.Gyp));
        B.gx[i] = -1.0 / o.Gxm + 1.0 / o.Gxp;
        B.gy[i] = -1.0 / o.Gym + 1.0 / o.Gyp;
    }
    __syncthreads();
}

// d(projected landmark i)/d(direction dv) as (dx, dy)
__device__ __forceinline__ void landmark_dxy(const FrameGPU& fr, const BarrierFrame& B, int i, const double* dv,
                                             double& dx, double& dy)
{
    const double vx = B.v[i][0], vy = B.v[i][1], vz = B.v[i][2];
    dx = ch_div(fr.phix * (dv[0] * vz - dv[2] * vx), B.zz[i], B.izz[i]);
    dy = ch_div(fr.phiy * (dv[1] * vz - dv[2] * vy), B.zz[i], B.izz[i]);
}

// Rows of the projected-landmark derivatives: dx of landmark i to column j at D[dxrow(i)][j], dy at
// D[dyrow(i)][j], for the geometric unknowns; the other columns are left as they are.
template <typename Store>
__device__ __forceinline__ void barrier_rows(const ModelGPU& m, const Layout& L, const FrameGPU& fr,
                                             const BarrierFrame& B, Store store)
{
    const int tid = threadIdx.x;
    // basis columns: the gathers of BATCH entries per thread are issued before the arithmetic
    constexpr int BATCH = 8;
    for (int blk = 0; blk < 2; ++blk) {
        const int nc = blk ? L.nexp : L.nid, off = blk ? L.off_exp : L.off_id, ld = blk ? m.exp_ld : m.id_ld;
        const float* basis = blk ? m.exp_basis : m.id_basis;
        for (int e0 = 0; e0 < NLMK * nc; e0 += 256 * BATCH) {
            float b[BATCH][3];
#pragma unroll
            for (int q = 0; q < BATCH; ++q) {
                const int e = min(e0 + 256 * q + tid, NLMK * nc - 1), i = e / nc, c = e - i * nc;
#pragma unroll
                for (int a = 0; a < 3; ++a) b[q][a] = basis[(size_t)(3 * B.id[i] + a) * ld + c];
            }
#pragma unroll
            for (int q = 0; q < BATCH; ++q) {
                const int e = e0 + 256 * q + tid, i = e / nc, c = e - i * nc;
                if (e >= NLMK * nc) continue;
                double dv[3], dx, dy;
#pragma unroll
                for (int a = 0; a < 3; ++a)
                    dv[a] = B.rt[a] * (double)b[q][0] + B.rt[3 + a] * (double)b[q][1] + B.rt[6 + a] * (double)b[q][2];
                landmark_dxy(fr, B, i, dv, dx, dy);
                store(i, off + c, dx, dy);
            }
        }
    }
    for (int e = tid; e < NLMK * 6; e += blockDim.x) {
        const int i = e / 6, c = e - 6 * i;
        double dv[3] = {0.0, 0.0, 0.0}, dx, dy;
        if (c < 3) {
            dv[0] = c == 0; dv[1] = c == 1; dv[2] = c == 2;
        } else {
            const double* d = B.dR + 9 * (c - 3);
            for (int a = 0; a < 3; ++a) dv[a] = d[a] * B.p[i][0] + d[3 + a] * B.p[i][1] + d[6 + a] * B.p[i][2];
        }
        landmark_dxy(fr, B, i, dv, dx, dy);
        store(i, L.off_pose + c, dx, dy);
    }
}

// Gradient and Hessian diagonal of the bounds of unknown j (zero where it has none).
__device__ __forceinline__ void bound_terms(const ModelGPU& m, const float* tf, int j, float& g, double& h)
{
    g = 0.f;
    h = 0.0;
    const float lbf = m.lb[j], ubf = m.ub[j];
    if (!(ubf < INFINITY) || !(lbf > -INFINITY)) return;
    const double x = tf[j], lb = lbf, ub = ubf;
    const double fub = x - ub, flb = lb - x;
    g = (float)(-1.0 / fub + 1.0 / flb);
    const double a = -1.0 / (fub + 1e-12), b = 1.0 / (flb + 1e-12);
    h = a * a + b * b;
}

constexpr int BAR_THREADS = 512;
constexpr int BAR_PARTS = BAR_THREADS / 128, BAR_LMK = (NLMK + BAR_PARTS - 1) / BAR_PARTS;   // landmarks per part

// Derivatives: H[f] += barrier Hessian, g[f] += barrier gradient, for K <= BMAXK.  A thread owns a
// column j and a part of the landmarks: projected-landmark derivatives, the gradient's partial sum, and
// the derivatives scaled by the square roots of the Gauss-Newton weights into dynamic LDS
// [2 NLMK][KS], KS = K padded to 4; then the landmark block sum_i ex ex^T + ey ey^T, four rows of a
// column per thread (lanes along the columns: conflict-free reads, the four rows' as broadcasts).
__global__ void __launch_bounds__(BAR_THREADS) k_barrier(ModelGPU m, Layout L, const FrameGPU* __restrict__ frames,
                                                          const int* __restrict__ act, int n,
                                                          const float* __restrict__ theta, const double* __restrict__ rt,
                                                          const double* __restrict__ P0, LmkArrays lm, int use_lmk,
                                                          double* __restrict__ H,
                                                          float* __restrict__ g)
{
    // one workgroup per listed frame (the grid has a workgroup per slot)
    if ((int)blockIdx.x >= fl_count(act, n)) return;
    const int f = fl_frame(act, blockIdx.x);
    const int K = L.K, KS = (K + 3) & ~3;
    const FrameGPU fr = frames[f];
    const float* tf = theta + (size_t)f * K;
    extern __shared__ double sdyn[];
    __shared__ BarrierFrame B;
    __shared__ double sbound[BMAXK];
    __shared__ double sg[BAR_PARTS][128];
    const int tid = threadIdx.x;
    double* Hf = H + (size_t)f * K * K;
    float gb = 0.f;
    if (tid < K) {                                   // K <= BMAXK < BAR_THREADS
        double hb;
        bound_terms(m, tf, tid, gb, hb);
        if (use_lmk) sbound[tid] = hb;
        else {
            g[(size_t)f * K + tid] += gb;
            Hf[(size_t)tid * K + tid] += hb;
        }
    }
    if (!use_lmk) return;
    barrier_frame(m, L, fr, f, tf, rt, P0, lm.base + (size_t)f * 6 * NLMK, B);
    {
        const int j = tid & 127, part = tid >> 7;
        const bool exp = j >= L.off_exp && j < L.off_pose, id = j >= L.off_id && j < L.off_exp;
        const bool trans = j >= L.off_pose && j < L.off_pose + 3, rot = j >= L.off_pose + 3 && j < L.off_light;
        const float* col = exp ? m.exp_basis + (j - L.off_exp) : m.id_basis + (j - L.off_id);
        const int ld = exp ? m.exp_ld : m.id_ld;
        float e[BAR_LMK][3];
#pragma unroll
        for (int q = 0; q < BAR_LMK; ++q) {
            const int i = min(part * BAR_LMK + q, NLMK - 1);
#pragma unroll
            for (int a = 0; a < 3; ++a) e[q][a] = exp || id ? col[(size_t)(3 * B.id[i] + a) * ld] : 0.f;
        }
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < BAR_LMK; ++q) {
            const int i = part * BAR_LMK + q;
            if (i >= NLMK) continue;
            double dv[3], dx, dy;
            if (exp || id) {
#pragma unroll
                for (int a = 0; a < 3; ++a)
                    dv[a] = B.rt[a] * (double)e[q][0] + B.rt[3 + a] * (double)e[q][1] + B.rt[6 + a] * (double)e[q][2];
            } else if (rot) {
                const double* d = B.dR + 9 * (j - L.off_pose - 3);
#pragma unroll
                for (int a = 0; a < 3; ++a) dv[a] = d[a] * B.p[i][0] + d[3 + a] * B.p[i][1] + d[6 + a] * B.p[i][2];
            } else {
#pragma unroll
                for (int a = 0; a < 3; ++a) dv[a] = trans && j - L.off_pose == a ? 1.0 : 0.0;
            }
            landmark_dxy(fr, B, i, dv, dx, dy);
            if (!(exp || id || trans || rot)) dx = dy = 0.0;   // at any depth, zero included
            s += B.gx[i] * dx + B.gy[i] * dy;
            if (j < KS) {
                sdyn[(2 * i) * KS + j] = dx * B.rx[i];
                sdyn[(2 * i + 1) * KS + j] = dy * B.ry[i];
            }
        }
        sg[part][j] = s;
    }
    __syncthreads();
    if (tid < K) {
        double s = sg[0][tid];
#pragma unroll
        for (int p = 1; p < BAR_PARTS; ++p) s += sg[p][tid];
        g[(size_t)f * K + tid] = g[(size_t)f * K + tid] + gb + (float)s;
    }
    // task t: row group I (rows 4 I .. 4 I + 3) and column b of the upper triangle
    const int T = KS / 4;
    for (int t = tid;; t += BAR_THREADS) {
        int I = 0, b = t;
        while (I < T && b >= K - 4 * I) { b -= K - 4 * I; ++I; }
        if (I >= T) break;
        b += 4 * I;
        // both triangles are read: the data term's mirrored entries differ in the last places
        double hv[4], hl[4], s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int a = min(4 * I + r, K - 1);
            hv[r] = Hf[(size_t)a * K + b];
            hl[r] = Hf[(size_t)b * K + a];
        }
#pragma unroll 3
        for (int i = 0; i < NLMK; ++i) {
            const double* dx = sdyn + (2 * i) * KS;
            const double* dy = dx + KS;
            const double xb = dx[b], yb = dy[b];
#pragma unroll
            for (int r = 0; r < 4; ++r) s[r] += dx[4 * I + r] * xb + dy[4 * I + r] * yb;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int a = 4 * I + r;
            if (a > b) continue;
            Hf[(size_t)a * K + b] = a == b ? hv[r] + sbound[a] + s[r] : hv[r] + s[r];
            if (a != b) Hf[(size_t)b * K + a] = hl[r] + s[r];
        }
    }
}

// ------------------------------------------------------------------ batched Cholesky
// One workgroup of four wavefronts per matrix, the lower triangle in LDS as 16 x 16 blocks (padded
// with the identity to a multiple of 16).  What bounds it is the chain of K dependent columns, so
// the steps on that chain stay inside one wavefront, in registers, with no barrier:
//   panel     wavefront 0 holds the panel's rows (lane l: rows l and l + 64 below the diagonal
//             block's first), 16 columns each; pivots and column entries pass by lane reads;
//   trailing  A22 -= L21 L21^T on the MFMA of the type (FP32 or FP64, four 16 x 16 x 4 steps per
//             block), the blocks dealt to the four wavefronts; two barriers per panel;
//   solves    wavefront 0, lane l holding entries l and l + 64, right-looking.
// A barrier pair and an LDS round trip per column (what it replaces) took 283 us for one matrix of
// 94 unknowns (mode 1 with the FP64 fallback) and 552 us for 448; this takes 91 and 98 us, mode 1 without
// the fallback 57 and 61, mode 0 36 and 39.  Each entry takes its products in the same order (an MFMA
// step is four FMAs in order) and the root and the divisions round alike (ch_root, ch_div).
__device__ __forceinline__ double ch_wave_sum(double v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// mode 0: FP64 factorisation and solve.  mode 1: FP32 factorisation of the equilibrated
// matrix D^-1/2 H D^-1/2 (D = diag H, which removes the scale spread between pose and coefficient
// columns) and solve, then one FP64 residual-refinement step (r = -g - H x computed in FP64,
// correction solved with the FP32 factor); when the FP32 factorisation breaks down or the
// correction exceeds 1e-3 of the solution (an ill-conditioned frame), the FP64 factorisation.
template <typename TH>
__global__ void __launch_bounds__(256) k_cholesky(int K, const TH* __restrict__ H, const float* __restrict__ g,
                                                   float* __restrict__ delta, int* __restrict__ status,
                                                   const int* __restrict__ mask, int mode)
{
    const int f = blockIdx.x;
    if (mask && !mask[f]) return;
    extern __shared__ double dsm[];
    // a pivot that is not positive, of the FP32 and of the FP64 factorisation: two flags, as the wavefronts
    // read the first after their last common barrier and nothing may write it from then on
    __shared__ int sbad[2];
    __shared__ int sdone;                        // the FP32 solution is good
    __shared__ double sb[CMAXK];                 // the residual
    __shared__ float sx[CMAXK];
    const TH* Hf = H + (size_t)f * K * K;
    const float* gf = g + (size_t)f * K;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nT = (K + CHB - 1) / CHB;
    const bool in0 = lane < K, in1 = lane + 64 < K;
    if (tid == 0) sbad[0] = sbad[1] = sdone = 0;
    if (mode != 0) {
        float* A = (float*)dsm;
        __shared__ float sdinv[CMAXK];
        for (int i = tid; i < CMAXK; i += blockDim.x) {
            const float d = i < K ? (float)Hf[(size_t)i * K + i] : 1.f;
            sdinv[i] = d > 0.f ? rsqrtf(d) : 1.f;
        }
        __syncthreads();
        ch_load<float, TH>(A, Hf, K, nT, sdinv);
        __syncthreads();
        if (ch_factor<float>(A, nT, &sbad[0])) {
            float x0 = 0.f, x1 = 0.f;            // wavefront 0: the FP32 solution
            if (wave == 0) {
                x0 = in0 ? -gf[lane] * sdinv[lane] : 0.f;
                x1 = in1 ? -gf[lane + 64] * sdinv[lane + 64] : 0.f;
                ch_solve<float, float>(A, nT, x0, x1);
                x0 = in0 ? x0 * sdinv[lane] : 0.f;     // x = D^-1/2 y
                x1 = in1 ? x1 * sdinv[lane + 64] : 0.f;
                if (in0) sx[lane] = x0;
                if (in1) sx[lane + 64] = x1;
            }
            __syncthreads();
            // residual -g - H x in FP64, a thread per row over the columns in order; the rows go
            // through LDS 16 columns at a time so that they are read in whole sectors
            double* sH = (double*)((float*)dsm + nT * (nT + 1) / 2 * CHN);
            const int hr = tid >> 4, hc = tid & 15;
            TH hv[CHT];
            auto fetch = [&](int J) {
#pragma unroll
                for (int I = 0; I < CHT; ++I)
                    if (I < nT) hv[I] = Hf[(size_t)min(CHB * I + hr, K - 1) * K + min(CHB * J + hc, K - 1)];
            };
            double r = tid < K ? -(double)gf[tid] : 0.0;
            fetch(0);
            for (int J = 0; J < nT; ++J) {
#pragma unroll
                for (int I = 0; I < CHT; ++I)
                    if (I < nT) sH[(CHB * I + hr) * CHP + hc] = (double)hv[I];
                __syncthreads();
                if (J + 1 < nT) fetch(J + 1);
                if (tid < K) {
#pragma unroll
                    for (int c = 0; c < CHB; ++c)
                        if (CHB * J + c < K) r = fma(-sH[tid * CHP + c], (double)sx[CHB * J + c], r);
                }
                __syncthreads();
            }
            if (tid < K) sb[tid] = r * (double)sdinv[tid];
            __syncthreads();
            if (wave == 0) {
                double c0 = in0 ? sb[lane] : 0.0, c1 = in1 ? sb[lane + 64] : 0.0;
                ch_solve<float, double>(A, nT, c0, c1);
                c0 = in0 ? c0 * (double)sdinv[lane] : 0.0;
                c1 = in1 ? c1 * (double)sdinv[lane + 64] : 0.0;
                // the correction measures the FP32 solution's error (about cond * 2^-24 of it); past
                // 1e-3 of the solution one refinement step leaves more than ~1e-6, and the FP64
                // factorisation below takes over
                const double cn = ch_wave_sum(c0 * c0 + c1 * c1);
                const double xn = ch_wave_sum((double)x0 * x0 + (double)x1 * x1);
                const bool good = cn <= 1e-6 * xn;
                if (good) {
                    if (in0) delta[(size_t)f * K + lane] = (float)((double)x0 + c0);
                    if (in1) delta[(size_t)f * K + lane + 64] = (float)((double)x1 + c1);
                    if (lane == 0) status[f] = TDI_OK;
                }
                if (lane == 0) sdone = good;
            }
        }
        __syncthreads();
        if (sdone) return;
    }
    // FP64 factorisation and solve (mode 0, and the fallback of mode 1)
    double* A = dsm;
    ch_load<double, TH>(A, Hf, K, nT, nullptr);
    __syncthreads();
    if (!ch_factor<double>(A, nT, &sbad[1])) {
        if (tid == 0) status[f] = TDI_NOT_PD;
        return;
    }
    if (wave == 0) {
        double x0 = in0 ? -(double)gf[lane] : 0.0, x1 = in1 ? -(double)gf[lane + 64] : 0.0;
        ch_solve<double, double>(A, nT, x0, x1);
        if (in0) delta[(size_t)f * K + lane] = (float)x0;
        if (in1) delta[(size_t)f * K + lane + 64] = (float)x1;
        if (lane == 0) status[f] = TDI_OK;
    }
}

// Up to TINY_MAXK unknowns: a thread per matrix, in registers (padded with the identity), FP64 in both
// modes with the bits of k_cholesky's mode 0.  k_cholesky does sixteen columns whatever their number: 4096
// matrices of 4 unknowns 29 us (mode 1: 48), of 8 the same, here 12; from 9 on it is the faster for few
// matrices.
constexpr int TINY_MAXK = 8, TINY_THREADS = 64;

template <typename TH>
__global__ void __launch_bounds__(TINY_THREADS) k_cholesky_tiny(int n, int K, const TH* __restrict__ H,
                                                                const float* __restrict__ g, float* __restrict__ delta,
                                                                int* __restrict__ status, const int* __restrict__ mask)
{
    const int f = blockIdx.x * TINY_THREADS + threadIdx.x;
    if (f >= n || (mask && !mask[f])) return;
    const TH* Hf = H + (size_t)f * K * K;
    const float* gf = g + (size_t)f * K;
    double A[TINY_MAXK][TINY_MAXK], b[TINY_MAXK], q[TINY_MAXK];
#pragma unroll
    for (int i = 0; i < TINY_MAXK; ++i) {
#pragma unroll
        for (int j = 0; j <= i; ++j) {
            const double x = (double)Hf[min(i, K - 1) * K + min(j, K - 1)];
            A[i][j] = i < K ? (i == j ? ch_finite(x) : x) : i == j ? 1.0 : 0.0;
        }
        const double x = -(double)gf[min(i, K - 1)];
        b[i] = i < K ? x : 0.0;
    }
    bool bad = false;
#pragma unroll
    for (int k = 0; k < TINY_MAXK; ++k) {
        double s, inv;
        bad = bad || !(A[k][k] > 0.0);
        ch_root(A[k][k], s, inv, [](int) {});
        A[k][k] = s;
        q[k] = 1.0 / s;
#pragma unroll
        for (int i = k + 1; i < TINY_MAXK; ++i) A[i][k] = ch_div(A[i][k], s, inv);
#pragma unroll
        for (int i = k + 1; i < TINY_MAXK; ++i)
#pragma unroll
            for (int j = k + 1; j <= i; ++j) A[i][j] = fma(-A[i][k], A[j][k], A[i][j]);
    }
    status[f] = bad ? TDI_NOT_PD : TDI_OK;
    if (bad) return;
#pragma unroll
    for (int i = 0; i < TINY_MAXK; ++i) {
        b[i] = ch_div(b[i], A[i][i], q[i]);
#pragma unroll
        for (int j = i + 1; j < TINY_MAXK; ++j) b[j] = fma(-A[j][i], b[i], b[j]);
    }
#pragma unroll
    for (int i = TINY_MAXK - 1; i >= 0; --i) {
        b[i] = ch_div(b[i], A[i][i], q[i]);
#pragma unroll
        for (int j = 0; j < i; ++j) b[j] = fma(-A[i][j], b[i], b[j]);
    }
#pragma unroll
    for (int i = 0; i < TINY_MAXK; ++i)
        if (i < K) delta[(size_t)f * K + i] = (float)b[i];
}

// ------------------------------------------------------------------ line-search state machine
// One wavefront per frame (delta . g is a sum over its lanes in a fixed order).
__global__ void __launch_bounds__(64) k_ls_init(int n, int K, FitState* __restrict__ st, const int* __restrict__ chol_status,
                                                 const float* __restrict__ delta, const float* __restrict__ g,
                                                 const double* __restrict__ obj, int* __restrict__ searching)
{
    const int f = blockIdx.x, lane = threadIdx.x;
    double dg = 0.0;
    for (int k = lane; k < K; k += 64) dg += (double)delta[(size_t)f * K + k] * (double)g[(size_t)f * K + k];
    dg = ch_wave_sum(dg);
    if (lane != 0) return;
    FitState s = st[f];
    searching[f] = 0;
    if (!s.active) return;
    s.iters++;
    s.fresh = 1;              // the full evaluation just rendered theta
    if (chol_status[f] != TDI_OK) {
        s.active = 0;
        s.stop |= TDI_STOP_NOT_PD;
        s.status = TDI_NOT_PD;
    } else if (isnan(delta[(size_t)f * K])) {
        s.active = 0;
        s.stop |= TDI_STOP_NAN;
        s.status = TDI_NAN;
    } else {
        s.dg = (float)dg;
        s.obj0 = obj[f];
        s.t = 1.f;
        s.inner = 0;
        s.searching = 1;
        searching[f] = 1;
    }
    st[f] = s;
}

// Trials theta + t delta; unknowns [hold0, hold1) keep theta's value (the finetune fit's pose,
// model_fitter.cu:502).  rt null: no evaluation follows, and theta's render and rotation stay.
__global__ void k_ls_propose(int n, int K, int off_pose, float t_min, FitState* __restrict__ st,
                             const float* __restrict__ theta, const float* __restrict__ delta,
                             float* __restrict__ theta_try, double* __restrict__ rt, int* __restrict__ searching,
                             int* __restrict__ evalmask, int hold0, int hold1)
{
    const int f = blockIdx.x, off_tz = off_pose + 2;
    if (f >= n) return;
    __shared__ int go;
    if (threadIdx.x == 0) {
        FitState s = st[f];
        int ev = 0;
        if (searching[f]) {
            if (s.t < t_min) {
                s.active = 0;
                s.searching = 0;
                s.stop |= TDI_STOP_STEP;
                searching[f] = 0;
            } else {
                const bool held = off_tz >= hold0 && off_tz < hold1;
                const float tz = theta[(size_t)f * K + off_tz] + (held ? 0.f : s.t * delta[(size_t)f * K + off_tz]);
                if (tz < 0.f) {
                    s.searching = 0;
                    searching[f] = 0;
                } else {
                    ev = 1;
                }
            }
            st[f] = s;
        }
        evalmask[f] = ev;
        go = ev;
    }
    __syncthreads();
    if (!go) return;
    const float t = st[f].t;
    __shared__ float pose[6];
    for (int k = threadIdx.x; k < K; k += blockDim.x) {
        const float x = (k >= hold0 && k < hold1) ? theta[(size_t)f * K + k]
                                                  : theta[(size_t)f * K + k] + t * delta[(size_t)f * K + k];
        theta_try[(size_t)f * K + k] = x;
        if (k >= off_pose && k < off_pose + 6) pose[k - off_pose] = x;
    }
    __syncthreads();
    // the trial's rotation and translation for the synthesis that follows
    if (threadIdx.x == 0 && rt) {
        double R[9];
        rodrigues_f64(pose + 3, R);
        for (int k = 0; k < 9; ++k) rt[(size_t)f * 12 + k] = R[k];
        for (int a = 0; a < 3; ++a) rt[(size_t)f * 12 + 9 + a] = pose[a];
    }
}

// One wavefront per frame; it also sums the frame's objective from the evaluation's partials.
__global__ void __launch_bounds__(64) k_ls_decide(int n, int K, FitState* __restrict__ st, const int* __restrict__ act,
                            const int* __restrict__ evalmask, int* __restrict__ searching, double* __restrict__ obj,
                            const double* __restrict__ objb, const double* __restrict__ objp, int col_nb,
                            const int* __restrict__ face_ok, float* __restrict__ theta,
                            const float* __restrict__ theta_try, tdi_fit_options o)
{
    const int f = blockIdx.x;
    if (f >= n || !evalmask[f]) return;
    __shared__ int accept;
    const double data = obj_partials(objp + (size_t)f * OBJ_PARTS, col_fpb(col_nb, act[0]));
    if (threadIdx.x == 0) {
        const double F = objb[f] + data;
        obj[f] = F;
        FitState s = st[f];
        int acc = 0;
        if (!face_ok[f] || isnan(objb[f])) {
            s.t *= o.armijo_beta;
        } else {
            s.inner++;
            s.ls_evals++;
            if (-s.dg < o.decrement_tol) {
                s.active = 0;
                s.searching = 0;
                s.stop |= TDI_STOP_DECREMENT;
            } else if (F < s.obj0 + (double)(o.armijo_alpha * s.t * s.dg)) {
                acc = 1;
                s.searching = 0;
            } else {
                s.t *= o.armijo_beta;
            }
            if (s.inner >= o.max_ls) s.searching = 0;
        }
        s.fresh = acc;        // the trial's render is in the workspace; it is theta's if accepted
        searching[f] = s.searching;
        st[f] = s;
        accept = acc;
    }
    __syncthreads();
    if (!accept) return;
    for (int k = threadIdx.x; k < K; k += blockDim.x) theta[(size_t)f * K + k] = theta_try[(size_t)f * K + k];
}

// Frame lists, built by one workgroup: per 1024-entry tile a wavefront ballot and popcount give each
// set entry its rank within the wave, the wave totals in LDS give the wave offsets, and a running
// count carries across tiles.
constexpr int CMP_THREADS = 1024;
constexpr int CMP_WAVES = CMP_THREADS / 64;

struct ListBuilder {
    int running = 0;
    // every thread of the workgroup calls it, with its entry and whether it is set (act null: count only)
    __device__ __forceinline__ void add(int f, bool set, int* __restrict__ act, int* swave)
    {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
        const unsigned long long b = __ballot(set);
        if (lane == 0) swave[wave] = __popcll(b);
        __syncthreads();
        int off = 0, total = 0;
#pragma unroll
        for (int w = 0; w < CMP_WAVES; ++w) {
            off += (w < wave) ? swave[w] : 0;
            total += swave[w];
        }
        if (set && act) act[1 + running + off + __popcll(b & lt)] = f;
        running += total;
        __syncthreads();
    }
};

// The lists of one evaluation: act_m the active frames, of these act_r with a stale and act_u with a
// reusable render in the workspace; mask the active frames.  all: every real frame counts as active.
__global__ void __launch_bounds__(CMP_THREADS) k_iter_lists(int n, const FitState* __restrict__ st, int all,
                                                              int* __restrict__ mask, int* __restrict__ act_m,
                                                              int* __restrict__ act_r, int* __restrict__ act_u)
{
    __shared__ int swave[CMP_WAVES];
    ListBuilder lm, lr, lu;
    for (int t0 = 0; t0 < n; t0 += CMP_THREADS) {
        const int f = t0 + threadIdx.x;
        const bool in = f < n;
        const int active = in && (all ? st[f].real : st[f].active), fresh = in && st[f].fresh;
        if (in) mask[f] = active;
        lm.add(f, active, act_m, swave);
        lr.add(f, active && !fresh, act_r, swave);
        lu.add(f, active && fresh, act_u, swave);
    }
    if (threadIdx.x == 0) {
        act_m[0] = lm.running;
        act_r[0] = lr.running;
        act_u[0] = lu.running;
    }
}

// act_e from evalmask, and what the host decides the next launches from, in its own memory: status[1]
// frames to evaluate, [2] active frames, [3] active frames with a stale render; then status[0], the
// number of this report (counted in *seq), which the host waits for.
__global__ void __launch_bounds__(CMP_THREADS) k_ls_status(int n, const FitState* __restrict__ st,
                                                             const int* __restrict__ evalmask, int* __restrict__ act_e,
                                                             int* __restrict__ seq, int* status)
{
    __shared__ int swave[CMP_WAVES];
    ListBuilder le, la, ls;
    for (int t0 = 0; t0 < n; t0 += CMP_THREADS) {
        const int f = t0 + threadIdx.x;
        const bool in = f < n;
        const int active = in && st[f].active, fresh = in && st[f].fresh;
        le.add(f, in && evalmask[f], act_e, swave);
        la.add(f, active, nullptr, swave);
        ls.add(f, active && !fresh, nullptr, swave);
    }
    if (threadIdx.x == 0) {
        act_e[0] = le.running;
        const int k = *seq + 1;
        *seq = k;
        volatile int* out = status;
        out[1] = le.running;
        out[2] = la.running;
        out[3] = ls.running;
        __threadfence_system();
        __hip_atomic_store(status, k, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// The barrier's derivative terms (k_barrier's) for frames with more unknowns than the
// landmark-derivative rows fit in LDS (the identity stage): the rows go to global scratch D
// [frame][2][NLMK][K] and the Gauss-Newton sum is formed over 32 x 32 tiles of H by a grid.
// Same formulas, FP64 throughout.
__global__ void __launch_bounds__(256) k_barrier_rows(ModelGPU m, Layout L, const FrameGPU* __restrict__ frames,
                                                       const int* __restrict__ act, int n, const float* __restrict__ theta,
                                                       const double* __restrict__ rt, const double* __restrict__ P0,
                                                       LmkArrays lm, int use_lmk, double* __restrict__ D,
                                                       double* __restrict__ H, float* __restrict__ g)
{
    if ((int)blockIdx.x >= fl_count(act, n)) return;
    const int f = fl_frame(act, blockIdx.x);
    const int K = L.K;
    const FrameGPU fr = frames[f];
    const float* tf = theta + (size_t)f * K;
    double* sdx = D + (size_t)f * 2 * NLMK * K;
    double* sdy = sdx + (size_t)NLMK * K;
    __shared__ BarrierFrame B;
    const int tid = threadIdx.x;
    for (int j = tid; j < K; j += blockDim.x) {
        float gb;
        double hb;
        bound_terms(m, tf, j, gb, hb);
        g[(size_t)f * K + j] += gb;
        H[(size_t)f * K * K + (size_t)j * K + j] += hb;
    }
    if (!use_lmk) return;
    barrier_frame(m, L, fr, f, tf, rt, P0, lm.base + (size_t)f * 6 * NLMK, B);
    // the columns without geometry (albedo, light) are zero
    const int ng = L.off_light - L.off_id;
    for (int e = tid; e < NLMK * (K - ng); e += blockDim.x) {
        const int i = e / (K - ng), c = e - i * (K - ng), j = c < L.off_id ? c : c + ng;
        sdx[(size_t)i * K + j] = sdy[(size_t)i * K + j] = 0.0;
    }
    barrier_rows(m, L, fr, B, [&](int i, int j, double dx, double dy) {
        sdx[(size_t)i * K + j] = dx;
        sdy[(size_t)i * K + j] = dy;
    });
    __syncthreads();
    for (int j = tid; j < K; j += blockDim.x) {
        double s = 0.0;
#pragma unroll 8
        for (int i = 0; i < NLMK; ++i) {
            const double dx = sdx[(size_t)i * K + j], dy = sdy[(size_t)i * K + j];
            s += B.gx[i] * dx + B.gy[i] * dy;
            sdx[(size_t)i * K + j] = dx * B.rx[i];
            sdy[(size_t)i * K + j] = dy * B.ry[i];
        }
        g[(size_t)f * K + j] += (float)s;
    }
}

constexpr int BH_T = 32;

// H += sum_i dx_i dx_i^T + dy_i dy_i^T over the tiles (I, J >= I) of 32 x 32; both halves written.
__global__ void __launch_bounds__(256) k_barrier_hess(int K, const int* __restrict__ act, int n,
                                                       const double* __restrict__ D, double* __restrict__ H)
{
    const int T = (K + BH_T - 1) / BH_T;
    int t = blockIdx.x, I = 0;
    while (t >= T - I) { t -= T - I; ++I; }
    const int J = I + t;
    __shared__ double sa[2][NLMK][BH_T], sb[2][NLMK][BH_T];
    const int nact = fl_count(act, n);
    for (int yi = blockIdx.y; yi < nact; yi += gridDim.y) {
        const int f = fl_frame(act, yi);
        const double* Df = D + (size_t)f * 2 * NLMK * K;
        for (int e = threadIdx.x; e < 2 * NLMK * BH_T; e += blockDim.x) {
            const int c = e % BH_T, i = (e / BH_T) % NLMK, q = e / (BH_T * NLMK);
            const int a = I * BH_T + c, b = J * BH_T + c;
            sa[q][i][c] = a < K ? Df[((size_t)q * NLMK + i) * K + a] : 0.0;
            sb[q][i][c] = b < K ? Df[((size_t)q * NLMK + i) * K + b] : 0.0;
        }
        __syncthreads();
        for (int e = threadIdx.x; e < BH_T * BH_T; e += blockDim.x) {
            const int r = e / BH_T, c = e - r * BH_T;
            const int a = I * BH_T + r, b = J * BH_T + c;
            if (a >= K || b >= K || (I == J && c < r)) continue;
            double sacc = 0.0;
            for (int i = 0; i < NLMK; ++i) sacc += sa[0][i][r] * sb[0][i][c] + sa[1][i][r] * sb[1][i][c];
            H[(size_t)f * K * K + (size_t)a * K + b] += sacc;
            if (a != b) H[(size_t)f * K * K + (size_t)b * K + a] += sacc;
        }
        __syncthreads();
    }
}

} // namespace

int launch_barrier_big(const ModelGPU& m, const Layout& L, const FrameGPU* frames, FrameList fl, const float* theta,
                       const double* rt, const double* P0, const LmkArrays& lm, int use_landmarks, double* D, double* H, float* g,
                       hipStream_t s)
{
    hipLaunchKernelGGL(k_barrier_rows, dim3(fl.n > 0 ? fl.n : 1), dim3(256), 0, s, m, L, frames, fl.act, fl.n, theta,
                       rt, P0, lm, use_landmarks, D, H, g);
    if (use_landmarks) {
        const int T = (L.K + BH_T - 1) / BH_T;
        hipLaunchKernelGGL(k_barrier_hess, dim3(T * (T + 1) / 2, grid_frames(fl.n, 1 << 16)), dim3(256), 0, s, L.K,
                           fl.act, fl.n, D, H);
    }
    TDI_HIP(hipGetLastError());
    return TDI_OK;
}

int launch_barrier_obj(const ModelGPU& m, const Layout& L, const FrameGPU* frames, FrameList fl, const float* theta,
                       const double* rt, const double* P0, const float4* vproj, const LmkArrays& lm, int use_landmarks,
                       float ref_face_size, double* obj, double* objb, int* face_ok, hipStream_t s)
{
    hipLaunchKernelGGL(k_barrier_obj, dim3(fl.n > 0 ? fl.n : 1), dim3(256), 0, s, m, L, frames, fl.act, fl.n, theta, rt,
                       P0, vproj, lm, use_landmarks, ref_face_size, obj, objb, face_ok);
    TDI_HIP(hipGetLastError());
    return TDI_OK;
}

int launch_barrier(const ModelGPU& m, const Layout& L, const FrameGPU* frames, FrameList fl, const float* theta,
                   const double* rt, const double* P0, const LmkArrays& lm, int use_landmarks, double* H, float* g, hipStream_t s)
{
    if (L.K > BMAXK) {
        if (!use_landmarks)              // bounds alone: no landmark rows to hold
            return launch_barrier_big(m, L, frames, fl, theta, rt, P0, lm, 0, nullptr, H, g, s);
        set_error("barrier: K=%d > %d (derivative terms: launch_barrier_big)", L.K, BMAXK);
        return TDI_ERR_ARG;
    }
    const size_t lds = use_landmarks ? sizeof(double) * 2 * NLMK * ((L.K + 3) & ~3) : 0;
    if (use_landmarks) {
        // with the static part (10 KB) above the default limit from 65 unknowns on: allow up to what K <= BMAXK
        // needs (91 KB)
        static std::atomic<unsigned long long> done{0};
        TDI_HIP(allow_lds(reinterpret_cast<const void*>(k_barrier), sizeof(double) * 2 * NLMK * BMAXK, done));
    }
    hipLaunchKernelGGL(k_barrier, dim3(fl.n > 0 ? fl.n : 1), dim3(BAR_THREADS), lds, s, m, L, frames, fl.act, fl.n, theta,
                       rt, P0, lm, use_landmarks, H, g);
    TDI_HIP(hipGetLastError());
    return TDI_OK;
}

template <typename TH>
static int launch_cholesky_t(int n, int K, const TH* H, const float* g, float* delta, int* status, int mode,
                             const int* mask, hipStream_t s)
{
    if (K > CMAXK) {
        set_error("cholesky: K=%d > %d", K, CMAXK);
        return TDI_ERR_ARG;
    }
    if (K <= TINY_MAXK) {
        hipLaunchKernelGGL(k_cholesky_tiny<TH>, dim3((n + TINY_THREADS - 1) / TINY_THREADS), dim3(TINY_THREADS), 0, s, n, K, H,
                           g, delta, status, mask);
        TDI_HIP(hipGetLastError());
        return TDI_OK;
    }
    const int nT = (K + CHB - 1) / CHB;
    // the FP64 blocks, or mode 1's FP32 blocks and 16 columns of H in FP64
    const size_t nb = (size_t)nT * (nT + 1) / 2 * CHN;
    const size_t lds = std::max(nb * sizeof(double), nb * sizeof(float) + (size_t)nT * CHN * sizeof(double));
    hipLaunchKernelGGL(k_cholesky<TH>, dim3(n), dim3(256), lds, s, K, H, g, delta, status, mask, mode);
    TDI_HIP(hipGetLastError());
    return TDI_OK;
}

int launch_cholesky(int n, int K, const float* H, const float* g, float* delta, int* status, int mode, const int* mask,
                    hipStream_t s)
{
    // above one workgroup's LDS: the blocked FP64 factorisation (every listed matrix)
    if (K > CMAXK && !mask) return launch_cholesky_big(n, K, H, g, delta, status, s);
    return launch_cholesky_t(n, K, H, g, delta, status, mode, mask, s);
}

int launch_cholesky(int n, int K, const double* H, const float* g, float* delta, int* status, int mode, const int* mask,
                    hipStream_t s)
{
    return launch_cholesky_t(n, K, H, g, delta, status, mode, mask, s);
}

int launch_ls_init(int n, int K, FitState* st, const int* chol_status, const float* delta, const float* g,
                   const double* obj, int* searching, hipStream_t s)
{
    hipLaunchKernelGGL(k_ls_init, dim3(n), dim3(64), 0, s, n, K, st, chol_status, delta, g, obj,
                       searching);
    TDI_HIP(hipGetLastError());
    return TDI_OK;
}

int launch_ls_propose(int n, const Layout& L, float t_min, FitState* st, const float* theta, const float* delta,
                      float* theta_try, double* rt, int* searching, int* evalmask, int hold0, int hold1, hipStream_t s)
{
    hipLaunchKernelGGL(k_ls_propose, dim3(n), dim3(64), 0, s, n, L.K, L.off_pose, t_min, st, theta, delta, theta_try,
                       rt, searching, evalmask, hold0, hold1);
    TDI_HIP(hipGetLastError());
    return TDI_OK;
}

int launch_ls_decide(int n, int K, FitState* st, const int* act, const int* evalmask, int* searching, double* obj,
                     const double* objb, const double* objp, const int* face_ok, float* theta, const float* theta_try,
                     const tdi_fit_options& o, hipStream_t s)
{
    hipLaunchKernelGGL(k_ls_decide, dim3(n), dim3(64), 0, s, n, K, st, act, evalmask, searching, obj, objb, objp,
                       col_blocks(n), face_ok, theta, theta_try, o);
    TDI_HIP(hipGetLastError());
    return TDI_OK;
}

int launch_iter_lists(int n, const FitState* st, int all, int* mask, int* act_m, int* act_r, int* act_u, hipStream_t s)
{
    hipLaunchKernelGGL(k_iter_lists, dim3(1), dim3(CMP_THREADS), 0, s, n, st, all, mask, act_m, act_r, act_u);
    TDI_HIP(hipGetLastError());
    return TDI_OK;
}

int launch_ls_status(int n, const FitState* st, const int* evalmask, int* act_e, int* seq, int* status, hipStream_t s)
{
    hipLaunchKernelGGL(k_ls_status, dim3(1), dim3(CMP_THREADS), 0, s, n, st, evalmask, act_e, seq, status);
    TDI_HIP(hipGetLastError());
    return TDI_OK;
}

} // namespace tdi
