// geometry.hip — vertex synthesis, view transform and projection on gfx950.
//
// Reference: Renderer::compute_nonrigid_shape2 (renderer.cu:806-861) does three cuBLAS
// SGEMVs per basis (X0 = X0_mean + IX alpha + EX eps, ...) and then
// view_transform_3d_pts_and_render_2d (funcs.cu:395-453): P = R P0 + tau,
// xp = phix X/Z + cx, yp = phiy Y/Z + cy.
//
// The basis product, rotation, translation and projection are FP64, rounded to FP32 once: the
// projected vertices then equal the correctly rounded values (what an FP64 computation rounded to
// FP32 gives), so the FP32 coverage test downstream sees the same inputs as an FP64 transcription
// would.  MI355X runs FP64 FMA and FP64 MFMA at the same 78.6 TFLOP/s, so this costs little next
// to the rest of an iteration.
//
//   k_synth_tile   — [3V x K] x [K x B] on v_mfma_f64_16x16x4f64; a workgroup owns 16 vertices,
//                    stages their basis rows in LDS and walks every frame of the list; the
//                    epilogue fuses mean, rotation, translation and projection from registers.
//   k_synth_one    — a single frame: a thread per vertex coordinate.
#include "common.h"

namespace tdi {

namespace {

constexpr int MAX_UNKNOWNS = 1024;
constexpr int MAXK_LDS = 1024;          // identity coefficients that k_id_shape holds in LDS

__device__ __forceinline__ void store_vertex(const FrameCam& cam, const double* R, const double* p, size_t o, double* P0,
                                             float* P, float4* vproj)
{
    // model-space vertices stay FP64: the shading normal is the cross product of edges of
    // about a millimetre between coordinates of about 100 mm, which FP32 would round to 1e-5
    P0[3 * o + 0] = p[0];
    P0[3 * o + 1] = p[1];
    P0[3 * o + 2] = p[2];
    double q[3];
    vproj[o] = project_vertex(cam, R, p, q);
    if (P) {                               // camera-space vertices only when asked for
        P[3 * o + 0] = (float)q[0];
        P[3 * o + 1] = (float)q[1];
        P[3 * o + 2] = (float)q[2];
    }
}

// FP64 rotation and translation of every listed frame, once per launch (the synthesis
// workgroups read them instead of evaluating Rodrigues' formula per workgroup).
__global__ void k_frame_rt(Layout L, const float* __restrict__ theta, const int* __restrict__ act, int n,
                           double* __restrict__ rt)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= fl_count(act, n)) return;
    const int f = fl_frame(act, i);
    const float* tf = theta + (size_t)f * L.K;
    double R[9];
    rodrigues_f64(tf + L.off_pose + 3, R);
    double* o = rt + (size_t)f * 12;
    for (int k = 0; k < 9; ++k) o[k] = R[k];
    for (int a = 0; a < 3; ++a) o[9 + a] = tf[L.off_pose + a];
}

// FP64 MFMA operand layout, v_mfma_f64_16x16x4f64 (one double per lane for A and B):
//   A[i][k]: lane = i + 16*k          B[k][j]: lane = j + 16*k
// Accumulator: lane l, element r (0..3) holds C[l/16 + 4*r][l % 16] (measured on gfx950;
// the FP32/BF16 16x16 forms use row 4*(l/16) + r instead).

typedef double v4d __attribute__((ext_vector_type(4)));

// Vertex tiles for v_mfma_f64_16x16x4f64: a workgroup owns SY_VERTS = 16 vertices and keeps one
// accumulator per coordinate, whose tile row i is vertex i (A = that coordinate's basis rows of the
// 16 vertices, B = the coefficients of 16 frames), so lane l, element r of the x, y and z
// accumulators holds vertex l/16 + 4 r for frame l%16: every MFMA row is a vertex coordinate
// (three MFMAs per k-step for 16 vertices); step q takes columns 4 q .. 4 q + 3, in that order.
//
// Long lists: the basis rows are staged in LDS (as FP64), SY_KMAX columns at a time, identity
// columns first.  With one such chunk (the per-frame fit: expression columns only) it is staged
// once and each wavefront walks its own groups of 16 list entries with no further barrier; with
// more, the workgroup stages every chunk for each four groups.
//
// One group (a list of up to 16 frames, such as the last line-search rounds of any batch): nothing
// is reused from LDS and latency is all there is, so three wavefronts take a coordinate each
// straight from memory and the four share the epilogue.  The sums run in the same order in all
// forms, so a frame's vertices do not depend on the frames around it.
//
// Every caller of several frames takes this kernel.  Single evaluations took a thread per vertex walking
// its own three rows before: a sector per lane and load, and the whole basis again for every frame.
// Measured at 53,361 vertices and 79 columns, that kernel against this one: 96 frames 2493 -> 104 us,
// 48 frames 1258 -> 55 us.  Bound by the FP64 matrix rate (31 us of the 104)
// and the stores (40 B per vertex, 44 us).  The one-group form took the mean launch of a one-frame fit
// from 10.2 to 6.9 us (its basis staging alone was 39 us of a launch: run-time divisors).
constexpr int SY_VERTS = 16;               // vertices per workgroup
constexpr int SY_KMAX = 80;                // columns held in LDS at a time

// this lane's B entries: columns kq + 4 q of a chunk of kc, every load issued
// unconditionally (clamped to a valid column) so the batch has no branches.  Nothing needs zeroing:
// the A entries past the chunk's columns are zero, and an output column depends on its own frame's
// B column only, so lanes without a live frame just skip the epilogue.
__device__ __forceinline__ void synth_coefs(const float* __restrict__ tb, int kq, int kc, float* bv)
{
#pragma unroll
    for (int q = 0; q < SY_KMAX / 4; ++q) bv[q] = tb[min(kq + 4 * q, kc - 1)];
}

// y[q] on the lanes of residue kq (lane / 16) = element kq of the lanes of residue q: a 4 x 4
// transpose over the four 16-lane rows of a wavefront.
__device__ __forceinline__ void transpose_residues(float4 x, float* y)
{
    unsigned a0 = __float_as_uint(x.x), a1 = __float_as_uint(x.y), a2 = __float_as_uint(x.z), a3 = __float_as_uint(x.w);
    // the upper half of the first with the lower half of the second, then the odd rows with the even
    const auto s02 = __builtin_amdgcn_permlane32_swap(a0, a2, false, false);
    const auto s13 = __builtin_amdgcn_permlane32_swap(a1, a3, false, false);
    const auto s01 = __builtin_amdgcn_permlane16_swap(s02[0], s13[0], false, false);
    const auto s23 = __builtin_amdgcn_permlane16_swap(s02[1], s13[1], false, false);
    y[0] = __uint_as_float(s01[0]);
    y[1] = __uint_as_float(s01[1]);
    y[2] = __uint_as_float(s23[0]);
    y[3] = __uint_as_float(s23[1]);
}

// Three wavefronts per SIMD (register budget 168): with four, 30 registers spill and 96 frames take
// 148 us instead of 98.  ONE: a single chunk of columns.
template <bool ONE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
k_synth_tile(ModelGPU m, Layout L, const FrameGPU* __restrict__ frames, const float* __restrict__ theta,
             const int* __restrict__ act, int n, const double* __restrict__ rt, const double* __restrict__ mean64,
             double* __restrict__ P0, float* __restrict__ P, float4* __restrict__ vproj)
{
    __shared__ double sA[3][SY_KMAX][16];              // [coordinate][column][vertex]
    __shared__ double smean[SY_VERTS * 3];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nact = fl_count(act, n);
    if (nact == 0) return;                   // an emptied list
    const int v0 = blockIdx.x * SY_VERTS;
    const int j = lane & 15, kq = lane >> 4;
    // the base shape: the model's mean, or a given FP64 shape that holds the identity already (the
    // identity stage's shared identity)
    for (int e = tid; e < SY_VERTS * 3; e += blockDim.x) {
        const int v = v0 + e / 3;
        smean[e] = v < m.V ? (mean64 ? mean64[3 * v0 + e] : (double)m.mean[3 * v0 + e]) : 0.0;
    }
    if (ONE && nact <= 16) {
        const bool live = j < nact;
        const int f = fl_frame(act, live ? j : 0);
        const FrameCam cam{frames[f].phix, frames[f].phiy, frames[f].cx, frames[f].cy};
        double R[12];
#pragma unroll
        for (int q = 0; q < 12; ++q) R[q] = rt[(size_t)f * 12 + q];
        double (*sacc)[64] = (double (*)[64]) & sA[0][0][0];   // [coordinate * 4 + element][lane]
        if (wave < 3) {
            const float* row = m.exp_basis + (3 * (size_t)min(v0 + j, m.V - 1) + wave) * m.exp_ld;
            // columns 16 t + 4 kq .. + 3 in one load, then transposed over the four residues into
            // columns 16 t + 4 q + kq (one load per column took 34.6 us of a one-frame launch)
            float A[SY_KMAX / 4], bv[SY_KMAX / 4];
            float4 ld4[SY_KMAX / 16];
#pragma unroll
            for (int t = 0; t < SY_KMAX / 16; ++t) ld4[t] = *(const float4*)(row + min(16 * t + 4 * kq, m.exp_ld - 4));
#pragma unroll
            for (int t = 0; t < SY_KMAX / 16; ++t) transpose_residues(ld4[t], A + 4 * t);
            synth_coefs(theta + (size_t)f * L.K + L.off_exp, kq, L.nexp, bv);
            v4d acc = (v4d){0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < SY_KMAX / 4; ++q) {
                if (4 * q >= L.nexp) continue;         // within ld: zero past the last column
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)A[q], (double)bv[q], acc, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) sacc[4 * wave + r][lane] = acc[r];
        }
        __syncthreads();
        const int vl = kq + 4 * wave, v = v0 + vl;
        if (live && v < m.V) {
            double p[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) p[a] = smean[3 * vl + a] + sacc[4 * a + wave][lane];
            store_vertex(cam, R, p, (size_t)f * m.V + v, P0, P, vproj);
        }
        return;
    }
    const int nid = mean64 ? 0 : L.nid;
    const int idc = (nid + SY_KMAX - 1) / SY_KMAX;                     // identity chunks
    const int nch = ONE ? 1 : idc + (L.nexp + SY_KMAX - 1) / SY_KMAX;
    if (nch == 0) __syncthreads();
    const int ngroups = (nact + 15) >> 4;
    for (int g0 = 0; g0 < ngroups; g0 += 4) {
        const int g = g0 + wave;
        const int c = 16 * g + j;
        const bool live = c < nact;
        const int f = fl_frame(act, live ? c : 0);
        // the epilogue's camera and pose, loaded before the products that hide their latency
        const FrameCam cam{frames[f].phix, frames[f].phiy, frames[f].cx, frames[f].cy};
        double R[12];
#pragma unroll
        for (int q = 0; q < 12; ++q) R[q] = rt[(size_t)f * 12 + q];
        v4d acc[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) acc[a] = (v4d){0, 0, 0, 0};
        for (int ch = 0; ch < nch; ++ch) {
            const bool id = !ONE && ch < idc;
            const int k0 = ONE ? 0 : SY_KMAX * (id ? ch : ch - idc);   // first column of the chunk in its basis
            const int kc = ONE ? L.nexp : min(SY_KMAX, (id ? nid : L.nexp) - k0);
            if (!ONE || g0 == 0) {
                // basis rows of the workgroup's vertices: item = (coordinate, four columns, vertex),
                // the 16 vertices on neighbouring lanes so that the LDS stores are contiguous; a
                // fixed count of 16-byte loads per thread from clamped addresses, zeroed by a select,
                // so that they are in flight together.  The rows are zero past their last column
                // up to ld, a multiple of 16.
                const float* basis = id ? m.id_basis : m.exp_basis;
                const int ld = id ? m.id_ld : m.exp_ld;
                constexpr int NC4 = SY_KMAX / 4, NIT = 3 * NC4 * 16, NST = (NIT + 255) / 256;
                float4 av[NST];
#pragma unroll
                for (int q = 0; q < NST; ++q) {
                    const int e = min(tid + 256 * q, NIT - 1);
                    const int i = e & 15, c4 = (e >> 4) % NC4, a = (e >> 4) / NC4;
                    av[q] = *(const float4*)(basis + (size_t)(3 * min(v0 + i, m.V - 1) + a) * ld +
                                             min(k0 + 4 * c4, ld - 4));
                }
                if (!ONE) __syncthreads();             // the previous chunk is no longer read
#pragma unroll
                for (int q = 0; q < NST; ++q) {
                    const int e = tid + 256 * q;
                    if (e < NIT) {
                        const int i = e & 15, c4 = (e >> 4) % NC4, a = (e >> 4) / NC4;
                        const bool in = k0 + 4 * c4 < ld && v0 + i < m.V;
                        sA[a][4 * c4 + 0][i] = in ? (double)av[q].x : 0.0;
                        sA[a][4 * c4 + 1][i] = in ? (double)av[q].y : 0.0;
                        sA[a][4 * c4 + 2][i] = in ? (double)av[q].z : 0.0;
                        sA[a][4 * c4 + 3][i] = in ? (double)av[q].w : 0.0;
                    }
                }
                __syncthreads();
            }
            if (g >= ngroups) continue;
            float bv[SY_KMAX / 4];
            synth_coefs(theta + (size_t)f * L.K + (id ? L.off_id : L.off_exp) + k0, kq, kc, bv);
#pragma unroll
            for (int q = 0; q < SY_KMAX / 4; ++q) {
                if (4 * q >= kc) continue;
                const double b = (double)bv[q];
#pragma unroll
                for (int a = 0; a < 3; ++a)
                    acc[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(sA[a][4 * q + kq][j], b, acc[a], 0, 0, 0);
            }
        }
        if (g < ngroups && live) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int vl = kq + 4 * r, v = v0 + vl;
                if (v < m.V) {
                    double p[3];
#pragma unroll
                    for (int a = 0; a < 3; ++a) p[a] = smean[3 * vl + a] + acc[a][r];
                    store_vertex(cam, R, p, (size_t)f * m.V + v, P0, P, vproj);
                }
            }
        }
    }
}

// One frame: 15 of a tile's 16 columns would be idle, and with more than 80 columns its chunks would be
// staged for that one, so a thread takes one row (a vertex coordinate) with its sum in the tiles' order, 64
// vertices per workgroup.  The latency of the loads bounds it.  The whole call by a thread per vertex, by
// tiles and by this (53,361 vertices): 79 columns 49, 53 and 44 us, 199 + 79 columns 80, 114 and 65, 200
// columns 64, 95 and 57; two frames by tiles are faster than two of these (79 columns: 55 us).
constexpr int ONE_VERTS = 64;

__device__ __forceinline__ double synth_row(const ModelGPU& m, const Layout& L, const float* __restrict__ tf, int r,
                                            const double* __restrict__ mean64)
{
    const double base = mean64 ? mean64[r] : (double)m.mean[r];
    double s = 0.0;
    for (int blk = 0; blk < 2; ++blk) {                    // identity columns first
        const int nc = blk ? L.nexp : mean64 ? 0 : L.nid, ld = blk ? m.exp_ld : m.id_ld;
        const float* row = (blk ? m.exp_basis : m.id_basis) + (size_t)r * ld;
        const float* tb = tf + (blk ? L.off_exp : L.off_id);
#pragma unroll 2
        for (int k0 = 0; k0 < nc; k0 += 16) {              // rows are padded to 16 columns with zeros
            float4 e[4];
            float c[16];
#pragma unroll
            for (int q = 0; q < 4; ++q) e[q] = *(const float4*)(row + k0 + 4 * q);
#pragma unroll
            for (int q = 0; q < 16; ++q) c[q] = tb[min(k0 + q, nc - 1)];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                s = fma((double)e[q].x, (double)c[4 * q + 0], s);
                s = fma((double)e[q].y, (double)c[4 * q + 1], s);
                s = fma((double)e[q].z, (double)c[4 * q + 2], s);
                s = fma((double)e[q].w, (double)c[4 * q + 3], s);
            }
        }
    }
    return base + s;
}

__global__ void __launch_bounds__(3 * ONE_VERTS) k_synth_one(ModelGPU m, Layout L, const FrameGPU* __restrict__ frames,
                                                             const float* __restrict__ theta, const int* __restrict__ act,
                                                             const double* __restrict__ rt,
                                                             const double* __restrict__ mean64, double* __restrict__ P0,
                                                             float* __restrict__ P, float4* __restrict__ vproj)
{
    __shared__ double sp[3 * ONE_VERTS];
    if (fl_count(act, 1) == 0) return;
    const int f = fl_frame(act, 0), tid = threadIdx.x;
    const int r0 = 3 * ONE_VERTS * blockIdx.x, r = min(r0 + tid, 3 * m.V - 1);
    sp[tid] = synth_row(m, L, theta + (size_t)f * L.K, r, mean64);
    __syncthreads();
    const int v = ONE_VERTS * blockIdx.x + tid;
    if (tid >= ONE_VERTS || v >= m.V) return;
    double R[12];
#pragma unroll
    for (int q = 0; q < 12; ++q) R[q] = rt[(size_t)f * 12 + q];
    const FrameCam cam{frames[f].phix, frames[f].phiy, frames[f].cx, frames[f].cy};
    store_vertex(cam, R, sp + 3 * tid, (size_t)f * m.V + v, P0, P, vproj);
}

// The landmark vertices alone, a frame per workgroup (the rest of P0 is left as it is).
__global__ void __launch_bounds__(192) k_landmark_vertices(ModelGPU m, Layout L, const float* __restrict__ theta,
                                                           double* __restrict__ P0)
{
    const int f = blockIdx.x, tid = threadIdx.x;
    if (tid >= 3 * NLMK) return;
    const int r = 3 * m.lmk_ids[tid / 3] + tid % 3;
    P0[(size_t)f * m.V * 3 + r] = synth_row(m, L, theta + (size_t)f * L.K, r, nullptr);
}

} // namespace

static int launch_frame_rt(const Layout& L, FrameList fl, const float* theta, double* rt, hipStream_t s)
{
    hipLaunchKernelGGL(k_frame_rt, dim3((fl.n + 255) / 256 > 0 ? (fl.n + 255) / 256 : 1), dim3(256), 0, s, L, theta,
                       fl.act, fl.n, rt);
    TDI_HIP(hipGetLastError());
    return TDI_OK;
}

// The vertices of the listed frames, from the model's mean or (mean64) a base shape that already
// holds the identity, then their albedos when the albedo is fitted.
static int synthesize(const ModelGPU& m, const Layout& L, const FrameGPU* frames, FrameList fl, const float* theta,
                      double* rt, const double* mean64, double* P0, float* P, float4* vproj, hipStream_t s)
{
    const dim3 grid((m.V + SY_VERTS - 1) / SY_VERTS);
    if (fl.n == 1)
        hipLaunchKernelGGL(k_synth_one, dim3((m.V + ONE_VERTS - 1) / ONE_VERTS), dim3(3 * ONE_VERTS), 0, s, m, L, frames, theta,
                           fl.act, rt, mean64, P0, P, vproj);
    else if ((mean64 || L.nid == 0) && L.nexp > 0 && L.nexp <= SY_KMAX)
        hipLaunchKernelGGL(k_synth_tile<true>, grid, dim3(256), 0, s, m, L, frames, theta, fl.act, fl.n, rt, mean64, P0,
                           P, vproj);
    else
        hipLaunchKernelGGL(k_synth_tile<false>, grid, dim3(256), 0, s, m, L, frames, theta, fl.act, fl.n, rt, mean64, P0,
                           P, vproj);
    TDI_HIP(hipGetLastError());
    if (m.alb && L.ntex) return launch_albedo(m, L, fl, theta, const_cast<float*>(m.alb), s);
    return TDI_OK;
}

int launch_landmark_vertices(const ModelGPU& m, const Layout& L, int n, const float* theta, double* rt, double* P0,
                             hipStream_t s)
{
    const int rc = launch_frame_rt(L, all_frames(n), theta, rt, s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_landmark_vertices, dim3(n), dim3(192), 0, s, m, L, theta, P0);
    TDI_HIP(hipGetLastError());
    return TDI_OK;
}

int launch_synthesize(const ModelGPU& m, const Layout& L, const FrameGPU* frames, FrameList fl, const float* theta,
                      double* rt, double* P0, float* P, float4* vproj, hipStream_t s, bool rt_ready)
{
    if (L.K > MAX_UNKNOWNS) {
        set_error("synthesize: K=%d exceeds %d", L.K, MAX_UNKNOWNS);
        return TDI_ERR_ARG;
    }
    const int rc = rt_ready ? TDI_OK : launch_frame_rt(L, fl, theta, rt, s);
    if (rc) return rc;
    return synthesize(m, L, frames, fl, theta, rt, nullptr, P0, P, vproj, s);
}

namespace {

// alb[f][v] = tex_mean[v] + sum_q tex_basis[v][q] beta_q, summed in q order with fmaf as the
// shading's per-pixel loop does, so that both give the same value.  A workgroup owns 64 vertices:
// their basis rows are staged in LDS 128 columns at a time (coalesced row segments), then its four
// wavefronts run the sums of four frames at once, lane = vertex (conflict-free LDS rows, the
// frame's coefficients broadcast); a sum carried over column chunks goes through alb itself.
constexpr int AL_V = 64, AL_Q = 128;

__global__ void __launch_bounds__(256) k_albedo(ModelGPU m, Layout L, const int* __restrict__ act, int n,
                                                 const float* __restrict__ theta, float* __restrict__ alb)
{
    __shared__ float sB[AL_V][AL_Q + 1];
    __shared__ float sbeta[4][AL_Q];
    const int v0 = blockIdx.x * AL_V;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int v = v0 + lane;
    const int nact = fl_count(act, n);
    for (int q0 = 0; q0 < L.ntex; q0 += AL_Q) {
        const int nq = min(AL_Q, L.ntex - q0);
        __syncthreads();   // the previous chunk's staging is no longer read
        for (int e = threadIdx.x; e < AL_V * nq; e += blockDim.x) {
            const int vl = e / nq, q = e - vl * nq;
            sB[vl][q] = v0 + vl < m.V ? m.tex_basis[(size_t)(v0 + vl) * m.tex_ld + q0 + q] : 0.f;
        }
        for (int yi0 = 0; yi0 < nact; yi0 += 4) {
            __syncthreads();
            for (int e = threadIdx.x; e < 4 * nq; e += blockDim.x) {
                const int w = e / nq, q = e - w * nq;
                const int yi = yi0 + w;
                sbeta[w][q] = yi < nact ? theta[(size_t)fl_frame(act, yi) * L.K + L.off_tex + q0 + q] : 0.f;
            }
            __syncthreads();
            const int yi = yi0 + wave;
            if (yi < nact && v < m.V) {
                const int f = fl_frame(act, yi);
                float r = q0 == 0 ? m.tex_mean[v] : alb[(size_t)f * m.V + v];
                for (int q = 0; q < nq; ++q) r = fmaf(sB[lane][q], sbeta[wave][q], r);
                alb[(size_t)f * m.V + v] = r;
            }
        }
    }
}

} // namespace

int launch_albedo(const ModelGPU& m, const Layout& L, FrameList fl, const float* theta, float* alb, hipStream_t s)
{
    if (L.ntex > 512) {
        set_error("albedo: k_tex %d > 512", L.ntex);
        return TDI_ERR_ARG;
    }
    hipLaunchKernelGGL(k_albedo, dim3((m.V + AL_V - 1) / AL_V), dim3(256), 0, s, m, L, fl.act, fl.n, theta, alb);
    TDI_HIP(hipGetLastError());
    return TDI_OK;
}

namespace {

// mean + identity basis x alpha in FP64 for every vertex, alpha of the first listed frame (the
// frames of an identity-stage evaluation share it).
__global__ void __launch_bounds__(256) k_id_shape(ModelGPU m, Layout L, const int* __restrict__ act, int n,
                                                   const float* __restrict__ theta, double* __restrict__ S)
{
    __shared__ float sa[MAXK_LDS];
    if (fl_count(act, n) == 0) return;
    const float* tf = theta + (size_t)fl_frame(act, 0) * L.K + L.off_id;
    for (int k = threadIdx.x; k < L.nid; k += blockDim.x) sa[k] = tf[k];
    __syncthreads();
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= m.V) return;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int r = 3 * v + a;
        double sacc = m.mean[r];
        const float* ib = m.id_basis + (size_t)r * m.id_ld;
        for (int k = 0; k < L.nid; ++k) sacc = fma((double)ib[k], (double)sa[k], sacc);
        S[r] = sacc;
    }
}

} // namespace

int launch_synthesize_shared_id(const ModelGPU& m, const Layout& L, const FrameGPU* frames, FrameList fl,
                                const float* theta, double* rt, double* P0, float* P, float4* vproj, double* idshape,
                                hipStream_t s)
{
    if (L.nid > MAXK_LDS) return launch_synthesize(m, L, frames, fl, theta, rt, P0, P, vproj, s);
    int rc = launch_frame_rt(L, fl, theta, rt, s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_id_shape, dim3((m.V + 255) / 256), dim3(256), 0, s, m, L, fl.act, fl.n, theta, idshape);
    TDI_HIP(hipGetLastError());
    return synthesize(m, L, frames, fl, theta, rt, idshape, P0, P, vproj, s);
}

} // namespace tdi
