// chol.h — Cholesky factorisation and solve of one small matrix by one workgroup of four wavefronts,
// the lower triangle in LDS as 16 x 16 blocks (see k_cholesky in solve.hip for the layout's reasons).
#pragma once

#include "common.h"

namespace tdi {

constexpr int CMAXK = 112;
constexpr int CHB = 16;                          // block edge
constexpr int CHP = CHB + 1;                     // LDS row stride
constexpr int CHN = CHB * CHP;                   // LDS elements per block
constexpr int CHT = CMAXK / CHB;                 // most blocks per side

__device__ __forceinline__ int ch_block(int I, int J) { return (I * (I + 1) / 2 + J) * CHN; }   // I >= J

__device__ __forceinline__ float lane_read(float v, int j)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j));
}
__device__ __forceinline__ double lane_read(double v, int j)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), j),
                            __builtin_amdgcn_readlane(__double2loint(v), j));
}

typedef float ch_v4f __attribute__((ext_vector_type(4)));
typedef double ch_v4d __attribute__((ext_vector_type(4)));
// accumulator element r of lane l: row 4 (l / 16) + r for FP32, l / 16 + 4 r for FP64; column l % 16
__device__ __forceinline__ ch_v4f ch_mma(float a, float b, ch_v4f c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ ch_v4d ch_mma(double a, double b, ch_v4d c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ int ch_row(float, int lane, int r) { return 4 * (lane >> 4) + r; }
__device__ __forceinline__ int ch_row(double, int lane, int r) { return (lane >> 4) + 4 * r; }
template <typename T> struct ChVec;
template <> struct ChVec<float> { typedef ch_v4f type; };
template <> struct ChVec<double> { typedef ch_v4d type; };

// An infinite diagonal entry makes its column of the factor and its unknown zero, where ch_root and ch_div
// would make them NaN: the largest number does it too.
template <typename T>
__device__ __forceinline__ T ch_finite(T x)
{
    const T top = sizeof(T) == 8 ? T(1.7976931348623157e308) : T(3.4028234e38);
    return x > top ? top : x;
}

// The lower blocks of H into LDS, scaled by sdinv on both sides when given; every load of the
// thread (one entry of each block) is issued before the stores.
template <typename T, typename TH>
__device__ __forceinline__ void ch_load(T* A, const TH* __restrict__ Hf, int K, int nT, const float* sdinv)
{
    const int r = threadIdx.x >> 4, c = threadIdx.x & 15;
    TH v[CHT * (CHT + 1) / 2];
#pragma unroll
    for (int I = 0; I < CHT; ++I)
#pragma unroll
        for (int J = 0; J <= I; ++J) {
            if (I >= nT) continue;
            v[I * (I + 1) / 2 + J] = Hf[(size_t)min(CHB * I + r, K - 1) * K + min(CHB * J + c, K - 1)];
        }
#pragma unroll
    for (int I = 0; I < CHT; ++I)
#pragma unroll
        for (int J = 0; J <= I; ++J) {
            if (I >= nT) continue;
            const int i = CHB * I + r, j = CHB * J + c;
            T x = (T)v[I * (I + 1) / 2 + J];
            if (sdinv) x = x * (T)sdinv[i] * (T)sdinv[j];
            if (i >= K || j >= K) x = i == j ? T(1) : T(0);
            if (i == j) x = ch_finite(x);
            A[ch_block(I, J) + r * CHP + c] = x;
        }
}

// s = sqrt(d) and y = 1 / s to an ulp, d positive, finite and normal, on the factorisation's critical path
// (see ch_div).  fill(i) is called after each dependent step i; returns their number.
template <typename F>
__device__ __forceinline__ int ch_root(float d, float& s, float& y, F fill)
{
    y = __builtin_amdgcn_rsqf(d);
    fill(0);
    s = d * y;
    fill(1);
    const float r = fmaf(-s, s, d);
    fill(2);
    s = fmaf(0.5f * y, r, s);
    fill(3);
    const float e = fmaf(-s, y, 1.f);
    fill(4);
    y = fmaf(e, y, y);
    fill(5);
    return 6;
}
template <typename F>
__device__ __forceinline__ int ch_root(double d, double& s, double& y, F fill)
{
    y = __builtin_amdgcn_rsq(d);               // about 24 bits: two Newton steps
    fill(0);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        double e = -d * y;
        fill(1 + 3 * i);
        e = fma(e, y, 1.0);
        fill(2 + 3 * i);
        y = fma(0.5 * y, e, y);
        fill(3 + 3 * i);
    }
    s = d * y;
    fill(7);
    const double r = fma(-s, s, d);
    fill(8);
    s = fma(0.5 * y, r, s);
    fill(9);
    const double e = fma(-s, y, 1.0);
    fill(10);
    y = fma(e, y, y);
    fill(11);
    return 12;
}

// A = L L^T in place; false (for every thread) at a pivot that is not positive.  *sflag: zero for every
// thread at the start.  On false a wavefront may return while another has yet to read *sflag, so
// neither it nor A may be written before the next barrier.
template <typename T>
__device__ __forceinline__ bool ch_factor(T* A, int nT, int* sflag)
{
    typedef typename ChVec<T>::type V4;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, kq = lane >> 4;
    for (int p = 0; p < nT; ++p) {
        if (wave == 0) {
            const int rows = CHB * (nT - p);          // rows of the panel, the diagonal block first
            const bool in0 = lane < rows, in1 = lane + 64 < rows;
            T* r0 = A + ch_block(p + (in0 ? lane >> 4 : 0), p) + l16 * CHP;
            T* r1 = A + ch_block(p + (in1 ? (lane + 64) >> 4 : 0), p) + l16 * CHP;
            T x0[CHB], x1[CHB];
#pragma unroll
            for (int k = 0; k < CHB; ++k) {
                x0[k] = r0[k];
                x1[k] = r1[k];
            }
            bool bad = false;
            // (the block's upper triangle becomes garbage and is never read; ln is opaque so that the
            // comparisons are made here, one instruction each, and not kept over the panels)
            int ln = lane;
            asm volatile("" : "+v"(ln));
            T dg = T(0);
#pragma unroll
            for (int k = 0; k < CHB; ++k) {
                const T d = lane_read(x0[k], k);
                bad = bad || !(d > T(0));
                // between the steps of that chain, the update by the column before (a dependent FP64
                // operation leaves its wavefront's issue slots free); the compiler would put them after it
                auto fill = [&](int i) {
                    const int j = k + 1 + i;
                    if (k > 0 && j < CHB) {
                        const T l = lane_read(x0[k - 1], j);
                        x0[j] = fma(-x0[k - 1], l, x0[j]);
                        x1[j] = fma(-x1[k - 1], l, x1[j]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                };
                T s, inv;
                const int used = ch_root(d, s, inv, fill);
                dg = ln == k ? s : dg;
                const T q0 = x0[k] * inv, q1 = x1[k] * inv;   // ch_div, both rows
                fill(used);
                const T e0 = fma(-s, q0, x0[k]), e1 = fma(-s, q1, x1[k]);
                fill(used + 1);
                x0[k] = fma(e0, inv, q0);
                x1[k] = fma(e1, inv, q1);
#pragma unroll
                for (int i = used + 2; k + 1 + i < CHB; ++i) fill(i);
                // and of this one's, column k + 1's
                if (k + 1 < CHB) {
                    const T l = lane_read(x0[k], k + 1);
                    x0[k + 1] = fma(-x0[k], l, x0[k + 1]);
                    x1[k + 1] = fma(-x1[k], l, x1[k + 1]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            // x1's steps would otherwise move into its stores' branch, after x0's and apart from them
#pragma unroll
            for (int k = 0; k < CHB; ++k) asm volatile("" : "+v"(x1[k]));
#pragma unroll
            for (int k = 0; k < CHB; ++k) {
                if (in0) r0[k] = x0[k];
                if (in1) r1[k] = x1[k];
            }
            if (lane < CHB) r0[lane] = dg;
            if (bad && lane == 0) *sflag = 1;
        }
        __syncthreads();
        if (*sflag) return false;
        int t = 0;
        for (int I = p + 1; I < nT; ++I)
            for (int J = p + 1; J <= I; ++J, ++t) {
                if ((t & 3) != wave) continue;
                T* C = A + ch_block(I, J) + l16;
                const T* a = A + ch_block(I, p) + l16 * CHP + kq;
                const T* b = A + ch_block(J, p) + l16 * CHP + kq;
                V4 acc;
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[r] = C[ch_row(T(0), lane, r) * CHP];
#pragma unroll
                for (int k = 0; k < CHB / 4; ++k) acc = ch_mma(-a[4 * k], b[4 * k], acc);
#pragma unroll
                for (int r = 0; r < 4; ++r) C[ch_row(T(0), lane, r) * CHP] = acc[r];
            }
        __syncthreads();
    }
    return true;
}

// One block of 16 steps of ch_solve: entry j of the lane's half (HI: 64 on) is divided and passed on to
// the entries after (before) it, whose column (row) of the factor is in l0 and l1, zero elsewhere.
template <typename T, typename TB, bool HI, bool BACK>
__device__ __forceinline__ void ch_solve_block(int J, const T* l0, const T* l1, TB d, TB q, TB& b0, TB& b1)
{
#pragma unroll
    for (int s = 0; s < CHB; ++s) {
        const int c = BACK ? CHB - 1 - s : s;
        const TB y = lane_read(ch_div(HI ? b1 : b0, d, q), (CHB * J + c) & 63);
        b0 = fma(-(TB)l0[c], y, b0);
        b1 = fma(-(TB)l1[c], y, b1);
    }
}

// L L^T x = b on one wavefront, in TB arithmetic: lane l holds entries l (b0) and l + 64 (b1).  An entry
// that is done takes products with zero and keeps its value until its division at the end, so a step is
// the division of one entry, its broadcast and the update.
template <typename T, typename TB>
__device__ __forceinline__ void ch_solve(const T* A, int nT, TB& b0, TB& b1)
{
    const int lane = threadIdx.x & 63, l16 = lane & 15;
    const int I0 = min(lane >> 4, nT - 1), I1 = min((lane + 64) >> 4, nT - 1);
    const TB d0 = A[ch_block(I0, I0) + l16 * CHP + l16], d1 = A[ch_block(I1, I1) + l16 * CHP + l16];
    const TB q0 = TB(1) / d0, q1 = TB(1) / d1;
#pragma unroll 1
    for (int J = 0; J < nT; ++J) {
        // column j of the rows below it
        const T* c0 = A + ch_block(max(I0, J), J) + l16 * CHP;
        const T* c1 = A + ch_block(max(I1, J), J) + l16 * CHP;
        T l0[CHB], l1[CHB];
#pragma unroll
        for (int c = 0; c < CHB; ++c) {
            l0[c] = lane > CHB * J + c ? c0[c] : T(0);
            l1[c] = lane + 64 > CHB * J + c ? c1[c] : T(0);
        }
        if (J < 4) ch_solve_block<T, TB, false, false>(J, l0, l1, d0, q0, b0, b1);
        else ch_solve_block<T, TB, true, false>(J, l0, l1, d1, q1, b0, b1);
    }
    b0 = ch_div(b0, d0, q0);
    b1 = ch_div(b1, d1, q1);
#pragma unroll 1
    for (int J = nT - 1; J >= 0; --J) {
        // row j, of the entries before it
        const T* c0 = A + ch_block(J, min(I0, J)) + l16;
        const T* c1 = A + ch_block(J, min(I1, J)) + l16;
        T l0[CHB], l1[CHB];
#pragma unroll
        for (int c = 0; c < CHB; ++c) {
            l0[c] = lane < CHB * J + c ? c0[c * CHP] : T(0);
            l1[c] = lane + 64 < CHB * J + c ? c1[c * CHP] : T(0);
        }
        if (J < 4) ch_solve_block<T, TB, false, true>(J, l0, l1, d0, q0, b0, b1);
        else ch_solve_block<T, TB, true, true>(J, l0, l1, d1, q1, b0, b1);
    }
    b0 = ch_div(b0, d0, q0);
    b1 = ch_div(b1, d1, q1);
}

} // namespace tdi
