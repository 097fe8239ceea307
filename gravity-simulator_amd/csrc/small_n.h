// small_n.h -- the FP64 direct sum of a few particles inside one workgroup.
//
// For the adaptive integrators' small systems (planets, three bodies) a force
// evaluation is a handful of pairs and the time is the launches around it; a
// whole step then runs in one workgroup, thread 3 k + d holding component d
// of particle k.  Same terms and same order of additions as k_direct_f64, so
// the same bits.
#pragma once

#include <hip/hip_runtime.h>

#include "fp64_inrange.h"

namespace gs {

// Particles one workgroup takes at most: its one CU forms n^2 terms at about
// 1.2e9/s (96 particles: 7.9 us), so 128 take about what the launches of an
// IAS15 evaluation over the whole chip do.  Each caller has its own limit.
constexpr int SN_MAX = 128;
constexpr int SN_TERMS = 2400;  // pair terms in LDS at a time (58 KB)

struct SmallN {
    int n = 0, cols = 0, row = 0;  // cols: sources per tile; row: LDS row of a (target, component)
    int block = 0;
    size_t lds = 0;

    static SmallN plan(int n)
    {
        SmallN s;
        s.n = n;
        s.cols = n * n <= SN_TERMS ? n : SN_TERMS / n;
        s.row = s.cols | 1;  // odd: the lanes' rows start in different banks
        const int want = n * s.cols > 3 * n ? n * s.cols : 3 * n;
        s.block = (want + 63) / 64 * 64;
        if (s.block > 1024) s.block = 1024;
        s.lds = sizeof(double) * (4 * static_cast<size_t>(n) + 3 * static_cast<size_t>(n) * s.row + 64);
        return s;
    }
};

struct SmallNLds {
    double *x, *m, *term, *red;
    __device__ SmallNLds(double *base, const SmallN &s)
        : x(base), m(base + 3 * s.n), term(m + s.n), red(term + 3 * s.n * s.row)
    {
    }
};

// Acceleration of this thread's component (0 for threads past 3 n) at the
// positions w.x, which every thread has written and which may be rewritten
// on return.  Call with the whole workgroup.
__device__ __forceinline__ double small_n_force(const SmallN &s, const SmallNLds &w, double G,
                                                double eps2, bool skip_massless)
{
    const int tid = threadIdx.x, block = blockDim.x;
    const bool g_in = numerator_in_range(G);
    double acc = 0.0;
    __syncthreads();
#pragma unroll 1
    for (int l0 = 0; l0 < s.n; l0 += s.cols) {
        const int cols = min(s.cols, s.n - l0);
        const int dk = block / cols, dc = block - dk * cols;
        int k = tid / cols, c = tid - k * cols;
#pragma unroll 1
        while (k < s.n) {
            const int l = l0 + c;
            const double R0 = w.x[3 * l] - w.x[3 * k];
            const double R1 = w.x[3 * l + 1] - w.x[3 * k + 1];
            const double R2 = w.x[3 * l + 2] - w.x[3 * k + 2];
            const double ms = w.m[l];
            const bool use = k != l && !(skip_massless && ms == 0.0);
            double r2[1] = {use ? R0 * R0 + R1 * R1 + R2 * R2 + eps2 : 1.0};
            double tv[1];
            if (__all(g_in && r2_in_range(r2[0]))) over_r3<1>(G, r2, tv);
            else tv[0] = over_r3_any(G, r2[0]);
            double *row = w.term + 3 * k * s.row + c;
            row[0] = use ? (tv[0] * R0) * ms : 0.0;
            row[s.row] = use ? (tv[0] * R1) * ms : 0.0;
            row[2 * s.row] = use ? (tv[0] * R2) * ms : 0.0;
            k += dk;
            c += dc;
            if (c >= cols) {
                c -= cols;
                k++;
            }
        }
        __syncthreads();
        if (tid < 3 * s.n) {
            const double *row = w.term + tid * s.row;
#pragma unroll 8
            for (int j = 0; j < cols; j++) acc = acc + row[j];
        }
        __syncthreads();
    }
    return acc;
}

// Workgroup maxima of two non-negative values (NaN ignored, as fmax does).
__device__ __forceinline__ void small_n_max2(const SmallNLds &w, double &a, double &b)
{
    for (int o = 32; o > 0; o >>= 1) {
        a = fmax(a, __shfl_xor(a, o));
        b = fmax(b, __shfl_xor(b, o));
    }
    const int wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        w.red[2 * wave] = a;
        w.red[2 * wave + 1] = b;
    }
    __syncthreads();
    a = w.red[0];
    b = w.red[1];
    for (int q = 1; q < waves; q++) {
        a = fmax(a, w.red[2 * q]);
        b = fmax(b, w.red[2 * q + 1]);
    }
    __syncthreads();
}

}  // namespace gs
