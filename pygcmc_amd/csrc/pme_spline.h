// pme_spline.h -- order-4 cardinal B-spline weights of the PME grid, shared by
// the PME kernels (spread / gather) and the engine's trial energies, so that
// both interpolate the same reciprocal potential.
#pragma once

#include <hip/hip_runtime.h>

namespace gcmc_spline {

// weights at fractional offset t in [0, 1) of the 4 grid points f, f-1, f-2, f-3
__device__ inline void weights4(float t, float w[4])
{
    const float t2 = t * t, t3 = t2 * t;
    const float s = 1.0f - t;
    w[0] = t3 * (1.0f / 6.0f);                                         // M4(t)
    w[1] = (-3.0f * t3 + 3.0f * t2 + 3.0f * t + 1.0f) * (1.0f / 6.0f);  // M4(t+1)
    w[2] = (3.0f * t3 - 6.0f * t2 + 4.0f) * (1.0f / 6.0f);              // M4(t+2)
    w[3] = s * s * s * (1.0f / 6.0f);                                   // M4(t+3)
}

// grid point f = floor(u) and offset t = u - f of a scaled coordinate u in
// [0, K) (scaled() below; a NaN gives point 0): no integer remainder, which
// costs more than the weights
__device__ inline int base4(float u, float &t)
{
    const float fl = floorf(u);
    t = u - fl;
    return fl > 0.0f ? (int)fl : 0;
}

// weights of the 4 grid points f, f-1, f-2, f-3 of scaled coordinate u in [0, K)
__device__ inline void spline4(float u, int &f, float w[4])
{
    float t;
    f = base4(u, t);
    weights4(t, w);
}

// scaled coordinate K * frac(x / L) in [0, K)
__device__ inline float scaled(float x, float L, int K)
{
    float fr = x / L;
    fr -= floorf(fr);
    const float u = fr * (float)K;
    return u >= (float)K ? 0.0f : u;
}

// element i of a 4-vector held in registers (no indexed registers)
__device__ inline float pick4(const float w[4], int i)
{
    const float a = (i & 1) ? w[1] : w[0], b = (i & 1) ? w[3] : w[2];
    return (i & 2) ? b : a;
}

// interpolated potential of grid Phi [K0][K1][K2] at (x, y, z) by 16 lanes (sub =
// lane & 15), each one z row of the 4 x 4; the rows are added in order, so every
// lane has the same value
__device__ inline float gather16(const float *Phi, const int K[3], const float L[3], float x, float y, float z, int sub)
{
    int f0, f1, f2;
    float w0[4], w1[4], w2[4];
    spline4(scaled(x, L[0], K[0]), f0, w0);
    spline4(scaled(y, L[1], K[1]), f1, w1);
    spline4(scaled(z, L[2], K[2]), f2, w2);
    int k0 = f0 - (sub >> 2), k1 = f1 - (sub & 3);
    k0 += k0 < 0 ? K[0] : 0;
    k1 += k1 < 0 ? K[1] : 0;
    const float *row = Phi + ((size_t)k0 * K[1] + k1) * K[2];
    float v[4], r = 0.0f;
#pragma unroll
    for (int i2 = 0; i2 < 4; ++i2) v[i2] = row[f2 - i2 + (f2 - i2 < 0 ? K[2] : 0)];
#pragma unroll
    for (int i2 = 0; i2 < 4; ++i2) r = fmaf(w2[i2], v[i2], r);
    const float w = pick4(w0, sub >> 2) * pick4(w1, sub & 3);
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < 16; ++j) s = fmaf(__shfl(w, j, 16), __shfl(r, j, 16), s);
    return s;
}

// d modulo K for d in [-2 K, 2 K) (no integer remainder: a slab below would
// spend 98 of them, some 4,000 instructions)
__device__ inline int wrapped(int d, int K)
{
    d += d < 0 ? K : 0;
    d += d < 0 ? K : 0;
    return d >= K ? d - K : d;
}

// Potential at x of a unit charge at y as the grid represents it:
// sum_{k, k'} W_x(k) W_y(k') Gk(k - k'), with Gk = IFFT(G) the periodic grid
// kernel.  The weights factor per axis, so the 64 x 64 terms collapse to
// 7 x 7 x 7 offsets d = (f_x - f_y) - (j - 3) with coefficients c_j =
// sum_{i - i' = j - 3} w_x[i] w_y[i'].  `j0` selects one slab of 49 offsets
// along the first axis (callers split the 7 slabs over threads).
__device__ inline float pair_kernel_slab(const float *Gk, const int K[3], const float L[3], const float x[3],
                                         const float y[3], int j0)
{
    int df[3];
    float c[3][7];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        int fx, fy;
        float wx[4], wy[4];
        spline4(scaled(x[a], L[a], K[a]), fx, wx);
        spline4(scaled(y[a], L[a], K[a]), fy, wy);
        df[a] = fx - fy;
#pragma unroll
        for (int j = 0; j < 7; ++j) c[a][j] = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int ii = 0; ii < 4; ++ii) c[a][i - ii + 3] += wx[i] * wy[ii];
    }
    const int d0 = wrapped(df[0] - (j0 - 3), K[0]);
    float c0 = c[0][0];
#pragma unroll
    for (int j = 1; j < 7; ++j) c0 = j == j0 ? c[0][j] : c0;
    int d2[7];
#pragma unroll
    for (int j2 = 0; j2 < 7; ++j2) d2[j2] = wrapped(df[2] - (j2 - 3), K[2]);
    float s = 0.0f;
#pragma unroll
    for (int j1 = 0; j1 < 7; ++j1) {
        const int d1 = wrapped(df[1] - (j1 - 3), K[1]);
        const float *row = Gk + ((size_t)d0 * K[1] + d1) * K[2];
        float r = 0.0f;
#pragma unroll
        for (int j2 = 0; j2 < 7; ++j2) r = fmaf(c[2][j2], row[d2[j2]], r);
        s = fmaf(c[1][j1], r, s);
    }
    return c0 * s;
}

}  // namespace gcmc_spline
