// pme.hip -- smooth particle-mesh Ewald, reciprocal part (Essmann et al.,
// J. Chem. Phys. 103, 8577 (1995)), for an orthorhombic box.  The reference
// declares a PME flag (gcmc/cpp/gcmc.h:91) that no kernel reads; these
// kernels give the engine's optional Ewald electrostatics.
//
// Units as calcEnergy (K = 1388.431112 kJ/mol A e^-2):
//   Q(k)   = sum_i q_i W_i(k)        order-4 cardinal B-spline weights W
//   G(m)   = K/(pi V) exp(-pi^2 |m~|^2/beta^2)/|m~|^2 B(m),  G(0) = 0
//            m~ = (m1'/L1, m2'/L2, m3'/L3), m' the signed frequency,
//            B(m) = prod_i 1/|sum_{k=0}^{2} M4(k+1) e^{2 pi i m_i k/K_i}|^2
//   Phi    = IFFT(G . FFT(Q))         (unnormalised inverse)
//   E_rec  = 1/2 sum_k Q(k) Phi(k) = 1/2 sum_m G(m) |FFT(Q)(m)|^2
//   phi(r) = sum_k W_r(k) Phi(k)      reciprocal potential at r (per unit charge)
//
// The charge grid accumulates in 32.32 fixed point (int64 atomics): sums are
// exact and order independent, so a run is reproducible and removing a
// charge (spreading -q at the same point) cancels it exactly.
//
// Kernels (HBM / atomic bound; no MFMA -- not a dense contraction):
//   k_pme_spread    a wave per charge, each lane one of its 64 grid points: few
//                   charges, or a list whose length only the GPU knows
//   k_pme_bin, k_pme_bin_scan, k_pme_bin_sort, k_pme_spread_tiles
//                   many charges: sorted by grid tile, each tile summed in
//                   LDS by the one workgroup that owns its points
//   k_pme_tofloat   fixed-point grid -> FP32 grid for the FFT
//   k_pme_convolve  X *= G over the half spectrum, energy terms (FP64 block
//                   sums, added up by k_pme_energy)
//   k_pme_gather    16 lanes per point, each one z row of 4 points of Phi
// The FFTs are hipFFT R2C / C2R plans on the caller's stream.
#include <hip/hip_runtime.h>
#include <hipfft/hipfft.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "../../include/pygcmc_hip.h"
#include "pme_spline.h"

namespace gcmc_internal {
int set_error(int code, const std::string &msg);
}

namespace gcmc_pme_k {

constexpr double KC = 1388.431112;

struct Geo {
    int K[3];
    float L[3];
};

using gcmc_spline::spline4;
using gcmc_spline::scaled;

constexpr double FIX = 4294967296.0;   // 2^32

// A charge's weights along the three axes.
struct Spline3 {
    int f[3];
    float w[3][4];
};

__device__ inline Spline3 splines(const float4 a, const Geo &g)
{
    Spline3 s;
    spline4(scaled(a.x, g.L[0], g.K[0]), s.f[0], s.w[0]);
    spline4(scaled(a.y, g.L[1], g.K[1]), s.f[1], s.w[1]);
    spline4(scaled(a.z, g.L[2], g.K[2]), s.f[2], s.w[2]);
    return s;
}

using gcmc_spline::pick4;

// The fixed-point term rint(w01 w2 2^32) of one grid point.  Adding 1.5 2^52 puts
// the rounded integer into the low bits of the sum (round half to even, as the
// conversion rounds), exact below 2^51: a quarter of the instructions of the
// 64-bit conversion, which larger charges take.
__device__ inline unsigned long long fixed_term(float w01, float w2)
{
    const float x = w01 * w2;
    constexpr double MAGIC = 6755399441055744.0;   // 1.5 2^52
    if (fabsf(x) < 262144.0f)
        return (unsigned long long)(__double_as_longlong(fma((double)x, FIX, MAGIC)) - __double_as_longlong(MAGIC));
    return (unsigned long long)__double2ll_rn((double)x * FIX);
}

// n charges, or *count of them when count is not null (n = capacity): a wave
// per charge, the grid's waves taking them in turn; lane (i0, i1, i2) adds its point's term.  A chain of 64 atomics
// per thread (one thread per charge) left a few thousand charges to a few
// waves: 8,111 charges took 33 us that way, 10 us this way.
__global__ __launch_bounds__(256) void k_pme_spread(int n, const int *count, const float4 *xyzq, Geo g,
                                                    unsigned long long *Q)
{
    const int lane = threadIdx.x & 63, i0 = lane >> 4, i1 = (lane >> 2) & 3, i2 = lane & 3;
    if (count) n = min(n, *count);
    for (long long i = blockIdx.x * 4ll + (threadIdx.x >> 6); i < n; i += gridDim.x * 4ll) {
        const float4 a = xyzq[i];
        if (a.w == 0.0f) continue;
        const Spline3 s = splines(a, g);
        int k0 = s.f[0] - i0, k1 = s.f[1] - i1, k2 = s.f[2] - i2;
        k0 += k0 < 0 ? g.K[0] : 0;
        k1 += k1 < 0 ? g.K[1] : 0;
        k2 += k2 < 0 ? g.K[2] : 0;
        const float w01 = a.w * pick4(s.w[0], i0) * pick4(s.w[1], i1);
        atomicAdd(Q + ((size_t)k0 * g.K[1] + k1) * g.K[2] + k2, fixed_term(w01, pick4(s.w[2], i2)));
    }
}

// ---- many charges: sorted by tile -------------------------------------------
// Scattered 64-bit atomics run at about 23 G/s on this card whatever the grid,
// so 300,000 charges' 19.2 M adds took 837 us.  Here a tile of 8 x 8 x 16 points
// belongs to one workgroup, which adds the terms that fall into it in LDS and
// writes its points back with plain coalesced stores: 85 us in all (bin 16,
// scan 6, sort 8, tiles 55, bound by the 64-bit LDS adds).  A charge touches points
// f - 3 .. f along each axis, so a tile's charges lie in its own bin and in the
// next bin along each axis (modulo the box): eight bins.
constexpr int TS0 = 8, TS1 = 8, TS2 = 16, TPTS = TS0 * TS1 * TS2;

struct Tiles {
    int n[3], total;
};

// Tiles' counters lie a cache line apart: atomics on one line run one after
// another (32 us instead of 16 for 300,000 charges when packed).
constexpr int CPAD = 16;

// A sorted charge: offsets in its grid cell, charge, and the cell.
struct Placed {
    float t[3], q;
    int f[3], pad;
};

__device__ inline Placed placed(const float4 a, const Geo &g)
{
    Placed p;
    p.f[0] = gcmc_spline::base4(scaled(a.x, g.L[0], g.K[0]), p.t[0]);
    p.f[1] = gcmc_spline::base4(scaled(a.y, g.L[1], g.K[1]), p.t[1]);
    p.f[2] = gcmc_spline::base4(scaled(a.z, g.L[2], g.K[2]), p.t[2]);
    p.q = a.w;
    p.pad = 0;
    return p;
}

__device__ inline int tile_of(const int f[3], const Tiles &t)
{
    return ((f[0] / TS0) * t.n[1] + f[1] / TS1) * t.n[2] + f[2] / TS2;
}

// tile and rank within the tile of every charge (charges of zero get none)
__global__ __launch_bounds__(256) void k_pme_bin(int n, const float4 *xyzq, Geo g, Tiles t, int *count, int2 *where)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float4 a = xyzq[i];
    int tile = -1, rank = 0;
    if (a.w != 0.0f) {
        const Placed p = placed(a, g);
        tile = tile_of(p.f, t);
        rank = atomicAdd(&count[(size_t)tile * CPAD], 1);
    }
    where[i] = make_int2(tile, rank);
}

// exclusive scan of the tiles' counts (one workgroup), counts cleared for the
// next call
__global__ __launch_bounds__(1024) void k_pme_bin_scan(int total, int *count, int *start)
{
    __shared__ int part[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int base = 0;
    for (int b = 0; b < total; b += 1024) {
        const int i = b + tid;
        const int v = i < total ? count[(size_t)i * CPAD] : 0;
        int x = v;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int y = __shfl_up(x, off, 64);
            if (lane >= off) x += y;
        }
        if (lane == 63) part[wave] = x;
        __syncthreads();
        int before = 0, all = 0;
        for (int w = 0; w < 16; ++w) {
            const int p = part[w];
            before += w < wave ? p : 0;
            all += p;
        }
        if (i < total) {
            start[i] = base + before + x - v;
            count[(size_t)i * CPAD] = 0;
        }
        base += all;
        __syncthreads();
    }
    if (tid == 0) start[total] = base;
}

__global__ __launch_bounds__(256) void k_pme_bin_sort(int n, const float4 *xyzq, Geo g, const int2 *where,
                                                      const int *start, Placed *sorted)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int2 w = where[i];
    if (w.x >= 0) sorted[start[w.x] + w.y] = placed(xyzq[i], g);
}

// One workgroup per tile: the charges of its bins one per thread, those that
// reach the tile queued in LDS, then 16 lanes per queued charge add its terms
// in LDS (each lane one z row), and at the end Q += tile.  Integer sums: the
// result does not depend on the order.  (Without the queue, every one of a
// charge's 16 lanes repeated its weights for each of the eight tiles that look
// at it: 280 us for 300,000 charges.)
__global__ __launch_bounds__(256) void k_pme_spread_tiles(const Placed *sorted, const int *start, Geo g, Tiles t,
                                                          unsigned long long *Q)
{
    // rows of 17: a charge's 16 rows fall on 16 different pairs of banks (rows of
    // 16 put them on two)
    constexpr int ROW = TS2 + 1;
    __shared__ unsigned long long acc[TS0 * TS1 * ROW];
    __shared__ float qw[256][13];   // q w0[4], w1[4], w2[4], (13: no bank conflicts)
    __shared__ int qa[256];         // cell relative to the tile, 10 bits per axis
    __shared__ int nq, rs[28], rb[28];
    const int tid = threadIdx.x;
    int b = blockIdx.x;
    const int t2 = b % t.n[2];
    b /= t.n[2];
    const int t1 = b % t.n[1], t0 = b / t.n[1];
    const int o[3] = {t0 * TS0, t1 * TS1, t2 * TS2};
    const int m[3] = {min(TS0, g.K[0] - o[0]), min(TS1, g.K[1] - o[1]), min(TS2, g.K[2] - o[2])};
    // the tile's bins (rs: first charge, rb: charges in the bins before), its
    // own and the next along each axis, modulo the box; an axis of one tile has
    // only that one.  Where the last tile is shorter than three points, charges
    // of the first tile reach past it, so the tile before it reads one more.
    if (tid < 64) {
        const int e[3] = {tid / 9, tid / 3 % 3, tid % 3}, q[3] = {t0, t1, t2}, ts[3] = {TS0, TS1, TS2};
        int c[3];
        bool there = tid < 27;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            c[d] = e[d] == 0 ? q[d] : (e[d] == 1 ? (q[d] + 1) % t.n[d] : 0);
            there &= e[d] == 0 || (e[d] == 1 && t.n[d] > 1) ||
                     (e[d] == 2 && t.n[d] > 2 && g.K[d] - (t.n[d] - 1) * ts[d] < 3 && q[d] == t.n[d] - 2);
        }
        int s0 = 0, v = 0;
        if (there) {
            const int bin = (c[0] * t.n[1] + c[1]) * t.n[2] + c[2];
            s0 = start[bin];
            v = start[bin + 1] - s0;
        }
        int x = v;   // charges of this bin and the bins before it
#pragma unroll
        for (int off = 1; off < 32; off <<= 1) {
            const int y = __shfl_up(x, off, 64);
            if (tid >= off) x += y;
        }
        if (tid < 27) {
            rs[tid] = s0;
            rb[tid] = x - v;
        }
        if (tid == 26) rb[27] = x;
        if (tid == 0) nq = 0;
    }
    for (int p = tid; p < TS0 * TS1 * ROW; p += 256) acc[p] = 0ull;
    __syncthreads();
    const int total = rb[27];
    if (total == 0) return;
    const int sub = tid & 15, i0 = sub >> 2, i1 = sub & 3;
    // this thread's charge of the batch at c0, loaded while the batch before is added
    auto charge = [&](int c, Placed &p) {
        if (c >= total) return;
        int k = 0;
        while (c >= rb[k + 1]) ++k;
        p = sorted[rs[k] + (c - rb[k])];
    };
    Placed next;
    charge(tid, next);
    for (int c0 = 0; c0 < total; c0 += 256) {
        const Placed p = next;
        charge(c0 + 256 + tid, next);
        if (c0 + tid < total) {
            int a[3];
            bool in = true;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                a[d] = p.f[d] - o[d];
                a[d] += a[d] < 0 ? g.K[d] : 0;
                in &= a[d] < m[d] + 3 || g.K[d] < m[d] + 3;
            }
            if (in) {
                float w[3][4];
#pragma unroll
                for (int d = 0; d < 3; ++d) gcmc_spline::weights4(p.t[d], w[d]);
                const int e = atomicAdd(&nq, 1);
                // a cell behind the tile's end is at most 2 points past it (or K
                // is below 19): 10 bits hold it
                qa[e] = a[0] | a[1] << 10 | a[2] << 20;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    qw[e][j] = p.q * w[0][j];
                    qw[e][4 + j] = w[1][j];
                    qw[e][8 + j] = w[2][j];
                }
            }
        }
        __syncthreads();
        const int ne = nq;
        for (int e = tid >> 4; e < ne; e += 16) {
            const int pa = qa[e];
            int k0 = (pa & 1023) - i0, k1 = (pa >> 10 & 1023) - i1;
            k0 += k0 < 0 ? g.K[0] : 0;
            k1 += k1 < 0 ? g.K[1] : 0;
            if (k0 >= m[0] || k1 >= m[1]) continue;
            const float w01 = qw[e][i0] * qw[e][4 + i1];
#pragma unroll
            for (int i2 = 0; i2 < 4; ++i2) {
                int k2 = (pa >> 20) - i2;
                k2 += k2 < 0 ? g.K[2] : 0;
                if (k2 < m[2]) atomicAdd(&acc[(k0 * TS1 + k1) * ROW + k2], fixed_term(w01, qw[e][8 + i2]));
            }
        }
        __syncthreads();
        if (tid == 0) nq = 0;
        __syncthreads();
    }
    for (int p = tid; p < TPTS; p += 256) {
        const int z = p % TS2, y = (p / TS2) % TS1, x = p / (TS2 * TS1);
        const unsigned long long v = acc[p / TS2 * ROW + z];
        if (x < m[0] && y < m[1] && z < m[2] && v != 0ull)
            Q[((size_t)(o[0] + x) * g.K[1] + o[1] + y) * g.K[2] + o[2] + z] += v;
    }
}

__global__ void k_pme_tofloat(const unsigned long long *Qi, float *Q, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) Q[i] = (float)((double)(long long)Qi[i] * (1.0 / FIX));
}

__global__ void k_pme_zero64(unsigned long long *p, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0ull;
}

// the influence function as a spectrum, for a plan's grid kernel
__global__ void k_pme_spectrum(const float *G, hipfftComplex *X, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    hipfftComplex x;
    x.x = G[i];
    x.y = 0.0f;
    X[i] = x;
}

// X: K0 x K1 x (K2/2+1) half spectrum; G same layout (real).  part (when the
// energy is wanted): each workgroup's energy sum, added up by k_pme_energy.  (One
// FP64 atomic per workgroup on a single address: 67 us on 150 x 150 x 120 points
// instead of 7.)
__global__ __launch_bounds__(256) void k_pme_convolve(size_t nh, unsigned K2h, unsigned K2, const float *G, hipfftComplex *X,
                                                      double *part)
{
    __shared__ double red[4];
    double e = 0.0;
    const size_t first = (size_t)blockIdx.x * 256 + threadIdx.x, step = (size_t)gridDim.x * 256;
    unsigned m2 = (unsigned)(first % K2h);   // i modulo K2h, stepped along
    const unsigned dm2 = (unsigned)(step % K2h);
    for (size_t i = first; i < nh; i += step) {
        const float gm = G[i];
        hipfftComplex x = X[i];
        if (part) {
            // entries 0 < m2 < K2/2 stand for two conjugate frequencies
            const double mult = (m2 == 0u || 2u * m2 == K2) ? 1.0 : 2.0;
            e += 0.5 * mult * (double)gm * ((double)x.x * x.x + (double)x.y * x.y);
        }
        x.x *= gm;
        x.y *= gm;
        X[i] = x;
        m2 += dm2;
        m2 -= m2 >= K2h ? K2h : 0u;
    }
    if (!part) return;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) e += __shfl_down(e, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = e;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// *energy = sum of the workgroups' parts (one workgroup, fixed order)
__global__ __launch_bounds__(256) void k_pme_energy(int n, const double *part, double *energy)
{
    __shared__ double red[4];
    double e = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) e += part[i];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) e += __shfl_down(e, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = e;
    __syncthreads();
    if (threadIdx.x == 0) *energy = red[0] + red[1] + red[2] + red[3];
}

// Potential at n points, 64 per workgroup: their weights once per point, kept in
// LDS, then 16 lanes per point, lane (i0, i1) one z row of four grid points -- one
// 16-byte load unless the row wraps -- summed across the lanes.  Bound by the
// lines of Phi that random points touch, 16 each: 60 us for 300,000 points (86
// with one thread per point and 64 separate 4-byte loads), 5 us for 8,111 (13;
// 17 with every lane computing the point's weights for itself).
struct __attribute__((packed, aligned(4))) Row4 {
    float v[4];
};
constexpr int GPTS = 64;

__global__ __launch_bounds__(256) void k_pme_gather(int n, const float *xyz, Geo g, const float *Phi, float *phi)
{
    __shared__ float4 w2s[GPTS];
    __shared__ float w01[GPTS][17];
    __shared__ int3 fs[GPTS];
    const int tid = threadIdx.x, i00 = blockIdx.x * GPTS;
    if (tid < GPTS && i00 + tid < n) {
        const float *x = xyz + 3 * (size_t)(i00 + tid);
        const Spline3 s = splines(make_float4(x[0], x[1], x[2], 0.f), g);
        fs[tid] = make_int3(s.f[0], s.f[1], s.f[2]);
        w2s[tid] = make_float4(s.w[2][0], s.w[2][1], s.w[2][2], s.w[2][3]);
#pragma unroll
        for (int j = 0; j < 16; ++j) w01[tid][j] = s.w[0][j >> 2] * s.w[1][j & 3];
    }
    __syncthreads();
    const int sub = tid & 15, i0 = sub >> 2, i1 = sub & 3;
#pragma unroll
    for (int q = tid >> 4; q < GPTS; q += 16) {
        if (i00 + q >= n) break;   // whole groups of 16 lanes
        const int3 f = fs[q];
        int k0 = f.x - i0, k1 = f.y - i1;
        k0 += k0 < 0 ? g.K[0] : 0;
        k1 += k1 < 0 ? g.K[1] : 0;
        const float *row = Phi + ((size_t)k0 * g.K[1] + k1) * g.K[2];
        Row4 v;   // points f - 3, f - 2, f - 1, f
        if (f.z >= 3) {
            v = *(const Row4 *)(row + f.z - 3);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) v.v[3 - j] = row[f.z - j + (f.z - j < 0 ? g.K[2] : 0)];
        }
        const float4 w2 = w2s[q];
        float r = w01[q][sub] * fmaf(w2.w, v.v[0], fmaf(w2.z, v.v[1], fmaf(w2.y, v.v[2], w2.x * v.v[3])));
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) r += __shfl_xor(r, off, 16);
        if (sub == 0) phi[i00 + q] = r;
    }
}

}  // namespace gcmc_pme_k

struct gcmc_pme {
    gcmc_pme_k::Geo geo{};
    float beta = 0.0f;
    size_t ngrid = 0, nhalf = 0;
    unsigned long long *Qi = nullptr;
    float *Q = nullptr, *Phi = nullptr, *G = nullptr;
    float *Gk = nullptr;   // real-space grid kernel IFFT(G): Phi = Gk (*) Q
    hipfftComplex *X = nullptr;
    hipfftHandle fwd = 0, inv = 0;
    bool have_fwd = false, have_inv = false;
    char *work = nullptr;     // the buffers below
    double *part = nullptr;   // energy sums of k_pme_convolve's workgroups
    // many charges: per-tile counts (zero between calls) and starts, and room
    // for `room` sorted charges; more are spread in pieces of that many, so a
    // call never allocates (it may be captured)
    gcmc_pme_k::Tiles tiles{};
    int *tcount = nullptr, *tstart = nullptr;
    int2 *where = nullptr;
    gcmc_pme_k::Placed *sorted = nullptr;
    int room = 0;
};

namespace {

using namespace gcmc_pme_k;

constexpr int CONV_WGS = 1024;   // workgroups of k_pme_convolve: four per CU, one energy part each

// Charges from which the tiles pay.  A wave per charge takes 4 us + 0.93 ns per
// charge whatever the grid; the tiles take four launches (15 us), 4 ns per tile
// (its counter in the scan, its workgroup) and 0.2 to 0.9 ns per charge where each
// CU has a tile.  In us, a wave per charge / tiles: 16,384 charges on 150 x 150 x 120
// points (2,888 tiles) 19 / 29, 32,768 34 / 32, 300,000 283 / 83; 131,072 charges on
// 256^3 (16,384 tiles) 126 / 115, 65,536 65 / 103; 300,000 on 400^3 (62,500 tiles) 289 /
// 450, a million 964 / 546.  With fewer tiles than CUs the others idle: 65,536 charges
// on 32^3 points (32 tiles) 65 / 336, 131,072 on 45 x 50 x 63 (168) 127 / 196, and on
// 64^3 (256) 126 / 104.
constexpr int TILED_FROM = 24576, TILES_FROM = 256, CHARGES_PER_TILE = 8;

Tiles tiles_of(const int K[3])
{
    Tiles t;
    t.n[0] = (K[0] + TS0 - 1) / TS0;
    t.n[1] = (K[1] + TS1 - 1) / TS1;
    t.n[2] = (K[2] + TS2 - 1) / TS2;
    t.total = t.n[0] * t.n[1] * t.n[2];
    return t;
}

bool tiles_pay(const Tiles &t, int n)
{
    return t.total >= TILES_FROM && n >= TILED_FROM && n / CHARGES_PER_TILE >= t.total;
}

// |b(m)|^2 of the order-4 spline for frequency m of K points
double bmod2(int m, int K)
{
    const double M4[3] = {1.0 / 6.0, 2.0 / 3.0, 1.0 / 6.0};
    double re = 0.0, im = 0.0;
    for (int k = 0; k < 3; ++k) {
        const double a = 2.0 * M_PI * (double)m * k / K;
        re += M4[k] * cos(a);
        im += M4[k] * sin(a);
    }
    return 1.0 / (re * re + im * im);
}

int pme_hip(hipError_t e, const char *what)
{
    return gcmc_internal::set_error(GCMC_E_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

int pme_fft(hipfftResult r, const char *what)
{
    return gcmc_internal::set_error(GCMC_E_HIP, std::string(what) + ": hipFFT status " + std::to_string((int)r));
}

}  // namespace

extern "C" {

int gcmc_pme_destroy(gcmc_pme *p)
{
    if (!p) return 0;
    if (p->have_fwd) hipfftDestroy(p->fwd);
    if (p->have_inv) hipfftDestroy(p->inv);
    if (p->Qi) (void)hipFree(p->Qi);
    if (p->Q) (void)hipFree(p->Q);
    if (p->Gk) (void)hipFree(p->Gk);
    if (p->Phi) (void)hipFree(p->Phi);
    if (p->G) (void)hipFree(p->G);
    if (p->X) (void)hipFree(p->X);
    if (p->work) (void)hipFree(p->work);
    delete p;
    return 0;
}

int gcmc_pme_create(gcmc_pme **out, const int *grid, const float *box, float beta)
{
    if (!out || !grid || !box) return gcmc_internal::set_error(GCMC_E_ARG, "null argument");
    *out = nullptr;
    for (int i = 0; i < 3; ++i) {
        if (grid[i] < 4 || grid[i] > 4096) return gcmc_internal::set_error(GCMC_E_ARG, "PME grid must be 4..4096");
        if (!(box[i] > 0.0f)) return gcmc_internal::set_error(GCMC_E_ARG, "box edges must be positive");
    }
    if (!(beta > 0.0f)) return gcmc_internal::set_error(GCMC_E_ARG, "beta must be positive");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
        return gcmc_internal::set_error(GCMC_E_DEVICE, "no HIP device");
    gcmc_pme *p = new gcmc_pme;
    for (int i = 0; i < 3; ++i) {
        p->geo.K[i] = grid[i];
        p->geo.L[i] = box[i];
    }
    p->beta = beta;
    const int K0 = grid[0], K1 = grid[1], K2 = grid[2], K2h = K2 / 2 + 1;
    p->ngrid = (size_t)K0 * K1 * K2;
    p->nhalf = (size_t)K0 * K1 * K2h;
    hipError_t e = hipMalloc(&p->Qi, p->ngrid * sizeof(unsigned long long));
    if (e == hipSuccess) e = hipMalloc(&p->Q, p->ngrid * sizeof(float));
    if (e == hipSuccess) e = hipMalloc(&p->Gk, p->ngrid * sizeof(float));
    if (e == hipSuccess) e = hipMalloc(&p->Phi, p->ngrid * sizeof(float));
    if (e == hipSuccess) e = hipMalloc(&p->G, p->nhalf * sizeof(float));
    if (e == hipSuccess) e = hipMalloc(&p->X, p->nhalf * sizeof(hipfftComplex));
    p->tiles = tiles_of(grid);
    // a quarter as many charges as grid points: more than water's density on a
    // 1 A grid (0.1 per point); 10 bytes per grid point.  None for grids of few tiles
    const bool tiled = p->tiles.total >= TILES_FROM;
    p->room = tiled ? (int)std::min<size_t>(std::max<size_t>(p->ngrid / 4, TILED_FROM), (size_t)1 << 24) : 0;
    // the work buffers in one allocation
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t o = at;
        at += (bytes + 255) & ~(size_t)255;
        return o;
    };
    const size_t counted = tiled ? (size_t)p->tiles.total : 0, count_bytes = counted * CPAD * sizeof(int);
    const size_t o_part = take(CONV_WGS * sizeof(double)), o_count = take(count_bytes),
                 o_start = take((counted + 1) * sizeof(int)),
                 o_where = take((size_t)p->room * sizeof(int2)), o_sorted = take((size_t)p->room * sizeof(Placed));
    if (e == hipSuccess) e = hipMalloc(&p->work, at);
    if (e == hipSuccess) {
        p->part = (double *)(p->work + o_part);
        p->tcount = (int *)(p->work + o_count);
        p->tstart = (int *)(p->work + o_start);
        p->where = (int2 *)(p->work + o_where);
        p->sorted = (Placed *)(p->work + o_sorted);
        if (tiled) e = hipMemset(p->tcount, 0, count_bytes);
    }
    if (e != hipSuccess) {
        gcmc_pme_destroy(p);
        return pme_hip(e, "PME buffers");
    }
    // influence function on the half spectrum (host, FP64, once)
    std::vector<float> G(p->nhalf);
    const double V = (double)box[0] * box[1] * box[2];
    const double b2 = (double)beta * beta;
    std::vector<double> B0(K0), B1(K1), B2(K2h);
    for (int m = 0; m < K0; ++m) B0[m] = bmod2(m, K0);
    for (int m = 0; m < K1; ++m) B1[m] = bmod2(m, K1);
    for (int m = 0; m < K2h; ++m) B2[m] = bmod2(m, K2);
    for (int a = 0; a < K0; ++a) {
        const double ma = (a <= K0 / 2 ? a : a - K0) / (double)box[0];
        for (int b = 0; b < K1; ++b) {
            const double mb = (b <= K1 / 2 ? b : b - K1) / (double)box[1];
            for (int c = 0; c < K2h; ++c) {
                const double mc = c / (double)box[2];
                const double m2 = ma * ma + mb * mb + mc * mc;
                double g = 0.0;
                if (a || b || c) g = KC / (M_PI * V) * exp(-M_PI * M_PI * m2 / b2) / m2 * B0[a] * B1[b] * B2[c];
                G[((size_t)a * K1 + b) * K2h + c] = (float)g;
            }
        }
    }
    e = hipMemcpy(p->G, G.data(), p->nhalf * sizeof(float), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        gcmc_pme_destroy(p);
        return pme_hip(e, "PME influence function");
    }
    hipfftResult r = hipfftPlan3d(&p->fwd, K0, K1, K2, HIPFFT_R2C);
    if (r != HIPFFT_SUCCESS) {
        gcmc_pme_destroy(p);
        return pme_fft(r, "PME forward plan");
    }
    p->have_fwd = true;
    r = hipfftPlan3d(&p->inv, K0, K1, K2, HIPFFT_C2R);
    if (r != HIPFFT_SUCCESS) {
        gcmc_pme_destroy(p);
        return pme_fft(r, "PME inverse plan");
    }
    p->have_inv = true;
    // grid kernel: the potential grid of a unit charge at grid point 0
    hipLaunchKernelGGL(k_pme_spectrum, dim3((unsigned)((p->nhalf + 255) / 256)), dim3(256), 0, nullptr,
                       (const float *)p->G, p->X, p->nhalf);
    e = hipGetLastError();
    if (e != hipSuccess) {
        gcmc_pme_destroy(p);
        return pme_hip(e, "PME grid kernel");
    }
    r = hipfftExecC2R(p->inv, p->X, p->Gk);
    if (r == HIPFFT_SUCCESS && hipDeviceSynchronize() != hipSuccess) r = HIPFFT_EXEC_FAILED;
    if (r != HIPFFT_SUCCESS) {
        gcmc_pme_destroy(p);
        return pme_fft(r, "PME grid kernel");
    }
    *out = p;
    return 0;
}

int gcmc_pme_clear(gcmc_pme *p, void *stream)
{
    if (!p) return gcmc_internal::set_error(GCMC_E_ARG, "null PME plan");
    hipLaunchKernelGGL(k_pme_zero64, dim3((unsigned)((p->ngrid + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       p->Qi, p->ngrid);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : pme_hip(e, "PME clear");
}

int gcmc_pme_spread(gcmc_pme *p, int n, const float *xyzq, void *stream)
{
    if (!p || n < 0 || (n > 0 && !xyzq)) return gcmc_internal::set_error(GCMC_E_ARG, "bad PME spread arguments");
    if (n == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const float4 *q = (const float4 *)xyzq;
    int o = 0;
    while (o < n && tiles_pay(p->tiles, n - o)) {
        const int m = std::min(n - o, p->room);
        const unsigned nb = (unsigned)((m + 255) / 256);
        hipLaunchKernelGGL(k_pme_bin, dim3(nb), dim3(256), 0, s, m, q + o, p->geo, p->tiles, p->tcount, p->where);
        hipLaunchKernelGGL(k_pme_bin_scan, dim3(1), dim3(1024), 0, s, p->tiles.total, p->tcount, p->tstart);
        hipLaunchKernelGGL(k_pme_bin_sort, dim3(nb), dim3(256), 0, s, m, q + o, p->geo,
                           (const int2 *)p->where, (const int *)p->tstart, p->sorted);
        hipLaunchKernelGGL(k_pme_spread_tiles, dim3((unsigned)p->tiles.total), dim3(256), 0, s,
                           (const Placed *)p->sorted, (const int *)p->tstart, p->geo, p->tiles, p->Qi);
        o += m;
    }
    if (o < n)
        hipLaunchKernelGGL(k_pme_spread, dim3((unsigned)(((size_t)(n - o) + 3) / 4)), dim3(256), 0, s, n - o,
                           (const int *)nullptr, q + o, p->geo, p->Qi);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : pme_hip(e, "PME spread");
}

int gcmc_host_pme_tiled(int n, const int *grid)
{
    return n > 0 && grid && tiles_pay(tiles_of(grid), n) ? 1 : 0;
}

int gcmc_pme_solve(gcmc_pme *p, double *energy, void *stream)
{
    if (!p) return gcmc_internal::set_error(GCMC_E_ARG, "null PME plan");
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(k_pme_tofloat, dim3((unsigned)((p->ngrid + 255) / 256)), dim3(256), 0, s,
                       (const unsigned long long *)p->Qi, p->Q, p->ngrid);
    hipfftResult r = hipfftSetStream(p->fwd, s);
    if (r == HIPFFT_SUCCESS) r = hipfftSetStream(p->inv, s);
    if (r == HIPFFT_SUCCESS) r = hipfftExecR2C(p->fwd, p->Q, p->X);
    if (r != HIPFFT_SUCCESS) return pme_fft(r, "PME forward FFT");
    const int K2h = p->geo.K[2] / 2 + 1;
    const unsigned wgs = (unsigned)std::min<size_t>((p->nhalf + 255) / 256, CONV_WGS);
    hipLaunchKernelGGL(k_pme_convolve, dim3(wgs), dim3(256), 0, s, p->nhalf, (unsigned)K2h,
                       (unsigned)p->geo.K[2], (const float *)p->G, p->X, energy ? p->part : nullptr);
    if (energy) hipLaunchKernelGGL(k_pme_energy, dim3(1), dim3(256), 0, s, (int)wgs, (const double *)p->part, energy);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pme_hip(e, "PME convolve");
    r = hipfftExecC2R(p->inv, p->X, p->Phi);
    if (r != HIPFFT_SUCCESS) return pme_fft(r, "PME inverse FFT");
    return 0;
}

int gcmc_pme_gather(gcmc_pme *p, int n, const float *xyz, float *phi, void *stream)
{
    if (!p || n < 0 || (n > 0 && (!xyz || !phi))) return gcmc_internal::set_error(GCMC_E_ARG, "bad PME gather arguments");
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_pme_gather, dim3((unsigned)(((size_t)n + GPTS - 1) / GPTS)), dim3(256), 0, (hipStream_t)stream, n, xyz, p->geo,
                       (const float *)p->Phi, phi);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : pme_hip(e, "PME gather");
}

}  // extern "C"

namespace gcmc_internal {
// for the engine's Ewald mode: potential grid, grid shape, spread of a
// device-counted list
const float *pme_phi(const gcmc_pme *p) { return p->Phi; }
const float *pme_kernel(const gcmc_pme *p) { return p->Gk; }
void pme_grid(const gcmc_pme *p, int K[3])
{
    for (int i = 0; i < 3; ++i) K[i] = p->geo.K[i];
}
int pme_spread_counted(gcmc_pme *p, int cap, const int *count, const float4 *xyzq, hipStream_t s)
{
    if (cap > 0)
        hipLaunchKernelGGL(gcmc_pme_k::k_pme_spread, dim3(std::min((cap + 3) / 4, 256)), dim3(256), 0, s, cap, count, xyzq, p->geo,
                           p->Qi);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : pme_hip(e, "PME spread");
}
}  // namespace gcmc_internal
