// adjoint_kernels.h -- interaction energy of given fragment poses with the
// environment of a replica, and its derivatives with respect to the fragment
// atom coordinates and to per-type parameters.  No counterpart in the
// reference (which has no gradients); the energy is calcEnergy's
// (gcmc/cpp/gcmc_energy.h:142-204: group-centre cutoff, LJ + Coulomb).
//
// Parameters per atom type t (all types of the pair table's column list):
//   eps[t]   CHARMM epsilon, kcal/mol   -> epsilon_t = 4.184 |eps[t]| kJ/mol
//   rmin[t]  CHARMM Rmin/2, A           -> sigma_t = rmin[t] 2^(5/6) / 10 nm
//   dq[t]    charge shift added to every atom of type t (fragment and
//            environment), e
// combined per pair as sigma = (sigma_a + sigma_b)/2, epsilon =
// sqrt(epsilon_a epsilon_b) (gcmc/python/simulation.py:63-72).  With dq = 0
// and the parameters the pair table was built from, the energy equals the
// engine's trial energy.
//
// One wave per pose (four share one when there are few): the candidate scan is
// the energy path's; the pair pass keeps per-fragment-atom gradient sums in
// registers (one lane per environment atom, fragment atoms unrolled, ordered by
// type so that a table entry and 1/sigma serve all atoms of a type), adds
// environment-type terms once per environment atom to LDS accumulators, and
// writes, per pose, dE/dx [nf][3] and the per-type derivatives [3][Y] (dq, eps,
// rmin).  FP32 terms, those of the derivatives inside sigma in FP64; the energy and
// the type sums in LDS accumulate in FP64, a lane's share of an atom's sums in FP32
// (all sums in FP32 left some eps gradients 1.3e-6 off 64 bits where four waves'
// shorter sums had been 6e-7 off), the charge derivatives' from batch to batch in
// FP64 (2,100 poses of nine species, five systems each: 1.30e-7 off 64 bits in the
// geometric mean, 1.51e-7 with one FP32 sum per lane and pose; no time).
// Bound by issue at low residency: the registers hold six sums per fragment atom,
// 116 in all for up to 4 atoms (four waves per SIMD), 161 for 8 (three), 205 for 12
// (two), 256 for 20 (one).
#pragma once

#include "engine_kernels.h"

namespace gcmc {

constexpr double SIGMA_PER_RMINHALF_D = 0.17817974362806785;  // 2^(5/6) / 10
constexpr float SIGMA_PER_RMINHALF = (float)SIGMA_PER_RMINHALF_D;

struct AdjLds {
    float4 *tab;    // [X*Y] (100 sigma^2 hi, 4 epsilon, 100 sigma^2 lo, 0) from the per-type parameters
    float *dq;      // [Y]
    float *inv2e;   // [Y] 1 / (2 |eps|), 0 where eps = 0
    double *gq, *ge, *gr; // [Y] per-type derivative sums of this wave's pose
    float *red;     // [5*MAXF] per-fragment-atom sums of a shared pose
};

// the tables, then per pose in hand the type sums and the per-atom sums
__host__ __device__ inline int adj_pose_bytes(int Y) { return (24 * Y + 4 * 5 * MAXF + 15) & ~15; }
__host__ __device__ inline int adj_lds_bytes(int X, int Y, int poses)
{
    auto up = [](int x) { return (x + 15) & ~15; };
    return up(16 * X * Y) + 2 * up(4 * Y) + poses * adj_pose_bytes(Y);
}

// own: which of the workgroup's poses these sums are for
__device__ inline AdjLds adj_carve(char *b, int X, int Y, int own)
{
    auto up = [](int x) { return (x + 15) & ~15; };
    AdjLds A;
    A.tab = (float4 *)b; b += up(16 * X * Y);
    A.dq = (float *)b; b += up(4 * Y);
    A.inv2e = (float *)b; b += up(4 * Y);
    b += own * adj_pose_bytes(Y);
    A.gq = (double *)b; b += 8 * Y;
    A.ge = (double *)b; b += 8 * Y;
    A.gr = (double *)b; b += 8 * Y;
    A.red = (float *)b;
    return A;
}

template <int NF>
struct AdjPass {
    AdjLds A;
    int spi, nf;
    double acc;
    float gx[NF], gy[NF], gz[NF], sr[NF], se[NF], sq[NF];   // in the order of Species::slot
    double qsum;                                            // lane f: the batches' sums of sq[f]

    __device__ __forceinline__ void run(CRep &C, const Lds &L, const WaveLds &W, int g, int At)
    {
        const int lane = threadIdx.x & 63;
        CSpecies &F = species_of(C, spi);
        const auto atom = gbl(C.atom);
        const auto atype = gbl(C.atype);
        const float4 *fs = (const float4 *)W.fragd;
        const float Lx = C.L[0], Ly = C.L[1], Lz = C.L[2];
        const float ix = C.invL[0], iy = C.invL[1], iz = C.invL[2];
        const bool mapped = At <= WL_ATOMS;
        int carry = 0;
        float4 an;
        int tn;
        auto fetch = [&](int base) {
            const int t = base + lane, tq = min(t, At - 1);
            int slot;
            if (mapped) {
                slot = max(wave_scan_max(W.amap[t]), carry);
                carry = __builtin_amdgcn_readlane(slot, 63);
            } else {
                slot = bsearch_off(W.goff, g, tq);
            }
            const int a = W.gdel[slot] + tq;
            an = atom[a];
            tn = atype[a];
        };
        fetch(0);
        for (int base = 0; base < At; base += 64) {
            const float4 at = an;
            const int ty = tn;
            if (base + 64 < At) fetch(base + 64);
            if (base + lane >= At) continue;
            const float qa = at.w + A.dq[ty];
            float tr = 0.f, te = 0.f, tq = 0.f, isg = 0.f;
            float4 pp = make_float4(0.f, 0.f, 0.f, 0.f);
            int row = -1;
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                if (f < nf) {
                    if (F.srow[f] != row) {
                        row = F.srow[f];
                        pp = A.tab[row + ty];
                        // 1/sigma_pair = 10/sqrt(pp.x), nm^-1
                        isg = pp.x > 0.0f ? 10.0f * __builtin_amdgcn_rsqf(pp.x) : 0.0f;
                    }
                    const float4 fr = fs[f];
                    float ex, ey, ez;
                    float dx = two_diff(at.x, fr.x, ex);
                    float dy = two_diff(at.y, fr.y, ey);
                    float dz = two_diff(at.z, fr.z, ez);
                    dx = fmaf(-rintf(dx * ix), Lx, dx);
                    dy = fmaf(-rintf(dy * iy), Ly, dy);
                    dz = fmaf(-rintf(dz * iz), Lz, dz);
                    const float r2h = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
                    const float r2c = fmaf(dz, ez, fmaf(dy, ey, dx * ex));
                    const float r2 = fmaf(2.0f, r2c, r2h);
                    float ir = __builtin_amdgcn_rsqf(r2);
                    ir = ir * fmaf(-0.5f * r2 * ir, ir, 1.5f);
                    const float ir2 = ir * ir;
                    const float rr = __builtin_amdgcn_rcpf(r2);
                    float s2 = pp.x * rr;
                    s2 = fmaf(fmaf(-s2, r2, pp.x) + pp.z, rr, s2);
                    const float s6 = s2 * s2 * s2;
                    const float s12 = s6 * s6;
                    const float lj = pp.y * (s12 - s6);
                    const float el = (fr.w * qa) * ir;
                    acc += (double)(lj + el);
                    // the derivatives' LJ terms; inside sigma, where s^12 carries six times
                    // the rounding of s^2 and one pair can outweigh all others, from FP64
                    float l = lj, h = pp.y * fmaf(2.0f, s12, -s6);   // 4 eps (s^12 - s^6), 4 eps (2 s^12 - s^6)
                    if (s2 > 1.0f) {
                        const double ux = (double)dx + (double)ex, uy = (double)dy + (double)ey,
                                     uz = (double)dz + (double)ez;
                        const double r2d = fma(uz, uz, fma(uy, uy, ux * ux));
                        double q = __builtin_amdgcn_rcp(r2d);
                        q = q * fma(-r2d, q, 2.0);
                        q = q * fma(-r2d, q, 2.0);
                        const double s2d = ((double)pp.x + (double)pp.z) * q, s6d = s2d * s2d * s2d;
                        const double e6 = (double)pp.y * s6d;
                        l = (float)fma(e6, s6d, -e6);
                        h = (float)fma(2.0 * e6, s6d, -e6);
                    }
                    // dE/d(r^2); with d = x_a - x_f, dE/dx_f = -2 dE/d(r^2) d
                    const float dr2 = fmaf(-3.0f, h, -0.5f * el) * ir2;
                    const float gs = -2.0f * dr2;
                    gx[f] = fmaf(gs, dx + ex, gx[f]);
                    gy[f] = fmaf(gs, dy + ey, gy[f]);
                    gz[f] = fmaf(gs, dz + ez, gz[f]);
                    // dE/dsigma_pair = 6 h / sigma_pair;
                    // dsigma_pair/drmin = 2^(5/6)/20 on each side
                    const float ds = 6.0f * h * isg * (0.5f * SIGMA_PER_RMINHALF);
                    sr[f] += ds;
                    tr += ds;
                    // dE/deps[t] = lj / (2 |eps[t]|) on each side
                    se[f] += l;
                    te += l;
                    // dE/dq: K q_a / r to the fragment side (K applied later), K q_f / r here
                    sq[f] = fmaf(qa, ir, sq[f]);
                    tq = fmaf(fr.w, ir, tq);
                }
            }
            atomicAdd(&A.gr[ty], (double)tr);
            atomicAdd(&A.ge[ty], (double)(te * A.inv2e[ty]));
            atomicAdd(&A.gq[ty], (double)tq);
        }
        // sq's sums cancel most (charges of both signs), so they go on in FP64 from here:
        // 16 terms of a lane at most are added in FP32
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            if (f < nf) {
                const double x = lane_d(wave_scan_add((double)sq[f]), 63);
                qsum += lane == f ? x : 0.0;
                sq[f] = 0.0f;
            }
        }
    }
};

// sum over the wave, in every lane
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_add_f(float x)
{
    return x + __int_as_float(dpp_i<CTRL, ROWS>(0, __float_as_int(x)));
}
__device__ __forceinline__ float wave_sum_f(float x)
{
    x = dpp_add_f<DPP_SHR1, 0xf>(x);
    x = dpp_add_f<DPP_SHR2, 0xf>(x);
    x = dpp_add_f<DPP_SHR4, 0xf>(x);
    x = dpp_add_f<DPP_SHR8, 0xf>(x);
    x = dpp_add_f<DPP_BC15, 0xa>(x);
    x = dpp_add_f<DPP_BC31, 0xc>(x);
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}

// poses [npose][nf][3], centres [npose][3]; outputs E [npose] (FP64),
// dEdx [npose][nf][3], partial [npose][3][Y] (dq, eps, rmin).  PARTS waves share
// a pose; every workgroup builds the pair table once and takes poses in turn.
template <int NT, int NF, int PARTS>
__global__ __launch_bounds__(NT) void k_adjoint(const Rep *reps, int r, int spi, int npose, const float *centres,
                                               const float *poses, const float *eps_kcal,
                                               const float *rmin_half, const float *dq, double *E,
                                               float *dEdx, float *partial, LdsLayout lay, int adj_off)
{
    extern __shared__ __align__(16) char smem[];
    constexpr int NW = NT / 64, PER = NW / PARTS;
    const Lds L = carve(smem, lay);
    CRep &C = rep_of(reps, r);
    const int X = C.X, Y = C.Y;
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform_i(tid >> 6), part = wave % PARTS;
    const WaveLds W = wave_lds(L, wave);
    AdjPass<NF> P;
    P.A = adj_carve(smem + adj_off, X, Y, wave / PARTS);
    CSpecies &F = species_of(C, spi);
    const int nf = F.nf;
    P.spi = spi;
    P.nf = nf;
    for (int t = tid; t < Y; t += NT) {
        const float ek = fabsf(eps_kcal[t]);
        P.A.inv2e[t] = ek > 0.0f ? 0.5f / ek : 0.0f;
        P.A.dq[t] = dq ? dq[t] : 0.0f;
    }
    load_species_table(C, L);
    if (tid == 0) L.misc[M_NEXT] = PER;
    // pair entries in FP64, rounded once to FP32 (as a host-built table is)
    for (int q = tid; q < X * Y; q += NT) {
        const int x = q / Y, y = q - x * Y;
        const double sg = 0.5 * ((double)rmin_half[x] + (double)rmin_half[y]) * (double)SIGMA_PER_RMINHALF_D;
        const double ee = 4.184 * 4.184 * fabs((double)eps_kcal[x]) * fabs((double)eps_kcal[y]);
        const double s2 = 100.0 * sg * sg;
        const float hi = (float)s2;
        P.A.tab[q] = make_float4(hi, (float)(4.0 * sqrt(ee)), (float)(s2 - (double)hi), 0.0f);
    }
    __syncthreads();
    // this workgroup's poses; with one wave per pose each takes the next one when
    // it is done
    const int p0 = (int)((long long)npose * blockIdx.x / gridDim.x);
    const int p1 = (int)((long long)npose * (blockIdx.x + 1) / gridDim.x);
    // a pose by one load per lane: 3 nf coordinates, the centre
    auto fetch = [&](int k) {
        const size_t q = (size_t)min(p0 + k, p1 - 1);
        const float *src = poses + q * 3 * nf + lane;
        if (lane >= 60) src = centres + 3 * q + min(lane - 60, 2);
        return lane < 3 * nf || lane >= 60 ? *src : 0.0f;
    };
    int k = wave / PARTS;
    if (p0 >= p1) return;
    float in = fetch(k);
    while (p0 + (PARTS == 1 ? k : k - wave / PARTS) < p1) {
        const int i = p0 + k;
        int kn = k + PER;
        if (PARTS == 1) {
            if (lane == 0) kn = atomicAdd(&L.misc[M_NEXT], 1);
            kn = uniform_i(kn);
        }
        const float v = in;
        in = fetch(kn);
        const float c[3] = {lane_f(v, 60), lane_f(v, 61), lane_f(v, 62)};
        const float px = __shfl(v, min(3 * lane, 63)), py = __shfl(v, min(3 * lane + 1, 63)),
                    pz = __shfl(v, min(3 * lane + 2, 63));
        if (lane < nf) {
            const float kq = dq ? KCOUL_F * (F.tmpl[lane].w + dq[F.ttype[lane]]) : F.kq[lane];
            ((float4 *)W.fragd)[F.slot[lane]] = make_float4(px, py, pz, kq);
        }
        if (part == 0) {
            for (int t = lane; t < 3 * Y; t += 64) P.A.gq[t] = 0.0;
            for (int t = lane; t < 5 * MAXF; t += 64) P.A.red[t] = 0.0f;
        }
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            P.gx[f] = P.gy[f] = P.gz[f] = 0.0f;
            P.sr[f] = P.se[f] = P.sq[f] = 0.0f;
        }
        P.acc = P.qsum = 0.0;
        if (PARTS > 1) __syncthreads();
        wave_sync();
        ScanSums o{};
        NoTicks nt;
        scan_groups(C, L, W, c, c, 1, -1, part, PARTS, P, o, nt);
        // lane f of the first wave: the sums of the atom in place f
        float s[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            if (f < nf) {
                const float v[5] = {P.gx[f], P.gy[f], P.gz[f], P.sr[f], P.se[f]};
#pragma unroll
                for (int k = 0; k < 5; ++k) {
                    const float x = wave_sum_f(v[k]);
                    if (lane == f) s[k] = x;
                }
            }
        }
        PoseSums ps{};
        ps.e[0] = lane_d(wave_scan_add(P.acc), 63);
        // the place's atom (Species::slot is the other way round)
        int a = 0, tf = 0;
        if (lane < nf) {
            for (int b = 0; b < nf; ++b) a = F.slot[b] == lane ? b : a;
            tf = F.ttype[a];
            atomicAdd(&P.A.gq[tf], P.qsum * (double)KCOUL_F);
        }
        if (PARTS > 1) {
            if (lane < nf)
                for (int k = 0; k < 5; ++k) atomicAdd(&P.A.red[5 * lane + k], s[k]);
            team_sum<NT>(L, ps);
            if (lane < nf)
                for (int k = 0; k < 5; ++k) s[k] = P.A.red[5 * lane + k];
        }
        wave_sync();
        if (part == 0 && i < p1) {
            if (lane < nf) {
                float *o = dEdx + ((size_t)i * nf + a) * 3;
                o[0] = s[0];
                o[1] = s[1];
                o[2] = s[2];
                atomicAdd(&P.A.gr[tf], (double)s[3]);
                atomicAdd(&P.A.ge[tf], (double)(s[4] * P.A.inv2e[tf]));
            }
            wave_sync();
            float *pp = partial + (size_t)i * 3 * Y;
            for (int t = lane; t < 3 * Y; t += 64) pp[t] = (float)P.A.gq[t];
            if (lane == 0) E[i] = ps.e[0];
        }
        wave_sync();
        if (PARTS > 1) __syncthreads();
        k = kn;
    }
}

// The backward in one launch, or two when there are many poses (three, with the
// chunks' sums one after another, took 13 us for 64 poses):
//   workgroups 0 .. nscale - 1: grad[p][k] = w[p] dEdx[p][k], 4096 elements each;
//   the others, 64 columns of a chunk of poses each, 16 poses at a time: the sum
//   over the chunk's poses of w[p] partial[p][j] (FP64), to `out` when there is one
//   chunk, else to tmp[chunk][j], which k_adjoint_chunksum adds up.
constexpr int BACK_SCALE = 4096;

template <class W>   // weights are rounded to FP32
__global__ __launch_bounds__(1024) void k_adjoint_back(int npose, int per, int m, int nscale, int nch,
                                                      const float *dEdx, const float *partial, const W *w,
                                                      float *grad, double *tmp, float *out)
{
    __shared__ double red[16][64];
    if ((int)blockIdx.x < nscale) {
        const size_t n = (size_t)npose * per;
#pragma unroll
        for (int k = 0; k < BACK_SCALE; k += 1024) {
            const size_t q = (size_t)blockIdx.x * BACK_SCALE + k + threadIdx.x;
            if (q < n) grad[q] = (w ? (float)w[q / per] : 1.0f) * dEdx[q];
        }
        return;
    }
    const int ncb = (m + 63) / 64, b = blockIdx.x - nscale, ch = b / ncb;
    const int j = (b - ch * ncb) * 64 + (threadIdx.x & 63), pl = threadIdx.x >> 6;
    const int each = (npose + nch - 1) / nch, p0 = ch * each, p1 = min(npose, p0 + each);
    double s = 0.0;
    if (j < m) {
#pragma unroll 4
        for (int p = p0 + pl; p < p1; p += 16) s += (double)(w ? (float)w[p] : 1.0f) * (double)partial[(size_t)p * m + j];
    }
    red[pl][threadIdx.x & 63] = s;
    __syncthreads();
    if (pl == 0 && j < m) {
        double t = 0.0;
#pragma unroll
        for (int q = 0; q < 16; ++q) t += red[q][threadIdx.x & 63];
        if (nch == 1) out[j] = (float)t;
        else tmp[(size_t)ch * m + j] = t;
    }
}

// out[j] = sum over the chunks of tmp[c][j]: 64 columns per workgroup, 16 chunks at
// a time (one thread per column: 8.4 us for 32 chunks)
__global__ __launch_bounds__(1024) void k_adjoint_chunksum(int nch, int m, const double *tmp, float *out)
{
    __shared__ double red[16][64];
    const int j = blockIdx.x * 64 + (threadIdx.x & 63), cl = threadIdx.x >> 6;
    double s = 0.0;
    if (j < m)
        for (int c = cl; c < nch; c += 16) s += tmp[(size_t)c * m + j];
    red[cl][threadIdx.x & 63] = s;
    __syncthreads();
    if (cl == 0 && j < m) {
        double t = 0.0;
#pragma unroll
        for (int q = 0; q < 16; ++q) t += red[q][threadIdx.x & 63];
        out[j] = (float)t;
    }
}

}  // namespace gcmc
