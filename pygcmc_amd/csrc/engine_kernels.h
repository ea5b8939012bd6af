// engine_kernels.h -- device phases of one GCMC move and the kernels that
// schedule them.
//
// A move of one replica is three phases, each run by one workgroup of NT
// threads (NT = 256, 512 or 1024, a tuning choice):
//   prep    decode moveArray[step]; pick slots (partial Fisher-Yates);
//           trial centres                      (gcmc_move_*.h host side)
//   item    one trial: build its pose (or old and new pose), scan the cell
//           list, group test, pair energies    (Gmove_*, calcEnergy), by one
//           wave, or by four in moves of few trials
//   accept  grouping of trials, selection, Metropolis in FP64, commit
//           (move_add/del/trn/rot host logic, Gupdate*)
// The plain form launches item and accept kernels per move; the batched form
// runs every replica in one persistent kernel where workgroups of an XCD
// claim items of that XCD's replicas and the workgroup finishing a replica's
// last item runs its accept and prep phases (no grid-wide barrier, replicas
// advance independently).
#pragma once

#include "engine_types.h"
#include "pme_spline.h"

namespace gcmc {

// The buffers a Rep points to are all in device global memory, but a pointer
// read out of a struct is generic to the compiler, and generic (flat) loads
// count against the LDS counter as well: a wait for an LDS read then also
// waits for every outstanding flat load.  gbl() restates the address space so
// the hot loads are global_load / global_store.  (The host pass only parses
// device functions; address space 1 means nothing there.)
#if defined(__HIP_DEVICE_COMPILE__)
template <class T>
using gptr = __attribute__((address_space(1))) T *;
#else
template <class T>
using gptr = T *;
#endif
template <class T>
__device__ __forceinline__ gptr<T> gbl(T *p)
{
    return (gptr<T>)p;
}

// A replica's Rep and species table are never written while kernels run.
// Read through the constant address space, a field at a wave-uniform address
// is a scalar load (scalar data cache) rather than a vector load through the
// texture path that the evaluations' gathers keep busy.
#if defined(__HIP_DEVICE_COMPILE__)
using CRep = const __attribute__((address_space(4))) Rep;
using CSpecies = const __attribute__((address_space(4))) Species;
#else
using CRep = const Rep;
using CSpecies = const Species;
#endif
// The same Rep behind an address the compiler cannot relate to C: fields read
// through it are loaded where they are used (scalar loads), instead of all at
// once ahead of the loops: k_batched (256 threads, FP64 terms) then spills 323
// scalar and 26 vector registers, 190 and 17 this way.
__device__ __forceinline__ CRep &fresh(CRep &C)
{
    CRep *p = &C;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(p));
#endif
    return *p;
}
// The lane index, and a wave-uniform value, as the compiler's own for this use:
// addresses built from them are not kept in registers through the whole kernel.
__device__ __forceinline__ int fresh_lane()
{
    int l = threadIdx.x & 63;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(l));
#endif
    return l;
}
__device__ __forceinline__ int fresh_uniform(int x)
{
    x = __builtin_amdgcn_readfirstlane(x);
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(x));
#endif
    return x;
}
__device__ __forceinline__ CRep &rep_of(const Rep *reps, int r) { return ((CRep *)reps)[r]; }
__device__ __forceinline__ CSpecies &species_of(CRep &C, int s) { return ((CSpecies *)C.sp)[s]; }

// scratch ints of a workgroup (Lds::misc)
enum Misc : int {
    M_TICKS = 74,    // [74, 78)  time of the claimed trials by phase, summed over the waves
    M_GN = 78,       // groups in the batch (select_groups)
    M_NEXT = 79,     // next of the claimed trials (eval_items)
    M_ACC = 80,      // accept: decision / count of accepted
    M_NG = 81,       //         groups
    M_N = 82,        //         species count after the move
    M_CNT = 83,      // batched: items claimed (consecutive, from M_ITEM)
    M_INV = 84,      //          the claim needs an L1 invalidate (cu_acquire_needed)
    M_FOUND = 88,    // batched: replica claimed (-1 none, -2 exit)
    M_ITEM = 89,     //          item claimed
    M_LAST = 90,     //          this workgroup finished the move's last item
    M_NX = 91,       // [91, 97)  next move, loaded during the accept phase:
                     //           end step, move, species count, conf, maxNum, startRes
};

struct Lds {
    char *wave;       // per-wave scratch of evaluations (WaveLds)
    void *team;       // sums of the waves that share a trial
    float4 *pair;
    int4 *spt;
    int *misc;
    int *members;
    double *w, *val;
    int2 *accl;
    uint32_t *adjl;   // adjacency rows staged for the accept phase (null: read C.adj)
    // accept, a batch of groups: member masks, first place of each mask's members
    // and of each group in `members`, lowest values (order_key)
    uint32_t *gmask, *drop;
    uint16_t *goff;
    int *gstart;
    unsigned long long *gmin;
    int *J;
};

__device__ inline Lds carve(char *b, const LdsLayout &l)
{
    Lds s;
    s.wave = b + l.wave;
    s.team = b + l.team;
    s.pair = (float4 *)(b + (l.pair >= 0 ? l.pair : 0));
    s.spt = (int4 *)(b + l.spt);
    s.misc = (int *)(b + l.misc);
    s.members = (int *)(b + l.members);
    s.w = (double *)(b + l.w);
    s.val = (double *)(b + l.val);
    s.accl = (int2 *)(b + l.accl);
    s.adjl = l.adjl >= 0 ? (uint32_t *)(b + l.adjl) : nullptr;
    s.gmask = (uint32_t *)(b + l.gmask);
    s.drop = (uint32_t *)(b + l.drop);
    s.goff = (uint16_t *)(b + l.goff);
    s.gstart = (int *)(b + l.gstart);
    s.gmin = (unsigned long long *)(b + l.gmin);
    s.J = (int *)(b + l.J);
    return s;
}

// A wave's scratch: the cells it scans, the batch of included groups (offset of
// its first atom in the batch << 2 | flags; atom index minus that offset), the
// batch's atom -> group marks, candidate -> cell marks, and up to two poses.
struct WaveLds {
    uint32_t *list;
    int *goff, *gdel;
    uint8_t *amap, *head;
    float4 *frag;      // [2][MAXF] (x, y, z, K q), atom order
    double4 *fragd;    // [2][MAXF] ordered by type: relative to the centre, K q (or float4, absolute)
};

__device__ __forceinline__ WaveLds wave_lds(const Lds &L, int wave)
{
    char *b = L.wave + wave * WL_BYTES;
    WaveLds w;
    w.fragd = (double4 *)b; b += 2 * MAXF * 32;
    w.frag = (float4 *)b; b += 2 * MAXF * 16;
    w.amap = (uint8_t *)b; b += WL_ATOMS;
    w.list = (uint32_t *)b; b += 4 * WL_CELLS;
    w.goff = (int *)b; b += 4 * WL_GROUPS;
    w.gdel = (int *)b; b += 4 * WL_GROUPS;
    w.head = (uint8_t *)b;
    return w;
}

__device__ inline void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// ---- wave-wide scans on DPP (every lane of the wave active) -----------------
// Inclusive scan: Hillis-Steele within each row of 16 lanes (row_shr 1, 2, 4,
// 8), then row 0's last lane into row 1 and row 2's into row 3 (row_bcast:15),
// then lane 31 into rows 2 and 3 (row_bcast:31).  Lanes without a source keep
// the identity.  Register moves between lanes instead of ds_bpermute round
// trips through the LDS crossbar.
enum : int { DPP_SHR1 = 0x111, DPP_SHR2 = 0x112, DPP_SHR4 = 0x114, DPP_SHR8 = 0x118, DPP_BC15 = 0x142, DPP_BC31 = 0x143 };

template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_i(int identity, int v)
{
    return __builtin_amdgcn_update_dpp(identity, v, CTRL, ROWS, 0xf, false);
}

template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_d(double identity, double v)
{
    const long long b = __double_as_longlong(v), o = __double_as_longlong(identity);
    const int lo = __builtin_amdgcn_update_dpp((int)o, (int)b, CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(b >> 32), CTRL, ROWS, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

template <class T, class Op>
__device__ __forceinline__ T wave_scan(T x, T id, Op op)
{
    if constexpr (sizeof(T) == 8) {
        x = op(x, dpp_d<DPP_SHR1, 0xf>(id, x));
        x = op(x, dpp_d<DPP_SHR2, 0xf>(id, x));
        x = op(x, dpp_d<DPP_SHR4, 0xf>(id, x));
        x = op(x, dpp_d<DPP_SHR8, 0xf>(id, x));
        x = op(x, dpp_d<DPP_BC15, 0xa>(id, x));
        x = op(x, dpp_d<DPP_BC31, 0xc>(id, x));
    } else {
        x = op(x, (T)dpp_i<DPP_SHR1, 0xf>((int)id, (int)x));
        x = op(x, (T)dpp_i<DPP_SHR2, 0xf>((int)id, (int)x));
        x = op(x, (T)dpp_i<DPP_SHR4, 0xf>((int)id, (int)x));
        x = op(x, (T)dpp_i<DPP_SHR8, 0xf>((int)id, (int)x));
        x = op(x, (T)dpp_i<DPP_BC15, 0xa>((int)id, (int)x));
        x = op(x, (T)dpp_i<DPP_BC31, 0xc>((int)id, (int)x));
    }
    return x;
}

__device__ __forceinline__ int wave_scan_add(int x)
{
    return wave_scan(x, 0, [](int a, int b) { return a + b; });
}
__device__ __forceinline__ uint32_t wave_scan_add(uint32_t x)
{
    return wave_scan(x, 0u, [](uint32_t a, uint32_t b) { return a + b; });
}
__device__ __forceinline__ double wave_scan_add(double x)
{
    return wave_scan(x, 0.0, [](double a, double b) { return a + b; });
}
// minimum over the wave, in every lane
__device__ __forceinline__ double wave_min(double x)
{
    const double m = wave_scan(x, __builtin_huge_val(), [](double a, double b) { return b < a ? b : a; });
    const long long bm = __double_as_longlong(m);
    const int lo = __builtin_amdgcn_readlane((int)bm, 63), hi = __builtin_amdgcn_readlane((int)(bm >> 32), 63);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ unsigned wave_min(unsigned x)
{
    const unsigned m = wave_scan(x, 0xFFFFFFFFu, [](unsigned a, unsigned b) { return b < a ? b : a; });
    return (unsigned)__builtin_amdgcn_readlane((int)m, 63);
}

// 64-bit wave values by lane index (idx uniform across the wave)
__device__ inline double lane_d(double v, int idx)
{
    const int i = __builtin_amdgcn_readfirstlane(idx);
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), i);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), i);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ inline unsigned long long lane_u64(unsigned long long v, int idx)
{
    const int i = __builtin_amdgcn_readfirstlane(idx);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, i);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), i);
    return ((unsigned long long)hi << 32) | lo;
}
__device__ inline int lane_i(int v, int idx)
{
    return __builtin_amdgcn_readlane(v, __builtin_amdgcn_readfirstlane(idx));
}
// lane r receives v of the lane whose dst is r (dst a permutation of 0..63)
__device__ inline double permute_d(int dst, double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_ds_permute(dst * 4, (int)(b & 0xffffffffll));
    const int hi = __builtin_amdgcn_ds_permute(dst * 4, (int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// largest e in [0, n) with a[e] >> 2 <= m (a[0] >> 2 = 0 <= m): the group an atom
// of a batch that is too large for its atom map belongs to
__device__ inline int bsearch_off(const int *a, int n, int m)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if ((a[mid] >> 2) <= m) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// a - b = s + e exactly (Knuth TwoSum of a and -b); returns s
__device__ inline float two_diff(float a, float b, float &e)
{
    const float s = a - b;
    const float bv = s - a;
    const float av = s - bv;
    e = (a - av) - (b + bv);
    return s;
}

__device__ __forceinline__ float uniform_f(float x)
{
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}
__device__ __forceinline__ int uniform_i(int x) { return __builtin_amdgcn_readfirstlane(x); }
// lanes below this one whose bit is set
__device__ __forceinline__ int rank_below(unsigned long long bal)
{
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)bal, 0u));
}
__device__ __forceinline__ int wave_scan_max(int x)
{
    return wave_scan(x, 0, [](int a, int b) { return b > a ? b : a; });
}
__device__ __forceinline__ int lane_up(int v, int src) { return __builtin_amdgcn_ds_bpermute(src * 4, v); }

// ---- pair energies of a batch of included groups ----------------------------
// One wave; lane <-> environment atom, U atoms per lane and round, the next
// round's atoms loaded while this one's terms are computed; loop over the
// fragment atoms held in LDS, ordered by type so that the pair-table entry of a
// lane's atom is fetched once per type, not once per fragment atom.  A batch's
// atoms serve one or two poses ("sets": the old and new pose of a translate or
// rotate trial); bit s of a group's flags says that it is within the cutoff of
// pose s's centre.  FP64 terms by default, FP32 terms (fp32_coulomb, Ewald)
// added up in FP64.
// Bound by FP64 issue (about 20 instructions and one FP32 rsq per pair).
enum Terms : int { T_FP64, T_FP32, T_EWALD };   // FP32 terms with plain or Ewald real-space Coulomb

template <bool STAGED, int TM>
struct EnergyPass {
    float x[2], y[2], z[2];   // centres of the poses (uniform)
    int first, nset;          // poses first .. first + nset - 1
    bool wrap;                // image shift per pair (else per environment atom)
    int spi;
    double acc[2];            // this lane's sums

    template <class T>
    __device__ __forceinline__ T entry(CRep &C, const Lds &L, int i) const
    {
        if constexpr (STAGED) return ((const T *)L.pair)[i];
        else return ((gptr<const T>)gbl(C.pair))[i];
    }

    // Every pair term in FP64.  The environment atom's position relative to the
    // trial centre, image-shifted once per atom, and the fragment atom's (W.fragd)
    // are exact differences of FP32 positions (to 2^-53); their difference needs
    // no further image shift when Rep::nowrap holds, else it takes one per pair.
    // 1/r: the FP32 estimate (relative error ~2^-22) and one FP64 Newton step
    // (~1.5 2^-44).  LJ as (A r^-6 - B) r^-6 from the table's A, B; Coulomb's
    // environment charge taken out of the sum.
    template <bool WRAP, int U>
    __device__ __forceinline__ void terms64(CRep &C, const Lds &L, const WaveLds &W, int s, const float4 *at,
                                            const int *ty, const int *fl)
    {
        const double Lx = C.Ld[0], Ly = C.Ld[1], Lz = C.Ld[2], ix = C.invLd[0], iy = C.invLd[1], iz = C.invLd[2];
        const double cx = s ? x[1] : x[0], cy = s ? y[1] : y[0], cz = s ? z[1] : z[0];
        CSpecies &F = species_of(C, spi);
        double ax[U], ay[U], az[U], lj[U], cq[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            ax[u] = (double)at[u].x - cx;
            ay[u] = (double)at[u].y - cy;
            az[u] = (double)at[u].z - cz;
            ax[u] = fma(-rint(ax[u] * ix), Lx, ax[u]);
            ay[u] = fma(-rint(ay[u] * iy), Ly, ay[u]);
            az[u] = fma(-rint(az[u] * iz), Lz, az[u]);
            lj[u] = cq[u] = 0.0;
        }
        const double4 *fd = W.fragd + s * MAXF;
        const int nrun = F.nrun;
        int f = 0, row = F.run_row[0], end = F.run_end[0];
        double4 qn = fd[0];
        double2 pn[U];
#pragma unroll
        for (int u = 0; u < U; ++u) pn[u] = entry<double2>(C, L, row + ty[u]);
        for (int r = 0; r < nrun; ++r) {
            double2 p[U];
            const int stop = end;
#pragma unroll
            for (int u = 0; u < U; ++u) p[u] = pn[u];
            if (r + 1 < nrun) {
                // the next type's entries arrive while this one's atoms are done
                row = F.run_row[r + 1];
                end = F.run_end[r + 1];
#pragma unroll
                for (int u = 0; u < U; ++u) pn[u] = entry<double2>(C, L, row + ty[u]);
            }
            for (; f < stop; ++f) {
                // the next atom's position arrives while this one's terms are computed
                const double4 q = qn;
                qn = fd[f + 1];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    double ux = ax[u] - q.x, uy = ay[u] - q.y, uz = az[u] - q.z;
                    if (WRAP) {
                        ux = fma(-rint(ux * ix), Lx, ux);
                        uy = fma(-rint(uy * iy), Ly, uy);
                        uz = fma(-rint(uz * iz), Lz, uz);
                    }
                    const double r2 = fma(uz, uz, fma(uy, uy, ux * ux));
                    double v = (double)__builtin_amdgcn_rsqf((float)r2);
                    v = v * fma(-0.5 * r2 * v, v, 1.5);
                    const double v2 = v * v, v6 = v2 * v2 * v2;
                    lj[u] = fma(fma(p[u].x, v6, -p[u].y), v6, lj[u]);
                    cq[u] = fma(q.w, v, cq[u]);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const double e = fma((double)at[u].w, cq[u], lj[u]);
            const double m = ((fl[u] >> s) & 1) ? e : 0.0;
            if (s) acc[1] += m;
            else acc[0] += m;
        }
    }

    // FP32 terms (fp32_coulomb, Ewald) from the TwoSum-exact displacement
    template <int U>
    __device__ __forceinline__ void terms32(CRep &C, const Lds &L, const WaveLds &W, int s, const float4 *at,
                                            const int *ty, const int *fl)
    {
        const float Lx = C.L[0], Ly = C.L[1], Lz = C.L[2], ix = C.invL[0], iy = C.invL[1], iz = C.invL[2];
        const float eb = C.ew_beta;
        CSpecies &F = species_of(C, spi);
        const float4 *fs = (const float4 *)(W.fragd + s * MAXF);
        double sum[U];
#pragma unroll
        for (int u = 0; u < U; ++u) sum[u] = 0.0;
        const int nrun = F.nrun;
        int f = 0;
        for (int r = 0; r < nrun; ++r) {
            const int row = F.run_row[r], stop = F.run_end[r];
            float4 pp[U];
#pragma unroll
            for (int u = 0; u < U; ++u) pp[u] = entry<float4>(C, L, row + ty[u]);
            for (; f < stop; ++f) {
                const float4 fr = fs[f];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    // displacement as an exact sum s + e (TwoSum); the image shift
                    // s - n L is exact for |n| <= 1 (Sterbenz)
                    float ex, ey, ez;
                    float dx = two_diff(at[u].x, fr.x, ex);
                    float dy = two_diff(at[u].y, fr.y, ey);
                    float dz = two_diff(at[u].z, fr.z, ez);
                    dx = fmaf(-rintf(dx * ix), Lx, dx);
                    dy = fmaf(-rintf(dy * iy), Ly, dy);
                    dz = fmaf(-rintf(dz * iz), Lz, dz);
                    const float r2h = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
                    const float r2c = fmaf(dz, ez, fmaf(dy, ey, dx * ex));
                    const float r2 = fmaf(2.0f, r2c, r2h);
                    float ir = __builtin_amdgcn_rsqf(r2);
                    ir = ir * fmaf(-0.5f * r2 * ir, ir, 1.5f);     // one Newton step
                    // s^2 = 100 sigma^2 / r^2 to ~0.5 ulp: 100 sigma^2 held exactly as
                    // pp.x + pp.z, quotient with one residual correction.  s^12
                    // multiplies the relative error of s^2 by six, and a rounded
                    // table value would err alike on every pair of a type pair.
                    const float rr = __builtin_amdgcn_rcpf(r2);
                    float s2 = pp[u].x * rr;
                    s2 = fmaf(fmaf(-s2, r2, pp[u].x) + pp[u].z, rr, s2);
                    const float s6 = s2 * s2 * s2;
                    float lj = pp[u].y * fmaf(s6, s6, -s6);        // 4 eps (s^12 - s^6)
                    if (s2 > 1.0f) {
                        // inside sigma s^12 dominates and carries six times the
                        // relative error of r^2: this rare pair's LJ term in FP64,
                        // from the exact displacement
                        const double ux = (double)dx + (double)ex, uy = (double)dy + (double)ey,
                                     uz = (double)dz + (double)ez;
                        const double r2d = fma(uz, uz, fma(uy, uy, ux * ux));
                        double q = __builtin_amdgcn_rcp(r2d);
                        q = q * fma(-r2d, q, 2.0);
                        q = q * fma(-r2d, q, 2.0);
                        const double s2d = ((double)pp[u].x + (double)pp[u].z) * q;
                        const double s6d = s2d * s2d * s2d;
                        sum[u] = fma((double)pp[u].y, fma(s6d, s6d, -s6d), sum[u]);
                        lj = 0.0f;
                    }
                    float el = (fr.w * at[u].w) * ir;              // K q_f q_a / r
                    if (TM == T_EWALD) el *= erfcf(eb * (r2 * ir));           // Ewald real-space part
                    sum[u] += (double)(lj + el);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const double m = ((fl[u] >> s) & 1) ? sum[u] : 0.0;
            if (s) acc[1] += m;
            else acc[0] += m;
        }
    }

    // g groups with A atoms in W's batch
    __device__ __forceinline__ void run(CRep &C0, const Lds &L, const WaveLds &W, int g, int A)
    {
        CRep &C = fresh(C0);
        constexpr int U = 1;   // (two: 56 vector registers spilled in k_batched instead of 17)
        const int lane = fresh_lane();
        const auto atom = gbl(C.atom);
        const auto atype = gbl(C.atype);
        const bool mapped = A <= WL_ATOMS;
        int carry = 0;
        float4 an[U];
        int tn[U], fn[U];
        auto fetch = [&](int base) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int t = base + u * 64 + lane, tq = min(t, A - 1);
                int slot;
                if (mapped) {
                    slot = max(wave_scan_max(W.amap[t]), carry);
                    carry = __builtin_amdgcn_readlane(slot, 63);
                } else {
                    slot = bsearch_off(W.goff, g, tq);
                }
                const int w = W.goff[slot], a = W.gdel[slot] + tq;
                fn[u] = t < A ? w : 0;
                an[u] = atom[a];
                tn[u] = atype[a];
            }
        };
        fetch(0);
        for (int base = 0; base < A; base += 64 * U) {
            float4 at[U];
            int ty[U], fl[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                at[u] = an[u];
                ty[u] = tn[u];
                fl[u] = fn[u];
            }
            if (base + 64 * U < A) fetch(base + 64 * U);
            for (int s = first; s < first + nset; ++s) {
                if constexpr (TM != T_FP64) terms32<U>(C, L, W, s, at, ty, fl);
                else if (wrap) terms64<true, U>(C, L, W, s, at, ty, fl);
                else terms64<false, U>(C, L, W, s, at, ty, fl);
            }
        }
    }
};

// species table in LDS (mobile group id -> atom range)
__device__ inline void load_species_table(CRep &C, const Lds &L)
{
    for (int s = threadIdx.x; s < C.T; s += blockDim.x) {
        CSpecies &F = species_of(C, s);
        L.spt[s] = make_int4(F.startRes, F.maxNum, F.atomBase, F.nf);
    }
}

// the replica's pair table (X x Y entries) into LDS, straight from global
// memory (global_load_lds: no registers); the caller waits (vmcnt) and
// synchronises before the first read
template <int NT>
__device__ inline void stage_pair_table(CRep &C, const Lds &L)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n = C.X * C.Y;
    const auto P = gbl(C.pair);
    for (int b = wave * 64; b < n; b += NT)
        if (b + lane < n) __builtin_amdgcn_global_load_lds((const void *)(P + b + lane), (void *)&L.pair[b], 16, 0, 0);
}

// tables of a replica into LDS, complete for every wave on return
template <int NT, bool STAGED>
__device__ inline void stage_tables(CRep &C, const Lds &L, bool rep, bool tab)
{
    if (rep) load_species_table(C, L);
    if (STAGED && tab) {
        stage_pair_table<NT>(C, L);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    if (rep || (STAGED && tab)) __syncthreads();
}

// The FP32 group test (within, gcmc_math.h) of a wave's lanes at once: without
// branches when no lane is past the shift table (one ballot), else literally.
// (3,000 moves of one system take 79.5 ms, 80.9 with branches per axis, of 64
// systems 123-127 and 129; k_batched spills 190 scalar registers both ways.)
struct GroupCut {
    AxisCut ax[3];
    float r2max;
};
__device__ __forceinline__ GroupCut group_cut(CRep &C)
{
    GroupCut g;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        g.ax[i].L = C.ax[i].L;
        g.ax[i].t[0] = C.ax[i].t[0];
        g.ax[i].t[1] = C.ax[i].t[1];
        g.ax[i].t[2] = C.ax[i].t[2];
    }
    g.r2max = C.r2max;
    return g;
}
__device__ __forceinline__ bool within_lanes(const float c[3], const float4 p, const GroupCut &g)
{
    const float d0 = c[0] - p.x, d1 = c[1] - p.y, d2 = c[2] - p.z;
    const bool far = axis_far(d0, g.ax[0]) | axis_far(d1, g.ax[1]) | axis_far(d2, g.ax[2]);
    float e0 = axis_near(d0, g.ax[0].L, g.ax[0].t[0], g.ax[0].t[1]);
    float e1 = axis_near(d1, g.ax[1].L, g.ax[1].t[0], g.ax[1].t[1]);
    float e2 = axis_near(d2, g.ax[2].L, g.ax[2].t[0], g.ax[2].t[1]);
    if (__builtin_expect(__ballot(far) != 0ull, 0)) {
        e0 = axis_delta(c[0], p.x, g.ax[0]);
        e1 = axis_delta(c[1], p.y, g.ax[1]);
        e2 = axis_delta(c[2], p.z, g.ax[2]);
    }
    return fmaf(e2, e2, fmaf(e1, e1, e0 * e0)) <= g.r2max;
}

// ---- candidate groups over the cell list --------------------------------------
// One wave (or, with parts > 1, wave `part` of several that deal the stencil's
// cells out among themselves): fixed and mobile groups of the stencil cells
// around the trial centre plus the overflow bucket; kept when gid != exclude and
// the FP32 distanceP test passes (gcmc_energy.h:152-191).  With two centres (a
// translation's old and new) a group is kept when it passes either test.
// Included groups are batched in W (slot -> atoms) for P.run.  Needs L.spt.
//
// No barriers: every step is a wave's own.  (With 256 threads per evaluation
// the barriers between the steps, and the rounds of a step that fill a part of
// the threads, left a third of the issue slots: 14.5 us per evaluation and
// workgroup on the 64-system workload.)
struct ScanSums {
    int nin[2], nat[2];       // groups and their atoms within the cutoff, per centre (this lane's)
    uint32_t hash[2];
};

// Time of a trial by phase (device ticks), added up in LDS for the workgroup:
// poses and adjacency, cells and their records, group tests, pair passes.  A read
// of the clock holds a wave up for some 100 ns, about seven times in a share of a
// trial, so one trial in TICKED is timed, picked by a hash of step and trial, and
// counts TICKED times: 400 one-trial moves take 5.40 ms, as without (5.39), 5.58
// with every trial timed.
enum Phase : int { S_POSE, S_LIST, S_TEST, S_PAIRS };
constexpr int TICKED_BITS = 3, TICKED = 1 << TICKED_BITS;
struct Ticks {
    int *sum;         // the workgroup's
    unsigned mark;    // when the present phase began
    bool on;
    __device__ __forceinline__ Ticks(int *s, int step, int t) : sum(s), mark(0u)
    {
        on = ((unsigned)step * 0x9E3779B1u + (unsigned)t * 0x85EBCA77u) >> (32 - TICKED_BITS) == 0u;
        if (on) mark = (unsigned)wall_clock64();
    }
    __device__ __forceinline__ void end(Phase p)
    {
        if (!on) return;
        const unsigned now = (unsigned)wall_clock64();
        if (fresh_lane() == 0) atomicAdd(&sum[p], (int)(now - mark));
        mark = now;
    }
};
struct NoTicks {
    __device__ __forceinline__ void end(Phase) {}
};

template <class Pass, class TK>
__device__ __forceinline__ void scan_groups(CRep &C0, const Lds &L, const WaveLds &W, const float c0[3],
                                            const float c1[3], int ncentre, int exclude, int part, int parts,
                                            Pass &P, ScanSums &o, TK &tk)
{
    CRep &C = fresh(C0);
    const int lane = fresh_lane();
    const bool two = ncentre == 2;
    int home[3];
    // the centres' positions relative to the first one's cell
    float base0[3], base1[3], hp[3];
    cell_coords(C.L, C.start, C.inv_h, C.nc, c0[0], c0[1], c0[2], home);
    {
        float u0[3];
        cell_offset(C.L, C.start, C.cell_h, home, c0[0], c0[1], c0[2], u0);
        stencil_base(u0, C.cell_h, two ? C.prune_wide : C.prune, base0, hp);
        for (int i = 0; i < 3; ++i) {
            const float d = c1[i] - c0[i];
            base0[i] = uniform_f(base0[i]);
            base1[i] = hp[i] == 0.0f ? 0.0f : uniform_f(moved_base(base0[i], d, C.L[i], C.invL[i]));
            home[i] = uniform_i(home[i]) - 128;
        }
    }
    const int nst = two ? C.nst_wide : C.nst, ne = nst + 1;
    int g = 0, A = 0;             // groups and atoms in the batch
    int b = 0, nl = 0, q0 = 0;    // next stencil entry; cells listed, cells taken from the list
    int r0 = 0, T = 0;            // candidates of the listed cells at hand: next, total
    int n = 0, off = 0, fixb = 0, thr = 0, mobb = 0, carry = 0;
    auto clear_map = [&]() { ((int4 *)W.amap)[lane] = make_int4(0, 0, 0, 0); };
    clear_map();
    while (true) {
        // ---- the next 128 candidates
        bool done = false;
        const bool list = r0 >= T;
        if (list && b > 0) tk.end(S_TEST);   // (the first list begins the scan)
        while (r0 >= T) {
            if (q0 >= nl) {
                if (b >= ne) {
                    done = true;
                    break;
                }
                // list the cells that can hold a group within the cutoff
                constexpr int I = WL_CELLS / 64;
                CRep &D = fresh(C);
                const auto stencil = gbl(D.stencil) + (two ? D.nst : 0);
                const int n0 = D.nc[0], n1 = D.nc[1], n2 = D.nc[2];
                const float reach2 = D.prune_r2;
                int code[I];
#pragma unroll
                for (int i = 0; i < I; ++i) {
                    const int e = b + (i * 64 + lane) * parts + part;
                    code[i] = e < nst ? stencil[e] : 0;
                }
                nl = 0;
#pragma unroll
                for (int i = 0; i < I; ++i) {
                    if (b + i * 64 * parts >= ne) continue;
                    const int e = b + (i * 64 + lane) * parts + part;
                    // cells whose box lies beyond rc + slack from the centre hold no
                    // group centre that passes the group test
                    bool live = stencil_cell_near(code[i], base0, hp, reach2);
                    if (two) live |= stencil_cell_near(code[i], base1, hp, reach2);
                    // offsets span at most one box per axis: wrap by one add
                    auto wrap = [](int q, int nq) {
                        const unsigned x = min((unsigned)q, (unsigned)(q + nq));
                        return min(x, x - (unsigned)nq);
                    };
                    const unsigned i0 = wrap(home[0] + (code[i] & 255), n0), i1 = wrap(home[1] + (code[i] >> 8 & 255), n1),
                                   i2 = wrap(home[2] + (code[i] >> 16 & 255), n2);
                    // at most 255 cells per axis: 24-bit products
                    int cell = (int)(__umul24(__umul24(i0, n1) + i1, n2) + i2);
                    live = e < nst ? live : e == nst;     // the last entry: the overflow bucket
                    cell = e < nst ? cell : D.ncell;
                    const unsigned long long bal = __ballot(live);
                    if (live) W.list[nl + rank_below(bal)] = (uint32_t)cell;
                    nl += __popcll(bal);
                }
                b += WL_CELLS * parts;
                q0 = 0;
                wave_sync();
                continue;
            }
            // one listed cell per lane: its fixed records and mobile entries
            int fs = 0, fc = 0, mc = 0;
            mobb = 0;
            if (q0 + lane < nl) {
                CRep &D = fresh(C);
                const auto cellv = gbl(D.cell);
                const int cell = (int)W.list[q0 + lane], last = D.ncell;
                const int2 ci = cellv[cell];
                const int next = cellv[min(cell + 1, last)].x;   // (the overflow bucket has no fixed records)
                fs = ci.x;
                mc = ci.y;
                fc = next - fs;
                mobb = cell == last ? D.ovf_base : cell * D.cap;
            }
            n = fc + mc;
            const int incl = wave_scan_add(n);
            off = incl - n;
            T = __builtin_amdgcn_readlane(incl, 63);
            // candidate m of this chunk: record m + fixb below thr, entry m + mobb from thr on
            fixb = fs - off;
            thr = off + fc;
            mobb -= thr;
            q0 += 64;
            r0 = 0;
            carry = 0;
        }
        if (list) tk.end(S_LIST);
        constexpr int R = 2;
        int2 rr[R];
        int flag[R], pos[R], at[R], ng = 0, tot = 0;
        if (!done) {
            // the cell of each candidate: cells mark their first candidate, a running
            // maximum carries the mark on
            ((uint16_t *)W.head)[lane] = 0;
            wave_sync();
            if (n > 0 && off >= r0 && off < r0 + 64 * R) W.head[off - r0] = (uint8_t)lane;
            wave_sync();
            float4 rec[R];
            bool fixed[R];
            CRep &D = fresh(C);
            const auto fix = gbl(D.fix);
            const auto mob_rec = gbl(D.mob_rec);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int own = max(wave_scan_max(W.head[r * 64 + lane]), carry);
                carry = __builtin_amdgcn_readlane(own, 63);
                const int m = r0 + r * 64 + lane;
                const int fb = lane_up(fixb, own), th = lane_up(thr, own), mb = lane_up(mobb, own);
                fixed[r] = m < th;
                rec[r] = make_float4(0.f, 0.f, 0.f, 0.f);
                rr[r] = make_int2(0, 0);
                if (m < T) {
                    if (fixed[r]) {
                        rec[r] = fix[m + fb].p;
                        rr[r] = fix[m + fb].rng;
                    } else {
                        rec[r] = mob_rec[m + mb];
                    }
                }
            }
            const GroupCut cut = group_cut(D);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float4 p = rec[r];
                const bool valid = r0 + r * 64 + lane < T;
                int gid = __float_as_int(p.w);
                if (valid && !fixed[r]) {
                    const int4 sp = L.spt[gid >> GID_BITS];   // (startRes, maxNum, atomBase, nf)
                    gid &= GID_MASK;
                    rr[r] = make_int2(sp.z + (gid - sp.x) * sp.w, sp.w);
                }
                const bool able = valid && gid != exclude;
                const uint32_t h = group_hash((uint32_t)gid);
                const bool in0 = able && within_lanes(c0, p, cut);
                const bool in1 = two ? able && within_lanes(c1, p, cut) : in0;
                o.nin[0] += in0 ? 1 : 0;
                o.nat[0] += in0 ? rr[r].y : 0;
                o.hash[0] += in0 ? h : 0u;
                if (two) {
                    o.nin[1] += in1 ? 1 : 0;
                    o.nat[1] += in1 ? rr[r].y : 0;
                    o.hash[1] += in1 ? h : 0u;
                }
                flag[r] = rr[r].y > 0 ? (in0 ? 1 : 0) | (in1 ? 2 : 0) : 0;
                const unsigned long long bal = __ballot(flag[r] != 0);
                const int na = flag[r] ? rr[r].y : 0;
                const int incl = wave_scan_add(na);
                pos[r] = ng + rank_below(bal);
                at[r] = tot + incl - na;
                ng += __popcll(bal);
                tot += __builtin_amdgcn_readlane(incl, 63);
            }
            r0 += 64 * R;
        }
        // ---- a full batch goes through the pair pass
        if (done || g + ng > WL_GROUPS || A + tot > WL_ATOMS) {
            if (g > 0) {
                wave_sync();
                tk.end(S_TEST);
                P.run(C, L, W, g, A);
                tk.end(S_PAIRS);
                wave_sync();
            }
            if (done) break;
            if (g > 0) clear_map();
            g = 0;
            A = 0;
            wave_sync();
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (flag[r]) {
                const int a = A + at[r];
                W.goff[g + pos[r]] = a << 2 | flag[r];
                W.gdel[g + pos[r]] = rr[r].x - a;
                if (a < WL_ATOMS) W.amap[a] = (uint8_t)(g + pos[r]);
            }
        }
        g += ng;
        A += tot;
    }
}

// ---- a pose, or a trial's two poses, against the environment --------------------
struct PoseSums {
    double e[2];
    int nin[2], nat[2];
    uint32_t hash[2];
};
static_assert(sizeof(PoseSums) <= TEAM_BYTES, "team slots");

// W.frag[s * MAXF + a] (x, y, z, K q) of pose s's atoms -> the copies the pair
// pass reads, in the order of F.slot (equal types side by side): FP64 relative
// to the pose's centre, or FP32 absolute.  Lane a of the pose's wave.
template <int TM>
__device__ __forceinline__ void order_pose(CRep &C, CSpecies &F, const WaveLds &W, int s, int a, const float4 q,
                                           const float c[3])
{
    W.frag[s * MAXF + a] = q;
    const int i = s * MAXF + F.slot[a];
    if (TM == T_FP64)
        W.fragd[i] = make_double4((double)q.x - (double)c[0], (double)q.y - (double)c[1], (double)q.z - (double)c[2],
                                  (double)q.w);
    else
        ((float4 *)(W.fragd + s * MAXF))[F.slot[a]] = q;
}

// Energies of the nset poses in W around centres c0 and c1 (equal for a
// rotation), by one wave or its part of the cells; uniform results.
// pose_near: the poses were generated from the species template or the
// molecule's atoms (within the species' extent of the centre, the bound
// Rep::nowrap rests on); poses given by a caller take the per-pair image shift.
template <bool STAGED, int TM, class TK>
__device__ __forceinline__ void eval_poses_wave(CRep &C, const Lds &L, const WaveLds &W, int spi, int nf, int nset,
                                                const float c0[3], const float c1[3], bool same_centre, int exclude,
                                                bool pose_near, int part, int parts, PoseSums &out, TK &tk)
{
    EnergyPass<STAGED, TM> P;
    for (int i = 0; i < 2; ++i) P.acc[i] = 0.0;
    P.x[0] = c0[0]; P.y[0] = c0[1]; P.z[0] = c0[2];
    P.x[1] = c1[0]; P.y[1] = c1[1]; P.z[1] = c1[2];
    P.wrap = !(pose_near && C.nowrap != 0);
    P.spi = spi;
    ScanSums o{};
    // two centres in one scan when the stencil is wide enough for both
    const bool both = nset == 1 || same_centre || C.nst_wide > 0;
    P.first = 0;
    P.nset = both ? nset : 1;
    for (int pass = 0; pass < (both ? 1 : 2); ++pass) {
        ScanSums q{};
        P.first = pass;
        scan_groups(C, L, W, pass ? c1 : c0, c1, nset == 2 && both && !same_centre ? 2 : 1, exclude, part, parts, P, q, tk);
        if (pass == 0) o = q;
        else {
            o.nin[1] = q.nin[0];
            o.nat[1] = q.nat[0];
            o.hash[1] = q.hash[0];
        }
    }
    if (nset == 2 && same_centre) {
        o.nin[1] = o.nin[0];
        o.nat[1] = o.nat[0];
        o.hash[1] = o.hash[0];
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        out.e[s] = lane_d(wave_scan_add(P.acc[s]), 63);
        out.nin[s] = __builtin_amdgcn_readlane(wave_scan_add(o.nin[s]), 63);
        out.nat[s] = __builtin_amdgcn_readlane(wave_scan_add(o.nat[s]), 63);
        out.hash[s] = (uint32_t)__builtin_amdgcn_readlane((int)wave_scan_add(o.hash[s]), 63);
    }
}

__device__ inline uint32_t pose_hash(const float4 *p, int nf)
{
    uint32_t h = 2166136261u;
    for (int a = 0; a < nf; ++a) {
        h = (h ^ __float_as_uint(p[a].x)) * 16777619u;
        h = (h ^ __float_as_uint(p[a].y)) * 16777619u;
        h = (h ^ __float_as_uint(p[a].z)) * 16777619u;
    }
    return h;
}

__device__ inline bool tracing(CRep &C, int step, int &row)
{
    row = step - C.tr.first;
    return C.tr.k != nullptr && row >= 0 && row < C.tr.max_steps;
}

// Replica data is read and written by workgroups of one XCD (batched form)
// or by consecutive kernels (plain form).  Counters shared by workgroups use
// L2 atomics of that XCD (LOCAL) or device-wide atomics.
template <bool LOCAL, class T>
__device__ inline void count_add(T *p, T v)
{
    if (LOCAL) __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// statistics of a wave's evaluations (counters of the replica's State), added
// up in registers and published once per claim
struct ItemStats {
    unsigned nat, nin, neval, nfat;
};

template <bool LOCAL>
__device__ inline void add_item_stats(State &W, const ItemStats &s, int nf)
{
    count_add<LOCAL>(&W.n_eval, (unsigned long long)s.neval);
    count_add<LOCAL>(&W.n_pair, (unsigned long long)s.nat * nf);
    count_add<LOCAL>(&W.n_atom, (unsigned long long)s.nat);
    count_add<LOCAL>(&W.n_group, (unsigned long long)s.nin);
    count_add<LOCAL>(&W.n_fatom, (unsigned long long)s.nfat);
}

// ---- Ewald reciprocal term of a pose ------------------------------------------
// sum_f q_f phi(x_f) over the pose in W.frag (set s), phi the PME potential of
// the current state.  When the molecule itself is in that state (base >= 0: its
// atoms y_g at C.atom[base..]), its own share of phi -- what the grid holds
// for its charges, periodic images and neutralising background included --
// is removed: sum_{f,g} q_f q_g Kgrid(x_f, y_g) (pme_spline.h).  What remains
// is the reciprocal interaction with every other charge; for a rigid
// molecule the Ewald self, intramolecular and self-image terms are constants
// of the species, left out alike on insertion and deletion.  One wave (or its
// part); every lane gets its sum.
__device__ inline double ewald_recip(CRep &C, CSpecies &F, const WaveLds &W, int s, int nf, int base, int part,
                                     int parts)
{
    const int lane = threadIdx.x & 63;
    double v = 0.0;
    const int K[3] = {C.pk[0], C.pk[1], C.pk[2]};
    const float Lb[3] = {C.L[0], C.L[1], C.L[2]};
    // 16 lanes per atom
    for (int f0 = part * 4; f0 < nf; f0 += 4 * parts) {
        const int f = f0 + (lane >> 4), q = min(f, nf - 1);
        const float4 x = W.frag[s * MAXF + q];
        const float phi = gcmc_spline::gather16(C.pme_phi, K, Lb, x.x, x.y, x.z, lane & 15);
        if ((lane & 15) == 0 && f < nf) v += (double)F.tmpl[q].w * (double)phi;
    }
    if (base >= 0) {
        const int nw = nf * nf * 7;
        for (int w = part * 64 + lane; w < nw; w += 64 * parts) {
            const int f = w / (7 * nf), g = (w / 7) % nf, j0 = w % 7;
            const float4 xf = W.frag[s * MAXF + f];
            const float4 yg = C.atom[base + g];
            const float xv[3] = {xf.x, xf.y, xf.z}, yv[3] = {yg.x, yg.y, yg.z};
            const float kv = gcmc_spline::pair_kernel_slab(C.pme_gk, K, Lb, xv, yv, j0);
            v -= (double)F.tmpl[f].w * (double)F.tmpl[g].w * (double)kv;
        }
    }
    return lane_d(wave_scan_add(v), 63);
}

// ---- one trial -----------------------------------------------------------------
// A move's items are its trials: an insertion's or deletion's pose, or a
// translation's or rotation's old and new pose in one pass over the neighbourhood.
// A move of at most COOP_TRIALS trials is on its replica's critical path: its
// trials' cells are shared by four waves.  In larger moves every trial is one
// wave's.  The rule depends on the move alone: every form sums a pose's energy in
// the same order.  Sharing pays where waves would idle and costs where none do, so
// the line is a compromise between few systems and many.  us per move of a water
// chain among 8,000 atoms, shared / not: one system 11.9 / 18.5 at one trial,
// 40 / 48 at 64, 55 / 59 at 100, 75 / 79 at 200, 104 / 103 at 400; eight systems
// 46 / 54, 66 / 64, 85 / 84 and 134 / 134 at 64, 100, 200 and 400; 64 systems
// 15 / 21, 47 / 44, 60 / 57, 81 / 74 and 148 / 100 at 1, 32, 64, 100 and 200.
constexpr int COOP_TRIALS = 100, COOP = 4;

struct Move {
    int kind, spi, k, step, nset, nitems;   // nset: poses per trial
    bool coop;
};

__device__ __forceinline__ Move make_move(int kind, int spi, int k, int step)
{
    Move m;
    m.kind = uniform_i(kind);
    m.spi = uniform_i(spi);
    m.k = uniform_i(k);
    m.step = uniform_i(step);
    m.nitems = m.k;
    m.nset = m.kind >= K_TRN ? 2 : 1;
    m.coop = m.k <= COOP_TRIALS;
    return m;
}
__device__ __forceinline__ Move move_of(const State &S) { return make_move(S.kind, S.sp, S.k, S.step); }

// Wave `part` of `parts`: the poses of trial t (0: the old one, or an insertion's
// or deletion's only one, 1: the new one), its share of the adjacency row and of
// the energies.
template <bool STAGED, int TM>
__device__ __forceinline__ void trial_wave(CRep &C0, const Move &mv, int t, int part, int parts, const Lds &L,
                                           const WaveLds &W, PoseSums &out)
{
    CRep &C = fresh(C0);
    const int lane = fresh_lane();
    Ticks tk(L.misc + M_TICKS, mv.step, t);
    const int kind = mv.kind, k = mv.k, step = mv.step;
    CSpecies &F = species_of(C, mv.spi);
    const int nf = F.nf;
    const auto tc = gbl(C.tc);
    const auto atom = gbl(C.atom);
    const float4 tcl = tc[t];
    const int slot = (kind == K_INS) ? -1 : uniform_i(gbl(C.tslot)[t]);
    const int gid = (kind == K_INS) ? -1 : F.startRes + slot;
    const float cn[3] = {uniform_f(tcl.x), uniform_f(tcl.y), uniform_f(tcl.z)};
    float co[3] = {cn[0], cn[1], cn[2]};
    if (kind >= K_TRN) {
        const float4 cold = gbl(C.res_pos)[gid];
        co[0] = uniform_f(cold.x);
        co[1] = uniform_f(cold.y);
        co[2] = uniform_f(cold.z);
    }
    if (lane < nf) {
        const int a = lane;
        const float4 tm = F.tmpl[a];
        const float kq = F.kq[a];
        float px, py, pz;
        if (kind == K_INS) {
            const u32x4 y = draw(C.seed, (uint32_t)step, (uint32_t)t, P_ROTATION);
            float R[9], v[3];
            rotation_matrix(u01f(y.x), u01f(y.y), u01f(y.z), u01f(y.w) * 0x1.921fb6p+2f, R);
            rotate(R, tm.x, tm.y, tm.z, v);
            px = v[0] + cn[0]; py = v[1] + cn[1]; pz = v[2] + cn[2];
        } else {
            const int base = F.atomBase + slot * nf;
            const float4 cur = atom[base + a];
            order_pose<TM>(C, F, W, 0, a, make_float4(cur.x, cur.y, cur.z, kq), co);
            if (kind == K_TRN) {
                const u32x4 x = draw(C.seed, (uint32_t)step, (uint32_t)t, P_JITTER);
                const float u[3] = {u01f(x.x), u01f(x.y), u01f(x.z)};
                float r[3];
                for (int i = 0; i < 3; ++i) {
                    float d = u[i] * C.dx;
                    if (co[i] + d > C.L[i] + C.start[i]) d = d - C.L[i];
                    if (co[i] + d < C.start[i]) d = d + C.L[i];
                    r[i] = d;
                }
                px = cur.x + r[0]; py = cur.y + r[1]; pz = cur.z + r[2];
            } else if (kind == K_ROT) {
                // each lane divides its own atom's coordinates, the sums run in
                // atom order
                const float fn = (float)nf;
                const float s0 = cur.x / fn, s1 = cur.y / fn, s2 = cur.z / fn;
                float cen0 = 0.f, cen1 = 0.f, cen2 = 0.f;
                for (int b = 0; b < nf; ++b) {
                    cen0 = cen0 + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s0), b));
                    cen1 = cen1 + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s1), b));
                    cen2 = cen2 + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s2), b));
                }
                const u32x4 y = draw(C.seed, (uint32_t)step, (uint32_t)t, P_ROTATION);
                float R[9], v[3];
                rotation_matrix(u01f(y.x), u01f(y.y), u01f(y.z), u01f(y.w) * 0x1.921fb6p+2f, R);
                rotate(R, cur.x - cen0, cur.y - cen1, cur.z - cen2, v);
                px = v[0] + cen0; py = v[1] + cen1; pz = v[2] + cen2;
            }
        }
        if (kind != K_DEL) {
            order_pose<TM>(C, F, W, kind == K_INS ? 0 : 1, a, make_float4(px, py, pz, kq), cn);
            if (part == 0) gbl(C.pose)[t * MAXF + a] = make_float4(px, py, pz, 0.f);
        }
    }
    wave_sync();
    // adjacency row of trial t over the trial centres (grouping of the accept
    // phase), the loads of four blocks of 64 at a time
    if (kind != K_DEL) {
        constexpr int B = 4;
        const GroupCut cut = group_cut(C);
        for (int j0 = part * 64; j0 < k; j0 += B * 64 * parts) {
            float4 cj[B];
#pragma unroll
            for (int q = 0; q < B; ++q) {
                const int j = j0 + q * 64 * parts + lane;
                cj[q] = tc[min(j, k - 1)];
            }
#pragma unroll
            for (int q = 0; q < B; ++q) {
                const int jq = j0 + q * 64 * parts, j = jq + lane;
                if (jq >= k) break;
                const bool b = within_lanes(cn, cj[q], cut) && j < k && j != t;
                const unsigned long long bal = __ballot(b);
                if (lane == 0) {
                    const int wi = jq >> 5;
                    gbl(C.adj)[t * ADJW + wi] = (uint32_t)bal;
                    gbl(C.adj)[t * ADJW + wi + 1] = (uint32_t)(bal >> 32);
                }
            }
        }
    }
    tk.end(S_POSE);
    // a rotation keeps the centre
    eval_poses_wave<STAGED, TM>(C, L, W, mv.spi, nf, mv.nset, co, cn, kind != K_TRN, gid, true, part, parts, out, tk);
    if (TM == T_EWALD) {
        // the moving molecule (delete, translate, rotate) is in the PME grid
        const int base = kind == K_INS ? -1 : F.atomBase + slot * nf;
        out.e[0] += ewald_recip(C, F, W, 0, nf, base, part, parts);
        if (mv.nset == 2) out.e[1] += ewald_recip(C, F, W, 1, nf, base, part, parts);
    }
}

// energies of a trial to the replica's buffers, statistics, trace (one lane)
__device__ inline void finish_trial(CRep &C, const Move &mv, int t, const WaveLds &W, const PoseSums &r, ItemStats &st)
{
    CSpecies &F = species_of(C, mv.spi);
    const int nf = F.nf;
    const bool two = mv.nset == 2;
    const auto E = gbl(C.E);
    E[t] = r.e[0];
    if (two) E[mv.k + t] = r.e[1];
    st.nat += (unsigned)(r.nat[0] + (two ? r.nat[1] : 0));
    st.nin += (unsigned)(r.nin[0] + (two ? r.nin[1] : 0));
    st.neval += mv.nset;
    st.nfat += mv.nset * nf;
    int row;
    if (tracing(C, mv.step, row) && t < C.tr.max_k) {
        const int q = row * C.tr.max_k + t;
        for (int s = 0; s < mv.nset; ++s) {
            C.tr.e[2 * q + s] = s ? r.e[1] : r.e[0];
            C.tr.ninc[2 * q + s] = s ? r.nin[1] : r.nin[0];
            C.tr.inchash[2 * q + s] = s ? r.hash[1] : r.hash[0];
        }
        const float4 tcv = gbl(C.tc)[t];
        C.tr.posehash[q] = pose_hash(W.frag + (mv.nset - 1) * MAXF, nf);
        C.tr.centre[3 * q + 0] = tcv.x;
        C.tr.centre[3 * q + 1] = tcv.y;
        C.tr.centre[3 * q + 2] = tcv.z;
        C.tr.idx[q] = mv.kind == K_INS ? -1 : gbl(C.tslot)[t];
    }
}

// four waves' shares of one pose (or two), added up in wave order; W's wave 0
// of the team gets the sums.  Two barriers of the whole workgroup.
template <int NT>
__device__ __forceinline__ void team_sum(const Lds &L, PoseSums &r)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    auto slot = [&](int w) { return (PoseSums *)((char *)L.team + w * TEAM_BYTES); };
    if (lane == 0) *slot(wave) = r;
    __syncthreads();
    if (wave % COOP == 0 && lane == 0) {
        for (int w = 1; w < COOP; ++w) {
            const PoseSums q = *slot(wave + w);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                r.e[s] += q.e[s];
                r.nin[s] += q.nin[s];
                r.nat[s] += q.nat[s];
                r.hash[s] += q.hash[s];
            }
        }
    }
    __syncthreads();
}

// cnt trials from `item` on by the whole workgroup: teams of four waves, or the
// waves each on their own, taking the next trial from L.misc[M_NEXT] (0 on
// entry, written before a barrier)
template <int NT, bool STAGED, int TM>
__device__ __forceinline__ void eval_items(CRep &C, const Move &mv, int item, int cnt, const Lds &L, ItemStats &st)
{
    constexpr int NW = NT / 64, TEAMS = NW / COOP;
    const int wave = fresh_uniform(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const WaveLds W = wave_lds(L, wave);
    // one call site: the trial's code is long
    int j0 = 0;
    while (true) {
        int j;
        if (mv.coop) {
            if (j0 >= cnt) break;
            j = j0 + wave / COOP;
            j0 += TEAMS;
        } else {
            j = 0;
            if (lane == 0) j = atomicAdd(&L.misc[M_NEXT], 1);
            j = uniform_i(j);
            if (j >= cnt) break;
        }
        const int t = item + min(j, cnt - 1), part = mv.coop ? wave % COOP : 0, parts = mv.coop ? COOP : 1;
        PoseSums r;
        trial_wave<STAGED, TM>(C, mv, t, part, parts, L, W, r);
        if (mv.coop) team_sum<NT>(L, r);
        if (lane == 0 && part == 0 && j < cnt) finish_trial(C, mv, t, W, r, st);
        wave_sync();
    }
}

// ---- cell-list maintenance (single thread) ----------------------------------
__device__ inline void cell_insert(CRep &C, int gid, int spi, float x, float y, float z)
{
    const int c = cell_index(C.L, C.start, C.inv_h, C.nc, x, y, z);
    const int n = C.cell[c].y;
    int pos;
    if (n < C.cap) {
        pos = c * C.cap + n;
        C.cell[c].y = n + 1;
    } else {
        const int o = C.cell[C.ncell].y;
        pos = C.ovf_base + o;
        C.cell[C.ncell].y = o + 1;
    }
    C.mob_slot[pos] = gid;
    C.mob_rec[pos] = make_float4(x, y, z, __int_as_float(mob_word(gid, spi)));
    C.mob_loc[gid] = pos;
}

__device__ inline void cell_remove(CRep &C, int gid)
{
    const int pos = C.mob_loc[gid];
    int c, base;
    if (pos >= C.ovf_base) {
        c = C.ncell;
        base = C.ovf_base;
    } else {
        c = pos / C.cap;
        base = c * C.cap;
    }
    const int n = C.cell[c].y - 1;
    const int moved = C.mob_slot[base + n];
    C.mob_slot[pos] = moved;
    C.mob_rec[pos] = C.mob_rec[base + n];
    C.mob_loc[moved] = pos;
    C.cell[c].y = n;
    C.mob_loc[gid] = -1;
}

// group `from` now lives in slot `to` (its centre and species are unchanged)
__device__ inline void cell_rename(CRep &C, int from, int to)
{
    const int pos = C.mob_loc[from];
    C.mob_slot[pos] = to;
    float4 r = C.mob_rec[pos];
    r.w = __int_as_float((__float_as_int(r.w) & ~GID_MASK) | to);
    C.mob_rec[pos] = r;
    C.mob_loc[to] = pos;
    C.mob_loc[from] = -1;
}

// ---- selection and Metropolis --------------------------------------------------
// Greedy grouping in ascending trial order: leader = first unused trial,
// members = unused trials within the cutoff of the leader; Boltzmann weights
// relative to the group minimum; cumulative pick; acceptance
//   insert:  min(1, cav/(m P)/(N+1) exp(B - beta E))   (gcmc_move_add.h:164-174)
//   move:    min(1, 1/(m P) exp(-beta dE))             (gcmc_move_trn.h:215-222)
// On accept the unused trials within the cutoff of the pick are dropped.
// Trial values are staged in L.val, adjacency rows in L.adjl (when the layout
// has room; else read from C.adj).
__device__ inline uint32_t adj_word(CRep &C, const Lds &L, int nw, int t, int w)
{
    return L.adjl ? L.adjl[t * nw + w] : C.adj[t * ADJW + w];
}

// A move's descriptor and the replica values its accept phase reads, loaded
// once at its start: every later phase would otherwise reload them after a
// barrier, one dependent L2 round trip each on the replica's serial path.
struct MoveCtx {
    int kind, spi, k, step, nf, N, maxN, startRes, atomBase;
    double B, energy;
};

__device__ inline MoveCtx move_ctx(CRep &C, const State &S)
{
    MoveCtx m;
    m.kind = S.kind;
    m.spi = S.sp;
    m.k = S.k;
    m.step = S.step;
    m.N = S.totalNum[m.spi];
    m.energy = S.energy;
    CSpecies &F = species_of(C, m.spi);
    m.nf = F.nf;
    m.maxN = F.maxNum;
    m.startRes = F.startRes;
    m.atomBase = F.atomBase;
    m.B = F.B;
    return m;
}

// the next move's descriptor into L.misc[M_NX..] (one thread; the accept
// phase's selection wave is busy meanwhile).  The species count is the one
// before the current move: prep takes the current move's result for its own
// species.
__device__ inline void load_next_move(CRep &C, const State &S, const Lds &L, const MoveCtx &m)
{
    const int end = S.end, step = m.step + 1;
    const int mv = step < end ? C.moves[step] : 0;
    CSpecies &F = species_of(C, mv >> 2);
    L.misc[M_NX + 0] = end;
    L.misc[M_NX + 1] = mv;
    L.misc[M_NX + 2] = S.totalNum[mv >> 2];
    L.misc[M_NX + 3] = F.conf;
    L.misc[M_NX + 4] = F.maxNum;
    L.misc[M_NX + 5] = F.startRes;
}

// FP64 keys whose unsigned order is the values' order
__device__ inline unsigned long long order_key(double v)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return b >> 63 ? ~b : b | 0x8000000000000000ull;
}
__device__ inline double key_value(unsigned long long k)
{
    return __longlong_as_double((long long)(k >> 63 ? k & 0x7fffffffffffffffull : ~k));
}

// Moves of more than 64 trials.  The groups depend on each other only through
// acceptances, so they are settled in batches as if none were: wave 0 forms a
// batch's groups (bit operations only), the workgroup computes the members'
// weights, and one lane per group sums them in trial order, picks and decides.
// An accepted pick drops its neighbours from the later groups: the groups before
// the first one that loses a member stand, the next batch starts there.  Batches
// grow from 8 to SEL_GROUPS groups while all of them stand and shrink to the pace
// at which they do not (insertions of eight fragments, 10 to 400 trials each, into
// 20,000 atoms: 34.0 us per move, 35.2 in batches of 8 throughout; 36.2 on another
// machine, 37.4 in batches of 64).
// (One wave taking the groups one after another, weights included, spent
// 1.3 us on each.)
template <int NT>
__device__ inline void select_groups(CRep &C, State &S, const Lds &L, int row, bool trace, const MoveCtx &mc)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int kind = mc.kind, k = mc.k;
    const bool ins = kind == K_INS;
    const int nw = (k + 31) >> 5;
    // wave 0: lane w holds the unused trials 32 w .. 32 w + 31
    uint32_t u = 0u;
    if (lane < nw) {
        const int hi = k - lane * 32;
        u = hi >= 32 ? 0xffffffffu : ((1u << hi) - 1u);
    }
    int N = mc.N, g0 = 0, na = 0, most = 8;
    const int maxN = mc.maxN;
    const double cav = (double)C.cav, B = ins ? mc.B : 0.0;
    double et = mc.energy;
    if (wave == 1) L.gmin[lane] = ~0ull;
    while (true) {
        uint32_t v = u;
        if (wave == 0) {
            int n = 0, base = 0;
            // the first unused trial and its row of the adjacency matrix
            auto leader = [&](int &it, int &f, uint32_t &rw) {
                const unsigned long long bal = __ballot(v != 0u);
                if (bal == 0ull) return false;
                f = __ffsll((long long)bal) - 1;
                it = f * 32 + __ffs(__builtin_amdgcn_readlane((int)v, f)) - 1;
                rw = lane < nw ? adj_word(C, L, nw, it, lane) : 0u;
                return true;
            };
            int it = 0, f = 0;
            uint32_t rw = 0u;
            bool more = leader(it, f, rw);
            while (more && n < most) {
                uint32_t m = rw & v;
                if (lane == f) m |= 1u << (it & 31);
                v &= ~m;
                more = leader(it, f, rw);   // its row arrives while this group is stored
                const int cnt = __popc(m), incl = wave_scan_add(cnt);
                if (lane < nw) {
                    L.gmask[n * nw + lane] = m;
                    L.goff[n * nw + lane] = (uint16_t)(base + incl - cnt);
                }
                if (lane == 0) L.gstart[n] = base;
                base += __builtin_amdgcn_readlane(incl, 63);
                ++n;
            }
            if (lane == 0) {
                L.gstart[n] = base;
                L.misc[M_GN] = n;
            }
        }
        __syncthreads();
        const int n = uniform_i(L.misc[M_GN]);
        if (n == 0) break;
        const int total = uniform_i(L.gstart[n]);
        // the batch's trials in group and trial order, and each group's lowest
        // value (NaN counts for none)
        for (int q = tid; q < n * nw; q += NT) {
            uint32_t m = L.gmask[q];
            if (m == 0u) continue;
            const int g = q / nw, t0 = (q - g * nw) * 32;
            int o = L.goff[q];
            for (; m; m &= m - 1u) {
                const int t = t0 + __ffs(m) - 1;
                const double x = L.val[t];
                L.members[o++] = t | g << 16;
                if (x == x) atomicMin(&L.gmin[g], order_key(x));
            }
        }
        __syncthreads();
        for (int p = tid; p < total; p += NT) {
            const int e = L.members[p];
            const unsigned long long key = L.gmin[e >> 16];
            const double emin = key == ~0ull ? __builtin_huge_val() : key_value(key);
            L.w[p] = exp(-BETA * (L.val[e & 0xffff] - emin));
        }
        __syncthreads();
        if (wave == 1) L.gmin[lane] = ~0ull;
        if (wave == 0) {
            // lane g: group g0 + g
            int pick = 0, rec = 0;
            double ea = 0.0, cp = 0.0, ran_acc = 1.0;
            if (lane < n) {
                const int s = L.gstart[lane], e = L.gstart[lane + 1], cnt = e - s;
                const u32x4 xr = draw(C.seed, (uint32_t)mc.step, (uint32_t)(g0 + lane), P_DECIDE);
                const double ran_sel = u01d(xr.x, xr.y);
                ran_acc = u01d(xr.z, xr.w);
                double sum = 0.0, P = 1.0;
                for (int p = s; p < e; p += 4) {
                    const double w0 = L.w[p], w1 = L.w[min(p + 1, e - 1)], w2 = L.w[min(p + 2, e - 1)],
                                 w3 = L.w[min(p + 3, e - 1)];
                    sum += w0;
                    sum += p + 1 < e ? w1 : 0.0;
                    sum += p + 2 < e ? w2 : 0.0;
                    sum += p + 3 < e ? w3 : 0.0;
                }
                int at = s;
                if (cnt > 1 && sum != 0.0) {
                    // first member with sum_{j<=q} w_j > ran_sel * sum (the last one
                    // when rounding leaves the target at the total)
                    const double target = ran_sel * sum;
                    double c = 0.0;
                    at = e - 1;
                    for (int p = s; p < e; p += 2) {
                        const double w0 = L.w[p], w1 = L.w[min(p + 1, e - 1)];
                        c += w0;
                        if (target < c) {
                            at = p;
                            break;
                        }
                        c += w1;
                        if (target < c) {
                            at = min(p + 1, e - 1);
                            break;
                        }
                    }
                    P = L.w[at] / sum;
                }
                pick = L.members[at] & 0xffff;
                ea = exp(B - BETA * L.val[pick]);
                cp = (ins ? cav : 1.0) / ((double)cnt * P);
            }
            auto decide = [&]() {
                const double pp = ins ? cp / ((double)N + 1.0) * ea : cp * ea;
                const double p = pp < 1.0 ? pp : 1.0;
                return __ballot(lane < n && ran_acc < p);
            };
            unsigned long long am = decide();
            int stand = n;
            uint32_t drop = 0u;   // lane w: neighbours of the accepted picks
            while (am != 0ull) {
                const int g = __ffsll((long long)am) - 1;
                const int ap = __builtin_amdgcn_readlane(pick, g);
                if (lane < nw) {
                    drop |= adj_word(C, L, nw, ap, lane);
                    L.drop[lane] = drop;
                }
                if (lane == g) rec = ins && N >= maxN ? 2 : 1;
                if (!(ins && N >= maxN)) {
                    if (lane == 0) L.accl[na] = make_int2(ap, ins ? N : C.tslot[ap]);
                    N += ins ? 1 : 0;
                    na += 1;
                    et += L.val[ap];
                    if (ins) am = decide();
                }
                wave_sync();   // other lanes' words of L.drop are read
                // the first later group that loses a member
                bool hit = false;
                if (lane > g && lane < stand)
                    for (int w = 0; w < nw; ++w) hit |= (L.gmask[lane * nw + w] & L.drop[w]) != 0u;
                const unsigned long long hm = __ballot(hit);
                if (hm) stand = __ffsll((long long)hm) - 1;
                // accepted groups still to take: after g, among those that stand
                am &= stand >= 64 ? ~0ull : (1ull << stand) - 1ull;
                am &= g >= 63 ? 0ull : ~0ull << (g + 1);
            }
            if (stand == n) {
                u = v & ~drop;
                most = min(4 * most, SEL_GROUPS);
            } else {
                for (int g = 0; g < stand; ++g)
                    if (lane < nw) u &= ~L.gmask[g * nw + lane];
                u &= ~drop;
                most = min(max(2 * stand, 8), SEL_GROUPS);
            }
            if (trace && lane < stand && g0 + lane < C.tr.max_k) {
                C.tr.gpick[row * C.tr.max_k + g0 + lane] = pick;
                C.tr.gacc[row * C.tr.max_k + g0 + lane] = rec;
            }
            g0 += stand;
        }
    }
    if (tid == 0) {
        L.misc[M_ACC] = na;
        L.misc[M_NG] = g0;
        L.misc[M_N] = N;
        S.energy = et;
        // counters only: an atomic add without return keeps the load of
        // the old value off the serial path
        if (na) count_add<false>(&S.acc[mc.spi * 4 + kind], (long long)na);
    }
}

// At most 64 trials, per-trial values in registers: lane t holds trial t's
// value, exp term, adjacency row (bit j: trial j within the cutoff) and slot,
// and group t's two variates.  Group members are compacted into lanes 0..m-1
// in trial order (ds_permute) and their weights summed by one scan.  Wave 0 only.
__device__ inline void greedy_select64(CRep &C, State &S, const Lds &L, int row, bool trace, const MoveCtx &mc,
                                       double val, double ea, double rsel, double racc, unsigned long long adj,
                                       int tslot)
{
    const int lane = threadIdx.x & 63;
    const int kind = mc.kind, k = mc.k;
    const bool ins = kind == K_INS;
    const unsigned long long below = (1ull << lane) - 1ull;
    unsigned long long U = k >= 64 ? ~0ull : ((1ull << k) - 1ull);
    int N = mc.N;
    const int maxN = mc.maxN;
    const double cav = (double)C.cav;
    int g = 0, na = 0;
    double et = mc.energy;
    while (U != 0ull) {
        const int it = __ffsll((long long)U) - 1;
        const unsigned long long M = (lane_u64(adj, it) & U) | (1ull << it);
        U &= ~M;
        const int mtot = __popcll(M);
        const double ran_sel = lane_d(rsel, g);
        const double ran_acc = lane_d(racc, g);
        int pick = it;
        double P = 1.0;
        if (mtot > 1) {
            const bool in = ((M >> lane) & 1ull) != 0ull;
            const double emin = wave_min(in ? val : __builtin_huge_val());
            const double wl = in ? exp(-BETA * (val - emin)) : 0.0;
            const int dst = in ? __popcll(M & below) : mtot + __popcll(~M & below);
            const double w = permute_d(dst, wl);                      // lane q: member q's weight
            const int tix = __builtin_amdgcn_ds_permute(dst * 4, lane);  // lane q: member q's trial
            const double part = lane < mtot ? w : 0.0;
            const double incl = wave_scan_add(part);
            const double sumP = lane_d(incl, 63);
            int pq = 0;
            if (sumP != 0.0) {
                const double target = ran_sel * sumP;
                const double excl = incl - part;
                const unsigned long long hit = __ballot(lane < mtot && excl <= target && target < incl);
                pq = hit ? __ffsll((long long)hit) - 1 : mtot - 1;
                pick = lane_i(tix, pq);
                P = lane_d(w, pq) / sumP;
            }
        }
        const double vp = lane_d(val, pick);
        const double eap = lane_d(ea, pick);
        double pp;
        if (ins)
            pp = (cav / ((double)mtot * P)) / ((double)N + 1.0) * eap;
        else
            pp = (1.0 / ((double)mtot * P)) * eap;
        const double p = pp < 1.0 ? pp : 1.0;
        const bool acc = ran_acc < p;
        int rec = acc ? 1 : 0;
        if (acc) {
            U &= ~lane_u64(adj, pick);
            if (ins) {
                if (N < maxN) {
                    if (lane == 0) L.accl[na] = make_int2(pick, N);
                    N += 1;
                    na += 1;
                    et += vp;
                } else {
                    rec = 2;
                }
            } else {
                const int sl = lane_i(tslot, pick);
                if (lane == 0) L.accl[na] = make_int2(pick, sl);
                na += 1;
                et += vp;
            }
        }
        if (trace && lane == 0 && g < C.tr.max_k) {
            C.tr.gpick[row * C.tr.max_k + g] = pick;
            C.tr.gacc[row * C.tr.max_k + g] = rec;
        }
        g += 1;
    }
    if (lane == 0) {
        L.misc[M_ACC] = na;
        L.misc[M_NG] = g;
        L.misc[M_N] = N;
        S.energy = et;
        // counters only: an atomic add without return keeps the load of
        // the old value off the serial path
        if (na) count_add<false>(&S.acc[mc.spi * 4 + kind], (long long)na);
    }
}

// ---- commit of the accepted trials (L.accl[0..na): trial, slot) ------------------
// GupdateAdd / GupdateTrn / GupdateRot: copy committed poses, then the group
// centres and cell-list entries in acceptance order (thread 0).
template <int NT, bool EW>
__device__ inline void commit_accepted(CRep &C, State &S, const Lds &L, int row, bool trace, const MoveCtx &mc)
{
    const int tid = threadIdx.x;
    const int kind = mc.kind, spi = mc.spi;
    CSpecies &F = species_of(C, spi);
    const int nf = mc.nf;
    const int na = L.misc[M_ACC];
    // GupdateAdd / GupdateTrn / GupdateRot: copy committed poses
    for (int idx = tid; idx < na * nf; idx += NT) {
        const int q = idx / nf, a = idx - q * nf;
        const int2 ts = L.accl[q];
        const int base = mc.atomBase + ts.y * nf;
        const float4 p = C.pose[ts.x * MAXF + a];
        float4 dst;
        if (kind == K_INS) {
            dst = make_float4(p.x, p.y, p.z, F.tmpl[a].w);
            C.atype[base + a] = F.ttype[a];
        } else {
            dst = C.atom[base + a];
            if (EW) C.pme_delta[2 * idx] = make_float4(dst.x, dst.y, dst.z, -F.tmpl[a].w);
            dst.x = p.x; dst.y = p.y; dst.z = p.z;
        }
        if (EW) {
            if (kind == K_INS) C.pme_delta[2 * idx] = make_float4(0.f, 0.f, 0.f, 0.f);
            C.pme_delta[2 * idx + 1] = make_float4(p.x, p.y, p.z, F.tmpl[a].w);
        }
        C.atom[base + a] = dst;
    }
    if (EW && tid == 0) *C.pme_ndelta = 2 * na * nf;
    if (tid == 0) {
        for (int q = 0; q < na; ++q) {
            const int2 ts = L.accl[q];
            const int gid = mc.startRes + ts.y;
            const float4 c = C.tc[ts.x];
            if (kind == K_INS) {
                C.res_pos[gid] = make_float4(c.x, c.y, c.z, 0.f);
                cell_insert(C, gid, spi, c.x, c.y, c.z);
                if (trace && ts.x < C.tr.max_k) C.tr.idx[row * C.tr.max_k + ts.x] = ts.y;
            } else if (kind == K_TRN) {
                const float4 old = C.res_pos[gid];
                C.res_pos[gid] = make_float4(c.x, c.y, c.z, old.w);
                cell_remove(C, gid);
                cell_insert(C, gid, spi, c.x, c.y, c.z);
            }
        }
        if (kind == K_INS) S.totalNum[spi] = L.misc[M_N];
    }
}

// ---- accept phase: decisions and commit ------------------------------------------
template <int NT, bool EW>
__device__ inline void accept_move(CRep &C, State &S, const Lds &L, const MoveCtx &mc, bool prefetch = false)
{
    const int tid = threadIdx.x;
    const int kind = mc.kind, spi = mc.spi, k = mc.k, step = mc.step;
    CSpecies &F = species_of(C, spi);
    const int nf = mc.nf;
    int row;
    const bool trace = tracing(C, step, row);
    // stage the trial values (E for insert/delete, E_new - E_old otherwise);
    // with at most 64 trials of an insert or move they stay in registers
    const bool in_regs = k <= 64 && kind != K_DEL;
    if (!in_regs)
        for (int t = tid; t < k; t += NT) L.val[t] = (kind == K_TRN || kind == K_ROT) ? C.E[k + t] - C.E[t] : C.E[t];
    if (tid == 0) {
        count_add<false>(&S.att[spi * 4 + kind], 1ll);
        L.misc[M_ACC] = 0;
        L.misc[M_NG] = 0;
        L.misc[M_N] = mc.N;
        if (EW) *C.pme_ndelta = 0;
    }
    __syncthreads();
    if (prefetch && tid == 64) load_next_move(C, S, L, mc);
    if (kind == K_DEL && k == 1) {
        const int N = mc.N;
        if (tid == 0) {
            const double E = L.val[0];
            const u32x4 x = draw(C.seed, (uint32_t)step, 0u, P_DECIDE);
            const double ran = u01d(x.z, x.w);
            const double pp = (double)N * exp(-mc.B - BETA * (-E));
            const double p = pp < 1.0 ? pp : 1.0;
            const int acc = ran < p;
            L.misc[M_ACC] = acc;
            L.misc[M_NG] = 1;
            if (trace) {
                C.tr.gpick[row * C.tr.max_k] = 0;
                C.tr.gacc[row * C.tr.max_k] = acc;
            }
            if (acc) {
                S.energy = mc.energy - E;
                count_add<false>(&S.acc[spi * 4 + kind], 1ll);
            }
        }
        __syncthreads();
        if (L.misc[M_ACC]) {
            // GupdateDel (gcmc_move_del.h:55-94): swap-remove with the last slot
            const int newN = N - 1;
            const int hole_slot = C.tslot[0];
            const int hole = F.startRes + hole_slot, last = F.startRes + newN;
            if (EW) {
                // the deleted molecule's charges leave the PME grid (the moved
                // last molecule keeps its coordinates)
                for (int a = tid; a < nf; a += NT) {
                    const float4 o = C.atom[F.atomBase + hole_slot * nf + a];
                    C.pme_delta[a] = make_float4(o.x, o.y, o.z, -F.tmpl[a].w);
                }
                if (tid == 0) *C.pme_ndelta = nf;
                __syncthreads();
            }
            if (newN > 0 && hole != last) {
                const int bh = F.atomBase + hole_slot * nf, bl = F.atomBase + newN * nf;
                for (int a = tid; a < nf; a += NT) {
                    const float4 src = C.atom[bl + a];
                    float4 dst = C.atom[bh + a];
                    dst.x = src.x; dst.y = src.y; dst.z = src.z;
                    C.atom[bh + a] = dst;
                }
            }
            if (tid == 0) {
                cell_remove(C, hole);
                if (newN > 0 && hole != last) {
                    const float4 pl = C.res_pos[last];
                    float4 ph = C.res_pos[hole];
                    ph.x = pl.x; ph.y = pl.y; ph.z = pl.z;
                    C.res_pos[hole] = ph;
                    cell_rename(C, last, hole);
                }
                S.totalNum[spi] = newN;
                L.misc[M_N] = newN;
            }
        }
    } else if (k > 0 && in_regs) {
        // lane t of wave 0 holds trial t's values (greedy_select64)
        if ((tid >> 6) == 0) {
            const int t = tid;
            double val = 0.0, ea = 0.0, rsel = 0.0, racc = 0.0;
            unsigned long long adj = 0ull;
            int sl = 0;
            if (t < k) {
                const auto E = gbl(C.E);
                val = (kind == K_TRN || kind == K_ROT) ? E[k + t] - E[t] : E[t];
                const auto A = gbl(C.adj);
                adj = (unsigned long long)A[t * ADJW];
                if (k > 32) adj |= (unsigned long long)A[t * ADJW + 1] << 32;
                if (kind != K_INS) sl = gbl(C.tslot)[t];
                const u32x4 xr = draw(C.seed, (uint32_t)step, (uint32_t)t, P_DECIDE);
                rsel = u01d(xr.x, xr.y);
                racc = u01d(xr.z, xr.w);
                ea = exp(((kind == K_INS) ? mc.B : 0.0) - BETA * val);
            }
            greedy_select64(C, S, L, row, trace, mc, val, ea, rsel, racc, adj, sl);
        }
        __syncthreads();
        commit_accepted<NT, EW>(C, S, L, row, trace, mc);
    } else if (k > 0 && kind != K_DEL) {
        if (L.adjl) {
            const int nw = (k + 31) >> 5;
            for (int q = tid; q < k * nw; q += NT) {
                const int t = q / nw, w = q - t * nw;
                L.adjl[q] = C.adj[t * ADJW + w];
            }
        }
        __syncthreads();
        select_groups<NT>(C, S, L, row, trace, mc);
        __syncthreads();
        commit_accepted<NT, EW>(C, S, L, row, trace, mc);
    }
    if (tid == 0) {
        if (trace) {
            C.tr.k[row] = k;
            C.tr.ngroups[row] = L.misc[M_NG];
            C.tr.naccept[row] = L.misc[M_ACC];
            C.tr.n_after[row] = S.totalNum[spi];
            C.tr.etot[row] = S.energy;
        }
        S.step = step + 1;
    }
    __syncthreads();
}

template <int NT, bool EW>
__device__ inline void accept_step(CRep &C, State &S, const Lds &L)
{
    const MoveCtx mc = move_ctx(C, S);
    accept_move<NT, EW>(C, S, L, mc);
}

// a move without trials (insertion into full slots, no molecule to move): an
// attempt, nothing else (accept_move's result for k = 0)
__device__ inline void skip_move(CRep &C, State &S)
{
    if (threadIdx.x == 0) {
        const int spi = S.sp, step = S.step;
        count_add<false>(&S.att[spi * 4 + S.kind], 1ll);
        int row;
        if (tracing(C, step, row)) {
            C.tr.k[row] = 0;
            C.tr.ngroups[row] = 0;
            C.tr.naccept[row] = 0;
            C.tr.n_after[row] = S.totalNum[spi];
            C.tr.etot[row] = S.energy;
        }
        S.step = step + 1;
    }
    __syncthreads();
}

// ---- prep phase: picks and trial centres of S.step ------------------------------
// pre: the move's descriptor loaded with the previous move (for the same
// species, the count that move's accept phase left in L.misc[M_N]), or null
// use_pre: the move after prev (species prev_spi) was loaded into L.misc[M_NX..]
template <int NT>
__device__ inline Move prep_step(CRep &C, State &S, const Lds &L, bool use_pre, int prev_step, int prev_spi)
{
    const int tid = threadIdx.x;
    int step, mv, N, conf, maxNum, startRes;
    if (use_pre) {
        step = prev_step + 1;
        mv = L.misc[M_NX + 1];
        N = ((mv >> 2) == prev_spi) ? L.misc[M_N] : L.misc[M_NX + 2];
        conf = L.misc[M_NX + 3];
        maxNum = L.misc[M_NX + 4];
        startRes = L.misc[M_NX + 5];
    } else {
        step = S.step;
        mv = C.moves[step];
        CSpecies &F0 = species_of(C, mv >> 2);
        N = S.totalNum[mv >> 2];
        conf = F0.conf;
        maxNum = F0.maxNum;
        startRes = F0.startRes;
    }
    const int spi = mv >> 2, kind = mv & 3;
    int k;
    if (kind == K_INS) k = (N >= maxNum) ? 0 : conf;
    else if (kind == K_DEL) k = (N == 0) ? 0 : 1;
    else k = conf < N ? conf : N;
    if (k > C.maxk) k = C.maxk;
    if (kind != K_INS && k > 0) {
        // partial Fisher-Yates (gcmc_move_trn.h:135-149): pick i takes the value at
        // position J[i] after the swaps 0..i-1, found by tracing the swaps back
        for (int i = tid; i < k; i += NT) {
            const u32x4 x = draw(C.seed, (uint32_t)step, (uint32_t)i, P_PICK);
            L.J[i] = i + (int)below(x.x, (uint32_t)(N - i));
        }
        __syncthreads();
        for (int i = tid; i < k; i += NT) {
            int p = L.J[i];
            for (int m = i - 1; m >= 0; --m) {
                const int jm = L.J[m];
                p = (p == m) ? jm : ((p == jm) ? m : p);
            }
            C.tslot[i] = p;
        }
    }
    __syncthreads();
    for (int t = tid; t < k; t += NT) {
        float c[3];
        if (kind == K_INS) {
            const u32x4 x = draw(C.seed, (uint32_t)step, (uint32_t)t, P_JITTER);
            const uint32_t g = below(x.w, (uint32_t)C.G);
            const float u[3] = {u01f(x.x), u01f(x.y), u01f(x.z)};
            for (int i = 0; i < 3; ++i) c[i] = C.grid[3 * g + i] + u[i] * C.dx;
        } else {
            const float4 r = C.res_pos[startRes + C.tslot[t]];
            c[0] = r.x; c[1] = r.y; c[2] = r.z;
            if (kind == K_TRN) {
                const u32x4 x = draw(C.seed, (uint32_t)step, (uint32_t)t, P_JITTER);
                const float u[3] = {u01f(x.x), u01f(x.y), u01f(x.z)};
                for (int i = 0; i < 3; ++i) {
                    float d = u[i] * C.dx;
                    if (c[i] + d > C.L[i] + C.start[i]) d = d - C.L[i];
                    if (c[i] + d < C.start[i]) d = d + C.L[i];
                    c[i] = c[i] + d;
                }
            }
        }
        C.tc[t] = make_float4(c[0], c[1], c[2], 0.f);
    }
    if (tid == 0) {
        S.kind = kind;
        S.sp = spi;
        S.k = k;
        S.nitems = k;
        S.done = 0;
    }
    __syncthreads();
    return make_move(kind, spi, k, step);
}

template <int NT>
__device__ inline Move prep_step(CRep &C, State &S, const Lds &L)
{
    return prep_step<NT>(C, S, L, false, 0, 0);
}

// Trials a workgroup takes with one claim of a move of nitems trials, unc of
// them unclaimed: of a small move (COOP_TRIALS) one per team, two while more than
// 4 are left; of a larger move two per wave, so that waves whose trials end
// early take over, and one per wave when few are left.  With few systems per XCD
// (nc < 4) the workgroups would idle while a few of them work through a move's
// trials, so a claim then takes no more than a fair share, ceil(unc / workgroups
// of the XCD).
template <int NT>
__device__ inline int claim_take(int nitems, int unc, int nc, int nwx)
{
    constexpr int NW = NT / 64;
    const int want = nitems <= COOP_TRIALS ? (unc > 4 ? 2 : 1) * (NW / COOP) : NW;
    if (nc >= 4) return want;
    const int share = (unc + nwx - 1) / nwx;
    return min(want, max(share, 1));
}

// XCD-local ordering.  Every workgroup touching a replica in the batched form
// runs on the same XCD, whose L2 is shared and whose L1s are write-through: a
// release waits until this thread's memory operations reached L2; an acquire
// invalidates the CU's L1 at device scope (sc1) so later loads read L2 -- a
// workgroup-scope invalidate (sc0) leaves L1 as it is, since one workgroup's
// waves share that L1.  No L2 write-back: replica data never leaves the XCD.
__device__ inline void xcd_release() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
__device__ inline void xcd_acquire() { asm volatile("buffer_inv sc1" ::: "memory"); }

// claim-word priority of a replica's published move: lower is claimed first,
// the replica with the most estimated work left first -- the run lasts as long
// as its slowest chain
__device__ inline int claim_prio(CRep &C, int step, int end)
{
    const uint32_t left = C.wcum[end] - C.wcum[step];
    return 0xFFFFFF - (int)(left < 0xFFFFFFu ? left : 0xFFFFFFu);
}

// Advance past empty moves, prepare the next move with trials and publish it
// (batched form), the first `keep` of its trials (claim_take of the move, nc and
// nwx as there) claimed for this workgroup, which goes on with them: a small
// move then needs neither the other workgroups' polls nor a claim, and nothing
// is published of a move that this workgroup takes whole.  None are kept where an
// XCD has more replicas (nc) than workgroups (nwx): those left out would start only
// when others have ended.
// use_pre: the move after prev_step (species prev_spi) is in L.misc[M_NX..]
// Returns the move (k = 0 at the end of the run) and the trials kept.
template <int NT>
__device__ inline Move advance_and_publish(CRep &C, State &S, Sched *sch, const Lds &L, bool use_pre,
                                           int prev_step, int prev_spi, int nc, int nwx, int &keep)
{
    Move mv;
    while (true) {
        if (use_pre ? prev_step + 1 >= L.misc[M_NX + 0] : S.step >= S.end) {
            xcd_release();
            __syncthreads();
            if (threadIdx.x == 0) {
                __hip_atomic_store(&S.claim, claim_word(0xFFFFFF, 0, 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_fetch_add(&sch->finished, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            mv.k = keep = 0;
            break;
        }
        int end;
        if (use_pre) end = L.misc[M_NX + 0];
        else end = S.end;
        mv = prep_step<NT>(C, S, L, use_pre, prev_step, prev_spi);
        use_pre = false;
        if (mv.k > 0) {
            keep = nc <= nwx ? min(claim_take<NT>(mv.nitems, mv.nitems, nc, nwx), mv.nitems) : 0;
            if (threadIdx.x == 0) {
                S.t_pub = wall_clock64();
                L.misc[M_NEXT] = 0;
            }
            if (keep < mv.nitems) {
                const int prio = claim_prio(C, mv.step, end);
                if (threadIdx.x == 0)
                    __hip_atomic_store(&S.done, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                xcd_release();
                __syncthreads();
                if (threadIdx.x == 0) {
                    // every thread's writes have completed: a CU whose L1 was
                    // invalidated after this time holds no older copy of them
                    S.t_data = wall_clock64();
                    xcd_release();
                    __hip_atomic_store(&S.claim, claim_word(prio, mv.nitems, keep), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            break;
        }
        skip_move(C, S);
    }
    __syncthreads();
    return mv;
}

// ---- kernels ---------------------------------------------------------------------

// start of a run: set the end step of every replica and reset the scheduler
__global__ void k_begin(State *st, const Rep *reps, int r0, int nrep, int nsteps, Sched *sch)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) {
        sch->finished = 0;
        sch->abort = 0;
        sch->progress = 0;
    }
    if (i < nrep) {
        State &S = st[r0 + i];
        const long long e = (long long)S.step + nsteps;
        S.end = (int)(e < reps[r0 + i].nmoves ? e : reps[r0 + i].nmoves);
    }
}

// prepare the current move of replicas r0 + blockIdx.x (batched: publish it)
template <int NT, bool STAGED>
__global__ __launch_bounds__(NT) void k_start(const Rep *reps, State *st, Sched *sch, LdsLayout lay,
                                             int r0, int batched)
{
    extern __shared__ __align__(16) char smem[];
    const Lds L = carve(smem, lay);
    const int r = r0 + blockIdx.x;
    int keep;
    // (Ewald) the last move's charge changes are in the grid by now
    if (rep_of(reps, r).ew && threadIdx.x == 0) *rep_of(reps, r).pme_ndelta = 0;
    if (batched) advance_and_publish<NT>(rep_of(reps, r), st[r], sch, L, false, 0, 0, 1, 0, keep);
    else if (st[r].step < st[r].end) prep_step<NT>(rep_of(reps, r), st[r], L);
}

// the current move's trials, as many per workgroup as it has teams or waves
template <int NT, bool STAGED, int TM>
__global__ __launch_bounds__(NT) void k_eval_plain(const Rep *reps, State *st, int r, LdsLayout lay)
{
    extern __shared__ __align__(16) char smem[];
    State &S = st[r];
    if (S.step >= S.end) return;
    const Move mv = move_of(S);
    const int per = mv.coop ? NT / 64 / COOP : NT / 64;
    const int item = blockIdx.x * per;
    if (item >= mv.nitems) return;
    const Lds L = carve(smem, lay);
    CRep &C = rep_of(reps, r);
    if (threadIdx.x == 0) L.misc[M_NEXT] = 0;
    if (threadIdx.x < 4) L.misc[M_TICKS + threadIdx.x] = 0;
    stage_tables<NT, STAGED>(C, L, true, true);
    ItemStats ist{};
    eval_items<NT, STAGED, TM>(C, mv, item, min(per, mv.nitems - item), L, ist);
    if ((threadIdx.x & 63) == 0 && ist.neval) add_item_stats<false>(S, ist, species_of(C, mv.spi).nf);
    __syncthreads();
    if (threadIdx.x < 4) {
        const int t = L.misc[M_TICKS + threadIdx.x];
        if (t != 0) count_add<false>(&S.t_sub[threadIdx.x], (unsigned long long)t * TICKED);
    }
}

template <int NT, bool STAGED, bool EW>
__global__ __launch_bounds__(NT) void k_accept_plain(const Rep *reps, State *st, int r, LdsLayout lay)
{
    extern __shared__ __align__(16) char smem[];
    State &S = st[r];
    if (S.step >= S.end) return;
    const Lds L = carve(smem, lay);
    accept_step<NT, EW>(rep_of(reps, r), S, L);
    if (S.step < S.end) prep_step<NT>(rep_of(reps, r), S, L);
}

// Which replicas a workgroup serves: the XCD it runs on (XCC_ID hardware
// register) selects a class; class c owns replicas cls_reps[cls_start[c] ..
// cls_start[c+1]).  xcc_class maps XCC ids to classes (-1: none).
struct XcdMap {
    int nclass;
    int xcc_class[16];
    const int *cls_start;
    const int *cls_reps;
    unsigned long long *cu_inv;   // [CU_SLOTS] time of each CU's last L1 invalidate (100 MHz ticks)
};

__device__ inline int my_xcc() { return (int)(__builtin_amdgcn_s_getreg((20) | (0 << 6) | (15 << 11)) & 0xf); }

// This CU's slot in XcdMap::cu_inv: XCC id, shader engine, shader array and
// CU id from the XCC_ID and HW_ID registers (distinct for distinct CUs).
constexpr int CU_SLOTS = 4096;
__device__ inline int my_cu_slot()
{
    const unsigned hw = __builtin_amdgcn_s_getreg((4) | (0 << 6) | (31 << 11));
    const unsigned cu = (hw >> 8) & 15u, sh = (hw >> 12) & 1u, se = (hw >> 13) & 7u;
    return (int)(((unsigned)my_xcc() << 8) | (se << 5) | (sh << 4) | cu);
}

// The acquire before evaluating a claimed move's items is a device-scope L1
// invalidate, which also empties the L1 of the CU's other workgroups.  It is
// needed only when the CU's L1 may hold lines older than the move's data:
// not when this CU's last invalidate came after the move's data was complete
// (State::t_data).  One thread asks; both times are read at device scope.
__device__ inline int cu_acquire_needed(const State &S, const unsigned long long *cu_inv, int slot)
{
    const unsigned long long td = __hip_atomic_load(&S.t_data, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long last = __hip_atomic_load(&cu_inv[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return last >= td ? 0 : 1;
}

// persistent form: workgroups of an XCD claim evaluations from that XCD's
// replicas; the workgroup completing a replica's last evaluation runs its
// accept and prep phases and publishes the next move.  A replica with Ewald
// electrostatics (TM == T_EWALD) stops after a move that changed its charges: the
// potential has to be solved anew first (moves that change nothing, about half
// of a slab's, go on at once).  Exits when `target` replicas (counted from the
// scheduler's reset) finished or stopped, or when no replica advanced during
// spin_limit polls (then sch->abort is set).
template <int NT, bool STAGED, int TM>
__global__ __launch_bounds__(NT, 3) void k_batched(const Rep *reps, State *st, int target, Sched *sch,
                                               LdsLayout lay, int spin_limit, XcdMap xm, int aff)
{
    extern __shared__ __align__(16) char smem[];
    const Lds L = carve(smem, lay);
    const int tid = threadIdx.x;
    const int cls = xm.xcc_class[my_xcc()];
    if (cls < 0) return;
    const int c0 = xm.cls_start[cls], nc = xm.cls_start[cls + 1] - c0;
    if (nc <= 0) return;
    const int rot = (int)(blockIdx.x / (unsigned)xm.nclass) % nc;
    const int nwx = max((int)(gridDim.x / (unsigned)xm.nclass), 1);   // workgroups per XCD
    const int slot = my_cu_slot();
    int idle = 0, seen = -1;
    // replica whose species table, and pair table (Rep::tab) that are in LDS
    int cached_rep = -1, cached_tab = -1;
    // the trials this workgroup kept of a move it published (advance_and_publish)
    int kept = 0, kept_rep = -1;
    Move mv;
    if (tid < 4) L.misc[M_TICKS + tid] = 0;   // (a claim's barriers come before the first use)
    while (true) {
        int found, item, cnt;
        if (kept > 0) {
            found = kept_rep;
            item = 0;
            cnt = kept;
        } else {
            if (tid < 64) {
                // wave 0 polls every replica of this XCD at once, one claim word
                // per lane.  Claim words are device-scope: a workgroup-scope load
                // may hit this CU's L1, which only a claiming workgroup invalidates,
                // so idle workgroups would keep seeing an old word.  Polls are
                // loads; an atomic is issued only to claim (read-modify-writes of
                // one address serialize).  The scheduler's words (progress,
                // finished, abort) are read only when nothing could be claimed:
                // a workgroup that finds work goes from its last item to its next
                // with two memory round trips (the claim words, the claim).
                const int lane = tid;
                int rfound = -1, ritem = 0, rcnt = 1;
                for (int b0 = 0; b0 < nc && rfound < 0; b0 += 64) {
                    int r = -1;
                    unsigned long long w = 0ull;
                    if (b0 + lane < nc) {
                        r = xm.cls_reps[c0 + (rot + b0 + lane) % nc];
                        w = __hip_atomic_load(&st[r].claim, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                    bool avail = r >= 0 && (w & 0xFFFFFull) < ((w >> 20) & 0xFFFFFull);
                    // Moves with few unclaimed items first (up to 4, then up to
                    // 16): a replica waiting on one or a few evaluations is on its
                    // own critical chain.  Within those classes and among the
                    // larger moves, the replica with the most estimated work left
                    // first (claim_prio): the run ends with its last replica, and
                    // a large move occupies the XCD's workgroups for several
                    // rounds whichever order they come in.  (Fewest unclaimed
                    // items first among the large moves too: 5 % slower.)
                    const unsigned long long unc = ((w >> 20) & 0xFFFFFull) - (w & 0xFFFFFull);
                    unsigned size = unc <= 4ull ? 0u : (unc <= 16ull ? 1u : 2u);
                    // affinity (aff > 0): a move of at least aff unclaimed items
                    // of the replica whose tables this workgroup holds in LDS
                    // comes before the other such moves (its species table and
                    // staged pair table are reused)
                    if (aff > 0 && unc >= (unsigned long long)aff) size = (r == cached_rep) ? 2u : 3u;
                    const unsigned prio = (unsigned)(w >> 40) >> 8;
                    const int take_lane = claim_take<NT>((int)((w >> 20) & 0xFFFFFull), (int)unc, nc, nwx);
                    while (__ballot(avail) != 0ull) {
                        const unsigned key =
                            wave_min(avail ? ((size << 22) | (prio << 6) | (unsigned)lane) : 0xFFFFFFFFu);
                        const int l = (int)(key & 63u);
                        const int rr = __shfl(r, l, 64);
                        const int take = __shfl(take_lane, l, 64);
                        unsigned long long old = 0ull;
                        if (lane == l)
                            old = __hip_atomic_fetch_add(&st[rr].claim, (unsigned long long)take, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_AGENT);
                        old = __shfl(old, l, 64);
                        const int c = (int)(old & 0xFFFFFull), n = (int)((old >> 20) & 0xFFFFFull);
                        if (c < n) {
                            rfound = rr;
                            ritem = c;
                            rcnt = min(take, n - c);
                            break;
                        }
                        if (lane == l) avail = false;
                    }
                }
                if (rfound == -1) {
                    int ctl[3] = {0, 0, 0};
                    if (lane == 0) {
                        ctl[0] = __hip_atomic_load(&sch->progress, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        ctl[1] = __hip_atomic_load(&sch->finished, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        ctl[2] = __hip_atomic_load(&sch->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                    const int prog = __shfl(ctl[0], 0, 64), fin = __shfl(ctl[1], 0, 64), ab = __shfl(ctl[2], 0, 64);
                    if (prog != seen) {
                        seen = prog;
                        idle = 0;
                    }
                    if (fin >= target || ab != 0) {
                        rfound = -2;
                    } else if (++idle > spin_limit) {
                        // no replica advanced during spin_limit polls: stop instead of hanging
                        if (lane == 0) __hip_atomic_store(&sch->abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        rfound = -2;
                    }
                }
                if (lane == 0) {
                    L.misc[M_FOUND] = rfound;
                    L.misc[M_ITEM] = ritem;
                    L.misc[M_CNT] = rcnt;
                    L.misc[M_NEXT] = 0;
                    L.misc[M_INV] = rfound >= 0 ? cu_acquire_needed(st[rfound], xm.cu_inv, slot) : 1;
                }
            }
            __syncthreads();
            // uniform across the workgroup: the replica's fields become scalar loads
            found = __builtin_amdgcn_readfirstlane(L.misc[M_FOUND]);
            item = __builtin_amdgcn_readfirstlane(L.misc[M_ITEM]);
            cnt = __builtin_amdgcn_readfirstlane(L.misc[M_CNT]);
            const int need_inv = __builtin_amdgcn_readfirstlane(L.misc[M_INV]);
            __syncthreads();
            if (found == -2) break;
            if (found == -1) {
                // about 0.9 us between polls of an idle workgroup (1.5 % faster
                // than 0.2 us on short runs of the 64-replica workload, equal to
                // 0.45-1.8 us on full runs; evaluation times do not change)
                __builtin_amdgcn_s_sleep(32);
                continue;
            }
            if (need_inv) {
                const unsigned long long tinv = wall_clock64();
                xcd_acquire();
                if (tid == 0) {
                    // recorded once this wave's invalidate has executed
                    xcd_release();
                    __hip_atomic_store(&xm.cu_inv[slot], tinv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            mv = move_of(st[found]);
        }
        CRep &C = rep_of(reps, found);
        State &S = st[found];
        const unsigned long long te0 = wall_clock64();
        const int tab = C.tab;
        // the species table stays in LDS while a workgroup keeps evaluating
        // trials of one replica, the pair table while it keeps to replicas with
        // that table
        stage_tables<NT, STAGED>(C, L, found != cached_rep, tab != cached_tab);
        ItemStats ist{};
        // a small move's evaluations are its replica's serial path: ahead of the
        // large moves' waves sharing the SIMDs (3 % of a pass)
        if (mv.k <= 16) __builtin_amdgcn_s_setprio(2);
        eval_items<NT, STAGED, TM>(C, mv, item, cnt, L, ist);
        __builtin_amdgcn_s_setprio(0);
        cached_rep = found;
        cached_tab = tab;
        kept = 0;
        const unsigned long long te1 = wall_clock64();
        bool last = cnt == mv.nitems;   // the whole move is this workgroup's
        if (!last) {
            xcd_release();
            __syncthreads();
            if (tid == 0) {
                const int old = __hip_atomic_fetch_add(&S.done, cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                L.misc[M_LAST] = (old + cnt == mv.nitems) ? 1 : 0;
            }
            __syncthreads();
            last = uniform_i(L.misc[M_LAST]) != 0;
            // other workgroups' energies and poses
            if (last) xcd_acquire();
        } else {
            __syncthreads();
        }
        // statistics after the completion count: the release above does not
        // wait for them
        if (tid == 0) count_add<true>(&S.t_eval, te1 - te0);
        if ((tid & 63) == 0 && ist.neval) add_item_stats<true>(S, ist, species_of(C, mv.spi).nf);
        if (last) {
            // accept and prep are this replica's serial critical path: issue
            // ahead of the evaluation waves sharing the SIMDs
            __builtin_amdgcn_s_setprio(3);
            const unsigned long long ta0 = wall_clock64();
            const unsigned long long tpub = S.t_pub;
            const MoveCtx mc = move_ctx(fresh(C), S);
            accept_move<NT, TM == T_EWALD>(fresh(C), S, L, mc, true);
            const unsigned long long ta1 = wall_clock64();
            if (TM == T_EWALD && uniform_i(L.misc[M_ACC]) != 0) {
                // stopped: k_start publishes the next move after the solve
                xcd_release();
                __syncthreads();
                if (tid == 0) {
                    __hip_atomic_store(&S.claim, claim_word(0xFFFFFF, 0, 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_fetch_add(&sch->finished, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            } else {
                mv = advance_and_publish<NT>(fresh(C), S, sch, L, true, mc.step, mc.spi, nc, nwx, kept);
                kept_rep = found;
            }
            if (tid == 0) {
                const unsigned long long ta2 = wall_clock64();
                // timers after the next move is published, off its path; the
                // workgroup that finishes that move may already be adding its
                // own, so these are atomic adds too
                count_add<true>(&S.t_step, ta0 - tpub);
                count_add<true>(&S.t_accept, ta1 - ta0);
                count_add<true>(&S.t_prep, ta2 - ta1);
                int row;
                if (tracing(C, mc.step, row)) {
                    C.tr.tick[4 * row + 0] = tpub;
                    C.tr.tick[4 * row + 1] = ta0;
                    C.tr.tick[4 * row + 2] = ta1;
                    C.tr.tick[4 * row + 3] = ta2;
                }
                __hip_atomic_fetch_add(&sch->progress, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            __builtin_amdgcn_s_setprio(0);
        }
        // the phases of this replica's trials, complete since the barrier after them:
        // when the workgroup leaves the replica (a kept move follows at once), and now
        // and then
        if ((kept == 0 || (mv.step & 255) == 0) && tid < 4) {
            const int t = L.misc[M_TICKS + tid];
            if (t != 0) {
                count_add<true>(&S.t_sub[tid], (unsigned long long)t * TICKED);
                L.misc[M_TICKS + tid] = 0;
            }
        }
        __syncthreads();
    }
}

// A replica's state as the caller holds it, one word per thread: head takes the
// species' counts and the group centres (x, y, z), atoms the records (x, y, z,
// charge, type).  (Copied as they lie here and converted by the host, the states
// of 64 systems of some 100,000 atom slots each took 38 ms.)
__global__ void k_pack_state(const Rep *reps, const State *st, int r, int nsp, int nres, int natom, int *head,
                             int *atoms)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    CRep &C = rep_of(reps, r);
    if (i < nsp) head[i] = st[r].totalNum[i];
    if (i < 3 * nres) head[nsp + i] = ((const int *)C.res_pos)[i / 3 * 4 + i % 3];
    if (i < 5 * natom) {
        const int a = i / 5, c = i - 5 * a;
        atoms[i] = c < 4 ? ((const int *)C.atom)[4 * a + c] : C.atype[a];
    }
}

// XCC id of each workgroup (engine set-up: which XCDs exist)
__global__ void k_xcc_probe(int *out)
{
    if (threadIdx.x == 0) out[blockIdx.x] = my_xcc();
}

// lane i's value, in every lane
__device__ __forceinline__ float lane_f(float x, int i)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), i));
}

// Energies of given poses: one wave per pose, or (few poses) four that share
// its cells.
template <int NT, bool STAGED, int TM, int PARTS>
__global__ __launch_bounds__(NT) void k_eval_poses(const Rep *reps, int r, int spi, int npose, const float *centres,
                                                  const float *poses, const int *excl, double *E, int *ninc,
                                                  uint32_t *hash, LdsLayout lay)
{
    extern __shared__ __align__(16) char smem[];
    constexpr int PER = NT / 64 / PARTS;
    const Lds L = carve(smem, lay);
    CRep &C = rep_of(reps, r);
    CSpecies &F = species_of(C, spi);
    const int nf = F.nf, lane = threadIdx.x & 63, wave = uniform_i(threadIdx.x >> 6), part = wave % PARTS;
    const WaveLds W = wave_lds(L, wave);
    if (threadIdx.x == 0) L.misc[M_NEXT] = PER;
    stage_tables<NT, STAGED>(C, L, true, true);
    // this workgroup's poses; with one wave per pose each takes the next one when
    // it is done (in turn: 133 us for 16,384 benzene poses, a wave with costly
    // ones last; so: 106)
    const int p0 = (int)((long long)npose * blockIdx.x / gridDim.x);
    const int p1 = (int)((long long)npose * (blockIdx.x + 1) / gridDim.x);
    // a pose by one load per lane: 3 nf coordinates, the centre, the excluded
    // molecule (the arrays may lie in host memory)
    auto fetch = [&](int k) {
        const size_t q = (size_t)min(p0 + k, p1 - 1);
        const int *src = (const int *)poses + q * 3 * nf + lane;
        if (lane >= 60) src = lane < 63 ? (const int *)centres + 3 * q + (lane - 60) : excl + q;
        return lane < 3 * nf || lane >= 60 ? *src : 0;
    };
    auto next = [&](int k) {
        if (PARTS > 1) return k + PER;
        int n = 0;
        if (lane == 0) n = atomicAdd(&L.misc[M_NEXT], 1);
        return uniform_i(n);
    };
    int k = wave / PARTS;
    if (p0 >= p1) return;
    int in = fetch(k);
    while (p0 + (PARTS == 1 ? k : k - wave / PARTS) < p1) {
        const int i = p0 + k, kn = next(k), v = in;
        in = fetch(kn);
        const float vf = __int_as_float(v), c[3] = {lane_f(vf, 60), lane_f(vf, 61), lane_f(vf, 62)};
        const int x = __builtin_amdgcn_readlane(v, 63);
        const float px = __shfl(vf, min(3 * lane, 63)), py = __shfl(vf, min(3 * lane + 1, 63)),
                    pz = __shfl(vf, min(3 * lane + 2, 63));
        if (lane < nf) order_pose<TM>(C, F, W, 0, lane, make_float4(px, py, pz, F.kq[lane]), c);
        wave_sync();
        PoseSums s;
        NoTicks nt;
        eval_poses_wave<STAGED, TM>(C, L, W, spi, nf, 1, c, c, true, x, false, part, PARTS, s, nt);
        if (TM == T_EWALD) {
            const bool own = x >= F.startRes && x < F.startRes + F.maxNum;
            s.e[0] += ewald_recip(C, F, W, 0, nf, own ? F.atomBase + (x - F.startRes) * nf : -1, part, PARTS);
        }
        if (PARTS > 1) team_sum<NT>(L, s);
        if (i < p1 && part == 0 && lane == 0) {
            E[i] = s.e[0];
            ninc[i] = s.nin[0];
            hash[i] = s.hash[0];
        }
        wave_sync();
        k = kn;
    }
}

}  // namespace gcmc
