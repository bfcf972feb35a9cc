// Plane means and flux relaxation of the optional FLUXES branches (FP64 form).
//
// HORIZONTAL_MEAN (3dmhdsub.f:3143-3223, NGRID=0 branch) is reproduced in the
// reference's own summation order for an NPEY-slab decomposition: each slab
// (rows j = s*NRY .. s*NRY+NRY-1 of a plane) is summed sequentially, rows
// outer and points inner, then divided by FLOAT(NPX*NPY), and the slab
// quotients are added in slab order.  One wavefront per (plane, slab) forms
// a slab's sum; one workgroup combines them per plane.  The means feed
//   ROM   density diffusion (ID, sub:1301-1371), with the ghost planes of RO
//         holding the mirrored planes 2 and npz-1 (ID or LREM);
//   TTM   Rempel conduction (LREM, sub:1536-1581) and the relaxation;
//   HRAD  the radiative heating of the mean profile (LREM, sub:1567-1573);
//   radd  RLAX*TFAC*CORRECT(K) of the flux relaxation (sub:1615-1765), whose
//         saved factor TFAC and maximum TTM_MAX live in RelaxState and whose
//         vertical integral runs rank by rank over an NPEZ-rank decomposition
//         as the reference's does.
// These run on the stage input before each stage kernel, in the reference's
// arithmetic order.

#include "mhd_kernels.h"

namespace rmhd {

namespace {

// The reference's sums are one sequential chain per slab (rows outer, points
// inner; the slab is a contiguous run of NRY*NPX points of the plane).  A
// workgroup per (plane, slab) stages the run through LDS in chunks of
// SUM_CHUNK values (coalesced, double-buffered) and its thread 0 adds them
// in order, so the chain runs at the latency of an FP64 add instead of that
// of a dependent global load (k_fconm_sums, whose summands change sign).
constexpr int SUM_T = 256, SUM_CHUNK = 1024;

// sum + v[0] + v[1] + ... + v[m-1], added one by one in this order; the LDS
// reads of a group of 8 are issued before its adds.
__device__ __forceinline__ double chain_add(double sum, const double *v, int m) {
    int i = 0;
    for (; i + 8 <= m; i += 8) {
        double x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = v[i + u];
#pragma unroll
        for (int u = 0; u < 8; ++u) sum = sum + x[u];
    }
    for (; i < m; ++i) sum = sum + v[i];
    return sum;
}

// The same chain by one wavefront, eight rows of 64 values at a time.  While the
// running sum s stays in one binade, where its unit in the last place is u,
// RN(s + x) = s + RN_u(x) unless x lies halfway between two multiples of u:
// rounding to a multiple of u does not depend on s.  So every lane rounds its
// values to multiples of u and those are added in any order, exactly; the result
// is the chain's bit for bit.  A row that may leave the binade, holds a halfway
// case or a value not of s's sign is added value by value in order, and the rest
// of its block is rounded again if the binade changed.  s doubles ever more
// rarely, and halfway cases die out as it outgrows the values: of the 144 rows of
// a 96x96 plane about 15 go value by value.  What bounds it is the instructions
// of the one wavefront (96x96: 67 us as a chain of adds behind LDS
// reads, 28 us so).
constexpr int SUM_ROWS = 8;

__device__ __forceinline__ double lane_value(double v, int lane) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}

// In every row of 16 lanes: s + x of its lane 0 + ... + x of its lane 15, one
// by one.  One instruction an add: x * 1 + s rounds once, x broadcast within the
// row on the way.  (The wait states around it are the hardware's: a lane's value
// read by DPP or by readlane right after it is written.)
__device__ __forceinline__ double chain16(double s, double x) {
    const double one = 1.0;
#define ADD_LANE(l) "v_fmac_f64_dpp %0, %1, %2 row_newbcast:" #l " row_mask:0xf bank_mask:0xf\n"
    asm("s_nop 1\n" ADD_LANE(0) ADD_LANE(1) ADD_LANE(2) ADD_LANE(3) ADD_LANE(4) ADD_LANE(5) ADD_LANE(6) ADD_LANE(7)
            ADD_LANE(8) ADD_LANE(9) ADD_LANE(10) ADD_LANE(11) ADD_LANE(12) ADD_LANE(13) ADD_LANE(14) ADD_LANE(15)
        "s_nop 1"
        : "+v"(s)
        : "v"(x), "v"(one));
#undef ADD_LANE
    return s;
}

// v of the lane that DPP control CTRL names.
constexpr int DPP_XOR1 = 0xb1, DPP_XOR2 = 0x4e, DPP_XOR7 = 0x141, DPP_XOR8 = 0x128;
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xf, 0xf, true);
    const unsigned hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}

// One step of a sum of several values over the lanes: a lane with `up` keeps b,
// its partner keeps a.
template <int CTRL>
__device__ __forceinline__ double fold(bool up, double a, double b) {
    return (up ? b : a) + dpp<CTRL>(up ? a : b);
}

// Row sums of m[0..7]: on return lane l holds the sum over all lanes of row
// 4 (l >> 2 & 1) + 2 (l & 1) + (l >> 1 & 1).
__device__ __forceinline__ double row_sums(const double *m, int lane) {
    const bool u4 = lane & 4, u1 = lane & 1, u2 = lane & 2;
    double a[4], b[2];
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] = fold<DPP_XOR7>(u4, m[r], m[r + 4]);
    b[0] = fold<DPP_XOR1>(u1, a[0], a[2]);
    b[1] = fold<DPP_XOR1>(u1, a[1], a[3]);
    double v = fold<DPP_XOR2>(u2, b[0], b[1]);
    v = v + dpp<DPP_XOR8>(v);
    v = v + __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}
__device__ __forceinline__ int row_lane(int r) { return (r & 4) | (r & 2) >> 1 | (r & 1) << 1; }

// s + x[0] + ... + x[7] (rows < nrows, each the wavefront's lanes in order).
__device__ __forceinline__ double add_rows(double s, double *x, int nrows, int lane) {
    int r0 = 0;
    for (;;) {
        // s in [lo, hi), both mirrored if s < 0; zero, tiny, huge, NaN: no row qualifies
        const unsigned long long sb = __builtin_bit_cast(unsigned long long, s), e = (sb >> 52) & 0x7ff;
        const bool ok = e > 60 && e < 0x7fd;
        const unsigned long long eu = ok ? e : 1023;
        auto exp2_of = [](unsigned long long n) { return __builtin_bit_cast(double, n << 52); };
        const double lo = exp2_of(eu), hi = exp2_of(eu + 1), half = exp2_of(eu - 53);
        const unsigned quarter = (unsigned)(eu - 2) << 20;
        const double big = 1.5 * lo, sg = (sb >> 63) ? -1.0 : 1.0;
        double m[SUM_ROWS];
        unsigned bad = 0;
#pragma unroll
        for (int r = 0; r < SUM_ROWS; ++r) {
            const double y = __builtin_bit_cast(double, __builtin_bit_cast(unsigned long long, x[r]) ^ (sb & (1ull << 63)));
            m[r] = (y + big) - big;  // RN_u(y): big's unit is u, y < lo / 4
            // 0 <= y < lo / 4, by the upper word (a sign or a NaN is above)
            const unsigned yh = (unsigned)(__builtin_bit_cast(unsigned long long, y) >> 32);
            const unsigned long long good = __builtin_amdgcn_ballot_w64(yh < quarter) &
                                            __builtin_amdgcn_ballot_w64(fabs(y - m[r]) != half);
            if (~good) bad |= 1u << r;
        }
        if (!ok) bad = 0xff;
        // every partial sum lies between s and s + the sums, its exact value within
        // u / 2 of it: below hi if those are (sums past 2^53 u are inexact, but
        // never come out below it)
        const double sums = row_sums(m, lane);
        double all = sums + dpp<DPP_XOR7>(sums);
        all = all + dpp<DPP_XOR1>(all);
        all = lane_value(all + dpp<DPP_XOR2>(all), 0);
        double sa = s * sg;
        if (!(bad >> r0) && sa + all < hi) return (sa + all) * sg;
#pragma unroll 1
        for (;; ++r0) {
            if (r0 == nrows) return sa * sg;
            const double t = sa + lane_value(sums, row_lane(r0));
            if (!(bad >> r0 & 1) && t < hi) {
                sa = t;
                continue;
            }
            double v = x[0];
#pragma unroll
            for (int g = 1; g < SUM_ROWS; ++g) v = r0 == g ? x[g] : v;
            s = sa * sg;
#pragma unroll
            for (int g = 0; g < 64; g += 16) s = lane_value(chain16(s, v), g);
            sa = s * sg;
            if (!(sa >= lo && sa < hi) || !ok) break;
        }
        // the binade has changed: the rows after r0 once more
        ++r0;
#pragma unroll
        for (int r = 0; r < SUM_ROWS; ++r) x[r] = r < r0 ? 0.0 : x[r];
        if (r0 == nrows) return s;
    }
}

// Slab sums of plane k (0..npz+1) of RO (WHAT & 1) and TT (WHAT & 2), one
// wavefront each.  means: a slab is the whole plane and nothing else follows,
// so the wavefront writes the plane's means itself (no k_plane_means, 5 us).
template <int WHAT>
__global__ __launch_bounds__(64) void k_slab_sums(const Params p, const double *__restrict__ q,
                                                  double *__restrict__ part, double *__restrict__ rom,
                                                  double *__restrict__ wwz, double *__restrict__ ttm, int means) {
    const int npl = p.npz + 2, nsl = p.npey;
    const int f = WHAT == 3 ? (int)(blockIdx.x & 1) : WHAT - 1;  // RO, TT
    const int b = WHAT == 3 ? (int)(blockIdx.x >> 1) : (int)blockIdx.x;  // b = k * nsl + sl
    const int k = b / nsl, sl = b - k * nsl;
    const int nry = p.npy / nsl;
    const long long fs = p.fsize, pl = p.plane, n = (long long)nry * p.npx;
    int kr = k;
    if (p.mirror && f == 0 && k == 0) kr = 2;
    if (p.mirror && f == 0 && k == p.npz + 1) kr = p.npz - 1;
    const double *src = q + (3 + f) * fs + (long long)kr * pl + (long long)sl * nry * p.npx;
    constexpr int BLOCK = 64 * SUM_ROWS;
    double x[SUM_ROWS], next[SUM_ROWS];
    auto load = [&](long long c0) __attribute__((always_inline)) {
        const double *at = src + c0;
        if (c0 + BLOCK <= n) {
#pragma unroll
            for (int r = 0; r < SUM_ROWS; ++r) next[r] = at[r * 64 + threadIdx.x];
        } else {
            const int m = (int)(n - c0);
#pragma unroll
            for (int r = 0; r < SUM_ROWS; ++r) {
                const int i = r * 64 + threadIdx.x;
                next[r] = at[i < m ? i : m - 1];
                if (i >= m) next[r] = 0.0;  // s + 0 is s: s is never -0
            }
        }
    };
    double s = 0.0;
    load(0);
    for (long long c = 0; c < n; c += BLOCK) {
#pragma unroll
        for (int r = 0; r < SUM_ROWS; ++r) x[r] = next[r];
        if (c + BLOCK < n) load(c + BLOCK);
        s = add_rows(s, x, c + BLOCK <= n ? SUM_ROWS : (int)((n - c + 63) / 64), threadIdx.x);
    }
    if (threadIdx.x != 0) return;
    if (!means) {
        part[(long long)f * npl * nsl + b] = s;
        return;
    }
    const double mean = s / (double)(float)(p.npx * p.npy);
    if (f == 0) {
        rom[k] = mean;
        if (p.id == 1) wwz[k] = 1.0 / mean;  // sub:1323-1325
    } else {
        ttm[k] = mean;
    }
}

// The slab quotients of plane k added in slab order.
__device__ __forceinline__ double slab_mean(const Params &p, const double *part, int k) {
    const double cnt = (double)(float)(p.npx * p.npy);
    double v = 0.0;
    for (int sl = 0; sl < p.npey; ++sl) {
        const double w = part[k * p.npey + sl] / cnt;
        v = sl == 0 ? w : v + w;
    }
    return v;
}

// One workgroup: ROM, WWZ (ID=1), TTM, then HRAD (LREM).
__global__ void k_plane_means(const Params p, const Metrics m, const double *__restrict__ part, double *rom,
                              double *wwz, double *ttm, double *hrad, int what) {
    const int npl = p.npz + 2;
    for (int k = threadIdx.x; k < npl; k += blockDim.x) {
        if (what & 1) {
            const double v = slab_mean(p, part, k);
            rom[k] = v;
            if (p.id == 1) wwz[k] = 1.0 / v;  // sub:1323-1325
        }
        if (what & 2) ttm[k] = slab_mean(p, part + (size_t)npl * p.npey, k);
    }
    __syncthreads();
    if (p.lrem) {
        for (int k = 1 + threadIdx.x; k <= p.npz; k += blockDim.x) {
            const double tp1 = ttm[k + 1], t0 = ttm[k], tm1 = ttm[k - 1];
            hrad[k] = ((tp1 - 2.0 * t0 + tm1) * p.h2z * m.dzzdz[k] * m.dzzdz[k] + (tp1 - tm1) * p.hz * m.d2zzdz2[k])
                          * m.rkapa[k]
                      + (tp1 - tm1) * p.hz * m.dzzdz[k] * m.dkapa[k];
        }
    }
}

// Slab sums of the convective-flux summand -RW*(2.5*(TT-TTM) + 0.5*|u|^2) of
// planes k = 1..npz+1 (sub:1653-1662); u = RU*(1/RO) as FLUXES forms it.  The
// summands are formed by the staging threads, the chain by thread 0, as in
// k_slab_sums.
__global__ __launch_bounds__(SUM_T) void k_fconm_sums(const Params p, const double *__restrict__ q,
                                                      const double *__restrict__ ttm, double *__restrict__ part) {
    __shared__ double buf[2][SUM_CHUNK];
    const int nsl = p.npey;
    const int b = blockIdx.x;  // b = (k - 1) * nsl + sl
    const int k = 1 + b / nsl, sl = b % nsl;
    const int nry = p.npy / nsl;
    const long long fs = p.fsize, pl = p.plane, n = (long long)nry * p.npx;
    const long long so = (long long)sl * nry * p.npx;
    const int kr = (p.mirror && k == p.npz + 1) ? p.npz - 1 : k;
    const double *ru = q + (long long)k * pl + so, *rv = q + fs + (long long)k * pl + so;
    const double *rw = q + 2 * fs + (long long)k * pl + so;
    const double *ro = q + 3 * fs + (long long)kr * pl + so, *tt = q + 4 * fs + (long long)k * pl + so;
    const double tm = ttm[k];
    auto stage = [&](long long c0, int slot) {
        for (int i = threadIdx.x; i < SUM_CHUNK; i += SUM_T) {
            const long long o = c0 + i;
            if (o < n) {
                const double ri = 1.0 / ro[o];
                const double uu = ru[o] * ri, vv = rv[o] * ri, ww = rw[o] * ri;
                buf[slot][i] = -(rw[o] * (2.5 * (tt[o] - tm) + 0.5 * (uu * uu + vv * vv + ww * ww)));
            }
        }
    };
    double sum = 0.0;
    const long long nch = (n + SUM_CHUNK - 1) / SUM_CHUNK;
    stage(0, 0);
    __syncthreads();
    for (long long c = 0; c < nch; ++c) {
        const int slot = (int)(c & 1);
        if (c + 1 < nch) stage((c + 1) * SUM_CHUNK, slot ^ 1);
        if (threadIdx.x == 0) sum = chain_add(sum, buf[slot], (int)min((long long)SUM_CHUNK, n - c * SUM_CHUNK));
        __syncthreads();
    }
    if (threadIdx.x == 0) part[k * nsl + sl] = sum;
}

// One thread: TFAC, FCONM, FRADM, ALPHA and the per-rank integral CORRECT,
// then radd[k] = (RLAX*TFAC)*CORRECT(K) (fixed-T top, fixed-flux bottom).
__global__ void k_relax(const Params p, const Metrics m, const double *__restrict__ zee,
                        const double *__restrict__ part, const double *__restrict__ ttm, double *__restrict__ work,
                        DevScalars *__restrict__ sc, RelaxState *__restrict__ rs, double *__restrict__ radd) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    const int npz = p.npz, npl = npz + 2;
    double *fconm = work, *fradm = work + npl, *corr = work + 2 * npl, *endval = work + 3 * npl;
    double tfac = rs->tfac;
    if (sc->timt > p.tstart && tfac > 1e-4) {
        // the bottom boundary plane's mean temperature (sub:1619-1630)
        const double dt = sc->dt;
        if (ttm[npz] <= rs->ttm_max) {
            tfac = tfac - dt / (3.0 * p.toff);
        } else {
            rs->ttm_max = ttm[npz];
            tfac = tfac + dt / (3.0 * p.toff);
            tfac = fmin(tfac, 2.0);
        }
        for (int k = 1; k <= npz + 1; ++k) fconm[k] = slab_mean(p, part, k);
        // radiative flux (sub:1665-1677): resident plane k is padded K = k+1
        for (int k = 2; k <= npz - 1; ++k)
            fradm[k] = (ttm[k + 1] - ttm[k - 1]) * p.hz * m.dzzdz[k] * m.rkapa[k] / p.repr;
        fradm[1] = (-3.0 * ttm[1] + 4.0 * ttm[2] - ttm[3]) * p.hz * m.dzzdz[1] * m.rkapa[1] / p.repr;
        fradm[npz] = (3.0 * ttm[npz] - 4.0 * ttm[npz - 1] + ttm[npz - 2]) * p.hz * m.dzzdz[npz] * m.rkapa[npz] / p.repr;
        const double ftot = p.lrem ? (double)(8.07f * 0.4f) * p.theta : p.theta / p.repr;
        // per rank, local planes 2..NZ (padded K = pz*NRZ + kl); the bottom
        // rank's last one is its ghost plane and is never used (sub:1693-1705)
        const int nrz = npz / p.npez, nzl = nrz + 2;
        for (int pz = 0; pz < p.npez; ++pz) {
            const int kl_end = pz == p.npez - 1 ? nzl - 1 : nzl;
            double c = 0.0, aprev = 0.0;
            for (int kl = 2; kl <= kl_end; ++kl) {
                const int kg = pz * nrz + kl, k = kg - 1;
                double a = 1.0 - (fconm[k] + fradm[k]) / ftot;
                a = a / (1.0 + 4.0 * fabs(a));
                if (kl == 2) c = 0.0;
                else c = c + 0.5 * (a + aprev) * (zee[kg - 1] - zee[kg - 2]);
                if (kl <= nzl - 1) corr[k] = c;
                aprev = a;
            }
            endval[pz] = c;
        }
        // offsets: the end values of the ranks above, in rank order (sub:1733-1752)
        for (int pz = 0; pz < p.npez; ++pz) {
            double sum = 0.0;
            for (int ipe = 1; ipe <= pz; ++ipe) sum = sum + endval[ipe - 1];
            for (int kl = 2; kl <= nzl - 1; ++kl) corr[pz * nrz + kl - 1] = corr[pz * nrz + kl - 1] + sum;
        }
    } else {
        for (int k = 1; k <= npz; ++k) corr[k] = 0.0;
    }
    rs->tfac = tfac;
    rs->icall = rs->icall + 1;
    const double rt = p.rlax * tfac;
    for (int k = 1; k <= npz; ++k) radd[k] = rt * corr[k];
}

}  // namespace

hipError_t launch_opt_means(const Params &p, const Metrics &m, const double *q, const OptBuffers &o,
                            DevScalars *sc, hipStream_t s) {
    const int npl = p.npz + 2;
    const int what = (p.id != 0 ? 1 : 0) | ((p.lrem || p.rlax > 0.0) ? 2 : 0);
    if (what) {
        const int n = npl * p.npey, means = p.npey == 1 && !p.lrem ? 1 : 0;
        auto sums = [&](auto kernel, int blocks) {
            hipLaunchKernelGGL(kernel, dim3(blocks), dim3(64), 0, s, p, q, o.part, o.rom, o.wwz, o.ttm, means);
        };
        if (what == 1) sums(k_slab_sums<1>, n);
        else if (what == 2) sums(k_slab_sums<2>, n);
        else sums(k_slab_sums<3>, 2 * n);
        if (!means) hipLaunchKernelGGL(k_plane_means, dim3(1), dim3(256), 0, s, p, m, o.part, o.rom, o.wwz, o.ttm, o.hrad, what);
    }
    if (p.rlax > 0.0) {
        const int n = (p.npz + 1) * p.npey;
        hipLaunchKernelGGL(k_fconm_sums, dim3(n), dim3(SUM_T), 0, s, p, q, o.ttm, o.part);
        hipLaunchKernelGGL(k_relax, dim3(1), dim3(64), 0, s, p, m, o.zee, o.part, o.ttm, o.work, sc, o.rs, o.radd);
    }
    return hipGetLastError();
}

}  // namespace rmhd
