// HIP kernels of the explicit compressible-MHD step for gfx950 (MI355X).
//
// K2 k_stage : right-hand side of FLUXES (3dmhdsub.f:1178-2637) fused with one
//              Wray RK3 stage update of STEP (3dmhdsub.f:926-969, 977-1067,
//              1075-1165), one launch per stage, with the boundary planes of
//              BCON (3dmhdsub.f:2751-2958).  Stage 3 also reduces the CFL
//              limits of the new state for the next step (sub:741-873), and
//              its last workgroup closes the step (DT, clock).
// K1 k_cfl   : stand-alone CFL / Mach reduction for the first step after an
//              upload (sub:741-873).
// K4 k_pack / k_unpack : conversion between the reference's padded arrays
//              and the resident layout, with the periodic ghost semantics of
//              COMM_MPI (3dmhdsub.f:3131-3138).
//
// Resident layout: field f of a register is a contiguous block of (npz+2)
// planes of npx*npy doubles, x fastest.  Plane 0 and npz+1 are the top and
// bottom z ghost planes, planes 1..npz the reference's K=2..NPZ+1.  There are
// no x/y ghost cells: neighbours wrap periodically.
//
// Stage kernel organisation.  A workgroup owns a 64 x TY column tile, or one of
// up to 256 points fitted to the box (TY = 0, see fit_tile), and marches down a
// chunk of planes.  LDS holds the raw fields of planes k and k+1 with a one-point
// halo (double buffer) and a three-plane ring of the velocities u,v,w (needed at
// (i+-1,k+-1) and (j+-1,k+-1) by the cross terms of the viscous stress).  Plane k+2 is loaded into registers while plane k
// is computed, and the Z register of the RK3 scheme is prefetched the same
// way, so each global load has a whole plane of arithmetic to hide behind.
// Outputs are written with non-temporal stores so that L2 keeps the halo
// rows that neighbouring tiles re-read.  What bounds it: at 512x512x256 HBM
// (2.86 / 3.59 / 3.13 ms for 12.9 / 17.2 / 12.9 GB of algorithmic bytes); on
// small boxes the latency of a plane's march (3.3 us with one workgroup on a
// CU) and of the launch, hence few planes per chunk (z_chunks) and three
// launches per step (64x64x32: 56 us per step, 132 with boundary, CFL and
// 8-plane launches of their own; 16x16x12 by single steps: 67 against 207).
//
// Arithmetic: every expression keeps the reference's left-to-right
// association and the file is compiled with -ffp-contract=off, so results
// are bit-identical to the reference's FP64 build.

#include "mhd_device.h"
#include <type_traits>

namespace rmhd {

constexpr int TX = 64;  // interior columns per tile (one wavefront row)

template <int TY_>
struct Tile {
    static constexpr int TY = TY_;
    static constexpr int NT = TX * TY;      // threads per workgroup
    static constexpr int SW = TX + 2;       // LDS row stride (1-point halo each side)
    static constexpr int SH = TY + 2;
    static constexpr int SP = SW * SH;      // points per LDS plane
    static constexpr int NHALO = SP - NT;   // halo points, one per thread for t < NHALO
    static_assert(NHALO <= NT, "one halo point per thread at most");
};
// Fitted tiles (Params::tile_w x tile_h, see fit_tile): 256 threads.
template <>
struct Tile<0> {
    static constexpr int TY = 4, NT = 256, SW = 0, SP = FIT_POINTS_FP64;
};

// Raw-field slots of the LDS planes (resident field order).
enum { S_RU = 0, S_RV, S_RW, S_RO, S_TT, S_BX, S_BY, S_BZ };

struct Raw {
    double v[NFIELD];
};

template <bool MAG>
__device__ __forceinline__ void load_raw(const double *__restrict__ q, long long fs, long long off, Raw &r) {
#pragma unroll
    for (int f = 0; f < (MAG ? 8 : 5); ++f) r.v[f] = q[f * fs + off];
}

// CFL limits of one point (sub:750-856).  mach = OGAMMA*UU/TT before the
// square root; w1..w4 the four pointwise limits.
template <bool MAG>
__device__ __forceinline__ void cfl_point(const Params &p, const double *q, double ddx, double ddy, double ddz,
                                          double rkap, double &mach, double &w1, double &w2, double &w3,
                                          double &w4) {
    const double ru = q[F_RU], rv = q[F_RV], rw = q[F_RW], ro = q[F_RO], tt = q[F_TT];
    const double r = 1.0 / ro;
    double uu = (ru * ru + rv * rv + rw * rw) * (r * r);
    const double mm = p.ogamma * uu / tt;
    if (mm > mach || !(mm == mm)) mach = mm;  // NaN propagates into the max
    if (MAG) {
        const double bx = q[F_BX], by = q[F_BY], bz = q[F_BZ];
        const double b2 = bx * bx + by * by + bz * bz;
        uu = uu + p.gamma * tt + b2 * p.obeta / ro + 2.0 * sqrt(uu * (p.gamma * tt + b2 * p.obeta / ro));
    } else {
        uu = uu + p.gamma * tt + 2.0 * sqrt(uu * p.gamma * tt);
    }
    double dd = fmin(fmin(ddx, ddy), ddz);
    const double a1 = dd / sqrt(uu);
    const double a2 = 0.5 * dd * dd * p.repr * p.cv * ro / rkap;
    const double a3 = 0.375 * dd * dd * p.re * ro;
    w1 = (a1 < w1 || !(a1 == a1)) ? a1 : w1;
    w2 = (a2 < w2 || !(a2 == a2)) ? a2 : w2;
    w3 = (a3 < w3 || !(a3 == a3)) ? a3 : w3;
    if (MAG) w4 = fmin(w4, 0.5 * dd * dd * p.rm);
}

// Workgroup reduction of the CFL accumulators, published as order-preserving
// keys (min/max are exact, so the order is irrelevant); workgroup seq of
// total.  The key of +NaN sorts above +Inf and wins the max, that of -NaN sorts
// below -Inf and wins the min, so a non-finite state cannot go unnoticed.
__device__ void cfl_reduce(double mach, double w1, double w2, double w3, double w4, double sf, int lmag,
                           int clock, DevScalars *__restrict__ sc, CflSlots *__restrict__ cs, int seq, int total,
                           DevScalars *report = nullptr) {
    __shared__ unsigned long long red[16][5];
    unsigned long long km = dkey(mach), k1 = dkey(w1), k2 = dkey(w2), k3 = dkey(w3), k4 = dkey(w4);
    // a NaN, of either sign, wins: the Mach number's as +NaN of the max, a limit's
    // as -NaN of the min reduction
    if (!(mach == mach)) km = ~0ull;
    if (!(w1 == w1)) k1 = 0;
    if (!(w2 == w2)) k2 = 0;
    if (!(w3 == w3)) k3 = 0;
    for (int off = 32; off > 0; off >>= 1) {
        unsigned long long o;
        o = __shfl_xor(km, off, 64); km = o > km ? o : km;
        o = __shfl_xor(k1, off, 64); k1 = o < k1 ? o : k1;
        o = __shfl_xor(k2, off, 64); k2 = o < k2 ? o : k2;
        o = __shfl_xor(k3, off, 64); k3 = o < k3 ? o : k3;
        o = __shfl_xor(k4, off, 64); k4 = o < k4 ? o : k4;
    }
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    if (lane == 0) {
        red[wv][0] = km; red[wv][1] = k1; red[wv][2] = k2; red[wv][3] = k3; red[wv][4] = k4;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int v = 1; v < nw; ++v) {
            km = red[v][0] > km ? red[v][0] : km;
            k1 = red[v][1] < k1 ? red[v][1] : k1;
            k2 = red[v][2] < k2 ? red[v][2] : k2;
            k3 = red[v][3] < k3 ? red[v][3] : k3;
            k4 = red[v][4] < k4 ? red[v][4] : k4;
        }
    }
    if (threadIdx.x < 64) {
        const unsigned long long k[CFL_KEYS] = {~km, k1, k2, k3, k4};
        cfl_publish(k, sc, cs, sf, lmag, clock, seq, total, report);
    }
}

// BCON on the boundary planes (top: plane 1, bot: plane npz) of one column of
// the freshly written register q, and the in-place 1/rho of the untouched z
// ghost planes that FLUXES performs (sub:1390) so that the resident ghosts
// follow the reference exactly.  A stage's workgroup calls it for the columns
// it owns when its chunk holds a boundary plane and so, with at least three
// planes, everything BCON reads: the conditions then need no launch of their
// own (5, 5 and 10 us of a 130 us step at 64x64x32, 8, 8 and 23 us of 1280
// at 256x256x128).  It is a chain of loads at the end of a workgroup's march:
// all of them are issued before the first store, which the compiler could not
// move them across itself (64x64x32, stage 3: 26.8 us with a wait per field,
// 21.3 so).  With CFL set (stage 3), the boundary planes' CFL limits of the
// final state are added to the accumulators.
template <bool MAG, bool CFL>
__device__ __forceinline__ void bcon_column(const Params &p, const Metrics &m, const double *__restrict__ qin,
                                            double *q, const DevScalars *sc, int i, int j, bool top, bool bot,
                                            double &c_mach, double &c_w1, double &c_w2, double &c_w3, double &c_w4) {
    const long long fs = p.fsize, pl = p.plane, idx = (long long)j * p.npx + i;
    const int nz = p.npz;
    const double C13 = p.c13, C23 = p.c23, C43 = p.c43;
    const double *ROi = qin + 3 * fs;
    // shear boundaries: RRT = 1, RRB = -1, RPP = 0 (sub:2751-2756)
    const double shear = p.lshr ? cos(0.0 * sc->timt) : 0.0;
#pragma unroll 1
    for (int side = 0; side < 2; ++side) {
        if (side ? !bot : !top) continue;
        const int k = side ? nz : 1, in = side ? -1 : 1;  // boundary plane, direction inwards
        const long long o = (long long)k * pl + idx, b = o + in * pl, c = b + in * pl;
        // everything that is read, before the first store (one wait, not one per
        // store): the plane's own values, RU, RV, RO, TT of the next two, and RO
        // of the ghost plane
        double v[8];
        v[F_RO] = q[3 * fs + o];
        v[F_TT] = q[4 * fs + o];
        if (MAG) {
#pragma unroll
            for (int f = F_BX; f <= F_BZ; ++f) v[f] = q[f * fs + o];
        }
        const double rub = q[b], ruc = q[c], rvb = q[fs + b], rvc = q[fs + c];
        const double rob = q[3 * fs + b], roc = q[3 * fs + c], ttb = q[4 * fs + b], ttc = q[4 * fs + c];
        // the z ghost plane of RO flips to 1/RO once per FLUXES call; with ID or
        // LREM it held the mirrored RO of the plane next to the boundary
        // (sub:1301-1310)
        const int kg = side ? nz + 1 : 0;
        const double rog = ROi[(long long)(p.mirror ? k + in : kg) * pl + idx];
        const double dz = p.dzf / m.dzzdz[k];
        if (p.lshr) {
            v[F_RU] = 0.0;
            v[F_RV] = (side ? -1.0 : 1.0) * shear * v[F_RO];
        } else {
            v[F_RU] = v[F_RO] * (C43 * rub / rob - C13 * ruc / roc);
            v[F_RV] = v[F_RO] * (C43 * rvb / rob - C13 * rvc / roc);
        }
        v[F_RW] = 0.0;
        bool sett = true;
        if (side) {  // sub:2873-2955
            if (p.izc == 0) v[F_TT] = p.tb;
            else if (p.lrem) v[F_TT] = C43 * ttb - C13 * ttc + p.dztb;
            else v[F_TT] = C43 * ttb - C13 * ttc + C23 * dz * p.theta / m.rkapa[nz];
        } else if (p.tp != 0.0 && (p.itc == 0 || p.itc == 1)) {
            // Gaussian top temperature or flux (sub:2790-2827)
            const double HH = p.hh, ex = p.gx[i + 1], ey = p.gy[j + 1];
            if (p.itc == 0) v[F_TT] = 1.0 - (1.0 - p.tpr) * ex / HH * ey / HH;
            else v[F_TT] = C43 * ttb - C13 * ttc - C23 * dz * (p.theta - (p.theta - p.tpr) * ex / HH * ey / HH);
        } else if (p.itc == 0 || p.itc == 2 || p.itc == 4) {
            // fixed T; TU with LREM; ITC=4: TP cooler on I <= NX/2 (sub:2828-2850)
            if (p.lrem) v[F_TT] = p.tu;
            else v[F_TT] = (p.itc == 4 && i + 2 <= (p.npx + 2) / 2) ? 1.0 - p.tp : 1.0;
        } else if (p.itc == 1) {
            if (p.lrem) v[F_TT] = C43 * ttb - C13 * ttc + p.dztu;
            else v[F_TT] = C43 * ttb - C13 * ttc - C23 * dz * p.theta;
        } else {
            sett = false;  // ITC=3: the top temperature is left to the equations
        }
        q[o] = v[F_RU];
        q[fs + o] = v[F_RV];
        q[2 * fs + o] = v[F_RW];
        if (sett) q[4 * fs + o] = v[F_TT];
        if (MAG && p.ibc == 0) {
            v[F_BZ] = 0.0;
            q[7 * fs + o] = 0.0;
        }
        q[3 * fs + (long long)kg * pl + idx] = 1.0 / rog;
        if (CFL)
            cfl_point<MAG>(p, v, m.ddx[i + 1], m.ddy[j + 1], m.ddz[k], m.rkcfl[k], c_mach, c_w1, c_w2, c_w3, c_w4);
    }
}

// Dynamic LDS bytes of a stage workgroup.
template <int TY, bool MAG>
constexpr int stage_lds_bytes() {
    return (2 * (MAG ? 8 : 5) + 9) * Tile<TY>::SP * (int)sizeof(double);
}

// One tile column chunk of a stage: interior columns i0..i0+TX-1, rows
// j0..j0+TY-1 (clipped to the box), planes kbeg..kend.  MODE 0 writes the
// right-hand side F to fout; MODE 1..3 performs RK3 stage s with the boundary
// conditions on the boundary planes it holds.  The whole workgroup calls it
// with the same arguments.
// OPT instantiates the optional branches of FLUXES (Params::opt; the per-plane
// tables come from mhd_opt.hip): 1 density diffusion alone, 2 any of density
// diffusion, Rempel conduction, shear boundaries, flux relaxation and embedded
// heat loss; the main path has none of their code.  Form 2 spills 60-90
// registers of each lane, form 1 none (96x96x48 with density diffusion, stages
// 1 to 3 in 64x4 tiles: 53, 81, 85 us as form 2, 35, 40, 44 us as form 1; 32, 35,
// 41 us in the fitted 48x5).
template <int TY, bool MAG, int MODE, int OPT = 0>
__device__ __forceinline__ void stage_tile(const Params &p, const Metrics &m, ArgPtr args,
                                           const double *__restrict__ qin,
                                           double *__restrict__ qout, double *__restrict__ zr,
                                           double *__restrict__ fout, DevScalars *__restrict__ sc,
                                           CflSlots *__restrict__ cs, int i0, int j0, int kbeg, int kend, int seq,
                                           int total, double *lds, int tw = 0, int th = 0) {
    using T = Tile<TY>;
    constexpr bool FIT = TY == 0;
    constexpr int SP = T::SP;
    const int W = FIT ? tw : TX, H = FIT ? th : TY, SW = FIT ? tw + 2 : T::SW;
    constexpr int NF = MAG ? 8 : 5;
    double *const s_cur = lds;                  // [2][NF][SP]: raw planes k, k+1 (by parity)
    double *const s_ring = lds + 2 * NF * SP;   // [3][3][SP]: u, v, w of planes k-1, k, k+1

    const int t = threadIdx.x;
    const int npx = p.npx, npy = p.npy, npz = p.npz;
    const long long fs = p.fsize, pl = p.plane;

    // own point
    // (threads past a fitted tile's last point double that point)
    const int own = FIT && t >= W * H ? W * H - 1 : t;
    const int oly = own / W + 1, olx = own - (oly - 1) * W + 1;
    const int opt = oly * SW + olx;
    const int gi = i0 + olx - 1, gj = j0 + oly - 1;
    const bool valid = (gi < npx) && (gj < npy) && (!FIT || t < W * H);
    const int gci = wrapc(gi, npx), gcj = wrapc(gj, npy);  // this lane's column
    const long long ooff = (long long)gcj * npx + gci;
    // halo point (t < NHALO): top row, bottom row, left column, right column
    int hpt = -1;
    long long hoff = 0;
    if (t < 2 * (SW + H)) {
        int hlx, hly;
        if (t < SW) { hlx = t; hly = 0; }
        else if (t < 2 * SW) { hlx = t - SW; hly = H + 1; }
        else if (t < 2 * SW + H) { hlx = 0; hly = t - 2 * SW + 1; }
        else { hlx = SW - 1; hly = t - 2 * SW - H + 1; }
        hpt = hly * SW + hlx;
        hoff = (long long)wrapc(j0 + hly - 1, npy) * npx + wrapc(i0 + hlx - 1, npx);
    }
    const bool has_h = hpt >= 0;

    auto cur = [&](int k, int f, int pt) -> double & { return s_cur[((k & 1) * NF + f) * SP + pt]; };
    auto ring = [&](int k, int c, int pt) -> double & { return s_ring[((k % 3) * 3 + c) * SP + pt]; };
    auto put_cur = [&](int k, int pt, const Raw &r) {
#pragma unroll
        for (int f = 0; f < NF; ++f) cur(k, f, pt) = r.v[f];
    };
    auto put_ring = [&](int k, int pt, const Raw &r) {
        const double ri = 1.0 / r.v[S_RO];     // sub:1390
        ring(k, 0, pt) = r.v[S_RU] * ri;        // sub:1414-1424
        ring(k, 1, pt) = r.v[S_RV] * ri;
        ring(k, 2, pt) = r.v[S_RW] * ri;
    };

    // the per-column values are on their way before the warm-up's loads
    const double HX = p.hx, H2X = p.h2x, HY = p.hy, H2Y = p.h2y, HZ = p.hz, H2Z = p.h2z;
    const double C43 = p.c43, OCV = p.ocv, ORE = p.ore, ORM = p.orm, OBETA = p.obeta;
    const int gix = gci + 1, gjy = gcj + 1;
    const double dx = m.dxxdx[gix], d2x = m.d2xxdx2[gix];
    const double dy = m.dyydy[gjy], d2y = m.d2yydy2[gjy];
    const double tmpy = HY * dy;
    const double tmpy1 = HY * d2y;
    const double tmpy2 = H2Y * dy * dy;
    double coefg = 0.0, coefz = 0.0;
    if (MODE > 0) {
        const double dt = sc->dt;
        coefg = (MODE == 1 ? p.gam1 : MODE == 2 ? p.gam2 : p.gam3) * dt;
        coefz = (MODE == 1 ? p.zeta1 : p.zeta2) * dt;
    }
    // CFL accumulators of the new state (stage 3 only)
    double c_mach = 0.0, c_w1 = INFINITY, c_w2 = INFINITY, c_w3 = INFINITY, c_w4 = INFINITY;
    const double c_ddx = MODE == 3 ? m.ddx[gix] : 0.0, c_ddy = MODE == 3 ? m.ddy[gjy] : 0.0;
    // the embedded heat loss's per-column Gaussians, read once
    const double c_gx = (OPT == 2 && p.itc == 2) ? p.gx[gix] : 0.0, c_gy = (OPT == 2 && p.itc == 2) ? p.gy[gjy] : 0.0;
    // Warm-up: planes kbeg-1 (own values + ring), kbeg and kbeg+1 (LDS + ring).
    // Every load is issued before the first is used: a chunk then pays one
    // memory latency before its march instead of three.
    Raw rm_, rp_o, rp_h;
    {
        Raw ro_[2], rh_[3];
        // with ID or LREM the ghost planes 0 and npz+1 hold RO of planes 2 and
        // npz-1 while FLUXES runs (sub:1303-1307)
        auto get = [&](int kk, long long off, Raw &r) __attribute__((always_inline)) {
            load_raw<MAG>(qin, fs, (long long)kk * pl + off, r);
            if (OPT && p.mirror && (kk == 0 || kk == npz + 1))
                r.v[S_RO] = qin[3 * fs + (long long)(kk == 0 ? 2 : npz - 1) * pl + off];
        };
        get(kbeg - 1, ooff, rm_);
        get(kbeg, ooff, ro_[0]);
        get(kbeg + 1, ooff, ro_[1]);
        if (has_h) {
#pragma unroll
            for (int n = 0; n < 3; ++n) get(kbeg - 1 + n, hoff, rh_[n]);
        }
        put_ring(kbeg - 1, opt, rm_);
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            put_cur(kbeg + n, opt, ro_[n]);
            put_ring(kbeg + n, opt, ro_[n]);
        }
        if (has_h) {
            put_ring(kbeg - 1, hpt, rh_[0]);
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                put_cur(kbeg + n, hpt, rh_[n + 1]);
                put_ring(kbeg + n, hpt, rh_[n + 1]);
            }
        }
    }

    // the per-column metrics arrive before the march, not inside its first plane
    settle(dx), settle(d2x), settle(dy), settle(d2y), settle(c_ddx), settle(c_ddy);
    if (OPT == 2) settle(c_gx), settle(c_gy);

    // One plane of the march.  BND instantiates the boundary-plane form
    // (one-sided z stencils, extra planes read directly); the interior form
    // has none of that code, so its loads are waited for only where used.
    auto plane = [&](const int k, auto bnd) __attribute__((always_inline)) {
        constexpr bool BND = decltype(bnd)::value;
        const bool pre = k < kend;
        const long long o = (long long)k * pl + ooff;
        if (pre) {
            load_raw<MAG>(qin, fs, (long long)(k + 2) * pl + ooff, rp_o);
            if (has_h) load_raw<MAG>(qin, fs, (long long)(k + 2) * pl + hoff, rp_h);
        }
        // Z of this point, read once (every lane: the wrapped column is in
        // range also for lanes outside the domain)
        double zk[8];
        if (MODE >= 2) {
#pragma unroll
            for (int f = 0; f < NF; ++f) zk[f] = __builtin_nontemporal_load(&zr[f * fs + o]);
        }
        const double dz = uload(m.dzzdz, k), d2z = uload(m.d2zzdz2, k);
        const double rk = uload(m.rkapa, k), dk = uload(m.dkapa, k);
        __syncthreads();
        if (valid) {
            const bool top = BND && k == 1, bot = BND && k == npz;
            const double tmpz = HZ * dz;
            const double tmpz1 = HZ * d2z;
            const double tmpz2 = H2Z * dz * dz;
#define CUR(f, d) cur(k, f, opt + (d))
#define NXT(f) cur(k + 1, f, opt)
#define RNG(kp, c, d) ring(kp, c, opt + (d))
            double q0[8];
#pragma unroll
            for (int f = 0; f < NF; ++f) q0[f] = CUR(f, 0);
            const double ro0 = q0[S_RO], tt0 = q0[S_TT];
            const double rinv = 1.0 / ro0;
            const double u0 = RNG(k, 0, 0), v0 = RNG(k, 1, 0), w0 = RNG(k, 2, 0);
            const double um = RNG(k - 1, 0, 0), vm = RNG(k - 1, 1, 0), wm = RNG(k - 1, 2, 0);
            const double up = RNG(k + 1, 0, 0), vp = RNG(k + 1, 1, 0), wp = RNG(k + 1, 2, 0);
            const double uxp = RNG(k, 0, 1), uxm = RNG(k, 0, -1);
            const double uyp = RNG(k, 0, SW), uym = RNG(k, 0, -SW);
            const double vxp = RNG(k, 1, 1), vxm = RNG(k, 1, -1);
            const double vyp = RNG(k, 1, SW), vym = RNG(k, 1, -SW);
            const double wxp = RNG(k, 2, 1), wxm = RNG(k, 2, -1);
            const double wyp = RNG(k, 2, SW), wym = RNG(k, 2, -SW);
            // own column, planes k-1 and k+1
            const double ru_m = rm_.v[S_RU], rv_m = rm_.v[S_RV], rw_m = rm_.v[S_RW], tt_m = rm_.v[S_TT];
            const double ru_p = NXT(S_RU), rv_p = NXT(S_RV), rw_p = NXT(S_RW), tt_p = NXT(S_TT);
            const double pm = rm_.v[S_RO] * tt_m, pp = NXT(S_RO) * tt_p;
            // pressure RO*TT at the in-plane neighbours (sub:1389)
            const double pxm = CUR(S_RO, -1) * CUR(S_TT, -1), pxp = CUR(S_RO, 1) * CUR(S_TT, 1);
            const double pym = CUR(S_RO, -SW) * CUR(S_TT, -SW), pyp = CUR(S_RO, SW) * CUR(S_TT, SW);

            // extra own-column values for the one-sided forms on the boundary planes
            double rwk2 = 0.0, wk2 = 0.0, bxk2 = 0.0, bxk3 = 0.0, byk2 = 0.0, byk3 = 0.0;
            if (top || bot) {
                const int ka = top ? k + 2 : k - 2;
                const int kb = top ? k + 3 : k - 3;
                const long long oa = (long long)ka * pl + ooff, ob = (long long)kb * pl + ooff;
                rwk2 = qin[2 * fs + oa];
                wk2 = rwk2 * (1.0 / qin[3 * fs + oa]);
                if (MAG) {
                    bxk2 = qin[5 * fs + oa];
                    byk2 = qin[6 * fs + oa];
                    bxk3 = qin[5 * fs + ob];
                    byk3 = qin[6 * fs + ob];
                }
            }

            // ---- continuity (sub:1252-1295)
            double fr = (CUR(S_RU, -1) - CUR(S_RU, 1)) * HX * dx;
            fr = fr - (CUR(S_RV, SW) - CUR(S_RV, -SW)) * tmpy;
            double wz;
            if (top) wz = (4.0 * rw_p - rwk2) * tmpz;
            else if (bot) wz = (rwk2 - 4.0 * rw_m) * tmpz;
            else wz = (rw_p - rw_m) * tmpz;
            fr = fr - wz;
            if (OPT && p.id != 0) {
                // diffusion of the density perturbations W1 = RO - ROM (sub:1319-1371)
                const double romk = uload(p.rom, k);
                const double d0 = ro0 - romk;
                if (p.dh != 0.0) {
                    const double dxp = CUR(S_RO, 1) - romk, dxm = CUR(S_RO, -1) - romk;
                    const double dyp = CUR(S_RO, SW) - romk, dym = CUR(S_RO, -SW) - romk;
                    const double ww2 = (dxp - dxm) * HX * d2x + (dxp - 2.0 * d0 + dxm) * H2X * dx * dx;
                    const double ww3 = (dyp - dym) * tmpy1 + (dyp - 2.0 * d0 + dym) * tmpy2;
                    fr = fr + (ww2 + ww3) * (p.dh * ORE * uload(p.wwz, k));
                }
                if (p.dv != 0.0) {
                    const double dzp = NXT(S_RO) - uload(p.rom, k + 1), dzm = rm_.v[S_RO] - uload(p.rom, k - 1);
                    const double ww2 = (dzp - dzm) * tmpz1 + (dzp - 2.0 * d0 + dzm) * tmpz2;
                    fr = fr + ww2 * (p.dv * ORE * uload(p.wwz, k));
                }
            }

            // ---- buoyancy and pressure gradient (sub:1379, 1401-1403)
            double fw = p.grav * ro0;
            fw = fw - (pp - pm) * tmpz;
            double fv = (pym - pyp) * tmpy;
            double fu = (pxm - pxp) * HX * dx;

            // ---- momentum advection (sub:1440-1481)
            fu = fu - (CUR(S_RU, 1) * uxp - CUR(S_RU, -1) * uxm) * HX * dx;
            fu = fu - (CUR(S_RU, SW) * vyp - CUR(S_RU, -SW) * vym) * tmpy;
            fu = fu - (ru_p * wp - ru_m * wm) * tmpz;
            fv = fv - (CUR(S_RV, 1) * uxp - CUR(S_RV, -1) * uxm) * HX * dx;
            fv = fv - (CUR(S_RV, SW) * vyp - CUR(S_RV, -SW) * vym) * tmpy;
            fv = fv - (rv_p * wp - rv_m * wm) * tmpz;
            fw = fw - (CUR(S_RW, 1) * uxp - CUR(S_RW, -1) * uxm) * HX * dx;
            fw = fw - (CUR(S_RW, SW) * vyp - CUR(S_RW, -SW) * vym) * tmpy;
            fw = fw - (rw_p * wp - rw_m * wm) * tmpz;

            // ---- temperature advection (sub:1500-1505)
            const double txp = CUR(S_TT, 1), txm = CUR(S_TT, -1);
            const double typ = CUR(S_TT, SW), tym = CUR(S_TT, -SW);
            const double tzp = tt_p, tzm = tt_m;
            double ft;
            if (OPT == 2 && p.lshr) {
                // no advection; FT keeps the previous evaluation's values (sub:1493)
                ft = p.ftacc[o];
            } else {
                ft = -(u0 * (txp - txm) * HX * dx);
                ft = ft - v0 * (typ - tym) * tmpy;
                ft = ft - w0 * (tzp - tzm) * tmpz;
            }

            // ---- conduction (sub:1584-1610)
            if (OPT == 2 && p.lrem) {
                // of the perturbations W1 = TT - TTM only, plus the mean profile's
                // radiative heating HRAD (sub:1536-1581)
                const double tc = p.t_cond, tmk = uload(p.ttm, k);
                const double e0 = tt0 - tmk, exp_ = txp - tmk, exm = txm - tmk, eyp = typ - tmk, eym = tym - tmk;
                const double ezp = tzp - uload(p.ttm, k + 1), ezm = tzm - uload(p.ttm, k - 1);
                ft = ft + ((exp_ - exm) * HX * d2x + (exp_ - 2.0 * e0 + exm) * H2X * dx * dx) * rinv * tc;
                ft = ft + ((eyp - eym) * tmpy1 + (eyp - 2.0 * e0 + eym) * tmpy2) * rinv * tc;
                ft = ft + ((ezp - ezm) * tmpz1 + (ezp - 2.0 * e0 + ezm) * tmpz2) * rinv * tc;
                ft = ft + rinv * tc * uload(p.hrad, k);
            } else {
                const double tc = p.t_cond;
                ft = ft + ((txp - txm) * HX * d2x + (txp - 2.0 * tt0 + txm) * H2X * dx * dx) * rinv * tc * rk;
                ft = ft + ((typ - tym) * tmpy1 + (typ - 2.0 * tt0 + tym) * tmpy2) * rinv * tc * rk;
                ft = ft + ((tzp - tzm) * tmpz1 + (tzp - 2.0 * tt0 + tzm) * tmpz2) * rinv * tc * rk;
                ft = ft + (tzp - tzm) * HZ * dz * rinv * tc * dk;
            }
            if (OPT == 2) {
                // flux relaxation (sub:1757-1765) and embedded heat loss (sub:1783-1806)
                if (p.rlax > 0.0) ft = ft + uload(p.radd, k);
                if (p.itc == 2) {
                    const double HH = p.hh;
                    if (p.tc != 0.0)
                        ft = ft - p.tp * OCV * 0.5 * p.ramp * rinv * c_gx / HH * c_gy / HH * uload(p.gz, k) / HH;
                    else
                        ft = ft - p.tp * OCV * rinv * c_gx / HH * c_gy / HH * uload(p.gz, k) / HH;
                }
            }
            // LSHR: no viscous or compressional heating (sub:1903-2101)
            const bool heat = !(OPT == 2 && p.lshr);

            // ---- viscous Laplacians (sub:1818-1886)
            fu = fu + ORE * (C43 * ((uxp - uxm) * HX * d2x + (uxp - 2.0 * u0 + uxm) * H2X * dx * dx)
                             + (uyp - uym) * tmpy1 + (uyp - 2.0 * u0 + uym) * tmpy2
                             + (up - um) * tmpz1 + (up - 2.0 * u0 + um) * tmpz2);
            fv = fv + ORE * ((vxp - vxm) * HX * d2x + (vxp - 2.0 * v0 + vxm) * H2X * dx * dx
                             + C43 * ((vyp - vym) * tmpy1 + (vyp - 2.0 * v0 + vym) * tmpy2)
                             + (vp - vm) * tmpz1 + (vp - 2.0 * v0 + vm) * tmpz2);
            fw = fw + ORE * ((wxp - wxm) * HX * d2x + (wxp - 2.0 * w0 + wxm) * H2X * dx * dx
                             + (wyp - wym) * tmpy1 + (wyp - 2.0 * w0 + wym) * tmpy2
                             + C43 * ((wp - wm) * tmpz1 + (wp - 2.0 * w0 + wm) * tmpz2));

            // ---- viscous and compressional heating, grad div u cross terms (sub:1891-2101)
            const double tv = p.t_visc, tv43 = p.t_visc43, tcr = p.t_cross;
            const double dxu = (uxp - uxm) * HX * dx;
            const double dxv = (vxp - vxm) * HX * dx;
            const double dxw = (wxp - wxm) * HX * dx;
            if (heat) {
                ft = ft + (C43 * dxu * dxu + dxv * dxv + dxw * dxw) * rinv * tv;
                ft = ft - OCV * dxu * tt0;
            }
            {
                const double dxv_jp = (RNG(k, 1, SW + 1) - RNG(k, 1, SW - 1)) * HX * dx;
                const double dxv_jm = (RNG(k, 1, -SW + 1) - RNG(k, 1, -SW - 1)) * HX * dx;
                fu = fu + tcr * (dxv_jp - dxv_jm) * HY * dy;
                const double dxu_jp = (RNG(k, 0, SW + 1) - RNG(k, 0, SW - 1)) * HX * dx;
                const double dxu_jm = (RNG(k, 0, -SW + 1) - RNG(k, 0, -SW - 1)) * HX * dx;
                fv = fv + tcr * (dxu_jp - dxu_jm) * HY * dy;
            }
            const double dyu = (uyp - uym) * HY * dy;
            const double dyv = (vyp - vym) * HY * dy;
            const double dzw = (wp - wm) * HZ * dz;
            if (heat) {
                ft = ft + (dyu * dyu + 2.0 * dyu * dxv) * rinv * tv;
                ft = ft + dyv * dyv * rinv * tv43;
                ft = ft - OCV * dyv * tt0;
                ft = ft + (dzw * dzw - dxu * dzw - dxu * dyv - dyv * dzw) * rinv * tv43;
                ft = ft - OCV * dzw * tt0;
            }
            {
                const double dzw_ip = (RNG(k + 1, 2, 1) - RNG(k - 1, 2, 1)) * HZ * dz;
                const double dzw_im = (RNG(k + 1, 2, -1) - RNG(k - 1, 2, -1)) * HZ * dz;
                fu = fu + tcr * (dzw_ip - dzw_im) * HX * dx;
                const double dzw_jp = (RNG(k + 1, 2, SW) - RNG(k - 1, 2, SW)) * HZ * dz;
                const double dzw_jm = (RNG(k + 1, 2, -SW) - RNG(k - 1, 2, -SW)) * HZ * dz;
                fv = fv + tcr * (dzw_jp - dzw_jm) * HY * dy;
            }
            const double dzu = (up - um) * HZ * dz;
            const double dzv = (vp - vm) * HZ * dz;
            const double dyw = (wyp - wym) * HY * dy;
            if (heat) ft = ft + (dzu * dzu + dzv * dzv + dyw * dyw + 2.0 * dzv * dyw) * rinv * tv;
            {
                const double dzu_ip = (RNG(k + 1, 0, 1) - RNG(k - 1, 0, 1)) * HZ * dz;
                const double dzu_im = (RNG(k + 1, 0, -1) - RNG(k - 1, 0, -1)) * HZ * dz;
                const double dzv_jp = (RNG(k + 1, 1, SW) - RNG(k - 1, 1, SW)) * HZ * dz;
                const double dzv_jm = (RNG(k + 1, 1, -SW) - RNG(k - 1, 1, -SW)) * HZ * dz;
                fw = fw + tcr * ((dzu_ip - dzu_im) * HX * dx + (dzv_jp - dzv_jm) * HY * dy);
            }
            if (heat) ft = ft + 2.0 * dzu * dxw * rinv * tv;

            // ---- Coriolis (sub:2106-2125)
            if (p.lrot) {
                fu = fu + p.omz * q0[S_RV];
                fv = fv - p.omz * q0[S_RU] + p.omx * q0[S_RW];
                fw = fw - p.omx * q0[S_RV];
            }

            // ---- induction, Lorentz force, Ohmic heating, resistive diffusion (sub:2129-2634)
            double w1 = 0.0, w2 = 0.0, w3 = 0.0;
            if (MAG) {
                const double bx0 = q0[S_BX], by0 = q0[S_BY], bz0 = q0[S_BZ];
                const double bxm = rm_.v[S_BX], bym = rm_.v[S_BY], bzm = rm_.v[S_BZ];
                const double bxp = NXT(S_BX), byp = NXT(S_BY), bzp = NXT(S_BZ);
                const double bxxp = CUR(S_BX, 1), bxxm = CUR(S_BX, -1);
                const double bxyp = CUR(S_BX, SW), bxym = CUR(S_BX, -SW);
                const double byxp = CUR(S_BY, 1), byxm = CUR(S_BY, -1);
                const double byyp = CUR(S_BY, SW), byym = CUR(S_BY, -SW);
                const double bzxp = CUR(S_BZ, 1), bzxm = CUR(S_BZ, -1);
                const double bzyp = CUR(S_BZ, SW), bzym = CUR(S_BZ, -SW);
                const double tm = p.t_ohm;

                w2 = bx0 * dxv - by0 * dxu;
                w3 = bx0 * dxw - bz0 * dxu;
                w1 = by0 * dyu - bx0 * dyv;
                w3 = w3 + by0 * dyw - bz0 * dyv;
                double dzw1;
                if (top) dzw1 = (4.0 * wp - wk2) * HZ * dz;
                else if (bot) dzw1 = (wk2 - 4.0 * wm) * HZ * dz;
                else dzw1 = dzw;
                w1 = w1 + bz0 * dzu - bx0 * dzw1;
                w2 = w2 + bz0 * dzv - by0 * dzw1;

                const double dxbx = (bxxp - bxxm) * HX * dx;
                const double dxby = (byxp - byxm) * HX * dx;
                const double dxbz = (bzxp - bzxm) * HX * dx;
                const double dybx = (bxyp - bxym) * HY * dy;
                fu = fu + OBETA * by0 * (dybx - dxby) - OBETA * bz0 * dxbz;
                fv = fv + OBETA * bx0 * (dxby - dybx);
                fw = fw + OBETA * bx0 * dxbz;
                ft = ft + (dybx * dybx + dxby * dxby + dxbz * dxbz - 2.0 * dxby * dybx) * rinv * tm;
                w1 = w1 - u0 * dxbx - v0 * dybx;
                w2 = w2 - u0 * dxby;
                w3 = w3 - u0 * dxbz;

                const double d2xbx = (bxxp - bxxm) * HX * d2x + (bxxp - 2.0 * bx0 + bxxm) * H2X * dx * dx;
                const double d2xby = (byxp - byxm) * HX * d2x + (byxp - 2.0 * by0 + byxm) * H2X * dx * dx;
                const double d2ybx = (bxyp - bxym) * HY * d2y + (bxyp - 2.0 * bx0 + bxym) * H2Y * dy * dy;
                w1 = w1 + ORM * (d2xbx + d2ybx);
                w2 = w2 + ORM * d2xby;
                const double d2xbz = (bzxp - bzxm) * HX * d2x + (bzxp - 2.0 * bz0 + bzxm) * H2X * dx * dx;
                w3 = w3 + ORM * d2xbz;

                const double dzbx = (bxp - bxm) * HZ * dz;
                const double dyby = (byyp - byym) * HY * dy;
                fu = fu + OBETA * bz0 * dzbx;
                fw = fw - OBETA * bx0 * dzbx;
                ft = ft + (dzbx * dzbx - 2.0 * dzbx * dxbz) * rinv * tm;
                w1 = w1 - w0 * dzbx;
                w2 = w2 - v0 * dyby;

                double d2zbx, d2zby;
                if (top) {
                    d2zbx = (-(3.0 * bx0) + 4.0 * bxp - bxk2) * HZ * d2z
                            + (2.0 * bx0 - 5.0 * bxp + 4.0 * bxk2 - bxk3) * H2Z * dz * dz;
                    d2zby = (-(3.0 * by0) + 4.0 * byp - byk2) * HZ * d2z
                            + (2.0 * by0 - 5.0 * byp + 4.0 * byk2 - byk3) * H2Z * dz * dz;
                } else if (bot) {
                    d2zbx = (3.0 * bx0 - 4.0 * bxm + bxk2) * HZ * d2z
                            + (2.0 * bx0 - 5.0 * bxm + 4.0 * bxk2 - bxk3) * H2Z * dz * dz;
                    d2zby = (3.0 * by0 - 4.0 * bym + byk2) * HZ * d2z
                            + (2.0 * by0 - 5.0 * bym + 4.0 * byk2 - byk3) * H2Z * dz * dz;
                } else {
                    d2zbx = (bxp - bxm) * HZ * d2z + (bxp - 2.0 * bx0 + bxm) * H2Z * dz * dz;
                    d2zby = (byp - bym) * HZ * d2z + (byp - 2.0 * by0 + bym) * H2Z * dz * dz;
                }
                const double d2yby = (byyp - byym) * HY * d2y + (byyp - 2.0 * by0 + byym) * H2Y * dy * dy;
                w1 = w1 + ORM * d2zbx;
                w2 = w2 + ORM * d2yby;

                const double dzby = (byp - bym) * HZ * dz;
                const double dybz = (bzyp - bzym) * HY * dy;
                const double jx = dzby - dybz;
                fv = fv + OBETA * bz0 * jx;
                fw = fw - OBETA * by0 * jx;
                ft = ft + (dzby * dzby + dybz * dybz - 2.0 * dzby * dybz) * rinv * tm;
                w2 = w2 - w0 * dzby;
                w3 = w3 - v0 * dybz;
                const double d2ybz = (bzyp - bzym) * HY * d2y + (bzyp - 2.0 * bz0 + bzym) * H2Y * dy * dy;
                w2 = w2 + ORM * d2zby;
                w3 = w3 + ORM * d2ybz;
                const double dzbz = (bzp - bzm) * HZ * dz;
                w3 = w3 - w0 * dzbz;
                const double d2zbz = (bzp - bzm) * HZ * d2z + (bzp - 2.0 * bz0 + bzm) * H2Z * dz * dz;
                w3 = w3 + ORM * d2zbz;
            }
#undef CUR
#undef NXT
#undef RNG
            // ---- output
            if (OPT == 2 && p.lshr) p.ftacc[o] = ft;
            // (the boundary conditions overwrite RU, RV and RW of a boundary plane
            // after every stage: their right-hand sides are not needed there)
            constexpr bool MOM = !BND || MODE == 0;
            const double F[8] = {MOM ? fu : 0.0, MOM ? fv : 0.0, MOM ? fw : 0.0, fr, ft, w1, w2, w3};
            if (MODE == 0) {
#pragma unroll
                for (int f = 0; f < NF; ++f) fout[f * fs + o] = F[f];
            } else {
                double qn[8];
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    // (Z is read only once this field's right-hand side exists)
                    const double zin = (MODE == 1) ? q0[f] : after(zk[f], F[f]);
                    qn[f] = zin + coefg * F[f];
                    __builtin_nontemporal_store(qn[f], &qout[f * fs + o]);
                    if (MODE < 3) __builtin_nontemporal_store(qn[f] + coefz * F[f], &zr[f * fs + o]);
                }
                if (MODE == 3 && !top && !bot)
                    cfl_point<MAG>(p, qn, c_ddx, c_ddy, uload(m.ddz, k), OPT == 2 ? uload(m.rkcfl, k) : rk, c_mach, c_w1,
                                   c_w2, c_w3, c_w4);
            }
            // own raw values of plane k become the k-1 values of the next plane
#pragma unroll
            for (int f = 0; f < NF; ++f) rm_.v[f] = q0[f];
            if (BND) settle(rwk2), settle(wk2), settle(bxk2), settle(byk2), settle(bxk3), settle(byk3);
        }
        // every load of this plane has arrived on every path out of it, so
        // none is still counted as outstanding in the next plane
        if (MODE >= 2) {
#pragma unroll
            for (int f = 0; f < NF; ++f) settle(zk[f]);
        }
        __syncthreads();
        // plane k+2 replaces plane k in LDS and enters the ring
        if (OPT && pre && p.mirror && k + 2 == npz + 1) {
            // ghost plane npz+1 holds RO of plane npz-1 = k (sub:1306-1307); each
            // thread reads the points it wrote itself
            rp_o.v[S_RO] = cur(k, S_RO, opt);
            if (has_h) rp_h.v[S_RO] = cur(k, S_RO, hpt);
        }
        if (pre) {
            put_cur(k + 2, opt, rp_o);
            put_ring(k + 2, opt, rp_o);
            if (has_h) {
                put_cur(k + 2, hpt, rp_h);
                put_ring(k + 2, hpt, rp_h);
            }
        }
    };
    int k0 = kbeg, k1 = kend;
    if (k0 == 1) plane(k0++, std::true_type{});
    const bool last_bnd = k1 == npz && k1 >= k0;
    if (last_bnd) --k1;
#pragma unroll 1
    for (int k = k0; k <= k1; ++k) plane(k, std::false_type{});
    if (last_bnd) plane(npz, std::true_type{});
    if (MODE > 0 && (kbeg == 1 || kend == npz) && valid) {
        const BoxArgs &l = late_args(args);
        bcon_column<MAG, MODE == 3>(l.p, l.m, qin, qout, sc, gi, gj, kbeg == 1, kend == npz, c_mach, c_w1, c_w2, c_w3,
                                    c_w4);
    }
    if (MODE == 3) {
        const BoxArgs &l = late_args(args);
        cfl_reduce(c_mach, c_w1, c_w2, c_w3, c_w4, l.p.sf, l.p.lmag, 1, sc, cs, seq, total, l.p.report);
    }
}

// Single box: workgroup -> (tile, z chunk), XCD-aware.
template <int TY, bool MAG, int MODE, int OPT>
__global__ __launch_bounds__(Tile<TY>::NT, 2) void k_stage(const BoxArgs b,
                                                  const double *__restrict__ qin,
                                                  double *__restrict__ qout,
                                                  double *__restrict__ zr,
                                                  double *__restrict__ fout,
                                                  DevScalars *__restrict__ sc, CflSlots *__restrict__ cs,
                                                  int nchunks) {
    extern __shared__ double lds[];
    const Params &p = b.p;
    const int W = TY ? TX : p.tile_w, H = TY ? TY : p.tile_h;
    const int ntx = (p.npx + W - 1) / W, nty = (p.npy + H - 1) / H;
    const TileChunk tc = tile_of(blockIdx.x, ntx * nty, nchunks);
    const int tz = tc.chunk, tyb = tc.tile / ntx, txb = tc.tile - tyb * ntx;
    const int kbeg = chunk_begin(p.npz, nchunks, tz), kend = chunk_begin(p.npz, nchunks, tz + 1) - 1;
    stage_tile<TY, MAG, MODE, OPT>(p, b.m, kernel_args(), qin, qout, zr, fout, sc, cs, txb * W, tyb * H, kbeg, kend,
                                   blockIdx.x, gridDim.x, lds, W, H);
}

// Ensemble: a persistent grid walks the work-item table of all boxes with a
// static stride (deterministic; every workgroup leaves after its last item).
// Register a of every box is the input, 1-a the output.
template <int TY, bool MAG, int MODE>
__global__ __launch_bounds__(Tile<TY>::NT, 2) void k_stage_batch(const BoxDev *__restrict__ boxes,
                                                        const StageItem *__restrict__ items, int nitems, int a) {
    extern __shared__ double lds[];
    const int slot = xcd_remap(blockIdx.x, gridDim.x);
    for (int w = slot; w < nitems; w += gridDim.x) {
        const StageItem it = items[w];
        const BoxDev &B = box_at(boxes, it.box);
        __syncthreads();  // the previous item's last LDS reads are done
        stage_tile<TY, MAG, MODE>(B.a.p, B.a.m, (ArgPtr)&B.a, B.q[a], B.q[1 - a], B.z, nullptr, B.sc, B.cs, it.i0, it.j0, it.kbeg,
                                  it.kend, it.seq, it.total, lds, it.w, it.h);
    }
}

// Stand-alone CFL reduction over planes 1..npz (first step after an upload).
template <bool MAG>
__global__ __launch_bounds__(256) void k_cfl(const Params p, const Metrics m, const double *__restrict__ q,
                                             DevScalars *__restrict__ sc, CflSlots *__restrict__ cs) {
    const long long fs = p.fsize, pl = p.plane;
    const long long n = (long long)p.npz * pl;
    double mach = 0.0, w1 = INFINITY, w2 = INFINITY, w3 = INFINITY, w4 = INFINITY;
    for (long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x; idx < n;
         idx += (long long)gridDim.x * blockDim.x) {
        const long long o = pl + idx;
        const int k = (int)(idx / pl) + 1;
        const long long r2 = idx - (long long)(k - 1) * pl;
        const int j = (int)(r2 / p.npx), i = (int)(r2 - (long long)j * p.npx);
        double v[8];
#pragma unroll
        for (int f = 0; f < (MAG ? 8 : 5); ++f) v[f] = q[f * fs + o];
        cfl_point<MAG>(p, v, m.ddx[i + 1], m.ddy[j + 1], m.ddz[k], m.rkcfl[k], mach, w1, w2, w3, w4);
    }
    cfl_reduce(mach, w1, w2, w3, w4, p.sf, p.lmag, 0, sc, cs, blockIdx.x, gridDim.x);
}

// Upload of all fields at once: thread (column, plane k = 0..npz+1) copies the
// padded arrays' point into q0, the z ghost planes (which no stage writes) into
// q1 too, and adds the point's limits to the CFL reduction; the stages write
// every other point of q1 before they read it.  One launch for what took a
// pack launch per field and register and k_cfl (64x64x32: 12 us, 17 launches of 59 before,
// mhd_step_noalloc 100 us, 171 before).
template <bool MAG>
__global__ __launch_bounds__(256) void k_load(const Params p, const Metrics m, const FieldSrc src,
                                              double *__restrict__ q0, double *__restrict__ q1,
                                              DevScalars *__restrict__ sc, CflSlots *__restrict__ cs) {
    constexpr int NF = MAG ? 8 : 5, PTS = 2;  // points per thread: fewer workgroups queue at the reduction
    const int k = blockIdx.y, nxp = p.npx + 2, nyp = p.npy + 2;
    double mach = 0.0, w1 = INFINITY, w2 = INFINITY, w3 = INFINITY, w4 = INFINITY;
    double v[PTS][8];
    int i[PTS], j[PTS];
    bool on[PTS];
    long long o[PTS];
#pragma unroll
    for (int t = 0; t < PTS; ++t) {
        const unsigned r = (blockIdx.x * PTS + t) * 256 + threadIdx.x;
        on[t] = r < (unsigned)p.plane;
        j[t] = r / (unsigned)p.npx;
        i[t] = r - j[t] * p.npx;
        o[t] = k * p.plane + r;
        const long long a = ((long long)k * nyp + (j[t] + 1)) * nxp + (i[t] + 1);
#pragma unroll
        for (int f = 0; f < NF; ++f)
            if (on[t]) v[t][f] = src.f[f][a];
    }
#pragma unroll
    for (int t = 0; t < PTS; ++t)
        if (on[t]) {
#pragma unroll
            for (int f = 0; f < NF; ++f) q0[f * p.fsize + o[t]] = v[t][f];
            if (k == 0 || k == p.npz + 1) {
#pragma unroll
                for (int f = 0; f < NF; ++f) q1[f * p.fsize + o[t]] = v[t][f];
            } else {
                cfl_point<MAG>(p, v[t], m.ddx[i[t] + 1], m.ddy[j[t] + 1], m.ddz[k], m.rkcfl[k], mach, w1, w2, w3, w4);
            }
        }
    cfl_reduce(mach, w1, w2, w3, w4, p.sf, p.lmag, 0, sc, cs, blockIdx.y * gridDim.x + blockIdx.x,
               gridDim.x * gridDim.y);
}

// Arms the reduction slots of one box per workgroup (a new handle).
__global__ __launch_bounds__(64) void k_cfl_arm(CflSlots *cs) { cfl_arm(cs + blockIdx.x, threadIdx.x); }

// padded Fortran (npx+2, npy+2, npz+2) -> resident field (x/y ghosts dropped)
__global__ void k_pack(const Params p, const double *__restrict__ padded, double *__restrict__ field) {
    const long long n = p.plane * (p.npz + 2);  // the field's values, not its padded stride
    const int nxp = p.npx + 2, nyp = p.npy + 2;
    for (long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x; idx < n;
         idx += (long long)gridDim.x * blockDim.x) {
        const long long k = idx / p.plane;
        const long long r = idx - k * p.plane;
        const int j = (int)(r / p.npx), i = (int)(r - (long long)j * p.npx);
        field[idx] = padded[(k * nyp + (j + 1)) * nxp + (i + 1)];
    }
}

// resident fields -> padded Fortran arrays (one field per blockIdx.z, planes
// over blockIdx.y: a point's column is one 32-bit division away); periodic
// ghost fill (mode 1) or zero ghosts and zero z ghost planes (mode 0, for
// right-hand sides)
__global__ void k_unpack(const Params p, const double *__restrict__ q, const FieldList l, int mode) {
    const double *__restrict__ const field = q + l.f[blockIdx.z] * p.fsize;
    double *__restrict__ const padded = l.dst[blockIdx.z];
    const unsigned nxp = p.npx + 2, nh = nxp * (unsigned)(p.npy + 2);
    for (unsigned r = blockIdx.x * blockDim.x + threadIdx.x; r < nh; r += gridDim.x * blockDim.x) {
        const int J = r / nxp, I = r - J * nxp;
        const int j = J == 0 ? p.npy - 1 : J > p.npy ? 0 : J - 1, i = I == 0 ? p.npx - 1 : I > p.npx ? 0 : I - 1;
        const bool ring = I == 0 || I > p.npx || J == 0 || J > p.npy;
        for (int k = blockIdx.y; k < p.npz + 2; k += gridDim.y) {
            const bool zero = mode == 0 && (ring || k == 0 || k > p.npz);
            padded[(long long)k * nh + r] = zero ? 0.0 : field[k * p.plane + (long long)j * p.npx + i];
        }
    }
}

// Box filter of nf resident fields (planes 1..npz) onto a coarse grid:
// out[f][K][J][I], I fastest.  Horizontally the mean of factor x factor
// blocks (coarse I covers fine i = factor*I .. factor*I + factor-1).
// Vertically, zmode 0: the mean of factor planes (coarse K covers fine
// planes factor*K+1 .. factor*K+factor); zmode 1 (vertex grids with npz =
// factor*(nzc-1)+1): coarse K sits on fine plane factor*K+1 and averages the
// planes within factor/2 of it with trapezoid weights (1/2 at both ends);
// the two boundary planes are taken as they are.
//
// A thread owns a coarse column over `depth` (BF_DEPTH) coarse planes; the fine
// plane that two of them share (zmode 1) is averaged once.  FACTOR 2, 4 and
// 8 read their rows in 16-byte pieces, all of a plane (of half a plane: 8) before
// the first is added; 0 is any other factor.  Bound by the read of the state:
// 8 fields of 256x256x125 by 4 in 115 us (4.6 TB/s), 156 us with a thread per
// coarse point and 8-byte loads.  More planes a thread save no time on a large box,
// where the shared plane is found in L2, and leave a small one with too few
// wavefronts (100x120x49 by 4 with its download: 91 us with 8 planes, 84 with 2;
// 288x288x145: 758, 742).
constexpr int BF_DEPTH = 2;
template <int FACTOR>
__global__ __launch_bounds__(256) void k_box_filter(const Params p, const double *__restrict__ q, int fct, int zmode,
                                                    int nxc, int nyc, int nzc, int depth, double *__restrict__ out) {
    const int factor = FACTOR ? FACTOR : fct;
    const unsigned col = blockIdx.x * 256 + threadIdx.x;
    if (col >= (unsigned)nxc * (unsigned)nyc) return;
    const int J = col / nxc, I = col - J * nxc, f = blockIdx.z;
    const double *qf = q + (long long)f * p.fsize + (long long)J * factor * p.npx + (long long)I * factor;
    auto hmean = [&](int k) {
        const double *at = qf + (long long)k * p.plane;
        double s = 0.0;
        if constexpr (FACTOR) {
            constexpr int ROWS = FACTOR == 8 ? 4 : FACTOR;
#pragma unroll
            for (int j0 = 0; j0 < FACTOR; j0 += ROWS) {
                double2 v[ROWS][FACTOR / 2];
#pragma unroll
                for (int jj = 0; jj < ROWS; ++jj)
#pragma unroll
                    for (int ii = 0; ii < FACTOR / 2; ++ii)
                        v[jj][ii] = *reinterpret_cast<const double2 *>(at + (long long)(j0 + jj) * p.npx + 2 * ii);
#pragma unroll
                for (int jj = 0; jj < ROWS; ++jj)
#pragma unroll
                    for (int ii = 0; ii < FACTOR / 2; ++ii) {
                        s += v[jj][ii].x;
                        s += v[jj][ii].y;
                    }
            }
        } else {
            for (int jj = 0; jj < factor; ++jj)
                for (int ii = 0; ii < factor; ++ii) s += at[(long long)jj * p.npx + ii];
        }
        return s / (double)(factor * factor);
    };
    const int hw = factor / 2;
    double shared = 0.0;  // zmode 1: the mean of the last plane of coarse plane K - 1
    const int K0 = blockIdx.y * depth, K1 = min(nzc, K0 + depth);
    for (int K = K0; K < K1; ++K) {
        double v = 0.0;
        if (zmode == 0) {
            for (int kk = 1; kk <= factor; ++kk) v += hmean(K * factor + kk);
            v /= (double)factor;
        } else if (K == 0 || K == nzc - 1) {
            v = hmean(K * factor + 1);
        } else {
            const int c = K * factor + 1;
            v += 0.5 * (K > K0 && K > 1 ? shared : hmean(c - hw));
            for (int d = 1 - hw; d < hw; ++d) v += 1.0 * hmean(c + d);
            shared = hmean(c + hw);
            v += 0.5 * shared;
            v /= (double)factor;
        }
        out[(((long long)f * nzc + K) * nyc + J) * nxc + I] = v;
    }
}

// ---------------------------------------------------------------------------
// launchers

template <int TY, bool MAG, int MODE, int OPT>
static hipError_t launch_stage_o(const Params &p, const Metrics &m, const double *qin, double *qout, double *z,
                                 double *fout, DevScalars *sc, CflSlots *cs, hipStream_t s) {
    constexpr int lds = stage_lds_bytes<TY, MAG>();
    static std::atomic<unsigned long long> attr{0};
    {
        hipError_t e = lds_limit_once(attr, reinterpret_cast<const void *>(&k_stage<TY, MAG, MODE, OPT>), lds);
        if (e != hipSuccess) return e;
    }
    const int nch = p.nchunks;
    hipLaunchKernelGGL((k_stage<TY, MAG, MODE, OPT>), dim3(tiles_of(p) * nch), dim3(Tile<TY>::NT), lds, s, BoxArgs{p, m, {}},
                       qin, qout, z, fout, sc, cs, nch);
    return hipGetLastError();
}

template <int TY, bool MAG, int MODE>
static hipError_t launch_stage_t(const Params &p, const Metrics &m, const double *qin, double *qout, double *z,
                                 double *fout, DevScalars *sc, CflSlots *cs, hipStream_t s) {
    if constexpr (TY != 0)  // (fitted tiles are chosen without form 2, see params_from_desc)
        if (p.opt == 2 || (p.opt && TY == 8)) return launch_stage_o<TY, MAG, MODE, 2>(p, m, qin, qout, z, fout, sc, cs, s);
    if constexpr (TY != 8)  // (8-row tiles are for trials: form 2 serves them)
        if (p.opt) return launch_stage_o<TY, MAG, MODE, 1>(p, m, qin, qout, z, fout, sc, cs, s);
    return launch_stage_o<TY, MAG, MODE, 0>(p, m, qin, qout, z, fout, sc, cs, s);
}

template <int TY>
static hipError_t launch_stage_ty(int mode, const Params &p, const Metrics &m, const double *qin, double *qout,
                                  double *z, double *fout, DevScalars *sc, CflSlots *cs, hipStream_t s) {
    if (p.lmag) {
        switch (mode) {
            case 0: return launch_stage_t<TY, true, 0>(p, m, qin, qout, z, fout, sc, cs, s);
            case 1: return launch_stage_t<TY, true, 1>(p, m, qin, qout, z, fout, sc, cs, s);
            case 2: return launch_stage_t<TY, true, 2>(p, m, qin, qout, z, fout, sc, cs, s);
            default: return launch_stage_t<TY, true, 3>(p, m, qin, qout, z, fout, sc, cs, s);
        }
    }
    switch (mode) {
        case 0: return launch_stage_t<TY, false, 0>(p, m, qin, qout, z, fout, sc, cs, s);
        case 1: return launch_stage_t<TY, false, 1>(p, m, qin, qout, z, fout, sc, cs, s);
        case 2: return launch_stage_t<TY, false, 2>(p, m, qin, qout, z, fout, sc, cs, s);
        default: return launch_stage_t<TY, false, 3>(p, m, qin, qout, z, fout, sc, cs, s);
    }
}

hipError_t launch_stage(int mode, const Params &p, const Metrics &m, const double *qin, double *qout,
                        double *z, double *fout, DevScalars *sc, CflSlots *cs, hipStream_t s) {
    if (p.tile_w) return launch_stage_ty<0>(mode, p, m, qin, qout, z, fout, sc, cs, s);
    if (p.tile_y == 8) return launch_stage_ty<8>(mode, p, m, qin, qout, z, fout, sc, cs, s);
    return launch_stage_ty<4>(mode, p, m, qin, qout, z, fout, sc, cs, s);
}

template <int TY, bool MAG, int MODE>
static hipError_t launch_batch_t(const BoxDev *boxes, const StageItem *items, int nitems, int grid, int a,
                                 hipStream_t s) {
    constexpr int lds = stage_lds_bytes<TY, MAG>();
    static std::atomic<unsigned long long> attr{0};
    {
        hipError_t e = lds_limit_once(attr, reinterpret_cast<const void *>(&k_stage_batch<TY, MAG, MODE>), lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((k_stage_batch<TY, MAG, MODE>), dim3(grid), dim3(Tile<TY>::NT), lds, s, boxes, items, nitems, a);
    return hipGetLastError();
}

template <int TY>
static hipError_t launch_batch_ty(int mode, int lmag, const BoxDev *boxes, const StageItem *items, int nitems,
                                  int grid, int a, hipStream_t s) {
    if (lmag) {
        if (mode == 1) return launch_batch_t<TY, true, 1>(boxes, items, nitems, grid, a, s);
        if (mode == 2) return launch_batch_t<TY, true, 2>(boxes, items, nitems, grid, a, s);
        return launch_batch_t<TY, true, 3>(boxes, items, nitems, grid, a, s);
    }
    if (mode == 1) return launch_batch_t<TY, false, 1>(boxes, items, nitems, grid, a, s);
    if (mode == 2) return launch_batch_t<TY, false, 2>(boxes, items, nitems, grid, a, s);
    return launch_batch_t<TY, false, 3>(boxes, items, nitems, grid, a, s);
}

hipError_t launch_stage_batch(int mode, int tile_y, int lmag, const BoxDev *boxes, const StageItem *items,
                              int nitems, int grid, int a, hipStream_t s) {
    if (tile_y == 8) return launch_batch_ty<8>(mode, lmag, boxes, items, nitems, grid, a, s);
    return launch_batch_ty<0>(mode, lmag, boxes, items, nitems, grid, a, s);
}

hipError_t launch_cfl(const Params &p, const Metrics &m, const double *q, DevScalars *sc, CflSlots *cs,
                      hipStream_t s) {
    const long long n = (long long)p.npz * p.plane;
    long long nb = (n + 255) / 256;
    if (nb > 2048) nb = 2048;
    dim3 grid((unsigned)nb), block(256);
    if (p.lmag) hipLaunchKernelGGL(k_cfl<true>, grid, block, 0, s, p, m, q, sc, cs);
    else hipLaunchKernelGGL(k_cfl<false>, grid, block, 0, s, p, m, q, sc, cs);
    return hipGetLastError();
}

hipError_t launch_cfl_arm(CflSlots *cs, int n, hipStream_t s) {
    hipLaunchKernelGGL(k_cfl_arm, dim3(n), dim3(64), 0, s, cs);
    return hipGetLastError();
}

hipError_t launch_pack(const Params &p, const double *padded, double *field, hipStream_t s) {
    long long nb = (p.plane * (p.npz + 2) + 255) / 256;
    if (nb > 8192) nb = 8192;
    hipLaunchKernelGGL(k_pack, dim3((unsigned)nb), dim3(256), 0, s, p, padded, field);
    return hipGetLastError();
}

hipError_t launch_load(const Params &p, const Metrics &m, const FieldSrc &src, double *q0, double *q1, DevScalars *sc,
                       CflSlots *cs, hipStream_t s) {
    if (p.plane > 0x7fffff00 || p.npz > 65533) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((p.plane + 511) / 512), (unsigned)(p.npz + 2));
    if (p.lmag) hipLaunchKernelGGL(k_load<true>, grid, dim3(256), 0, s, p, m, src, q0, q1, sc, cs);
    else hipLaunchKernelGGL(k_load<false>, grid, dim3(256), 0, s, p, m, src, q0, q1, sc, cs);
    return hipGetLastError();
}

hipError_t launch_unpack(const Params &p, const double *q, const FieldList &l, int mode, hipStream_t s) {
    const long long nh = (long long)(p.npx + 2) * (p.npy + 2);
    const unsigned gx = (unsigned)((nh + 255) / 256 > 4096 ? 4096 : (nh + 255) / 256);
    const unsigned gy = (unsigned)(p.npz + 2 > 4096 ? 4096 : p.npz + 2);
    hipLaunchKernelGGL(k_unpack, dim3(gx, gy, l.n), dim3(256), 0, s, p, q, l, mode);
    return hipGetLastError();
}

hipError_t launch_box_filter(const Params &p, const double *q, int nf, int factor, int zmode, int nxc, int nyc, int nzc,
                             double *out, hipStream_t s) {
    const long long cols = (long long)nxc * nyc;
    const int depth = nzc / BF_DEPTH < 32768 ? BF_DEPTH : nzc / 32768 + 1;
    const dim3 grid((unsigned)((cols + 255) / 256), (unsigned)((nzc + depth - 1) / depth), (unsigned)nf);
    if (cols > 0x7fffffff) return hipErrorInvalidValue;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, p, q, factor, zmode, nxc, nyc, nzc, depth, out);
        return hipGetLastError();
    };
    // (the register's base and field stride are multiples of 16 bytes, and every
    // row of a block starts at a multiple of the factor: npx is one too)
    static_assert(FIELD_PAD % 2 == 0, "fields of an even plane start on 16 bytes");
    if (factor == 2) return go(k_box_filter<2>);
    if (factor == 4) return go(k_box_filter<4>);
    if (factor == 8) return go(k_box_filter<8>);
    return go(k_box_filter<0>);
}

}  // namespace rmhd
