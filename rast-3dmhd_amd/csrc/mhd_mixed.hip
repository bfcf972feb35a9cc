// Mixed-precision form of the step (no counterpart in the reference).
//
// The state is carried as FP32 perturbations h about an FP64 hydrostatic
// background (rho0(z), T0(z); zero momentum and field), and the right-hand
// side is evaluated in FP32 in perturbation form: F(bg + h) = F_bg(z) + F'(h),
// where F_bg (nonzero only for the momentum z component and the temperature)
// is the background's own discrete residual, formed once per plane in FP64.
//
// Stored variables: RU, RV, RW, rho', P', BX, BY, BZ, where P' is the
// pressure perturbation rho T - rho0 T0 = rho0 T' + T0 rho' + rho' T'.  In
// low-Mach flow P' is a small residual of rho0 T' and T0 rho'; storing it
// directly keeps the pressure gradient, which drives the horizontal flow,
// accurate to the FP32 precision of P' itself, and T' = (P' - T0 rho')/rho
// follows without cancellation.  (Storing T' instead leaves the horizontal
// momentum several times 1e-6 off the FP64 result after 1000 steps.)
//
// The RK3 accumulation runs in FP64 in registers, on the same variables as
// the FP64 form (T, not P): X = value + D + gamma dt F, where the value of
// the temperature slot is T'(rho', P') as the stencil computes it (trep).  The second
// register D (FP32) carries, per Wray's low-storage scheme, the zeta*dt*F
// increment of the next stage plus the rounding residual of the stored
// value (for T: X_T - T'(new rho', new P')).  After the last stage only the
// residual is left, at most a few FP32 ulps of the value: it is kept in a
// third register R as BF16, two fields per 32-bit word (8 significant bits
// of a residual of relative size 2^-24, i.e. the state to about 2^-33), so
// that (h, R) is a
// compensated pair and the storage rounding does not accumulate from step
// to step.  Stage 1 reads R, stages 1-2 write D, stage 3 writes R.
// The CFL reduction, the boundary planes and the background are FP64.
// The file is compiled without FMA contraction; the FP32 right-hand side
// and the FP64 accumulation of the stage body opt in (#pragma clang fp
// contract), everything that packs, unpacks or reconstructs stored values
// (trep, pprime, the residuals) rounds each operation separately.
//
// Traffic per zone (8 fields): stage 1 reads h (4 B) and R (2 B) and writes
// h and D (4 + 4 B); stage 2 reads and writes h and D; stage 3 reads h and D
// and writes h and R: 112 + 128 + 112 = 352 B/zone/step (FP64: 640).

#include "mhd_device.h"
#include <type_traits>

namespace rmhd {

constexpr int MTX = 64;

// Arithmetic type of the perturbation right-hand side (storage stays FP32).
typedef float rhs_t;

// Tile of MTX columns x TY rows, one point per thread; TY = 0: fitted tiles of
// at most 256 points (Params::tile_w x tile_h, see fit_tile).
template <int TY_>
struct MTile {
    static constexpr int NT = MTX * TY_;
    static constexpr int SW = MTX + 2;
    static constexpr int SP = SW * (TY_ + 2);
    static_assert(SP - NT <= NT, "one halo point per thread at most");
};
template <>
struct MTile<0> {
    static constexpr int NT = 256, SW = 0, SP = FIT_POINTS_MIXED;
};

// LDS: raw planes k, k+1 (2 x NF fields) and a three-plane ring of u, v, w, T'.
// Lean: T' takes the place of rho', of which only a point's own value is read (it
// stays in registers, as does T' of plane k-1), 25 instead of 28 values a point.
// Stage 1, whose registers allow it, so has four workgroups of 64x4 on a CU
// (512x512x256: 1634 -> 1573 us); the others keep three either way, and stage 3
// is 1% slower lean (256x256x128).
template <int MODE>
constexpr bool lean_lds = MODE == 1;
template <int TY, bool MAG, int MODE>
constexpr int mixed_lds_bytes() {
    return (2 * (MAG ? 8 : 5) + (lean_lds<MODE> ? 9 : 12)) * MTile<TY>::SP * (int)sizeof(float);
}

// P' of temperature perturbation tp at density perturbation rh.  The
// stored P' is formed from the exact (FP64) rho', not from its FP32
// rounding: T0 times the rounding error of rho' would be comparable to P'.
__host__ __device__ __forceinline__ double pprime(double r0, double t0, double rh, double tp) {
    return r0 * tp + t0 * rh + rh * tp;
}

// CFL limits of the mixed form (FP64), accumulated in monotone transformed
// form so that a point costs two divisions and one square root:
//   min dd/sqrt(U)               = 1/sqrt(max U/dd^2)
//   min 0.5 dd^2 REPR CV rho/kap = 0.5 REPR CV min(rho dd^2 / kap)
//   min 0.375 dd^2 RE rho        = 0.375 RE min(rho dd^2)
//   min 0.5 dd^2 RM              = 0.5 RM min(dd^2)
// (U the fast-mode speed squared of sub:750-856).  The workgroup converts
// back once and publishes the same keys as cfl_reduce.  NaN sticks.
struct CflFast {
    double mach, q1, s2, s3, d2;
};

__device__ __forceinline__ double nmax(double a, double b) { return (b > a || !(b == b)) ? b : a; }
__device__ __forceinline__ double nmin(double a, double b) { return (b < a || !(b == b)) ? b : a; }

__device__ __forceinline__ CflFast cflf_init() { return CflFast{0.0, 0.0, INFINITY, INFINITY, INFINITY}; }

template <bool MAG>
__device__ __forceinline__ void cflf_point(const Params &p, const double *q, double dd2, double idd2, double irk,
                                           CflFast &c) {
    const double ro = q[F_RO], tt = q[F_TT];
    const double ri = 1.0 / ro;
    const double uu = (q[F_RU] * q[F_RU] + q[F_RV] * q[F_RV] + q[F_RW] * q[F_RW]) * (ri * ri);
    c.mach = nmax(c.mach, p.ogamma * uu / tt);
    double cs = p.gamma * tt;
    if (MAG) cs += (q[F_BX] * q[F_BX] + q[F_BY] * q[F_BY] + q[F_BZ] * q[F_BZ]) * p.obeta * ri;
    const double u2 = uu + cs + 2.0 * sqrt(uu * cs);
    c.q1 = nmax(c.q1, u2 * idd2);
    const double rd = ro * dd2;
    c.s2 = nmin(c.s2, rd * irk);
    c.s3 = nmin(c.s3, rd);
    if (MAG) c.d2 = nmin(c.d2, dd2);
}

// dd^2 = min(ddx, ddy, ddz)^2 and its inverse for one point
struct DdPair {
    double dd2, idd2;
};
__device__ __forceinline__ DdPair ddpair(double ddx, double ddy, double ddz) {
    const double a = ddx * ddx, b = ddy * ddy, c = ddz * ddz;
    const double d2 = fmin(fmin(a, b), c);
    return DdPair{d2, 1.0 / d2};
}

// d2extra: a min(dd^2) contribution computed elsewhere (the grid-only term
// of the stage kernel, which does not reduce it per point).
__device__ void cflf_reduce(const Params &p, CflFast c, int clock, DevScalars *__restrict__ sc,
                            CflSlots *__restrict__ cs, int seq, int total, double d2extra = INFINITY) {
    __shared__ double red[16][5];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        c.mach = nmax(c.mach, __shfl_xor(c.mach, off, 64));
        c.q1 = nmax(c.q1, __shfl_xor(c.q1, off, 64));
        c.s2 = nmin(c.s2, __shfl_xor(c.s2, off, 64));
        c.s3 = nmin(c.s3, __shfl_xor(c.s3, off, 64));
        c.d2 = nmin(c.d2, __shfl_xor(c.d2, off, 64));
    }
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    if (lane == 0) {
        red[wv][0] = c.mach; red[wv][1] = c.q1; red[wv][2] = c.s2; red[wv][3] = c.s3; red[wv][4] = c.d2;
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        for (int v = 1; v < nw; ++v) {
            c.mach = nmax(c.mach, red[v][0]);
            c.q1 = nmax(c.q1, red[v][1]);
            c.s2 = nmin(c.s2, red[v][2]);
            c.s3 = nmin(c.s3, red[v][3]);
            c.d2 = nmin(c.d2, red[v][4]);
        }
        c.d2 = nmin(c.d2, d2extra);
        const double w[4] = {1.0 / sqrt(c.q1), 0.5 * p.repr * p.cv * c.s2, 0.375 * p.re * c.s3, 0.5 * p.rm * c.d2};
        unsigned long long k[CFL_KEYS];
        // a NaN, of either sign, wins: as in cfl_reduce
        k[0] = c.mach == c.mach ? ~dkey(c.mach) : 0ull;
        for (int n = 0; n < 4; ++n) k[n + 1] = (w[n] == w[n]) ? dkey(w[n]) : 0ull;
        cfl_publish(k, sc, cs, p.sf, p.lmag, clock, seq, total, clock ? p.report : nullptr);
    }
}

struct RawF {
    float v[NFIELD];
};

template <bool MAG>
__device__ __forceinline__ void load_rawf(const float *__restrict__ q, long long fs, long long off, RawF &r) {
#pragma unroll
    for (int f = 0; f < (MAG ? 8 : 5); ++f) r.v[f] = q[f * fs + off];
}

// BCON of the mixed form on the boundary planes (top: plane 1, bot: plane
// npz) of one column, in FP64 on the full state bg + value (+ R after the
// last stage, where R holds the rounding residual); called by the stage
// workgroup that owns the column and the planes (see bcon_column of the FP64
// form).  New boundary values are split again into stored values and the
// residual (D after stages 1-2, R after stage 3); a new boundary temperature
// is stored as the P' of the plane's stored rho'.  LAST also accumulates the
// boundary planes' CFL limits.
template <bool MAG, bool LAST>
__device__ __forceinline__ void bcon_column_m(const Params &p, const Metrics &m, const Background &bg, float *h,
                                              float *dr, unsigned *rr, int i, int j, bool top, bool bot,
                                              CflFast &cfl) {
    const long long fs = p.fsize, pl = p.plane, idx = (long long)j * p.npx + i;
    const int nz = p.npz;
    const double C13 = p.c13, C23 = p.c23, C43 = p.c43;
#pragma unroll 1
    for (int side = 0; side < 2; ++side) {
        if (side ? !bot : !top) continue;
        const int a = side ? nz : 1, in = side ? -1 : 1, b = a + in, c = b + in;
        // everything that is read, before the first store (one wait, not one per
        // store): stored values (and R words) of the plane and the next two
        float ha[8], hb[5], hc[5];
        unsigned wa[4], wb[3], wc[3];
        const long long oa = (long long)a * pl + idx, ob = (long long)b * pl + idx, oc = (long long)c * pl + idx;
#pragma unroll
        for (int f = 0; f < (MAG ? 8 : 5); ++f) ha[f] = h[f * fs + oa];
#pragma unroll
        for (int f = 0; f < 5; ++f)
            if (f != 2) {
                hb[f] = h[f * fs + ob];
                hc[f] = h[f * fs + oc];
            }
        if (LAST) {
#pragma unroll
            for (int w = 0; w < (MAG ? 4 : 3); ++w) wa[w] = rr[w * fs + oa];
#pragma unroll
            for (int w = 0; w < 3; ++w) {
                wb[w] = rr[w * fs + ob];
                wc[w] = rr[w * fs + oc];
            }
        }
        // full value of field f of plane k from its stored values and R words
        auto full = [&](int f, int k, const float *hv, const unsigned *wv) __attribute__((always_inline)) {
            double v = f == 4 ? (double)trep(bg.ro32[k], bg.tt32[k], hv[3], hv[4]) : (double)hv[f];
            if (LAST) v += (double)r_half(wv[f >> 1], f);
            if (f == 3) v += bg.ro[k];
            if (f == 4) v += bg.tt[k];
            return v;
        };
        // new value v of field f of the boundary plane: its split
        auto put = [&](int f, double v) __attribute__((always_inline)) {
            float hn, r;
            if (f == 4) {
                const double tp = v - bg.tt[a];
                const double rhx = LAST ? (double)ha[3] + (double)r_half(wa[1], 3) : (double)ha[3];
                hn = (float)pprime(bg.ro[a], bg.tt[a], rhx, tp);
                r = (float)(tp - (double)trep(bg.ro32[a], bg.tt32[a], ha[3], hn));
            } else {
                hn = (float)v;
                r = (float)(v - (double)hn);
            }
            ha[f] = hn;
            h[f * fs + oa] = hn;
            if (LAST) {
                const unsigned rb = to_bf16(r);
                unsigned &w = wa[f >> 1];
                w = (f & 1) ? ((w & 0x0000ffffu) | (rb << 16)) : ((w & 0xffff0000u) | rb);
            } else {
                dr[f * fs + oa] = r;
            }
        };
        const double roa = full(3, a, ha, wa), rob = full(3, b, hb, wb), roc = full(3, c, hc, wc);
        put(0, roa * (C43 * full(0, b, hb, wb) / rob - C13 * full(0, c, hc, wc) / roc));
        put(1, roa * (C43 * full(1, b, hb, wb) / rob - C13 * full(1, c, hc, wc) / roc));
        put(2, 0.0);
        const int code = side ? p.izc : p.itc;
        double tnew;
        if (code == 0) {
            tnew = side ? p.tb : 1.0;
        } else {
            const double dz = p.dzf / m.dzzdz[a];
            const double tb = full(4, b, hb, wb), tc = full(4, c, hc, wc);
            tnew = side ? C43 * tb - C13 * tc + C23 * dz * p.theta / m.rkapa[a] : C43 * tb - C13 * tc - C23 * dz * p.theta;
        }
        put(4, tnew);
        if (MAG && p.ibc == 0) put(7, 0.0);
        if (LAST) {
#pragma unroll
            for (int w = 0; w < (MAG ? 4 : 3); ++w) rr[w * fs + oa] = wa[w];
            double v[8];
#pragma unroll
            for (int f = 0; f < (MAG ? 8 : 5); ++f) v[f] = full(f, a, ha, wa);
            const DdPair d = ddpair(m.ddx[i + 1], m.ddy[j + 1], m.ddz[a]);
            cflf_point<MAG>(p, v, d.dd2, d.idd2, 1.0 / m.rkapa[a], cfl);
        }
    }
}

// One tile column chunk of mixed stage s = MODE (1..3); see stage_tile of
// the FP64 form for the tile organisation.
// Per-plane values (z metrics, background, coefficients) from the
// records of Background::planes: one table pointer for the march.
#define PLM(F, K) uload(&bg.planes[K].F, 0)
#define PLB(F, K) uload(&bg.planes[K].F, 0)
#define PLP(F, K) uload(&bg.planes[K].F, 0)

template <int TY, bool MAG, int MODE>
__device__ __forceinline__ void stage_tile_m(const Params &p, const Metrics &m, const Background &bg, ArgPtr args,
                                             const float *__restrict__ hin, float *__restrict__ hout,
                                             float *__restrict__ dr, unsigned *__restrict__ rr,
                                             DevScalars *__restrict__ sc, CflSlots *__restrict__ cs, int i0, int j0,
                                             int kbeg, int kend, int seq, int total, float *ldsf, int tw, int th) {
    using T = MTile<TY>;
    constexpr bool FIT = TY == 0;
    constexpr int SP = T::SP;
    const int W = FIT ? tw : MTX, H = FIT ? th : TY, SW = FIT ? tw + 2 : T::SW;
    constexpr int NF = MAG ? 8 : 5;
    constexpr bool LEAN = lean_lds<MODE>;
    float *const s_cur = ldsf;
    float *const s_ring = ldsf + 2 * NF * SP;

    const int t = threadIdx.x;
    const int npx = p.npx, npy = p.npy, npz = p.npz;
    const long long fs = p.fsize, pl = p.plane;

    // (threads past a fitted tile's last point double that point)
    const int own = FIT && t >= W * H ? W * H - 1 : t;
    const int oly = own / W + 1, olx = own - (oly - 1) * W + 1;
    const int opt = oly * SW + olx;
    const int gi = i0 + olx - 1, gj = j0 + oly - 1;
    const bool valid = (gi < npx) && (gj < npy) && (!FIT || t < W * H);
    const int gci = wrapc(min(gi, npx), npx), gcj = wrapc(gj, npy);  // this lane's column
    const long long ooff = (long long)gcj * npx + gci;
    int hpt = -1;
    long long hoff = 0;
    {
        const int ht = min(t, 2 * (SW + H) - 1);
        int hlx, hly;
        if (ht < SW) { hlx = ht; hly = 0; }
        else if (ht < 2 * SW) { hlx = ht - SW; hly = H + 1; }
        else if (ht < 2 * SW + H) { hlx = 0; hly = ht - 2 * SW + 1; }
        else { hlx = SW - 1; hly = ht - 2 * SW - H + 1; }
        hpt = hly * SW + hlx;
        hoff = (long long)wrapc(j0 + hly - 1, npy) * npx + wrapc(i0 + hlx - 1, npx);
    }
    const bool has_h = t < 2 * (SW + H);

    auto cur = [&](int k, int f, int pt) -> float & { return s_cur[((k & 1) * NF + f) * SP + pt]; };
    auto ring = [&](int k, int c, int pt) -> float & { return s_ring[((k % 3) * (LEAN ? 3 : 4) + c) * SP + pt]; };
    auto tprime = [&](int k, const RawF &r) { return trep(PLB(ro32, k), PLB(tt32, k), r.v[3], r.v[4]); };
    auto put_cur = [&](int k, int pt, const RawF &r) {
#pragma unroll
        for (int f = 0; f < NF; ++f) cur(k, f, pt) = LEAN && f == 3 ? tprime(k, r) : r.v[f];
    };
    auto put_ring = [&](int k, int pt, const RawF &r) {
        const float ri = rcp32(PLB(ro32, k) + r.v[3]);
        ring(k, 0, pt) = r.v[0] * ri;
        ring(k, 1, pt) = r.v[1] * ri;
        ring(k, 2, pt) = r.v[2] * ri;
        if (!LEAN) ring(k, 3, pt) = tprime(k, r);  // temperature perturbation
    };

    // the per-column values are on their way before the warm-up's loads
    const rhs_t HX = (rhs_t)p.hx, H2X = (rhs_t)p.h2x, HY = (rhs_t)p.hy, H2Y = (rhs_t)p.h2y;
    const rhs_t HZ = (rhs_t)p.hz, H2Z = (rhs_t)p.h2z;
    const int gix = gci + 1, gjy = gcj + 1;
    const rhs_t dx = (rhs_t)m.dxxdx[gix], d2x = (rhs_t)m.d2xxdx2[gix];
    const rhs_t dy = (rhs_t)m.dyydy[gjy], d2y = (rhs_t)m.d2yydy2[gjy];
    const rhs_t hxdx = HX * dx, hydy = HY * dy;
    const rhs_t h2xdx2 = H2X * dx * dx, h2ydy2 = H2Y * dy * dy;
    const rhs_t hxd2x = HX * d2x, hyd2y = HY * d2y;
    const double dt = sc->dt;
    const double coefg = (MODE == 1 ? p.gam1 : MODE == 2 ? p.gam2 : p.gam3) * dt;
    const double coefz = (MODE == 1 ? p.zeta1 : p.zeta2) * dt;
    // stage 3: this column's part of min(dd^2) and its inverse; per plane
    // the CFL takes dd^2 = min(c_d2, ddz^2) and 1/dd^2 = max(c_id2, 1/ddz^2),
    // which is 1/min(...) exactly (correctly rounded division is monotone)
    double c_d2 = 0.0, c_id2 = 0.0;
    if (MODE == 3) {
        const double ddx = m.ddx[gix], ddy = m.ddy[gjy];
        c_d2 = fmin(ddx * ddx, ddy * ddy);
        c_id2 = 1.0 / c_d2;
    }
    // warm-up: planes kbeg-1 .. kbeg+1, every load issued before the first is
    // used (lanes without a halo point re-read their own)
    RawF rm_, rp_o, rp_h;  // planes k-1 (lean: T' in the place of rho'), k+2
    float rho_k = 0.0f, rho_n = 0.0f;  // lean: own rho' of planes k, k+1
    {
        RawF ro_[2], rh_[3];
        const long long ho = hoff;
        load_rawf<MAG>(hin, fs, (long long)(kbeg - 1) * pl + ooff, rm_);
#pragma unroll
        for (int n = 0; n < 2; ++n) load_rawf<MAG>(hin, fs, (long long)(kbeg + n) * pl + ooff, ro_[n]);
#pragma unroll
        for (int n = 0; n < 3; ++n) load_rawf<MAG>(hin, fs, (long long)(kbeg - 1 + n) * pl + ho, rh_[n]);
        put_ring(kbeg - 1, opt, rm_);
        if (LEAN) {
            rm_.v[3] = tprime(kbeg - 1, rm_);
            rho_k = ro_[0].v[3];
            rho_n = ro_[1].v[3];
        }
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

    // stage 3: this thread's running CFL maxima/minima over its column
    CflFast cfl_acc = cflf_init();
    const bool frc = bg.force != nullptr && *bg.force_on != 0;

    // One plane of the march.  BND instantiates the boundary-plane form
    // (one-sided z stencils, extra planes read directly); the interior form
    // has none of that code, so its loads are waited for only where used.
    auto plane = [&](const int k, auto bnd) __attribute__((always_inline)) {
        constexpr bool BND = decltype(bnd)::value;
        const bool pre = k < kend;
        const long long o = (long long)k * pl + ooff;
        // D (stages 2, 3) or the packed R words (stage 1) of this point, read
        // once; R is unpacked where it is used, so that no wait for these
        // loads comes before the plane's arithmetic.  Every load of the plane
        // is issued on every path (lanes outside the box read their wrapped
        // column, which is in range; the last plane of a chunk and the lanes
        // without a halo point re-read points of their own), D first: the
        // number of loads in flight is then the same on all paths, and the
        // wait for D at the accumulation does not also wait for the prefetch.
        float dk_[8];
        unsigned rk_[4];
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            if (MODE != 1) dk_[f] = __builtin_nontemporal_load(&dr[f * fs + o]);
            else if (!(f & 1)) rk_[f >> 1] = __builtin_nontemporal_load(&rr[(f >> 1) * fs + o]);
        }
        {
            const long long kp = (long long)(pre ? k + 2 : k) * pl;
            load_rawf<MAG>(hin, fs, kp + ooff, rp_o);
            load_rawf<MAG>(hin, fs, kp + hoff, rp_h);
        }
        __syncthreads();
        if (valid) {
            const bool top = BND && k == 1, bot = BND && k == npz;
            const rhs_t C43 = PLP(c43, k), OCV = PLP(ocv, k), ORE = PLP(ore, k), ORM = PLP(orm, k);
            const rhs_t OBETA = PLP(obeta, k), GRAV = PLP(grav, k);
            const rhs_t dz = (rhs_t)PLM(dzzdz, k), d2z = (rhs_t)PLM(d2zzdz2, k);
            const rhs_t rk = (rhs_t)PLM(rkapa, k), dkap = (rhs_t)PLM(dkapa, k);
            const rhs_t hzdz = HZ * dz, hzd2z = HZ * d2z, h2zdz2 = H2Z * dz * dz;
            const rhs_t r0 = PLB(ro32, k), t0 = PLB(tt32, k);
#define CUR(f, d) cur(k, f, opt + (d))
#define NXT(f) cur(k + 1, f, opt)
#define RNG(kp, c, d) ring(kp, c, opt + (d))
#define TP(d) (LEAN ? CUR(3, d) : RNG(k, 3, d))
            float h0[8];
            rhs_t q0[8];
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                h0[f] = LEAN && f == 3 ? rho_k : CUR(f, 0);
                q0[f] = h0[f];
            }
            const rhs_t rh0 = q0[3], th0 = TP(0);
            const rhs_t tf0 = t0 + th0;                    // full temperature
            const rhs_t rinv = rcp32(r0 + rh0);                // 1/rho
            const rhs_t u0 = RNG(k, 0, 0), v0 = RNG(k, 1, 0), w0 = RNG(k, 2, 0);
            const rhs_t um = RNG(k - 1, 0, 0), vm = RNG(k - 1, 1, 0), wm = RNG(k - 1, 2, 0);
            const rhs_t up = RNG(k + 1, 0, 0), vp = RNG(k + 1, 1, 0), wp = RNG(k + 1, 2, 0);
            const rhs_t uxp = RNG(k, 0, 1), uxm = RNG(k, 0, -1), uyp = RNG(k, 0, SW), uym = RNG(k, 0, -SW);
            const rhs_t vxp = RNG(k, 1, 1), vxm = RNG(k, 1, -1), vyp = RNG(k, 1, SW), vym = RNG(k, 1, -SW);
            const rhs_t wxp = RNG(k, 2, 1), wxm = RNG(k, 2, -1), wyp = RNG(k, 2, SW), wym = RNG(k, 2, -SW);
            const rhs_t ru_m = rm_.v[0], rv_m = rm_.v[1], rw_m = rm_.v[2];
            const rhs_t ru_p = NXT(0), rv_p = NXT(1), rw_p = NXT(2);
            const rhs_t th_m = LEAN ? rm_.v[3] : RNG(k - 1, 3, 0), th_p = LEAN ? NXT(3) : RNG(k + 1, 3, 0);
            // stored pressure perturbation at the six neighbours
            const rhs_t pm = rm_.v[4], pp = NXT(4);
            const rhs_t pxm = CUR(4, -1), pxp = CUR(4, 1), pym = CUR(4, -SW), pyp = CUR(4, SW);

            rhs_t rwk2 = rhs_t(0), wk2 = rhs_t(0), bxk2 = rhs_t(0), bxk3 = rhs_t(0), byk2 = rhs_t(0), byk3 = rhs_t(0);
            if (top || bot) {
                const int ka = top ? k + 2 : k - 2;
                const int kb = top ? k + 3 : k - 3;
                const long long oa = (long long)ka * pl + ooff, ob = (long long)kb * pl + ooff;
                rwk2 = hin[2 * fs + oa];
                wk2 = rwk2 * rcp32((rhs_t)PLB(ro32, ka) + (rhs_t)hin[3 * fs + oa]);
                if (MAG) {
                    bxk2 = hin[5 * fs + oa];
                    byk2 = hin[6 * fs + oa];
                    bxk3 = hin[5 * fs + ob];
                    byk3 = hin[6 * fs + ob];
                }
            }

            // The FP32 right-hand side is evaluated with its multiply-adds
            // fused (one rounding instead of two).  The mixed form is judged
            // by its error against the FP64 form, not bit for bit; fusion is
            // decided per source expression, so every kernel that inlines
            // this body computes the same values.
            rhs_t fr, fw, fv, fu, ft, w1 = rhs_t(0), w2 = rhs_t(0), w3 = rhs_t(0);
            {
#pragma clang fp contract(on)
                // continuity
                fr = (CUR(0, -1) - CUR(0, 1)) * hxdx - (CUR(1, SW) - CUR(1, -SW)) * hydy;
                if (top) fr -= (rhs_t(4) * rw_p - rwk2) * hzdz;
                else if (bot) fr -= (rwk2 - rhs_t(4) * rw_m) * hzdz;
                else fr -= (rw_p - rw_m) * hzdz;
                // buoyancy and pressure gradient of the perturbation
                fw = GRAV * rh0 - (pp - pm) * hzdz;
                fv = (pym - pyp) * hydy;
                fu = (pxm - pxp) * hxdx;
                // momentum advection
                fu -= (CUR(0, 1) * uxp - CUR(0, -1) * uxm) * hxdx + (CUR(0, SW) * vyp - CUR(0, -SW) * vym) * hydy
                      + (ru_p * wp - ru_m * wm) * hzdz;
                fv -= (CUR(1, 1) * uxp - CUR(1, -1) * uxm) * hxdx + (CUR(1, SW) * vyp - CUR(1, -SW) * vym) * hydy
                      + (rv_p * wp - rv_m * wm) * hzdz;
                fw -= (CUR(2, 1) * uxp - CUR(2, -1) * uxm) * hxdx + (CUR(2, SW) * vyp - CUR(2, -SW) * vym) * hydy
                      + (rw_p * wp - rw_m * wm) * hzdz;
                // temperature advection, the background gradient included
                const rhs_t txp = TP(1), txm = TP(-1), typ = TP(SW), tym = TP(-SW);
                const rhs_t dtz = (th_p - th_m) * hzdz;
                ft = -(u0 * (txp - txm) * hxdx + v0 * (typ - tym) * hydy + w0 * (dtz + PLB(dt0dz32, k)));
                // conduction of T': (1/rho) c [kappa lap T' + kappa' dT'/dz]; plus the
                // change of the background's conduction with 1/rho: -rho'/(rho rho0) S0
                {
                    const rhs_t lap = (txp - txm) * hxd2x + (txp - rhs_t(2) * th0 + txm) * h2xdx2
                                      + (typ - tym) * hyd2y + (typ - rhs_t(2) * th0 + tym) * h2ydy2
                                      + (th_p - th_m) * hzd2z + (th_p - rhs_t(2) * th0 + th_m) * h2zdz2;
                    ft += rinv * PLP(t_cond, k) * (rk * lap + dkap * dtz) - rh0 * rinv * PLB(rinv0_32, k) * PLB(s0_32, k);
                }
                // viscous Laplacians
                fu += ORE * (C43 * ((uxp - uxm) * hxd2x + (uxp - rhs_t(2) * u0 + uxm) * h2xdx2)
                             + (uyp - uym) * hyd2y + (uyp - rhs_t(2) * u0 + uym) * h2ydy2
                             + (up - um) * hzd2z + (up - rhs_t(2) * u0 + um) * h2zdz2);
                fv += ORE * ((vxp - vxm) * hxd2x + (vxp - rhs_t(2) * v0 + vxm) * h2xdx2
                             + C43 * ((vyp - vym) * hyd2y + (vyp - rhs_t(2) * v0 + vym) * h2ydy2)
                             + (vp - vm) * hzd2z + (vp - rhs_t(2) * v0 + vm) * h2zdz2);
                fw += ORE * ((wxp - wxm) * hxd2x + (wxp - rhs_t(2) * w0 + wxm) * h2xdx2
                             + (wyp - wym) * hyd2y + (wyp - rhs_t(2) * w0 + wym) * h2ydy2
                             + C43 * ((wp - wm) * hzd2z + (wp - rhs_t(2) * w0 + wm) * h2zdz2));
                // heating and grad div u cross terms
                const rhs_t tv = PLP(t_visc, k), tv43 = PLP(t_visc43, k), tcr = PLP(t_cross, k);
                const rhs_t dxu = (uxp - uxm) * hxdx, dxv = (vxp - vxm) * hxdx, dxw = (wxp - wxm) * hxdx;
                const rhs_t dyu = (uyp - uym) * hydy, dyv = (vyp - vym) * hydy, dyw = (wyp - wym) * hydy;
                const rhs_t dzu = (up - um) * hzdz, dzv = (vp - vm) * hzdz, dzw = (wp - wm) * hzdz;
                ft += (C43 * dxu * dxu + dxv * dxv + dxw * dxw + dyu * dyu + rhs_t(2) * dyu * dxv) * rinv * tv
                      + (dyv * dyv + dzw * dzw - dxu * dzw - dxu * dyv - dyv * dzw) * rinv * tv43
                      + (dzu * dzu + dzv * dzv + dyw * dyw + rhs_t(2) * dzv * dyw + rhs_t(2) * dzu * dxw) * rinv * tv
                      - OCV * (dxu + dyv + dzw) * tf0;
                fu += tcr * (((RNG(k, 1, SW + 1) - RNG(k, 1, SW - 1)) - (RNG(k, 1, -SW + 1) - RNG(k, 1, -SW - 1))) * hxdx * hydy
                             + ((RNG(k + 1, 2, 1) - RNG(k - 1, 2, 1)) - (RNG(k + 1, 2, -1) - RNG(k - 1, 2, -1))) * hzdz * hxdx);
                fv += tcr * (((RNG(k, 0, SW + 1) - RNG(k, 0, SW - 1)) - (RNG(k, 0, -SW + 1) - RNG(k, 0, -SW - 1))) * hxdx * hydy
                             + ((RNG(k + 1, 2, SW) - RNG(k - 1, 2, SW)) - (RNG(k + 1, 2, -SW) - RNG(k - 1, 2, -SW))) * hzdz * hydy);
                fw += tcr * (((RNG(k + 1, 0, 1) - RNG(k - 1, 0, 1)) - (RNG(k + 1, 0, -1) - RNG(k - 1, 0, -1))) * hzdz * hxdx
                             + ((RNG(k + 1, 1, SW) - RNG(k - 1, 1, SW)) - (RNG(k + 1, 1, -SW) - RNG(k - 1, 1, -SW))) * hzdz * hydy);
                // Coriolis
                if (p.lrot) {
                    const rhs_t omx = PLP(omx, k), omz = PLP(omz, k);
                    fu += omz * q0[1];
                    fv += -omz * q0[0] + omx * q0[2];
                    fw -= omx * q0[1];
                }
                // MHD
                if (MAG) {
                    const rhs_t bx0 = q0[5], by0 = q0[6], bz0 = q0[7];
                    const rhs_t bxm = rm_.v[5], bym = rm_.v[6], bzm = rm_.v[7];
                    const rhs_t bxp = NXT(5), byp = NXT(6), bzp = NXT(7);
                    const rhs_t bxxp = CUR(5, 1), bxxm = CUR(5, -1), bxyp = CUR(5, SW), bxym = CUR(5, -SW);
                    const rhs_t byxp = CUR(6, 1), byxm = CUR(6, -1), byyp = CUR(6, SW), byym = CUR(6, -SW);
                    const rhs_t bzxp = CUR(7, 1), bzxm = CUR(7, -1), bzyp = CUR(7, SW), bzym = CUR(7, -SW);
                    rhs_t dzw1 = dzw;
                    if (top) dzw1 = (rhs_t(4) * wp - wk2) * hzdz;
                    else if (bot) dzw1 = (wk2 - rhs_t(4) * wm) * hzdz;
                    const rhs_t dxbx = (bxxp - bxxm) * hxdx, dxby = (byxp - byxm) * hxdx, dxbz = (bzxp - bzxm) * hxdx;
                    const rhs_t dybx = (bxyp - bxym) * hydy, dyby = (byyp - byym) * hydy, dybz = (bzyp - bzym) * hydy;
                    const rhs_t dzbx = (bxp - bxm) * hzdz, dzby = (byp - bym) * hzdz, dzbz = (bzp - bzm) * hzdz;
                    // induction (B.grad) u - B div u - (u.grad) B
                    w1 = by0 * dyu - bx0 * dyv + bz0 * dzu - bx0 * dzw1 - u0 * dxbx - v0 * dybx - w0 * dzbx;
                    w2 = bx0 * dxv - by0 * dxu + bz0 * dzv - by0 * dzw1 - u0 * dxby - v0 * dyby - w0 * dzby;
                    w3 = bx0 * dxw - bz0 * dxu + by0 * dyw - bz0 * dyv - u0 * dxbz - v0 * dybz - w0 * dzbz;
                    // Lorentz force
                    fu += OBETA * (by0 * (dybx - dxby) - bz0 * dxbz + bz0 * dzbx);
                    fv += OBETA * (bx0 * (dxby - dybx) + bz0 * (dzby - dybz));
                    fw += OBETA * (bx0 * dxbz - bx0 * dzbx - by0 * (dzby - dybz));
                    // Ohmic heating |J|^2 / rho
                    ft += ((dybx - dxby) * (dybx - dxby) + dxbz * dxbz + dzbx * dzbx - rhs_t(2) * dzbx * dxbz
                           + (dzby - dybz) * (dzby - dybz)) * rinv * PLP(t_ohm, k);
                    // resistive diffusion, one-sided in z on the boundary planes for BX, BY
                    rhs_t d2zbx, d2zby;
                    if (top) {
                        d2zbx = (-rhs_t(3) * bx0 + rhs_t(4) * bxp - bxk2) * hzd2z + (rhs_t(2) * bx0 - rhs_t(5) * bxp + rhs_t(4) * bxk2 - bxk3) * h2zdz2;
                        d2zby = (-rhs_t(3) * by0 + rhs_t(4) * byp - byk2) * hzd2z + (rhs_t(2) * by0 - rhs_t(5) * byp + rhs_t(4) * byk2 - byk3) * h2zdz2;
                    } else if (bot) {
                        d2zbx = (rhs_t(3) * bx0 - rhs_t(4) * bxm + bxk2) * hzd2z + (rhs_t(2) * bx0 - rhs_t(5) * bxm + rhs_t(4) * bxk2 - bxk3) * h2zdz2;
                        d2zby = (rhs_t(3) * by0 - rhs_t(4) * bym + byk2) * hzd2z + (rhs_t(2) * by0 - rhs_t(5) * bym + rhs_t(4) * byk2 - byk3) * h2zdz2;
                    } else {
                        d2zbx = (bxp - bxm) * hzd2z + (bxp - rhs_t(2) * bx0 + bxm) * h2zdz2;
                        d2zby = (byp - bym) * hzd2z + (byp - rhs_t(2) * by0 + bym) * h2zdz2;
                    }
                    const rhs_t d2zbz = (bzp - bzm) * hzd2z + (bzp - rhs_t(2) * bz0 + bzm) * h2zdz2;
                    w1 += ORM * ((bxxp - bxxm) * hxd2x + (bxxp - rhs_t(2) * bx0 + bxxm) * h2xdx2
                                 + (bxyp - bxym) * hyd2y + (bxyp - rhs_t(2) * bx0 + bxym) * h2ydy2 + d2zbx);
                    w2 += ORM * ((byxp - byxm) * hxd2x + (byxp - rhs_t(2) * by0 + byxm) * h2xdx2
                                 + (byyp - byym) * hyd2y + (byyp - rhs_t(2) * by0 + byym) * h2ydy2 + d2zby);
                    w3 += ORM * ((bzxp - bzxm) * hxd2x + (bzxp - rhs_t(2) * bz0 + bzxm) * h2xdx2
                                 + (bzyp - bzym) * hyd2y + (bzyp - rhs_t(2) * bz0 + bzym) * h2ydy2 + d2zbz);
                }
#undef CUR
#undef NXT
#undef TP
#undef RNG
            }
            // FP64 accumulation: F = F_bg(z) + F', X = value + D + gamma dt F
            // (the temperature slot's value is T'(rho', P')); store the new
            // FP32 values and carry the residual (+ zeta dt F) in D.  The
            // products dt F are fused into their sums; the residual itself
            // (X minus its stored representation) is exact either way.
            // (The boundary conditions overwrite RU, RV, RW and T of a boundary
            // plane after every stage: their right-hand sides are not needed.)
            double Fd[8] = {BND ? 0.0f : fu, BND ? 0.0f : fv, BND ? 0.0f : fw, fr, BND ? 0.0f : ft, w1, w2, w3};
            Fd[2] += PLB(fwbg, k);
            Fd[4] += PLB(ftbg, k);
            if (frc) {
                // (two 16-byte loads; the stages took 44, 50 and 54 us with seven of
                // 4 bytes, 40, 42 and 48 so, 128x128x64)
                const float4 *g = reinterpret_cast<const float4 *>(bg.force) + 2 * (o - pl);
                const float4 g0 = g[0];
                Fd[0] += (double)g0.x;
                Fd[1] += (double)g0.y;
                Fd[2] += (double)g0.z;
                Fd[4] += (double)g0.w;
                if (MAG) {
                    const float4 g1 = g[1];
                    Fd[5] += (double)g1.x;
                    Fd[6] += (double)g1.y;
                    Fd[7] += (double)g1.z;
                }
            }
            const double r0d = PLB(ro, k), t0d = PLB(tt, k);
            double xq[8];
            float hn[8];
#pragma unroll
            for (int f = 0; f < NF; ++f) {
#pragma clang fp contract(on)
                const double v = f == 4 ? (double)th0 : (double)h0[f];
                // (read only once this field's right-hand side exists)
                const float dkf = MODE == 1 ? r_half(after(rk_[f >> 1], Fd[f]), f) : after(dk_[f], Fd[f]);
                xq[f] = (v + (double)dkf) + coefg * Fd[f];
                if (f != 4) hn[f] = (float)xq[f];
            }
            hn[4] = (float)pprime(r0d, t0d, xq[3], xq[4]);
            float rs[8];
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                const double r = xq[f] - (f == 4 ? (double)trep(PLB(ro32, k), PLB(tt32, k), hn[3], hn[4]) : (double)hn[f]);
                __builtin_nontemporal_store(hn[f], &hout[f * fs + o]);
                if (MODE < 3) {
#pragma clang fp contract(on)
                    __builtin_nontemporal_store((float)(r + coefz * Fd[f]), &dr[f * fs + o]);
                } else {
                    rs[f] = (float)r;
                }
            }
            if (MODE == 3) {
                // the residuals as BF16 pairs (an odd last field with a zero high half)
#pragma unroll
                for (int w = 0; w < (NF + 1) / 2; ++w)
                    __builtin_nontemporal_store(pack_bf16x2(rs[2 * w], 2 * w + 1 < NF ? rs[2 * w + 1] : 0.0f),
                                                &rr[w * fs + o]);
            }
            if (MODE == 3 && !top && !bot) {
                double full[8];
#pragma unroll
                for (int f = 0; f < NF; ++f) full[f] = xq[f];
                full[3] += PLB(ro, k);
                full[4] += PLB(tt, k);
                const double ddz = PLM(ddz, k);
                const double dd2 = fmin(c_d2, ddz * ddz), idd2 = fmax(c_id2, PLB(iddz2, k));
                // (min(dd^2) is not accumulated per point: see the reduction)
                CflFast c{cfl_acc.mach, cfl_acc.q1, cfl_acc.s2, cfl_acc.s3, INFINITY};
                cflf_point<MAG>(p, full, dd2, idd2, PLB(irk, k), c);
                cfl_acc = c;
            }
#pragma unroll
            for (int f = 0; f < NF; ++f) rm_.v[f] = LEAN && f == 3 ? th0 : h0[f];
        }
        if (LEAN) {
            rho_k = rho_n;
            rho_n = rp_o.v[3];
        }
        __syncthreads();
        if (pre) {
            put_cur(k + 2, opt, rp_o);
            put_ring(k + 2, opt, rp_o);
            if (has_h) {
                put_cur(k + 2, hpt, rp_h);
                put_ring(k + 2, hpt, rp_h);
            }
        }
    };
#pragma unroll 1
    for (int k = kbeg; k <= kend; ++k) {
        if (k == 1 || k == npz) plane(k, std::true_type{});
        else plane(k, std::false_type{});
    }
    if ((kbeg == 1 || kend == npz) && valid) {
        const BoxArgs &l = late_args(args);
        bcon_column_m<MAG, MODE == 3>(l.p, l.m, l.bg, hout, dr, rr, gi, gj, kbeg == 1, kend == npz, cfl_acc);
    }
    if (MODE == 3) {
        // min(dd^2) depends on the grid only: its minimum over all points
        // comes with the metrics
        cflf_reduce(late_args(args).p, CflFast{cfl_acc.mach, cfl_acc.q1, cfl_acc.s2, cfl_acc.s3, INFINITY}, 1, sc, cs, seq, total,
                    MAG ? sc->dd2min : INFINITY);
    }
}

template <int TY, bool MAG, int MODE>
__global__ __launch_bounds__(MTile<TY>::NT, 3) void k_stage_m(const BoxArgs b,
                                                     const float *__restrict__ hin, float *__restrict__ hout,
                                                     float *__restrict__ dr, unsigned *__restrict__ rr,
                                                     DevScalars *__restrict__ sc, CflSlots *__restrict__ cs,
                                                     int nchunks) {
    extern __shared__ float ldsf[];
    const Params &p = b.p;
    const int W = TY ? MTX : p.tile_w, H = TY ? TY : p.tile_h;
    const int ntx = (p.npx + W - 1) / W, nty = (p.npy + H - 1) / H;
    const TileChunk tc = tile_of(blockIdx.x, ntx * nty, nchunks);
    const int tz = tc.chunk, tyb = tc.tile / ntx, txb = tc.tile - tyb * ntx;
    const int kbeg = chunk_begin(p.npz, nchunks, tz), kend = chunk_begin(p.npz, nchunks, tz + 1) - 1;
    stage_tile_m<TY, MAG, MODE>(p, b.m, b.bg, kernel_args(), hin, hout, dr, rr, sc, cs, txb * W, tyb * H, kbeg, kend,
                                blockIdx.x, gridDim.x, ldsf, W, H);
}

// Ensemble: persistent grid over the work items of all boxes (static stride);
// each item carries its tile's shape.
// Stage 1 of 64x8 tiles, 512 threads: at most 128 registers a lane, so that two
// workgroups fit a CU (a step of 8 boxes of 128x128x64 with 8 planes a chunk: 912
// us with 129 registers, 881 so; 16 of 64x64x64: 439, 418).
template <int TY, bool MAG, int MODE>
__global__ __launch_bounds__(MTile<TY>::NT, TY == 8 && MODE == 1 ? 4 : 3) void k_stage_m_batch(const BoxDev *__restrict__ boxes,
                                                           const StageItem *__restrict__ items, int nitems, int a) {
    extern __shared__ float ldsf[];
    const int slot = xcd_remap(blockIdx.x, gridDim.x);
    for (int w = slot; w < nitems; w += gridDim.x) {
        const StageItem it = items[w];
        const BoxDev &B = box_at(boxes, it.box);
        __syncthreads();  // the previous item's last LDS reads are done
        stage_tile_m<TY, MAG, MODE>(B.a.p, B.a.m, B.a.bg, (ArgPtr)&B.a, B.h[a], B.h[1 - a], B.dr, B.rr, B.sc, B.cs, it.i0, it.j0,
                                    it.kbeg, it.kend, it.seq, it.total, ldsf, it.w, it.h);
    }
}

// Stand-alone CFL of the mixed state (first step after an upload).
template <bool MAG>
__global__ __launch_bounds__(256) void k_cfl_m(const Params p, const Metrics m, const Background bg,
                                               const float *__restrict__ h, const unsigned *__restrict__ rr,
                                               DevScalars *__restrict__ sc, CflSlots *__restrict__ cs) {
    const long long fs = p.fsize, pl = p.plane;
    const long long n = (long long)p.npz * pl;
    CflFast cfl = cflf_init();
    for (long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x; idx < n;
         idx += (long long)gridDim.x * blockDim.x) {
        const long long o = pl + idx;
        const int k = (int)(idx / pl) + 1;
        const long long r2 = idx - (long long)(k - 1) * pl;
        const int j = (int)(r2 / p.npx), i = (int)(r2 - (long long)j * p.npx);
        double v[8];
        for (int f = 0; f < (MAG ? 8 : 5); ++f) {
            const double x = f == 4 ? (double)trep(bg.ro32[k], bg.tt32[k], h[3 * fs + o], h[4 * fs + o]) : (double)h[f * fs + o];
            v[f] = x + (double)r_get(rr, fs, f, o);
        }
        v[3] += bg.ro[k];
        v[4] += bg.tt[k];
        const DdPair d = ddpair(m.ddx[i + 1], m.ddy[j + 1], m.ddz[k]);
        cflf_point<MAG>(p, v, d.dd2, d.idd2, 1.0 / m.rkapa[k], cfl);
    }
    cflf_reduce(p, cfl, 0, sc, cs, blockIdx.x, gridDim.x);
}

// padded FP64 field f -> (stored value, R = rounding residual) in the
// registers hreg, rreg (all fields); the temperature is stored as the P' of
// the already packed rho' of the same register.
__global__ void k_pack_m(const Params p, const double *__restrict__ padded, int field, const Background bg,
                         float *__restrict__ hreg, unsigned *__restrict__ rreg) {
    const long long n = p.plane * (p.npz + 2), fs = p.fsize;  // n: the field's values
    const int nxp = p.npx + 2, nyp = p.npy + 2;
    float *const h = hreg + field * fs;
    for (long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x; idx < n;
         idx += (long long)gridDim.x * blockDim.x) {
        const long long k = idx / p.plane;
        const long long r = idx - k * p.plane;
        const int j = (int)(r / p.npx), i = (int)(r - (long long)j * p.npx);
        double v = padded[(k * nyp + (j + 1)) * nxp + (i + 1)];
        if (field == 4) {
            const double tp = v - bg.tt[k];
            const float rh = hreg[3 * fs + idx];
            const float hp = (float)pprime(bg.ro[k], bg.tt[k], (double)rh + (double)r_get(rreg, fs, 3, idx), tp);
            h[idx] = hp;
            r_put(rreg, fs, 4, idx, (float)(tp - (double)trep(bg.ro32[k], bg.tt32[k], rh, hp)));
            continue;
        }
        if (field == 3) v -= bg.ro[k];
        const float hn = (float)v;
        h[idx] = hn;
        r_put(rreg, fs, field, idx, (float)(v - (double)hn));
    }
}

// fields of (stored value, R) -> padded FP64 fields with periodic ghosts (one
// field per blockIdx.y)
__global__ void k_unpack_m(const Params p, const float *__restrict__ hreg, const unsigned *__restrict__ rreg,
                           const FieldList l, const Background bg) {
    const int field = l.f[blockIdx.y];
    double *__restrict__ const padded = l.dst[blockIdx.y];
    const int nxp = p.npx + 2, nyp = p.npy + 2, nzp = p.npz + 2;
    const long long n = (long long)nxp * nyp * nzp, fs = p.fsize;
    for (long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x; idx < n;
         idx += (long long)gridDim.x * blockDim.x) {
        const long long k = idx / ((long long)nxp * nyp);
        const long long r = idx - k * nxp * nyp;
        const int J = (int)(r / nxp), I = (int)(r - (long long)J * nxp);
        const long long o = k * p.plane + (long long)wrapi(J - 1, p.npy) * p.npx + wrapi(I - 1, p.npx);
        double v;
        if (field == 4) v = bg.tt[k] + (double)trep(bg.ro32[k], bg.tt32[k], hreg[3 * fs + o], hreg[4 * fs + o]);
        else v = (double)hreg[field * fs + o] + (field == 3 ? bg.ro[k] : 0.0);
        padded[idx] = v + (double)r_get(rreg, fs, field, o);
    }
}

// Re-centring of the background (mhd_rebase): rho and T of every interior
// point, reconstructed about the old background ob exactly as k_unpack_m
// does, are split about the new background nb exactly as k_pack_m does
// (rho' before T', whose stored P' uses the new rho' + R).  The other fields
// do not depend on the background; the z ghost planes keep their background.
__global__ void k_rebase_m(const Params p, const Background ob, const Background nb, float *__restrict__ hreg,
                           unsigned *__restrict__ rreg) {
    const long long fs = p.fsize, n = (long long)p.npz * p.plane;
    for (long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x; v < n;
         v += (long long)gridDim.x * blockDim.x) {
        const long long idx = p.plane + v;
        const int k = (int)(idx / p.plane);
        const float h3 = hreg[3 * fs + idx], h4 = hreg[4 * fs + idx];
        const double ro = ((double)h3 + ob.ro[k]) + (double)r_get(rreg, fs, 3, idx);
        const double tt = (ob.tt[k] + (double)trep(ob.ro32[k], ob.tt32[k], h3, h4)) + (double)r_get(rreg, fs, 4, idx);
        const double rp = ro - nb.ro[k];
        const float n3 = (float)rp;
        hreg[3 * fs + idx] = n3;
        r_put(rreg, fs, 3, idx, (float)(rp - (double)n3));
        const double tp = tt - nb.tt[k];
        const float n4 = (float)pprime(nb.ro[k], nb.tt[k], (double)n3 + (double)r_get(rreg, fs, 3, idx), tp);
        hreg[4 * fs + idx] = n4;
        r_put(rreg, fs, 4, idx, (float)(tp - (double)trep(nb.ro32[k], nb.tt32[k], n3, n4)));
    }
}

// Network inputs of the closure from the state (h, R) about the background: a
// plane per blockIdx.y, one 16-byte store a point.  Bound by the FP64 logarithms
// and divisions (128x128x64: 18 us; 22 with 64-bit divisions for the plane and
// eight 2-byte stores).
template <bool MAG>
__global__ __launch_bounds__(256) void k_closure_inputs(const Params p, const Background bg, const float *__restrict__ h,
                                                        const unsigned *__restrict__ rr,
                                                        const float *__restrict__ nrm, __bf16 *__restrict__ x,
                                                        int *__restrict__ force_on) {
    const long long fs = p.fsize;
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *force_on = 1;  // (the network's last layer clears it)
    for (int k = blockIdx.y + 1; k <= p.npz; k += gridDim.y)
        for (long long c0 = (long long)blockIdx.x * 256 + threadIdx.x; c0 < p.plane; c0 += (long long)gridDim.x * 256) {
            const long long o = k * p.plane + c0;
            float hv[8];
            unsigned w[4];
#pragma unroll
            for (int f = 0; f < (MAG ? 8 : 5); ++f) hv[f] = h[f * fs + o];
#pragma unroll
            for (int n = 0; n < (MAG ? 4 : 3); ++n) w[n] = rr[n * fs + o];
            auto val = [&](int f) { return (double)hv[f] + (double)r_half(w[f >> 1], f); };
            const double ro = bg.ro[k] + val(3);
            const double tt = bg.tt[k] + (double)trep(bg.ro32[k], bg.tt32[k], hv[3], hv[4]) + (double)r_half(w[2], 4);
            const double ri = 1.0 / ro;
            double c[8];
            c[0] = ro;
            c[1] = val(0) * ri;
            c[2] = val(1) * ri;
            c[3] = val(2) * ri;
            c[4] = log(tt) / (p.gamma - 1.0) - log(ro);
#pragma unroll
            for (int f = 5; f < 8; ++f) c[f] = MAG ? val(f) : 0.0;
            // nrm: per-plane means [8][npz], then 1/std [8]
            typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
            bf16x8 v;
#pragma unroll
            for (int f = 0; f < 8; ++f)
                v[f] = (__bf16)(float)((c[f] - (double)nrm[f * p.npz + k - 1]) * (double)nrm[8 * p.npz + f]);
            *reinterpret_cast<bf16x8 *>(x + (o - p.plane) * 8) = v;
        }
}

// ---------------------------------------------------------------------------

template <int TY, bool MAG, int MODE>
static hipError_t launch_m(const Params &p, const Metrics &m, const Background &bg, const float *hin, float *hout,
                           float *dr, unsigned *rr, DevScalars *sc, CflSlots *cs, hipStream_t s) {
    constexpr int lds = mixed_lds_bytes<TY, MAG, MODE>();
    static std::atomic<unsigned long long> attr{0};
    {
        hipError_t e = lds_limit_once(attr, reinterpret_cast<const void *>(&k_stage_m<TY, MAG, MODE>), lds);
        if (e != hipSuccess) return e;
    }
    const int nch = p.nchunks;
    hipLaunchKernelGGL((k_stage_m<TY, MAG, MODE>), dim3(tiles_of(p) * nch), dim3(MTile<TY>::NT), lds, s, BoxArgs{p, m, bg}, hin, hout,
                       dr, rr, sc, cs, nch);
    return hipGetLastError();
}

template <int TY>
static hipError_t launch_m_ty(int mode, const Params &p, const Metrics &m, const Background &bg, const float *hin,
                              float *hout, float *dr, unsigned *rr, DevScalars *sc, CflSlots *cs, hipStream_t s) {
    if (p.lmag) {
        if (mode == 1) return launch_m<TY, true, 1>(p, m, bg, hin, hout, dr, rr, sc, cs, s);
        if (mode == 2) return launch_m<TY, true, 2>(p, m, bg, hin, hout, dr, rr, sc, cs, s);
        return launch_m<TY, true, 3>(p, m, bg, hin, hout, dr, rr, sc, cs, s);
    }
    if (mode == 1) return launch_m<TY, false, 1>(p, m, bg, hin, hout, dr, rr, sc, cs, s);
    if (mode == 2) return launch_m<TY, false, 2>(p, m, bg, hin, hout, dr, rr, sc, cs, s);
    return launch_m<TY, false, 3>(p, m, bg, hin, hout, dr, rr, sc, cs, s);
}

hipError_t launch_stage_mixed(int mode, const Params &p, const Metrics &m, const Background &bg, const float *hin,
                              float *hout, float *dr, unsigned *rr, DevScalars *sc, CflSlots *cs, hipStream_t s) {
    if (p.tile_w) return launch_m_ty<0>(mode, p, m, bg, hin, hout, dr, rr, sc, cs, s);
    if (p.tile_y == 8) return launch_m_ty<8>(mode, p, m, bg, hin, hout, dr, rr, sc, cs, s);
    return launch_m_ty<4>(mode, p, m, bg, hin, hout, dr, rr, sc, cs, s);
}

hipError_t launch_cfl_mixed(const Params &p, const Metrics &m, const Background &bg, const float *h,
                            const unsigned *rr, DevScalars *sc, CflSlots *cs, hipStream_t s) {
    const long long n = (long long)p.npz * p.plane;
    long long nb = (n + 255) / 256;
    if (nb > 2048) nb = 2048;
    if (p.lmag) hipLaunchKernelGGL(k_cfl_m<true>, dim3((unsigned)nb), dim3(256), 0, s, p, m, bg, h, rr, sc, cs);
    else hipLaunchKernelGGL(k_cfl_m<false>, dim3((unsigned)nb), dim3(256), 0, s, p, m, bg, h, rr, sc, cs);
    return hipGetLastError();
}

hipError_t launch_pack_mixed(const Params &p, const double *padded, int field, const Background &bg, float *hreg,
                             unsigned *rreg, hipStream_t s) {
    long long nb = (p.plane * (p.npz + 2) + 255) / 256;
    if (nb > 8192) nb = 8192;
    hipLaunchKernelGGL(k_pack_m, dim3((unsigned)nb), dim3(256), 0, s, p, padded, field, bg, hreg, rreg);
    return hipGetLastError();
}

hipError_t launch_unpack_mixed(const Params &p, const float *hreg, const unsigned *rreg, const FieldList &l,
                               const Background &bg, hipStream_t s) {
    const long long n = (long long)(p.npx + 2) * (p.npy + 2) * (p.npz + 2);
    long long nb = (n + 255) / 256;
    if (nb > 8192) nb = 8192;
    hipLaunchKernelGGL(k_unpack_m, dim3((unsigned)nb, l.n), dim3(256), 0, s, p, hreg, rreg, l, bg);
    return hipGetLastError();
}

hipError_t launch_rebase_mixed(const Params &p, const Background &ob, const Background &nb, float *hreg,
                               unsigned *rreg, hipStream_t s) {
    const long long n = (long long)p.npz * p.plane;
    long long nb_ = (n + 255) / 256;
    if (nb_ > 8192) nb_ = 8192;
    hipLaunchKernelGGL(k_rebase_m, dim3((unsigned)nb_), dim3(256), 0, s, p, ob, nb, hreg, rreg);
    return hipGetLastError();
}

template <int TY, bool MAG, int MODE>
static hipError_t launch_mb(const BoxDev *boxes, const StageItem *items, int nitems, int grid, int a,
                            hipStream_t s) {
    constexpr int lds = mixed_lds_bytes<TY, MAG, MODE>();
    static std::atomic<unsigned long long> attr{0};
    {
        hipError_t e = lds_limit_once(attr, reinterpret_cast<const void *>(&k_stage_m_batch<TY, MAG, MODE>), lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((k_stage_m_batch<TY, MAG, MODE>), dim3(grid), dim3(MTile<TY>::NT), lds, s, boxes, items, nitems,
                       a);
    return hipGetLastError();
}

template <int TY>
static hipError_t launch_mb_ty(int mode, int lmag, const BoxDev *boxes, const StageItem *items, int nitems,
                               int grid, int a, hipStream_t s) {
    if (lmag) {
        if (mode == 1) return launch_mb<TY, true, 1>(boxes, items, nitems, grid, a, s);
        if (mode == 2) return launch_mb<TY, true, 2>(boxes, items, nitems, grid, a, s);
        return launch_mb<TY, true, 3>(boxes, items, nitems, grid, a, s);
    }
    if (mode == 1) return launch_mb<TY, false, 1>(boxes, items, nitems, grid, a, s);
    if (mode == 2) return launch_mb<TY, false, 2>(boxes, items, nitems, grid, a, s);
    return launch_mb<TY, false, 3>(boxes, items, nitems, grid, a, s);
}

// 64x8 tiles, or tiles of at most 256 points of the items' own shapes.
hipError_t launch_stage_batch_mixed(int mode, int tile_x, int tile_y, int lmag, const BoxDev *boxes,
                                    const StageItem *items, int nitems, int grid, int a, hipStream_t s) {
    if (tile_x == 64 && tile_y == 8) return launch_mb_ty<8>(mode, lmag, boxes, items, nitems, grid, a, s);
    return launch_mb_ty<0>(mode, lmag, boxes, items, nitems, grid, a, s);
}

hipError_t launch_closure_inputs(const Params &p, const Background &bg, const float *h, const unsigned *rr,
                                 const float *nrm, __bf16 *x, int *force_on, hipStream_t s) {
    const long long nb = (p.plane + 255) / 256;
    const dim3 grid((unsigned)(nb > 4096 ? 4096 : nb), (unsigned)(p.npz > 4096 ? 4096 : p.npz));
    if (p.lmag) hipLaunchKernelGGL(k_closure_inputs<true>, grid, dim3(256), 0, s, p, bg, h, rr, nrm, x, force_on);
    else hipLaunchKernelGGL(k_closure_inputs<false>, grid, dim3(256), 0, s, p, bg, h, rr, nrm, x, force_on);
    return hipGetLastError();
}

}  // namespace rmhd
