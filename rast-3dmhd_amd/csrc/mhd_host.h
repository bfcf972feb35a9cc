// Host-side helpers shared by the single-box and the ensemble C-ABI.
#pragma once

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../include/rast3dmhd.h"
#include "mhd_copy.h"
#include "mhd_kernels.h"

namespace rmhd {

// Records an error for mhd_last_error(NULL) (the message of calls without a
// handle) and returns code (mhd_capi.hip).
int global_fail(int code, const char *fmt, ...);

// Whether a descriptor switches on any optional branch of FLUXES/BCON.
inline bool desc_branches(const mhd_desc *d) {
    return d->id != 0 || d->lrem || d->lshr || d->rlax > 0.0 || d->itcon > 1 || d->tp != 0.0;
}

// Branches whose kernels read the coordinate tables (EXX, WYY, ZEE).
inline bool desc_needs_coords(const mhd_desc *d) {
    return (d->tp != 0.0 && (d->itcon == 0 || d->itcon == 1)) || d->itcon == 2 || d->id == 2 || d->rlax > 0.0;
}

// Checks a descriptor; on failure writes a message to msg and returns the
// MHD_ERR_* code.
inline int check_desc(const mhd_desc *d, char *msg, size_t len) {
    if (d->npx < 3 || d->npy < 3 || d->npz < 4) {
        snprintf(msg, len, "box %dx%dx%d too small (need npx,npy>=3, npz>=4)", d->npx, d->npy, d->npz);
        return MHD_ERR_ARG;
    }
    if (d->izcon != 0 && d->izcon != 1) {
        snprintf(msg, len, "IZCON=%d (BCON: Invalid IZCON)", d->izcon);
        return MHD_ERR_SCOPE;
    }
    if (d->itcon < 0 || d->itcon > 4) {
        snprintf(msg, len, "ITCON=%d not supported (0..4)", d->itcon);
        return MHD_ERR_SCOPE;
    }
    if (d->precision != MHD_FP64 && d->precision != MHD_MIXED) {
        snprintf(msg, len, "precision %d unknown", d->precision);
        return MHD_ERR_ARG;
    }
    if (d->id < 0 || d->id > 2) {
        snprintf(msg, len, "ID=%d not supported (0..2)", d->id);
        return MHD_ERR_SCOPE;
    }
    if (d->rlax > 0.0 && !(d->itcon == 0 && d->izcon == 1)) {
        // the reference stops for other pairs (sub:1642-1646), and its fixed-flux
        // top / fixed-T bottom integral reads FRADM(NZ), which it never sets on
        // the bottom rank (sub:1679-1691, 1745-1748)
        snprintf(msg, len, "flux relaxation (RLAX > 0) needs ITCON=0 and IZCON=1");
        return MHD_ERR_SCOPE;
    }
    if (d->lshr && (d->lrem || d->rlax > 0.0)) {
        snprintf(msg, len, "LSHR with LREM or RLAX (the reference uses a stale TTM there)");
        return MHD_ERR_SCOPE;
    }
    const int npey = d->npey > 0 ? d->npey : 1, npez = d->npez > 0 ? d->npez : 1;
    if (d->npy % npey || d->npz % npez) {
        snprintf(msg, len, "NPEY=%d / NPEZ=%d do not divide NPY=%d / NPZ=%d", npey, npez, d->npy, d->npz);
        return MHD_ERR_ARG;
    }
    if (desc_branches(d) && d->precision != MHD_FP64) {
        snprintf(msg, len, "the optional FLUXES/BCON branches (ID, LREM, LSHR, RLAX, ITCON 2..4, TP) are built "
                           "in the MHD_FP64 form only");
        return MHD_ERR_SCOPE;
    }
    return MHD_OK;
}

// z chunks of a box's stage launches.  A launch is a number of rounds in
// which every CU holds `occ` workgroups, and a last round with fewer; a
// workgroup's time is its planes plus about 1.5 planes of warm-up, times the
// time of a plane, which grows with the workgroups that share the CU (FP64:
// 3.3 us alone, 5.7 us with two; mixed: 2.6, 3.5, 4.4 us).  The count with
// the least sum wins: small boxes split until the chip is about full (64x64x32
// FP64: 11 chunks of up to 3 planes, stages of 16, 17 and 22 us against 38 with 4
// chunks on 64 of 256 CUs), larger ones take whole rounds (256x256x128 mixed: 6 chunks, two
// full rounds, 230 us against 254 with 16 chunks of 5.3 rounds).  Chunks are
// at most 32 planes: over a longer march the tiles that share halo rows drift
// apart and re-read them from HBM (512x512x256 FP64, 128 planes: 14% more
// bytes fetched).
struct ZSplit {
    int nc;
    double time;  // of a launch, us
};
inline ZSplit z_chunks(int npz, int ntiles, int occ, double alone, double more) {
    constexpr int CUS = 256;
    ZSplit best{0, 0.0};
    for (int nc = (npz + 31) / 32; nc <= max_chunks(npz) || !best.nc; ++nc) {
        const long long n = (long long)ntiles * nc, slots = (long long)CUS * occ;
        const long long rest = (n % slots + CUS - 1) / CUS;
        const double round = alone + (occ - 1) * more, last = rest ? alone + (rest - 1) * more : 0.0;
        const double t = (chunk_depth(npz, nc) + 1.5) * ((double)(n / slots) * round + last);
        if (!best.nc || t < best.time) best = ZSplit{nc, t};
    }
    return best;
}

// The tile of a box: 64x4, or one of at most 256 points fitted to its width if
// that saves 5% (mixed: 12%) of time(tiles) times a tile's own cost.  64-column
// tiles leave up to half of the lanes of a narrow or ragged box idle (a 40-column
// box: 24 of 64).  Fitted tiles are npx / m columns wide, so that whole rows of a
// narrow box are one contiguous run of memory.  Against them speak the ends of a
// tile's rows that are not on 64 bytes, where two tiles write a piece each (3% of
// a tile's time per end in FP64, 9% in the mixed form: 320x320x100 mixed, 64x4 2.1
// us a tile, 54x4 3.1, 40x6 3.3), and more, shorter rows (5% each).  Steps from
// 64x4 to fitted, FP64: 40x72x54 64 -> 55 us (40x6), 72x200x64 249 -> 200 (72x3),
// 130x90x41 hydro 91 -> 85 (44x5); mixed: 72x200x64 164 -> 119 (72x3), 150x300x100
// 628 -> 559 (75x3).  Left at 64x4: 300x300x100 FP64 (1595; 50x5: 1852),
// 160x160x64 mixed (185; 80x3: 189).
template <class Time>
inline TileShape fit_tile(int npx, int npy, bool mixed, Time time) {
    const int esz = mixed ? 4 : 8, points = mixed ? FIT_POINTS_MIXED : FIT_POINTS_FP64;
    auto cost = [&](TileShape t) {
        const bool rows = t.w == npx;  // whole rows: the ends are the tile's two
        const long long run = (long long)t.w * (rows ? t.h : 1) * esz, pitch = rows ? 64 : (long long)npx * esz;
        int unit = 64;
        while (run % unit || pitch % unit) unit /= 2;
        const double ends = (rows ? 2 : 2 * t.h) * (1.0 - unit / 64.0);
        const double more = rows || t.h < 4 ? 0.0 : 0.05 * (t.h - 4);
        return time(tile_count(npx, npy, t)) * (1.0 + (mixed ? 0.09 : 0.03) * ends + more);
    };
    TileShape best{64, 4};
    double least = (mixed ? 0.88 : 0.95) * cost(best);
    for (int m = (npx + 95) / 96; m <= npx; ++m) {
        const int w = (npx + m - 1) / m;
        if (m > 1 && w < 32) break;
        int h = 256 / w < npy ? 256 / w : npy;
        while ((w + 2) * (h + 2) > points) --h;
        const int n = (npy + h - 1) / h;
        const TileShape t{w, (npy + n - 1) / n};
        const double c = cost(t);
        if (c < least) {
            least = c;
            best = t;
        }
    }
    return best;
}

// Kernel parameters of a box.  The products the reference forms once per
// FLUXES / STEP call are formed here with the same association.
inline Params params_from_desc(const mhd_desc *d) {
    Params p{};
    p.npx = d->npx; p.npy = d->npy; p.npz = d->npz;
    p.lmag = d->lmag ? 1 : 0; p.lrot = d->lrot ? 1 : 0;
    p.izc = d->izcon; p.itc = d->itcon; p.ibc = d->ibcon;
    p.tile_y = 4;
    if (const char *ty = getenv("RAST3DMHD_TILE_Y")) p.tile_y = atoi(ty) == 8 ? 8 : 4;
    p.plane = (long long)d->npx * d->npy;
    p.fsize = p.plane * (d->npz + 2) + FIELD_PAD;
    p.hx = d->hx; p.h2x = d->h2x; p.hy = d->hy; p.h2y = d->h2y; p.hz = d->hz; p.h2z = d->h2z;
    p.c13 = d->c13; p.c23 = d->c23; p.c43 = d->c43;
    p.gam1 = d->gam1; p.gam2 = d->gam2; p.gam3 = d->gam3; p.zeta1 = d->zeta1; p.zeta2 = d->zeta2;
    p.cv = d->cv; p.ocv = d->ocv; p.ore = d->ore; p.re = d->re; p.repr = d->repr;
    p.theta = d->theta; p.grav = d->grav; p.sf = d->sf; p.gamma = d->gamma;
    p.omx = d->lrot ? d->omx : 0.0; p.omz = d->lrot ? d->omz : 0.0;
    p.orm = d->orm; p.rm = d->rm; p.obeta = d->obeta; p.tb = d->tb; p.dzf = d->dzf;
    p.ogamma = 1.0 / d->gamma;             // sub:744
    p.t_cond = d->ocv / d->repr;           // sub:1584
    p.t_visc = d->ocv * d->ore;            // sub:1904
    p.t_visc43 = d->c43 * d->ocv * d->ore; // sub:1962
    p.t_cross = d->c13 * d->ore;           // sub:1930
    p.t_ohm = d->obeta * d->orm * d->ocv;  // sub:2287
    p.id = d->id; p.lrem = d->lrem ? 1 : 0; p.lshr = d->lshr ? 1 : 0;
    p.mirror = (d->id != 0 || d->lrem) ? 1 : 0;
    p.npey = d->npey > 0 ? d->npey : 1; p.npez = d->npez > 0 ? d->npez : 1;
    p.dh = d->dh; p.dv = d->dv; p.tu = d->tu; p.dztu = d->dztu; p.dztb = d->dztb;
    p.rlax = d->rlax; p.tstart = d->tstart; p.toff = d->toff; p.tp = d->tp; p.tc = d->tc; p.hh = d->hh;
    p.tpr = d->tp;
    p.opt = p.lrem || p.lshr || p.rlax > 0.0 || p.itc == 2 ? 2 : p.id != 0 ? 1 : 0;
    {
        // workgroups per CU by LDS and registers (64x8 tiles: half)
        const bool mixed = d->precision == MHD_MIXED;
        const int occ = (mixed ? (d->lmag ? 3 : 4) : 2) / (p.tile_y == 8 ? 2 : 1);
        auto split = [&](int ntiles) { return z_chunks(d->npz, ntiles, occ, mixed ? 2.6 : 3.3, mixed ? 0.9 : 2.4); };
        if (p.tile_y == 4 && p.opt != 2) {
            const TileShape t = fit_tile(d->npx, d->npy, mixed, [&](int ntiles) { return split(ntiles).time; });
            if (t.w != 64 || t.h != 4) {
                p.tile_w = t.w;
                p.tile_h = t.h;
            }
        }
        p.nchunks = split(tiles_of(p)).nc;
    }
    return p;
}

// Initial device scalars: clocks zero.
inline DevScalars initial_scalars() {
    DevScalars s{};
    s.dd2min = INFINITY;
    return s;
}

// min over the points i = 1..npx, j = 1..npy, k = 1..npz of
// min(DDX_i, DDY_j, DDZ_k)^2, the grid-only term of the magnetic CFL limit
// (the same squares and minimum the per-point reduction forms).
inline double dd2_min(const Params &p, const double *ddx, const double *ddy, const double *ddz) {
    double m = INFINITY;
    for (int i = 1; i <= p.npx; ++i) m = std::fmin(m, ddx[i] * ddx[i]);
    for (int j = 1; j <= p.npy; ++j) m = std::fmin(m, ddy[j] * ddy[j]);
    for (int k = 1; k <= p.npz; ++k) m = std::fmin(m, ddz[k] * ddz[k]);
    return m;
}

// Number of doubles of the 11 metric arrays of a box.
inline size_t metric_len(const Params &p) {
    return 3 * (size_t)(p.npx + 2) + 3 * (size_t)(p.npy + 2) + 5 * (size_t)(p.npz + 2);
}

// Lengths of the 11 metric arrays in the order dxxdx, d2xxdx2, ddx, dyydy,
// d2yydy2, ddy, dzzdz, d2zzdz2, ddz, rkapa, dkapa.
inline void metric_lengths(const Params &p, size_t len[11]) {
    const size_t lx = p.npx + 2, ly = p.npy + 2, lz = p.npz + 2;
    const size_t l[11] = {lx, lx, lx, ly, ly, ly, lz, lz, lz, lz, lz};
    for (int n = 0; n < 11; ++n) len[n] = l[n];
}

// Points the Metrics table into a packed device block of metric_len doubles
// (same order) and returns each array's length in len[11].
inline Metrics metric_table(const Params &p, const double *base, size_t len[11]) {
    metric_lengths(p, len);
    const double *a[11];
    size_t off = 0;
    for (int n = 0; n < 11; ++n) {
        a[n] = base + off;
        off += len[n];
    }
    Metrics m;
    m.dxxdx = a[0]; m.d2xxdx2 = a[1]; m.ddx = a[2];
    m.dyydy = a[3]; m.d2yydy2 = a[4]; m.ddy = a[5];
    m.dzzdz = a[6]; m.d2zzdz2 = a[7]; m.ddz = a[8];
    m.rkapa = a[9]; m.dkapa = a[10];
    m.rkcfl = a[9];
    return m;
}

// Host tables of the mixed form's background for planes 0..npz+1:
// dbl = [ro | tt | fwbg | ftbg], flt = [ro32 | tt32 | dt0dz32 | rinv0_32 | s0_32].
// The background actually used is the given profile rounded to FP32
// values, so that the FP32 copies the perturbation stencil multiplies with
// are exact: the perturbation pressure rho0 T' + rho' (T0 + T') is a small
// residual of nearly cancelling terms in low-Mach flow, and different
// rounding errors of rho0 and T0 would leave a systematic error in it.
// fwbg, ftbg are the background's own discrete residuals of the momentum z
// and temperature equations (conduction S0 / rho0), formed in FP64 with the
// same stencils as the step.  iddz2 = 1/ddz^2 and irk = 1/rkapa are per-plane
// factors of the CFL limits, divided here once instead of per point (IEEE
// division on host and device alike).  Returns the first plane with
// rho0 <= 0, or -1.
constexpr int BG_DBL = 6, BG_FLT = 5;  // FP64 and FP32 tables of npz+2 entries
inline int background_tables(const Params &p, const double *dzzdz, const double *d2zzdz2, const double *ddz,
                             const double *rkapa, const double *dkapa, const double *ro0, const double *tt0,
                             std::vector<double> &dbl, std::vector<float> &flt, std::vector<PlaneM> &pl) {
    const int nz = p.npz + 2;
    dbl.assign(BG_DBL * (size_t)nz, 0.0);
    flt.assign(BG_FLT * (size_t)nz, 0.0f);
    double *ro = dbl.data(), *tt = ro + nz, *fw = tt + nz, *ft = fw + nz, *iz = ft + nz, *irk = iz + nz;
    float *ro32 = flt.data(), *tt32 = ro32 + nz, *dtz = tt32 + nz, *ri = dtz + nz, *s0 = ri + nz;
    for (int k = 0; k < nz; ++k) {
        if (!(ro0[k] > 0.0) || !((float)ro0[k] > 0.0f)) return k;
        ro32[k] = (float)ro0[k];
        tt32[k] = (float)tt0[k];
        ro[k] = (double)ro32[k];
        tt[k] = (double)tt32[k];
        ri[k] = (float)(1.0 / ro[k]);
    }
    for (int k = 1; k <= p.npz; ++k) {
        const double dz = dzzdz[k], d2z = d2zzdz2[k];
        const double g0 = (tt[k + 1] - tt[k - 1]) * p.hz * dz;
        const double l0 = (tt[k + 1] - tt[k - 1]) * p.hz * d2z + (tt[k + 1] - 2.0 * tt[k] + tt[k - 1]) * p.h2z * dz * dz;
        const double sz = p.t_cond * (rkapa[k] * l0 + dkapa[k] * g0);
        dtz[k] = (float)g0;
        s0[k] = (float)sz;
        ft[k] = sz / ro[k];
        fw[k] = p.grav * ro[k] - (ro[k + 1] * tt[k + 1] - ro[k - 1] * tt[k - 1]) * p.hz * dz;
        iz[k] = 1.0 / (ddz[k] * ddz[k]);
        irk[k] = 1.0 / rkapa[k];
    }
    pl.assign((size_t)nz, PlaneM{});
    for (int k = 0; k < nz; ++k) {
        PlaneM &q = pl[k];
        q.dzzdz = dzzdz[k];
        q.d2zzdz2 = d2zzdz2[k];
        q.rkapa = rkapa[k];
        q.dkapa = dkapa[k];
        q.ddz = ddz[k];
        q.ro = ro[k];
        q.tt = tt[k];
        q.fwbg = fw[k];
        q.ftbg = ft[k];
        q.iddz2 = iz[k];
        q.irk = irk[k];
        q.ro32 = ro32[k];
        q.tt32 = tt32[k];
        q.dt0dz32 = dtz[k];
        q.rinv0_32 = ri[k];
        q.s0_32 = s0[k];
        q.c43 = (float)p.c43;
        q.ocv = (float)p.ocv;
        q.ore = (float)p.ore;
        q.orm = (float)p.orm;
        q.obeta = (float)p.obeta;
        q.grav = (float)p.grav;
        q.t_cond = (float)p.t_cond;
        q.t_visc = (float)p.t_visc;
        q.t_visc43 = (float)p.t_visc43;
        q.t_cross = (float)p.t_cross;
        q.t_ohm = (float)p.t_ohm;
        q.omx = (float)p.omx;
        q.omz = (float)p.omz;
    }
    return -1;
}

// Fields of the device staging buffer of a box (its size in padded fields):
// as many as fit 16 MiB, and at least one: the download of a small box is then
// one launch, of a large one a launch per field beside the copy of the last.
inline int stage_fields(int nf, size_t field_bytes) {
    const size_t n = ((size_t)16 << 20) / field_bytes;
    return n < 1 ? 1 : n > (size_t)nf ? nf : (int)n;
}

// Download of the padded fields f = 0..nf-1 with dst[f] set: unpack(list)
// queues the launch that writes the listed fields into the staging buffer
// (room fields of field_bytes).
template <class Unpack>
hipError_t download_fields(double *const *dst, int nf, size_t field_bytes, double *stage, int room, Unpack unpack,
                           hipStream_t s) {
    struct Ctx {
        int n = 0, f[NFIELD];
        double *stage;
        size_t field_bytes;
        int room;
        Unpack *unpack;
    } c;
    HostSpan spans[NFIELD];
    for (int f = 0; f < nf; ++f)
        if (dst[f]) {
            spans[c.n] = HostSpan{dst[f], field_bytes};
            c.f[c.n++] = f;
        }
    c.stage = stage;
    c.field_bytes = field_bytes;
    c.room = room;
    c.unpack = &unpack;
    const FillFn fill = [](void *ctx, int i, const char **src, hipError_t *err) {
        const Ctx &x = *static_cast<Ctx *>(ctx);
        FieldList l{};
        for (l.n = 0; l.n < x.room && i + l.n < x.n; ++l.n) {
            l.f[l.n] = x.f[i + l.n];
            l.dst[l.n] = x.stage + (size_t)l.n * (x.field_bytes / sizeof(double));
        }
        *src = reinterpret_cast<const char *>(x.stage);
        *err = (*x.unpack)(l);
        return *err == hipSuccess ? l.n : 0;
    };
    return c.n ? copy_out(spans, c.n, fill, &c, s) : hipSuccess;
}

// Download of one contiguous device array that work queued on s produces.
inline hipError_t download_array(void *dst, const void *src, size_t bytes, hipStream_t s) {
    const HostSpan span{dst, bytes};
    const FillFn fill = [](void *ctx, int, const char **out, hipError_t *) {
        *out = static_cast<const char *>(ctx);
        return 1;
    };
    return copy_out(&span, 1, fill, const_cast<void *>(src), s);
}

// Background table pointers into device blocks laid out as background_tables.
inline Background background_view(int npz, const double *bgd, const float *bgf) {
    const int nz = npz + 2;
    Background bg{};
    bg.ro = bgd;
    bg.tt = bgd + nz;
    bg.fwbg = bgd + 2 * nz;
    bg.ftbg = bgd + 3 * nz;
    bg.iddz2 = bgd + 4 * nz;
    bg.irk = bgd + 5 * nz;
    bg.ro32 = bgf;
    bg.tt32 = bgf + nz;
    bg.dt0dz32 = bgf + 2 * nz;
    bg.rinv0_32 = bgf + 3 * nz;
    bg.s0_32 = bgf + 4 * nz;
    return bg;
}

}  // namespace rmhd
