// Horizontal means and mean flux profiles of the resident state (a
// diagnostic beside the step): the reference's HORIZONTAL_MEAN
// (3dmhdsub.f:3143-3223) of T and rho, and the mean convective flux FCONM
// (3dmhdsub.f:1650-1661), the horizontal mean of
//     -RW (2.5 (T - TTM) + 0.5 |u|^2),   u = RU (1/RO),
// on every interior plane.  The sums are formed by PROF_SEGS workgroups per plane
// in one pass over the state: the flux with the mean T0 of 64 of the plane's points
// in the place of TTM, whose difference times the sum of RW is added at the end (T0
// is as near as a sample allows, so the terms cancel as those about TTM do).  Each
// sum runs in a fixed order (per-thread strides with the rounding errors beside, a
// fixed reduction tree, the workgroups in order), so the result is the same on
// every run.  (The
// reference sums sequentially; the two orders agree to rounding.)  Bound by the
// read of five fields: 256x256x125 70 us, 155 with two passes by one workgroup per
// plane.

#include "mhd_device.h"

namespace rmhd {

constexpr int PROF_THREADS = 256;

// A sum with the rounding errors of its additions summed beside it (Knuth's
// two-sum): free beside the loads.  The flux about T0 ends in a difference and a
// product more than the flux about TTM; so carried, it is no further from the
// exact mean (FCONM of 48x48x25 to 144x144x73, largest error over largest value:
// 2.1e-16 in two plain passes, 3.7e-16 in one plain pass).
struct Sum {
    double s, c;
    __device__ void add(double x) {
        const double t = s + x, b = t - s;
        c += (s - (t - b)) + (x - b);
        s = t;
    }
    __device__ void add(const Sum &o) {
        add(o.s);
        c += o.c;
    }
    // a sum that is not finite has no rounding error to add
    __device__ double value() const { return isfinite(s) ? s + c : s; }
};
struct Sums {
    Sum t, r, w, f;  // T, RO, RW, flux about T0
};

// Deterministic workgroup sum: wavefront butterflies, then the wavefront
// partials in order.  Thread 0 returns the total.
__device__ Sum block_sum(Sum v, Sum *red) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        Sum o;
        o.s = __shfl_xor(v.s, off, 64);
        o.c = __shfl_xor(v.c, off, 64);
        v.add(o);
    }
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) red[wv] = v;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < PROF_THREADS / 64; ++w) v.add(red[w]);
    return v;
}

// Values of the state at offset o of plane k, FP64 form (register q).
struct StateFp64 {
    const double *q;
    long long fs;
    __device__ double get(int f, int, long long o) const { return q[f * fs + o]; }
};

// Mixed form: stored values h and resting residual R about the background.
struct StateMixed {
    const float *h;
    const unsigned *rr;
    Background bg;
    long long fs;
    __device__ double get(int f, int k, long long o) const {
        if (f == 4)
            return bg.tt[k] + (double)trep(bg.ro32[k], bg.tt32[k], h[3 * fs + o], h[4 * fs + o]) +
                   (double)r_get(rr, fs, 4, o);
        const double v = (double)h[f * fs + o] + (double)r_get(rr, fs, f, o);
        return f == 3 ? bg.ro[k] + v : v;
    }
};

// part[k-1][segment] = sums of T, RO, RW and of the flux about T0 over the points
// of segment blockIdx.y of plane k = blockIdx.x + 1.  T0 goes to out's place of FCONM.
template <class S>
__global__ __launch_bounds__(PROF_THREADS) void k_flux_sums(const Params p, const S st, Sums *__restrict__ part,
                                                            double *__restrict__ out) {
    __shared__ Sum red[4][PROF_THREADS / 64];
    const int k = blockIdx.x + 1;
    const long long pl = p.plane, base = (long long)k * pl;
    double t0 = st.get(4, k, base + (threadIdx.x & 63) * pl / 64);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) t0 += __shfl_xor(t0, off, 64);
    t0 /= 64.0;
    Sums a{};
#pragma unroll 4
    for (long long v = (long long)blockIdx.y * PROF_THREADS + threadIdx.x; v < pl; v += PROF_SEGS * PROF_THREADS) {
        const long long o = base + v;
        const double ro = st.get(3, k, o), tt = st.get(4, k, o);
        const double ri = 1.0 / ro;
        const double rw = st.get(2, k, o);
        const double uu = st.get(0, k, o) * ri, vv = st.get(1, k, o) * ri, ww = rw * ri;
        a.t.add(tt);
        a.r.add(ro);
        a.w.add(rw);
        a.f.add(-(rw * (2.5 * (tt - t0) + 0.5 * (uu * uu + vv * vv + ww * ww))));
    }
    a.t = block_sum(a.t, red[0]);
    a.r = block_sum(a.r, red[1]);
    a.w = block_sum(a.w, red[2]);
    a.f = block_sum(a.f, red[3]);
    if (threadIdx.x == 0 && blockIdx.y == 0) out[2 * p.npz + k - 1] = t0;
    if (threadIdx.x == 0) part[(long long)blockIdx.x * PROF_SEGS + blockIdx.y] = a;
}

// out: [3][npz] = TTM, ROM, FCONM of the planes k = 1..npz.
__global__ __launch_bounds__(64) void k_flux_profiles(const Params p, const Sums *__restrict__ part,
                                                      double *__restrict__ out) {
    const int k = blockIdx.x * 64 + threadIdx.x + 1;
    if (k > p.npz) return;
    const double cnt = (double)(float)(p.npx * p.npy);
    Sums a = part[(long long)(k - 1) * PROF_SEGS];
    for (int n = 1; n < PROF_SEGS; ++n) {
        const Sums x = part[(long long)(k - 1) * PROF_SEGS + n];
        a.t.add(x.t);
        a.r.add(x.r);
        a.w.add(x.w);
        a.f.add(x.f);
    }
    const double ttm = a.t.value() / cnt, t0 = out[2 * p.npz + k - 1];
    out[k - 1] = ttm;
    out[p.npz + k - 1] = a.r.value() / cnt;
    // RW (T - TTM) = RW (T - T0) - RW (TTM - T0), with what the division rounded off TTM
    const double d = 2.5 * ((ttm - t0) + (fma(-ttm, cnt, a.t.s) + a.t.c) / cnt), w = a.w.value();
    // (RW infinite: the flux about any T is; the correction would make it a NaN)
    if (isfinite(w) || !isfinite(d)) {
        const double x = d * w;
        a.f.add(x);
        a.f.c += fma(d, w, -x);
    }
    out[2 * p.npz + k - 1] = a.f.value() / cnt;
}

template <class S>
static hipError_t profiles(const Params &p, const S &st, double *out, hipStream_t s) {
    static_assert(sizeof(Sums) == 8 * sizeof(double), "prof_len");
    Sums *const part = reinterpret_cast<Sums *>(out + 3 * (size_t)p.npz);
    hipLaunchKernelGGL(k_flux_sums<S>, dim3(p.npz, PROF_SEGS), dim3(PROF_THREADS), 0, s, p, st, part, out);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_flux_profiles, dim3((p.npz + 63) / 64), dim3(64), 0, s, p, part, out);
    return hipGetLastError();
}

hipError_t launch_flux_profiles(const Params &p, const double *q, double *out, hipStream_t s) {
    return profiles(p, StateFp64{q, p.fsize}, out, s);
}

hipError_t launch_flux_profiles_mixed(const Params &p, const float *h, const unsigned *rr, const Background &bg,
                                      double *out, hipStream_t s) {
    return profiles(p, StateMixed{h, rr, bg, p.fsize}, out, s);
}

}  // namespace rmhd
