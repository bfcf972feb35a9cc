// Device helpers shared by the FP64 and the mixed-precision kernels.
#pragma once

#include "mhd_kernels.h"

namespace rmhd {

__device__ __forceinline__ int wrapi(int x, int n) {
    int r = x % n;
    return r < 0 ? r + n : r;
}

// The same without a division where x lies in [-n, 2n); further right it is
// some column of the box (lanes of a tile past the box's right neighbour,
// whose values nothing uses).
__device__ __forceinline__ int wrapc(int x, int n) {
    return x < 0 ? x + n : x < n ? x : x < 2 * n ? x - n : n - 1;
}

// XCD-aware block order.  The hardware deals consecutive workgroup ids to
// the 8 XCDs in turn; remap so that each XCD receives a contiguous run of
// tiles (tiles that share halo rows then share an L2).  A bijection for any
// grid size.
__device__ __forceinline__ int xcd_remap(int bid, int nb) {
    const int x = bid & 7, local = bid >> 3;
    const int q = nb >> 3, r = nb & 7;
    return x * q + (x < r ? x : r) + local;
}
// Tile and z chunk of workgroup bid of a stage launch over ntiles tiles and
// nch chunks.  Where the tiles divide by the 8 XCDs, each XCD gets a
// contiguous run of tiles in every chunk, chunk after chunk: tiles that share
// halo rows share an L2, and the chunks with the boundary planes, which do
// more work, are spread over all XCDs (as one contiguous run over all chunks,
// the two boundary chunks of 512x512x256 fell to two XCDs: FP64 stage 2 took
// 3.67 ms).  Other counts take the contiguous run.
struct TileChunk {
    int tile, chunk;
};
__device__ __forceinline__ TileChunk tile_of(int bid, int ntiles, int nch) {
    if (ntiles % 8 == 0) {
        const int per = ntiles / 8, local = bid >> 3;
        const int c = local / per;
        return TileChunk{(bid & 7) * per + local - c * per, c};
    }
    const int id = xcd_remap(bid, ntiles * nch);
    return TileChunk{id % ntiles, id / ntiles};
}

// Entry i of a read-only per-plane table (grid metrics, background
// profiles) at a workgroup-uniform index: read through the constant
// address space, so the compiler issues a scalar load.  A vector load here
// would share the in-order vector-memory counter with the plane prefetch
// and the wait for it would also wait for every load issued before it.
// The tables are written only between kernels (host copies, or earlier
// kernels on the stream, such as the plane means of the optional branches).
template <class T>
__device__ __forceinline__ T uload(const T *p, int i) {
    return ((const __attribute__((address_space(4))) T *)p)[i];
}


// x, held back until y has been computed: an empty asm that reads y and
// may change x, so that nothing derived from x is scheduled before y.  Used
// to keep the first use of a loaded value (and so the wait for the load,
// which also waits for every load issued before it) late in a plane.
template <class X, class Y>
__device__ __forceinline__ X after(X x, Y y) {
    asm volatile("" : "+v"(x) : "v"(y));
    return x;
}

// x is needed here: an empty asm that reads x, so the wait for the load of
// x happens at this point (once, before a loop) rather than at its first use
// inside the loop, where it would be repeated on every iteration.
template <class X>
__device__ __forceinline__ void settle(X x) {
    asm volatile("" ::"v"(x));
}

// A box's arguments for the code after a march (boundary conditions, CFL
// reduction), read anew from memory: the empty asm hides where the pointer
// comes from, so that the values are not loaded before the march and held in
// scalar registers through it (which spilled 50-60 more of them).
typedef const __attribute__((address_space(4))) BoxArgs *ArgPtr;
__device__ __forceinline__ const BoxArgs &late_args(ArgPtr a) {
    asm volatile("" : "+s"(a));
    return *(const BoxArgs *)a;
}
// Entry b of the ensemble's box table, read through the constant address
// space (it is written by host copies between launches only): its members
// arrive by scalar loads also after the stores of an earlier work item.
__device__ __forceinline__ const BoxDev &box_at(const BoxDev *boxes, int b) {
    return *(const BoxDev *)((const __attribute__((address_space(4))) BoxDev *)boxes + b);
}
// The kernel's first argument in the kernel-argument segment.
__device__ __forceinline__ ArgPtr kernel_args() { return (ArgPtr)__builtin_amdgcn_kernarg_segment_ptr(); }

// Value of key slot n between reductions (the neutral element of its min).
__host__ __device__ inline unsigned long long cfl_key_init(int n) { return n == 0 ? ~dkey(0.0) : dkey(INFINITY); }

__device__ __forceinline__ void cfl_arm(CflSlots *cs, int lane) {
    const int n = lane / CFL_REP, r = lane % CFL_REP;
    unsigned long long *const w = n < CFL_KEYS ? &cs->key[n][r].v : n == CFL_KEYS ? &cs->count[r].v : &cs->done.v;
    if (lane <= (CFL_KEYS + 1) * CFL_REP)
        __hip_atomic_store(w, n < CFL_KEYS ? cfl_key_init(n) : 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// End of a reduction: DT = SF*MIN(...), UMACH = SQRT(MAX(...)) (sub:761,
// 868-872).  A positive fixed_dt replaces the CFL DT.  With clock set this
// also closes the step that just ran: NIT, TIMC, TIMT (sub:1171-1173) with
// the DT it used, which is kept as dt_used / umach_used.
__device__ __forceinline__ void cfl_final(DevScalars *sc, const unsigned long long *k, double sf, int lmag, int clock,
                                          DevScalars *report) {
    DevScalars s = *sc;
    if (clock) {
        s.nit = s.nit + 1;
        s.timc = s.timc + s.dt;
        s.timt = s.timi + s.timc;
        s.dt_used = s.dt;
        s.umach_used = s.umach;
    }
    const double mach = dunkey(~k[0]);
    double mn = INFINITY;
    bool bad = !(mach == mach);
    for (int n = 0; n < 4; ++n) {
        const double w = dunkey(k[n + 1]);
        s.cflmin[n] = w;
        if (n < 3 || lmag) {
            mn = fmin(mn, w);
            bad = bad || !(w == w);
        }
    }
    s.umach = sqrt(mach);
    const double dcfl = sf * mn;
    s.dt = s.fixed_dt > 0.0 ? s.fixed_dt : dcfl;
    if (bad || dcfl == INFINITY) s.nonfinite |= 1;
    *sc = s;
    // for the host, which reads it once the stream is done: a copy less per call
    // (16x16x12 by single steps: 9 us of then 82; 67 now)
    if (report) *report = s;
}

// A workgroup's part of a CFL reduction, called by its first wavefront (all
// 64 lanes); k[0..4] of lane 0 are its keys (the complement of the Mach key,
// then the four limits).  Workgroup seq of total adds them to copy seq %
// CFL_REP of the slots and counts itself in; the last of the copy counts the
// copy in, and the last copy's workgroup combines the copies, re-arms the
// slots and closes the reduction, so that no launch of its own is needed
// (a one-thread launch takes 4.8 us in a step that may be 50 us long).
// Atomics and key reads are at device scope (coherent across the XCDs' L2s).
// The counter is raised after this wavefront's key updates have returned,
// so the last workgroup reads every key complete.  Until it is re-armed a
// key only falls: a workgroup whose value cannot move it skips the atomic,
// and a stale read there can only cost one that was not needed.
__device__ __forceinline__ void cfl_publish(const unsigned long long *k, DevScalars *sc, CflSlots *cs, double sf,
                                            int lmag, int clock, int seq, int total, DevScalars *report) {
    const int lane = threadIdx.x & 63, rep = seq % CFL_REP;
    unsigned long long v = 0;
#pragma unroll
    for (int n = 0; n < CFL_KEYS; ++n) {
        const unsigned long long x = __shfl(k[n], 0, 64);
        if (lane == n) v = x;
    }
    unsigned long long old = 0;
    if (lane < (lmag ? CFL_KEYS : CFL_KEYS - 1)) {
        unsigned long long *const w = &cs->key[lane][rep].v;
        // (a small launch has few atomics per line, and the read would only
        // lengthen its tail)
        if (total <= 512 || v < __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            old = __hip_atomic_fetch_min(w, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // the key updates have been performed: their results are here
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(old)::"memory");
    int last = 0;
    if (lane == 0) {
        const unsigned long long in_copy = (unsigned long long)((total - rep + CFL_REP - 1) / CFL_REP);
        const unsigned long long copies = total < CFL_REP ? total : CFL_REP;
        if (total <= 256)  // one counter: few enough to queue there, and one round trip less
            last = __hip_atomic_fetch_add(&cs->done.v, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 ==
                   (unsigned long long)total;
        else if (__hip_atomic_fetch_add(&cs->count[rep].v, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == in_copy)
            last = __hip_atomic_fetch_add(&cs->done.v, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == copies;
    }
    if (!__shfl(last, 0, 64)) return;
    asm volatile("" ::: "memory");
    unsigned long long x = ~0ull;
    if (lane < CFL_KEYS * CFL_REP)
        x = __hip_atomic_load(&cs->key[lane / CFL_REP][lane % CFL_REP].v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int off = CFL_REP / 2; off > 0; off >>= 1) {
        const unsigned long long y = __shfl_xor(x, off, 64);
        x = y < x ? y : x;
    }
    unsigned long long kk[CFL_KEYS];
#pragma unroll
    for (int n = 0; n < CFL_KEYS; ++n) kk[n] = __shfl(x, n * CFL_REP, 64);
    cfl_arm(cs, lane);
    if (lane == 0) cfl_final(sc, kk, sf, lmag, clock, report);
}

// Stored values of the mixed form (mhd_mixed.hip) as other kernels read them.

// 1/x of the FP32 perturbation arithmetic by the hardware reciprocal
// (v_rcp_f32, within 1 ulp) instead of the correctly rounded division
// sequence (about ten instructions).  The mixed form is judged by its error
// against the FP64 form, where one ulp of 1/rho is far below the FP32
// rounding of the stored values; every use (stencil, packing, unpacking,
// boundary planes) goes through this function, so they stay consistent.
__device__ __forceinline__ float rcp32(float x) { return __builtin_amdgcn_rcpf(x); }

// T' represented by a stored (rho', P') pair: (P' - T0 rho') / (rho0 + rho')
// in FP32.  Every kernel that needs T' of a stored pair calls this function
// (the stencil's ring included), so the value the residual compensates
// against is bit-identical to the value the right-hand side sees.
__device__ __forceinline__ float trep(float r0, float t0, float rh, float pp) {
    const float ri = rcp32(r0 + rh);
    return (pp - t0 * rh) * ri;
}

// BF16 bit patterns of the resting residual R: round to nearest even
// (v_cvt_pk_bf16_f32; NaN stays NaN), and back (exact).
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned short to_bf16(float x) { return __builtin_bit_cast(unsigned short, (__bf16)x); }
// Two residuals in one 32-bit word: lo in the low half, hi in the high half.
__device__ __forceinline__ unsigned pack_bf16x2(float lo, float hi) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2_t){lo, hi}, bf16x2_t));
}
__host__ __device__ __forceinline__ float from_bf16(unsigned short b) { return __uint_as_float((unsigned)b << 16); }

// R packs the BF16 residuals of two fields per 32-bit word: word
// (f/2)*fs + o holds field f in its low (f even) or high (f odd) half.
__device__ __forceinline__ float r_half(unsigned w, int f) {
    return from_bf16((unsigned short)((f & 1) ? (w >> 16) : (w & 0xffffu)));
}
__device__ __forceinline__ float r_get(const unsigned *__restrict__ rr, long long fs, int f, long long o) {
    return r_half(rr[(f >> 1) * fs + o], f);
}
__device__ __forceinline__ void r_put(unsigned *__restrict__ rr, long long fs, int f, long long o, float r) {
    unsigned *const w = &rr[(f >> 1) * fs + o];
    const unsigned b = to_bf16(r);
    *w = (f & 1) ? ((*w & 0x0000ffffu) | (b << 16)) : ((*w & 0xffff0000u) | b);
}

}  // namespace rmhd
