// Subgrid-closure network: three 3x3x3 convolutions cin -> width -> width
// -> cout with GELU after the first two, on BF16 MFMA with FP32
// accumulation (include/rast3dmhd_closure.h; no counterpart in the
// reference).  Training (forward, backward, Adam) and inference run on the
// device.
//
// Layout: activations channel-last, a[z][y][x][c] (BF16, c contiguous),
// periodic in x and y, zero padding in z.  Master parameters FP32 in the
// order W1[co][tap][ci], b1, W2, b2, W3, b3 with tap = 9(dz+1)+3(dy+1)+(dx+1).
//
// k_conv: implicit GEMM D[co][voxel] = sum_k W[co][k] A[voxel][k] with
//   k = tap*CIN + ci, on v_mfma_f32_16x16x32_bf16 (lane l holds
//   first[l%16][8(l/16)..+7], second[l%16][8(l/16)..+7],
//   D[4(l/16)..+3][l%16]).  A workgroup owns a 64 x 4 column
//   tile and marches down a z chunk with a ring of input planes (halo 1) in
//   LDS; a wavefront computes 16 columns x 4 rows (4 tiles).
//   - Weights stay in registers for the march; the only LDS is the input ring.
//     32 -> 32 channels: 8 wavefronts, each half of the output channels, so
//     that two share a SIMD and one's GELU (vector unit) runs beside the
//     other's products; within one wavefront the two add up.
//   - With 32 input channels a K block is one tap, so the fragment of an input
//     row serves the three output rows it touches: 54 reads per plane instead
//     of 108 (at 108 the LDS was as busy as the matrix cores).
//   - Output channels are the first operand, so that a lane ends with 4 or 8
//     consecutive channels of one voxel: one 8- or 16-byte store where the
//     other order needs as many of 2 bytes.
//   - Loads and stores are buffer accesses whose bounds check replaces the
//     branches at the volume's edges, and the epilogue of a plane runs in
//     pieces between the K blocks of the next.
//   What bounds it: the vector work of the GELU (22 instructions a value, two
//   of them at quarter rate) about as long as the products, and the LDS reads.
//   Measured at 128x128x64 (before): 8 -> 32 35 us (60), 32 -> 32 60 us (90),
//   32 -> 7 32 us (56); forward 127 us (204), 64x64x64 49 us (72).
//   The backward pass for the input reuses it with the flipped, transposed
//   kernel.
// k_dw: weight gradient dW[co][tap][ci] = sum_v G[v][co] X[v+off][ci] as
//   D[co][ci] over K = voxels, and the bias gradient sum_v G[v][co] beside it;
//   per-workgroup partials, reduced in a fixed order (deterministic) by
//   k_update, which in training also takes the Adam step and writes the BF16
//   weight panels.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <new>
#include <type_traits>
#include <vector>

#include "../../include/rast3dmhd_closure.h"
#include "mhd_kernels.h"

namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

constexpr int CTX = 64, CTY = 4;          // conv output tile per plane
constexpr int LW = CTX + 2, LH = CTY + 2; // LDS plane with halo
constexpr int DSEG = 64;                  // dW: voxels per segment (two K blocks)
constexpr int DS = DSEG + 8;              // dW: LDS row stride (odd number of 16-byte units)
constexpr int DRING = 6;                  // dW: ring slots of X rows (4 in use, 2 arriving)
constexpr int DBLK = 256;                 // dW: workgroups at most (one per CU)

// Shape of a convolution's workgroup.  32 -> 32 channels: 8 wavefronts, each
// half of the output channels, so that two share a SIMD (the weights of all 32
// are 216 registers a lane); 32 -> 8: three ring slots, so that two workgroups
// fit a CU's LDS.
template <int CIN, int NT>
struct ConvShape {
    static constexpr int HALVES = CIN == 32 && NT == 2 ? 2 : 1;
    static constexpr int NTW = NT / HALVES;  // 16-channel tiles of a wavefront
    static constexpr int THREADS = 256 * HALVES;
    static constexpr int SLOTS = CIN == 32 && NT == 1 ? 3 : 4;
    static constexpr int LDS = SLOTS * LW * LH * CIN * 2;  // bytes
};

// 16-byte unit of an LDS voxel that holds channel group u of column col.  The
// 16 lanes that the LDS serves together read one group of 16 consecutive
// columns, or two groups of 8 columns each, and so hit distinct banks.
template <int CIN>
__device__ __forceinline__ int unit_of(int u, int col) {
    return CIN == 32 ? u ^ ((0x78 >> (2 * ((col >> 2) & 3))) & 3) : u;
}

__device__ __forceinline__ int wrapn(int x, int n) {
    int r = x % n;
    return r < 0 ? r + n : r;
}

// erf by Abramowitz & Stegun, Handbook of Mathematical Functions, 7.1.26
// (absolute error below 1.5e-7, far under the BF16 rounding of the
// activations): branch-free, one hardware reciprocal and one exponential.
__device__ __forceinline__ float erf_as(float u) {
    const float s = fabsf(u);
    const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.3275911f, s, 1.0f));
    float q = __builtin_fmaf(1.061405429f, t, -1.453152027f);
    q = __builtin_fmaf(q, t, 1.421413741f);
    q = __builtin_fmaf(q, t, -0.284496736f);
    q = __builtin_fmaf(q, t, 0.254829592f);
    const float e = 1.0f - q * t * __expf(-s * s);
    return copysignf(e, u);
}
__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erf_as(x * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float x) {
    return 0.5f * (1.0f + erf_as(x * 0.70710678118654752f)) + x * __expf(-0.5f * x * x) * 0.39894228040143268f;
}

// EPI 0: out32 = acc + bias.  EPI 1: zout = acc + bias, out16 = gelu(zout).
// EPI 2: out16 = acc * gelu'(zprev).  EPI 3: out32 = acc.
// EPI 4: out16 = gelu(acc + bias) (inference: the pre-activation, which only
// the backward pass reads, is not stored).
// EPI 5: out32 = (acc + bias) * std + mean of channel and plane (the forcing of
// the closure-corrected step; nrm: mean[cout][nz], std[cout]), *finite cleared
// if one is not.  It saves a launch that read out32 back and wrote it again
// (128x128x64: 39 us; 34 without it, and 10 for that launch).
template <int CIN, int NT, int EPI>
__global__ __launch_bounds__((ConvShape<CIN, NT>::THREADS)) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_conv(const bf16 *__restrict__ x, const bf16 *__restrict__ wt, int kp,
                                              const float *__restrict__ bias, const float *__restrict__ zprev,
                                              bf16 *__restrict__ out16, float *__restrict__ out32,
                                              float *__restrict__ zout, int cout, int ostride, int nx, int ny,
                                              int nz, int kchunk, const float *__restrict__ nrm,
                                              int *__restrict__ finite) {
    using S = ConvShape<CIN, NT>;
    constexpr int PLANE = LW * LH * CIN;
    constexpr int NCH = CIN / 8, NTHR = S::THREADS, NTW = S::NTW;
    constexpr int NLOAD = (LW * LH * NCH + NTHR - 1) / NTHR;
    constexpr int KTOT = 27 * CIN, KB = (KTOT + 31) / 32;
    constexpr bool BIAS = EPI == 0 || EPI == 1 || EPI == 4 || EPI == 5;
    constexpr int NCL = 4 * NTW;  // channels of a lane, consecutive
    extern __shared__ uint4 lds_raw[];
    bf16 *const lds = reinterpret_cast<bf16 *>(lds_raw);

    const int t = threadIdx.x, lane = t & 63, wv = (t >> 6) & 3, half = t >> 8, lr = lane & 15, lg = lane >> 4;
    const int ntx = (nx + CTX - 1) / CTX, nty = (ny + CTY - 1) / CTY;
    const int bid = blockIdx.x;
    const int tz = bid / (ntx * nty);
    const int rem = bid - tz * (ntx * nty);
    const int x0 = (rem % ntx) * CTX, y0 = (rem / ntx) * CTY;
    const int zb = tz * kchunk, ze = min(nz, zb + kchunk);
    if (zb >= nz) return;

    constexpr unsigned NREC = 0xfffffff0u, OUT = 0xffffffffu;  // bytes of a buffer, an offset past them
    // this thread's 16-byte pieces of an input plane with halo: byte offsets in
    // a plane of x (OUT: no piece) and offsets in an LDS plane, computed once
    unsigned goff[NLOAD];
    int loff[NLOAD];
#pragma unroll
    for (int i = 0; i < NLOAD; ++i) {
        const int c = t + NTHR * i;
        goff[i] = OUT;
        loff[i] = 0;
        if (c < LW * LH * NCH) {
            const int vox = c / NCH, part = c - vox * NCH;
            const int row = vox / LW, col = vox - row * LW;
            const int gy = wrapn(y0 + row - 1, ny), gx = wrapn(x0 + col - 1, nx);
            goff[i] = ((unsigned)(gy * nx + gx) * CIN + part * 8) * (unsigned)sizeof(bf16);
            loff[i] = vox * CIN + unit_of<CIN>(part, col) * 8;
        }
    }
    const long long pstride = (long long)nx * ny * CIN;
    typedef u32x4 Piece[NLOAD];
    auto fetch = [&](int zz, Piece &pre) __attribute__((always_inline)) {
        // a plane outside the volume, like a lane without a piece, reads past
        // the buffer's end: zeros
        const bool in = zz >= 0 && zz < nz;
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16 *>(x + (in ? zz : 0) * pstride), 0,
                                                          in ? NREC : 0u, 0x00020000);
#pragma unroll
        for (int i = 0; i < NLOAD; ++i)
            pre[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, goff[i], 0, 0);
    };
    auto store = [&](int sl, const Piece &pre) __attribute__((always_inline)) {
        bf16 *pl = lds + sl * PLANE;
#pragma unroll
        for (int i = 0; i < NLOAD; ++i)  // (only the last piece is missing in some lanes)
            if (i + 1 < NLOAD || goff[i] != OUT) *reinterpret_cast<u32x4 *>(pl + loff[i]) = pre[i];
    };
    // planes zb-1, zb, zb+1 into slots 0, 1, 2, their loads issued together (the
    // first plane of the march waits for one memory latency, not for three)
    {
        Piece first[3];
#pragma unroll
        for (int n = 0; n < 3; ++n) fetch(zb - 1 + n, first[n]);
#pragma unroll
        for (int n = 0; n < 3; ++n) store(n, first[n]);
    }
    // the layer's weights of this lane, held in registers for the whole march.
    // Row m of tile nt is channel 8 (m/4) + 4 nt + m%4 with two tiles, m (plus 16
    // in the second half) with one.
    bf16x8 wb[KB][NTW];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) {
            const int row = NTW == 2 ? 8 * (lr >> 2) + 4 * nt + (lr & 3) : 16 * half + lr;
            wb[kb][nt] = *reinterpret_cast<const bf16x8 *>(wt + (long long)row * kp + kb * 32 + lg * 8);
        }
    const int co0 = 16 * half + NCL * lg;  // this lane's channels co0 .. co0 + NCL - 1
    float bco[NCL];
#pragma unroll
    for (int c = 0; c < NCL; ++c) bco[c] = BIAS && co0 + c < cout ? bias[co0 + c] : 0.f;
    // EPI 5: std and the means of the planes held in prv and acc
    float sd[NCL], mprv[NCL], macc[NCL];
    bool bad = false;
    auto means = [&](int z, float *m) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < NCL; ++c) m[c] = co0 + c < cout ? nrm[(co0 + c) * nz + z] : 0.f;
    };
    if (EPI == 5)
#pragma unroll
        for (int c = 0; c < NCL; ++c) sd[c] = co0 + c < cout ? nrm[cout * nz + co0 + c] : 0.f;
    const int gx = x0 + 16 * wv + lr;
    const bool vx = gx < nx && co0 < ostride;
    // this lane's column in an LDS row for dx = 0, 1, 2 (CIN = 32: its channels)
    int vcol[3];
#pragma unroll
    for (int dx = 0; dx < 3; ++dx) {
        const int col = 16 * wv + lr + dx;
        vcol[dx] = CIN == 32 ? col * CIN + unit_of<CIN>(lg, col) * 8 : col * CIN;
    }
    // CIN = 8: a K block holds four taps, one per lane group; the lane's offset
    // of each block within a plane and its plane
    int toff[CIN == 8 ? KB : 1], tdz[CIN == 8 ? KB : 1];
    if (CIN == 8) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            const int tap = min(4 * kb + lg, 26);  // (there is no tap 27: zero)
            tdz[kb] = tap / 9;
            toff[kb] = ((tap / 3) % 3 * LW + tap % 3) * CIN;
        }
    }

    f32x4 acc[CTY][NTW], prv[CTY][NTW];
    // Pieces of the epilogue of the plane held in prv: piece e < 4 NT CTY is one
    // channel of row e / (4 NT); a row's last piece stores it.  Lanes and
    // rows outside the volume access past the buffer's end, which the hardware
    // drops: no branch splits the code that the products are mixed with.
    constexpr int NPIECE = NCL * CTY;
    auto row_of = [&](const void *base, int size, int zp, int gy) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc(
            const_cast<char *>(static_cast<const char *>(base)) + ((((long long)zp * ny + gy) * nx + x0) * ostride) * size, 0, NREC,
            0x00020000);
    };
    const unsigned eo = (unsigned)((gx - x0) * ostride + co0);  // element offset of this lane in the tile's row
    bf16 o16[NCL];
    float o32[NCL], zrow[NCL];
    auto piece = [&](int e, int zp) __attribute__((always_inline)) {
        const int row = e / NCL, c = e % NCL;
        const int gy = y0 + row;
        const unsigned o2 = vx && gy < ny ? eo * 2 : OUT, o4 = vx && gy < ny ? eo * 4 : OUT;
        if (EPI == 2 && c == 0) {
            const auto rs = row_of(zprev, 4, zp, gy);
#pragma unroll
            for (int n = 0; n < NCL; n += 4) {
                const f32x4 z4 = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, o4, 4 * n, 0));
#pragma unroll
                for (int r = 0; r < 4; ++r) zrow[n + r] = z4[r];
            }
        }
        const float v = prv[row][c / 4][c % 4];
        if (EPI == 2) {
            o16[c] = (bf16)(v * gelu_grad(zrow[c]));
        } else {
            o32[c] = v + bco[c];
            if (EPI == 1 || EPI == 4) o16[c] = (bf16)gelu(o32[c]);
            if (EPI == 5) {
                o32[c] = o32[c] * sd[c] + mprv[c];
                bad = bad || (vx && gy < ny && co0 + c < cout && !(o32[c] - o32[c] == 0.0f));
            }
        }
        if (c == NCL - 1) {
            if (EPI == 0 || EPI == 1 || EPI == 3 || EPI == 5) {
                const auto rs = row_of(EPI == 1 ? zout : out32, 4, zp, gy);
#pragma unroll
                for (int n = 0; n < NCL; n += 4)
                    __builtin_amdgcn_raw_buffer_store_b128(
                        __builtin_bit_cast(u32x4, (f32x4){o32[n], o32[n + 1], o32[n + 2], o32[n + 3]}), rs, o4, 4 * n, 0);
            }
            if (EPI == 1 || EPI == 2 || EPI == 4) {
                typedef __bf16 out_t __attribute__((ext_vector_type(NCL)));
                out_t w;
#pragma unroll
                for (int n = 0; n < NCL; ++n) w[n] = o16[n];
                const auto rs = row_of(out16, 2, zp, gy);
                if constexpr (NCL == 8)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, w), rs, o2, 0, 0);
                else
                    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, w), rs, o2, 0, 0);
            }
        }
    };

    // plane z + 2 enters the fourth slot while plane z is computed (with three:
    // the slot of plane z - 1 after it)
    __syncthreads();
    int s0 = 0, s1 = 1, s2 = 2, s3 = S::SLOTS == 4 ? 3 : 0;  // slots of planes z-1 .. z+2
    auto plane = [&](int z, auto late_) __attribute__((always_inline)) {
        constexpr bool late = decltype(late_)::value;  // the plane before waits in prv
        const bool more = z + 1 < ze;
        Piece next;
        if (EPI == 5) means(z, macc);
        if (more) fetch(z + 2, next);
#pragma unroll
        for (int row = 0; row < CTY; ++row)
#pragma unroll
            for (int nt = 0; nt < NTW; ++nt) acc[row][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
        // K loop, software-pipelined: the LDS reads of the next unit are issued
        // before the products of this one, which cover their latency (one
        // wavefront per SIMD: nothing else would)
        if constexpr (CIN == 32) {
            // unit u: input row u % 6 of plane u / 6, three fragments (dx)
            bf16x8 fa[2][3];
            auto frag = [&](int u, bf16x8 *a) __attribute__((always_inline)) {
                const int dz = u / 6, yin = u % 6;
                const bf16 *pl = lds + (dz == 0 ? s0 : dz == 1 ? s1 : s2) * PLANE;
#pragma unroll
                for (int dx = 0; dx < 3; ++dx)
                    a[dx] = *reinterpret_cast<const bf16x8 *>(pl + yin * LW * CIN + vcol[dx]);
            };
            frag(0, fa[0]);
#pragma unroll
            for (int u = 0; u < 18; ++u) {
                const int c = u & 1, dz = u / 6, yin = u % 6;
                if (u + 1 < 18) frag(u + 1, fa[c ^ 1]);
                if (late && u < NPIECE) piece(u, z - 1);
#pragma unroll
                for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                    for (int row = 0; row < CTY; ++row) {
                        const int dy = yin - row;
                        if (dy < 0 || dy > 2) continue;
#pragma unroll
                        for (int nt = 0; nt < NTW; ++nt)
                            acc[row][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[dz * 9 + dy * 3 + dx][nt], fa[c][dx],
                                                                                   acc[row][nt], 0, 0, 0);
                    }
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            // unit u: K block u, the fragments of the four output rows
            bf16x8 fa[2][CTY];
            auto frag = [&](int u, bf16x8 *a) __attribute__((always_inline)) {
                const int p0 = s0, p1 = s1, p2 = s2;
                const int sl = tdz[u] == 0 ? p0 : tdz[u] == 1 ? p1 : p2;
                const bf16 *pl = lds + sl * PLANE + toff[u] + vcol[0];
#pragma unroll
                for (int row = 0; row < CTY; ++row) {
                    a[row] = *reinterpret_cast<const bf16x8 *>(pl + row * LW * CIN);
                    if (u == KB - 1 && lg == 3) a[row] = bf16x8{};  // (no tap 27)
                }
            };
            frag(0, fa[0]);
#pragma unroll
            for (int u = 0; u < KB; ++u) {
                const int c = u & 1;
                if (u + 1 < KB) frag(u + 1, fa[c ^ 1]);
                constexpr int PER = (NPIECE + KB - 1) / KB;
#pragma unroll
                for (int e = 0; e < PER; ++e)
                    if (late && u * PER + e < NPIECE) piece(u * PER + e, z - 1);
#pragma unroll
                for (int row = 0; row < CTY; ++row)
#pragma unroll
                    for (int nt = 0; nt < NTW; ++nt)
                        acc[row][nt] =
                            __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[u][nt], fa[c][row], acc[row][nt], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int row = 0; row < CTY; ++row)
#pragma unroll
            for (int nt = 0; nt < NTW; ++nt) prv[row][nt] = acc[row][nt];
        if (EPI == 5)
#pragma unroll
            for (int c = 0; c < NCL; ++c) mprv[c] = macc[c];
        if (S::SLOTS == 3) __syncthreads();  // plane z - 1 is done with
        if (more) store(s3, next);
        __syncthreads();
        const int s = s0;
        s0 = s1;
        s1 = s2;
        s2 = s3;
        s3 = S::SLOTS == 4 ? s : s0;
    };
    plane(zb, std::false_type{});
#pragma unroll 1
    for (int z = zb + 1; z < ze; ++z) plane(z, std::true_type{});
#pragma unroll
    for (int e = 0; e < NPIECE; ++e) piece(e, ze - 1);
    if (EPI == 5 && bad) *finite = 0;
}

// Weight gradient partials.  The operands want 8 consecutive voxels of one
// channel per lane, so rows of 64 voxels are kept transposed in LDS,
// [channel][voxel].  A workgroup marches along y over pairs of rows of one
// (z, x segment): a ring holds the X rows of the planes z-1, z, z+1, so each
// row is transposed once per plane that uses it instead of once per tap row.
// The x offset goes to G, kept in three shifted copies, which leaves every
// fragment an aligned 16-byte read shared by three taps.  Wavefront (dz, half
// h of the 16-channel tiles, K block kb) accumulates the 9 taps of its dz for
// its half; the two K blocks are added through LDS at the end.  The rows of
// the next pair are loaded while this one is computed.
// What bounds it: the latency of those loads (one workgroup per CU); 64x64x64,
// 32 x 32 channels 33 us against 97 with rows transposed per segment for every
// tap and 2-byte LDS accesses; partials of 256 workgroups instead of 512.
template <int CI, int CO>  // padded to multiples of 16
constexpr int dw_lds_bytes() {
    return (DRING * 3 * CI + 2 * 2 * 3 * CO) * DS * 2;
}

template <int CI, int CO>
__global__ __launch_bounds__(768, 3) void k_dw(const bf16 *__restrict__ x, int cis, const bf16 *__restrict__ g, int cos_,
                                               int co_real, int nx, int ny, int nz, float *__restrict__ partial,
                                               float *__restrict__ partial_b) {
    constexpr int MT = CO / 16, NT = CI / 16;
    constexpr int M = NT == 2 ? MT : 1;  // tiles of a wavefront
    static_assert(MT * NT == 2 * M, "two halves");
    extern __shared__ uint4 lds_raw[];
    bf16 *const tx = reinterpret_cast<bf16 *>(lds_raw);  // [slot][dz][ci][DS]
    bf16 *const tg = tx + DRING * 3 * CI * DS;           // [buffer][row][dx][co][DS]
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, lr = lane & 15, lg = lane >> 4;
    const int dz = w % 3, h = (w / 3) % 2, kb = w / 6;
    const int nseg = (nx + DSEG - 1) / DSEG, npair = (ny + 1) / 2;
    const long long total = (long long)nz * nseg * npair;
    const long long p0 = total * blockIdx.x / gridDim.x, p1 = total * (blockIdx.x + 1) / gridDim.x;
    // padding channels stay zero
    for (int e = t; e < dw_lds_bytes<CI, CO>() / 16; e += 768) lds_raw[e] = make_uint4(0, 0, 0, 0);

    f32x4 acc[9][M];
#pragma unroll
    for (int s = 0; s < 9; ++s)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[s][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    float db[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    // X task e: row, dz, voxel pair, channel group (fastest); G task: row, pair, group
    const int nc = cis / 8, ng = cos_ / 8;
    struct XPiece { uint4 v[2]; };
    struct GPiece { uint4 v[4]; };
    auto load_x = [&](int e, int z, int sx0, int row0) __attribute__((always_inline)) {
        const int c8 = e % nc, pr = e / nc % 32, d = e / (32 * nc) % 3, row = row0 + e / (96 * nc);
        const int zz = z + d - 1, yy = wrapn(row, ny);
        XPiece q;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const int xx = sx0 + 2 * pr + n;
            q.v[n] = make_uint4(0, 0, 0, 0);
            if (zz >= 0 && zz < nz && xx < nx)
                q.v[n] = *reinterpret_cast<const uint4 *>(x + (((long long)zz * ny + yy) * nx + xx) * cis + c8 * 8);
        }
        return q;
    };
    // two voxels of 8 channels -> 8 words of (first, second) of one channel each
    auto put_pair = [&](bf16 *row, int c8, int pr, const uint4 &a, const uint4 &b) __attribute__((always_inline)) {
        const unsigned av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            unsigned *const lo = reinterpret_cast<unsigned *>(row + (c8 * 8 + 2 * q) * DS + 2 * pr);
            unsigned *const hi = reinterpret_cast<unsigned *>(row + (c8 * 8 + 2 * q + 1) * DS + 2 * pr);
            *lo = __builtin_amdgcn_perm(bv[q], av[q], 0x05040100);
            *hi = __builtin_amdgcn_perm(bv[q], av[q], 0x07060302);
        }
    };
    auto slot = [](int row) { return (row + 1) % DRING; };  // row >= -1
    auto store_x = [&](int e, int row0, const XPiece &q) __attribute__((always_inline)) {
        const int c8 = e % nc, pr = e / nc % 32, d = e / (32 * nc) % 3, row = row0 + e / (96 * nc);
        put_pair(tx + (slot(row) * 3 + d) * CI * DS, c8, pr, q.v[0], q.v[1]);
    };
    const int gtasks = 2 * 32 * ng;
    auto load_g = [&](int z, int sx0, int row0) __attribute__((always_inline)) {
        GPiece q{};
        if (t < gtasks) {
            const int c8 = t % ng, pr = t / ng % 32, yy = wrapn(row0 + t / (32 * ng), ny);
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                const int xx = wrapn(sx0 + 2 * pr - 1 + n, nx);
                q.v[n] = *reinterpret_cast<const uint4 *>(g + (((long long)z * ny + yy) * nx + xx) * cos_ + c8 * 8);
            }
        }
        return q;
    };
    auto store_g = [&](int sx0, int row0, int buf, const GPiece &q) __attribute__((always_inline)) {
        if (t < gtasks) {
            const int c8 = t % ng, pr = t / ng % 32, r = t / (32 * ng);
            bf16 *const row = tg + (buf * 2 + r) * 3 * CO * DS;
            // (zero where X is past the row's end: 0 times an infinite G is a NaN)
            const uint4 none = make_uint4(0, 0, 0, 0);
            const bool in0 = sx0 + 2 * pr < nx, in1 = sx0 + 2 * pr + 1 < nx;
#pragma unroll
            for (int dx = 0; dx < 3; ++dx)
                put_pair(row + dx * CO * DS, c8, pr, in0 ? q.v[2 - dx] : none, in1 ? q.v[3 - dx] : none);
            if (row0 + r < ny) {
#pragma unroll
                for (int n = 0; n < 2; ++n)
                    if (sx0 + 2 * pr + n < nx) {
                        const bf16x8 v = __builtin_bit_cast(bf16x8, q.v[1 + n]);
#pragma unroll
                        for (int c = 0; c < 8; ++c) db[c] += (float)v[c];
                    }
            }
        }
    };

    for (long long p = p0; p < p1;) {
        const long long zs = p / npair;
        int j = (int)(p - zs * npair);
        const int z = (int)(zs / nseg), sx0 = (int)(zs % nseg) * DSEG;
        const int jend = (int)min((long long)npair, j + (p1 - p));
        p += jend - j;
        __syncthreads();  // the last run's fragments are read
        for (int e = t; e < 4 * 96 * nc; e += 768) store_x(e, 2 * j - 1, load_x(e, z, sx0, 2 * j - 1));
        store_g(sx0, 2 * j, 0, load_g(z, sx0, 2 * j));
        __syncthreads();
        for (int buf = 0; j < jend; ++j, buf ^= 1) {
            const bool more = j + 1 < jend;
            XPiece xn{};
            GPiece gn{};
            if (more) {
                if (t < 2 * 96 * nc) xn = load_x(t, z, sx0, 2 * j + 3);
                gn = load_g(z, sx0, 2 * j + 2);
            }
            const int k0 = kb * 32 + lg * 8;
            // X fragments of rows 2j-1 .. 2j+2 of plane z + dz - 1
            auto xfrag = [&](int row, int nt) __attribute__((always_inline)) {
                return *reinterpret_cast<const bf16x8 *>(tx + ((slot(row) * 3 + dz) * CI + 16 * nt + lr) * DS + k0);
            };
            bf16x8 xf[4];
#pragma unroll
            for (int n = 0; n < 4; ++n) xf[n] = xfrag(2 * j - 1 + n, NT == 2 ? h : 0);
#pragma unroll
            for (int r = 0; r < 2; ++r)
                if (2 * j + r < ny) {
#pragma unroll
                    for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                        for (int m = 0; m < M; ++m) {
                            const int mt = NT == 2 ? m : h;
                            const bf16x8 a = *reinterpret_cast<const bf16x8 *>(
                                tg + (((buf * 2 + r) * 3 + dx) * CO + 16 * mt + lr) * DS + k0);
#pragma unroll
                            for (int dy = 0; dy < 3; ++dy)
                                acc[3 * dy + dx][m] =
                                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, xf[r + dy], acc[3 * dy + dx][m], 0, 0, 0);
                        }
                }
            if (more) {
                if (t < 2 * 96 * nc) store_x(t, 2 * j + 3, xn);
                store_g(sx0, 2 * j + 2, buf ^ 1, gn);
            }
            __syncthreads();
        }
    }

    // add the two K blocks: those of kb = 1 pass theirs through LDS
    f32x4 *const comb = reinterpret_cast<f32x4 *>(lds_raw);
    static_assert(6 * 9 * M * 64 * 16 <= dw_lds_bytes<CI, CO>(), "the combined sums fit");
    if (kb == 1)
#pragma unroll
        for (int s = 0; s < 9; ++s)
#pragma unroll
            for (int m = 0; m < M; ++m) comb[((w - 6) * 9 * M + s * M + m) * 64 + lane] = acc[s][m];
    __syncthreads();
    // partial[blk][tap][co][ci]
    if (kb == 0)
#pragma unroll
        for (int s = 0; s < 9; ++s)
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const f32x4 v = acc[s][m] + comb[(w * 9 * M + s * M + m) * 64 + lane];
                const int mt = NT == 2 ? m : h, nt = NT == 2 ? h : 0;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    partial[(((long long)blockIdx.x * 27 + 9 * dz + s) * CO + 16 * mt + 4 * lg + r) * CI + 16 * nt + lr] = v[r];
            }
    __syncthreads();
    // bias partials: the sums of the threads that staged a channel, in thread order
    float *const bred = reinterpret_cast<float *>(lds_raw);
    if (t < gtasks)
#pragma unroll
        for (int c = 0; c < 8; ++c) bred[t * 8 + c] = db[c];
    __syncthreads();
    if (t < co_real) {
        float v = 0.f;
        for (int e = t / 8; e < gtasks; e += ng) v += bred[e * 8 + t % 8];
        partial_b[(long long)blockIdx.x * 32 + t] = v;
    }
}

// One layer as k_update sees it.
struct LayerDev {
    long long woff, boff;                    // in the parameter vector
    int co, ci, co_pad, ci_pad, cis, cos_;   // channels, paddings of the partials, storage strides
    int kpf, kpb;
    const float *pw, *pb;                    // partials of k_dw
    bf16 *wf, *wb;                           // weight panels
};
struct UpdateArgs {
    LayerDev l[3];
};

// Gradient of every parameter as the sum of its nblk partials; with train
// also the Adam step and the parameter's entries of the BF16 panels (the
// padding of the panels was written by k_pack_w and stays).  A workgroup takes
// 32 consecutive parameters: its 8 thread groups sum the partials c, c+8, ...
// and the 8 sums are added in order (deterministic).  One launch in place of
// three reductions, three bias reductions, Adam and three packings (62 + 26 +
// 5 + 14 us of a 548 us iteration at 64x64x64; 13 us).
constexpr int UPD_OUT = 32, UPD_GRP = 8;
__global__ __launch_bounds__(UPD_OUT *UPD_GRP) void k_update(const UpdateArgs a, int nblk, long long nparam,
                                                            float *__restrict__ grad, int train, float *__restrict__ p,
                                                            float *__restrict__ am, float *__restrict__ av, float lr,
                                                            float b1, float b2, float eps, float c1, float c2) {
    __shared__ float red[UPD_GRP][UPD_OUT];
    const int j = threadIdx.x % UPD_OUT, c = threadIdx.x / UPD_OUT;
    const long long e = (long long)blockIdx.x * UPD_OUT + j;
    const LayerDev &L = e < a.l[1].woff ? a.l[0] : e < a.l[2].woff ? a.l[1] : a.l[2];
    const bool bias = e >= L.boff;
    const int ew = (int)(e - L.woff);
    const int co = bias ? (int)(e - L.boff) : ew / (27 * L.ci);
    const int rem = bias ? 0 : ew - co * 27 * L.ci, tap = rem / L.ci, ci = rem - tap * L.ci;
    float s = 0.f;
    if (e < nparam) {
        const float *src = bias ? L.pb + co : L.pw + ((long long)tap * L.co_pad + co) * L.ci_pad + ci;
        const long long step = bias ? 32 : 27LL * L.co_pad * L.ci_pad;
#pragma unroll 8
        for (int b = c; b < nblk; b += UPD_GRP) s += src[b * step];
    }
    red[c][j] = s;
    __syncthreads();
    if (c != 0 || e >= nparam) return;
    float gr = red[0][j];
    for (int q = 1; q < UPD_GRP; ++q) gr += red[q][j];
    grad[e] = gr;
    if (!train) return;
    const float mm = b1 * am[e] + (1.f - b1) * gr;
    const float vv = b2 * av[e] + (1.f - b2) * gr * gr;
    am[e] = mm;
    av[e] = vv;
    const float pn = p[e] - lr * (mm / c1) / (sqrtf(vv / c2) + eps);
    p[e] = pn;
    if (!bias) {
        L.wf[(long long)co * L.kpf + tap * L.cis + ci] = (bf16)pn;
        L.wb[(long long)ci * L.kpb + (26 - tap) * L.cos_ + co] = (bf16)pn;
    }
}

// BF16 weight panels of one layer from the FP32 master W[co][tap][ci]:
// forward wf[co_pad][kpf] at k = tap*ci_str + ci; backward (input
// gradient) wb[ci_pad][kpb] at k = tap'*co_str + co with tap' = 26 - tap.
__global__ void k_pack_w(const float *__restrict__ w, int co_real, int ci_real, int ci_str, int co_str,
                         bf16 *__restrict__ wf, int co_pad, int kpf, bf16 *__restrict__ wb, int ci_pad, int kpb) {
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long nf = (long long)co_pad * kpf, nb = (long long)ci_pad * kpb;
    if (e < nf) {
        const int co = (int)(e / kpf), k = (int)(e - (long long)co * kpf);
        const int tap = k / ci_str, ci = k - tap * ci_str;
        float v = 0.f;
        if (co < co_real && tap < 27 && ci < ci_real) v = w[((long long)co * 27 + tap) * ci_real + ci];
        wf[e] = (bf16)v;
    }
    if (e < nb) {
        const int ci = (int)(e / kpb), k = (int)(e - (long long)ci * kpb);
        const int tp = k / co_str, co = k - tp * co_str;
        float v = 0.f;
        if (ci < ci_real && tp < 27 && co < co_real) v = w[((long long)co * 27 + (26 - tp)) * ci_real + ci];
        wb[e] = (bf16)v;
    }
}

// MSE loss of y against t (first cout channels of stride 8) and its
// gradient g = 2 (y - t) / (n cout) as BF16 with stride 8 (channel >= cout
// zero); per-block partial sums of the squared error.
__global__ __launch_bounds__(256) void k_loss(const float *__restrict__ y, const float *__restrict__ tgt, int cout,
                                              long long nvox, float gscale, bf16 *__restrict__ g,
                                              double *__restrict__ partial) {
    __shared__ double red[256];
    double s = 0.0;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < nvox * 8;
         e += (long long)gridDim.x * blockDim.x) {
        const int c = (int)(e & 7);
        float d = 0.f;
        if (c < cout) {
            d = y[e] - tgt[e];
            s += (double)d * (double)d;
        }
        if (g) g[e] = (bf16)(gscale * d);
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ void k_f32_to_bf16(const float *__restrict__ a, bf16 *__restrict__ b, long long n, int cin, int cstr) {
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n * cstr) return;
    const long long v = e / cstr;
    const int c = (int)(e - v * cstr);
    b[e] = (bf16)(c < cin ? a[v * cin + c] : 0.f);
}

struct Sample {
    int nx, ny, nz;
    bf16 *x;   // [v][8]
    float *t;  // [v][8]
};

struct Layer {
    int ci, co;          // real channel counts
    int cis, cos_;       // storage strides of input / output activations (multiples of 8)
    int co_pad, ci_pad;  // MFMA paddings (multiples of 16)
    int kpf, kpb;
    long long woff, boff;  // offsets into the parameter vector
    bf16 *wf = nullptr, *wb = nullptr;
};

}  // namespace

struct mhd_net {
    int dev = 0;
    hipStream_t stream = nullptr;
    int cin = 0, width = 0, cout = 0;
    long long nparam = 0;
    Layer L[3];
    float *p = nullptr, *grad = nullptr, *am = nullptr, *av = nullptr;
    int adam_t = 0;
    // workspace for volumes up to cap voxels
    long long cap = 0;
    bf16 *a0 = nullptr, *a1 = nullptr, *a2 = nullptr, *g1 = nullptr, *g2 = nullptr, *g3 = nullptr;
    float *z1 = nullptr, *z2 = nullptr, *y = nullptr, *tmp32 = nullptr, *dx32 = nullptr;
    float *partial = nullptr;  // of the three layers: weights, then biases
    double *lpart = nullptr;
    std::vector<Sample> samples;
    char err[512] = {0};
};

static char g_net_err[512];

static int nfail(mhd_net_t *n, int code, const char *fmt, ...) {
    char *buf = n ? n->err : g_net_err;
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, 512, fmt, ap);
    va_end(ap);
    return code;
}

#define NHIP(n, x)                                                                         \
    do {                                                                                   \
        hipError_t r_ = (x);                                                               \
        if (r_ != hipSuccess)                                                              \
            return nfail((n), MHD_ERR_HIP, "%s: %s (%s:%d)", #x, hipGetErrorString(r_),    \
                         __FILE__, __LINE__);                                              \
    } while (0)

// z chunk per workgroup so that the grid has about `target` workgroups.
static int kchunk_for(int nx, int ny, int nz, int target, int *nblocks) {
    const int tiles = ((nx + CTX - 1) / CTX) * ((ny + CTY - 1) / CTY);
    int nc = (target + tiles - 1) / tiles;
    if (nc > nz) nc = nz;
    if (nc < 1) nc = 1;
    const int kc = (nz + nc - 1) / nc;
    *nblocks = tiles * ((nz + kc - 1) / kc);
    return kc;
}

template <int CIN, int NT, int EPI>
static hipError_t conv(hipStream_t s, const bf16 *x, const bf16 *w, int kp, const float *bias, const float *zprev,
                       bf16 *out16, float *out32, float *zout, int cout, int ostride, int nx, int ny, int nz,
                       const float *nrm = nullptr, int *finite = nullptr) {
    using S = ConvShape<CIN, NT>;
    constexpr int lds = S::LDS;
    if (kp != 32 * ((27 * CIN + 31) / 32)) return hipErrorInvalidValue;  // the kernel's K blocks
    if (NT == 2 ? cout != 32 || ostride != 32 : cout > 8 || ostride != 8) return hipErrorInvalidValue;
    static_assert(lds <= 160 * 1024, "the LDS of a CU");
    if ((long long)nx * ny * CIN > 0x7fffffffLL) return hipErrorInvalidValue;  // in-plane byte offsets are 32-bit
    static std::atomic<unsigned long long> attr{0};
    hipError_t e = rmhd::lds_limit_once(attr, reinterpret_cast<const void *>(&k_conv<CIN, NT, EPI>), lds);
    if (e != hipSuccess) return e;
    // as many workgroups as fit the CUs at once (LDS and registers): each
    // streams a longer z chunk, which amortises its prologue (three planes +
    // the weights); per device
    static std::atomic<int> resident[64];
    int dev = 0;
    if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    int res = resident[dev].load(std::memory_order_relaxed);
    if (!res) {
        int per_cu = 0, ncu = 0;
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(&k_conv<CIN, NT, EPI>),
                                                         S::THREADS, lds);
        if (e == hipSuccess) e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
        if (e != hipSuccess) return e;
        res = std::max(1, per_cu) * std::max(1, ncu);
        resident[dev].store(res, std::memory_order_relaxed);
    }
    int nb;
    const int kc = kchunk_for(nx, ny, nz, res, &nb);
    hipLaunchKernelGGL((k_conv<CIN, NT, EPI>), dim3(nb), dim3(S::THREADS), lds, s, x, w, kp, bias, zprev, out16, out32, zout,
                       cout, ostride, nx, ny, nz, kc, nrm, finite);
    return hipGetLastError();
}

// Buffers for a volume of nvox voxels.  Whoever uses them calls this first: an
// allocation that failed leaves none (cap 0), also for volumes that fitted.
static int ensure_workspace(mhd_net_t *n, long long nvox) {
    if (nvox <= n->cap) return MHD_OK;
    n->cap = 0;
    void **bufs[11] = {(void **)&n->a0, (void **)&n->a1, (void **)&n->a2, (void **)&n->g1, (void **)&n->g2,
                       (void **)&n->g3, (void **)&n->z1, (void **)&n->z2, (void **)&n->y, (void **)&n->tmp32,
                       (void **)&n->dx32};
    for (auto b : bufs)
        if (*b) {
            (void)hipFree(*b);
            *b = nullptr;
        }
    const size_t w = (size_t)n->width;
    NHIP(n, hipMalloc(&n->a0, nvox * 8 * sizeof(bf16)));
    NHIP(n, hipMalloc(&n->a1, nvox * w * sizeof(bf16)));
    NHIP(n, hipMalloc(&n->a2, nvox * w * sizeof(bf16)));
    NHIP(n, hipMalloc(&n->g1, nvox * w * sizeof(bf16)));
    NHIP(n, hipMalloc(&n->g2, nvox * w * sizeof(bf16)));
    NHIP(n, hipMalloc(&n->g3, nvox * 8 * sizeof(bf16)));
    NHIP(n, hipMalloc(&n->z1, nvox * w * sizeof(float)));
    NHIP(n, hipMalloc(&n->z2, nvox * w * sizeof(float)));
    NHIP(n, hipMalloc(&n->y, nvox * 8 * sizeof(float)));
    NHIP(n, hipMalloc(&n->tmp32, nvox * 8 * sizeof(float)));
    NHIP(n, hipMalloc(&n->dx32, nvox * 8 * sizeof(float)));
    n->cap = nvox;
    return MHD_OK;
}

static hipError_t pack_weights(mhd_net_t *n) {
    for (int l = 0; l < 3; ++l) {
        const Layer &L = n->L[l];
        const long long tot = std::max((long long)L.co_pad * L.kpf, (long long)L.ci_pad * L.kpb);
        hipLaunchKernelGGL(k_pack_w, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, n->stream, n->p + L.woff, L.co,
                           L.ci, L.cis, L.cos_, L.wf, L.co_pad, L.kpf, L.wb, L.ci_pad, L.kpb);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// forward of a BF16 input x (stride 8) into n->y (FP32, stride 8) on stream s;
// keep: also store the pre-activations z1, z2 the backward pass reads
static hipError_t forward_on(mhd_net_t *n, hipStream_t s, const bf16 *x, int nx, int ny, int nz, bool keep,
                             const float *nrm = nullptr, float *force = nullptr, int *force_on = nullptr) {
    const Layer *L = n->L;
    hipError_t e = keep ? conv<8, 2, 1>(s, x, L[0].wf, L[0].kpf, n->p + L[0].boff, nullptr, n->a1, nullptr, n->z1,
                                        L[0].co, L[0].cos_, nx, ny, nz)
                        : conv<8, 2, 4>(s, x, L[0].wf, L[0].kpf, n->p + L[0].boff, nullptr, n->a1, nullptr, nullptr,
                                        L[0].co, L[0].cos_, nx, ny, nz);
    if (e == hipSuccess)
        e = keep ? conv<32, 2, 1>(s, n->a1, L[1].wf, L[1].kpf, n->p + L[1].boff, nullptr, n->a2, nullptr, n->z2,
                                  L[1].co, L[1].cos_, nx, ny, nz)
                 : conv<32, 2, 4>(s, n->a1, L[1].wf, L[1].kpf, n->p + L[1].boff, nullptr, n->a2, nullptr, nullptr,
                                  L[1].co, L[1].cos_, nx, ny, nz);
    if (e == hipSuccess && force)
        return conv<32, 1, 5>(s, n->a2, L[2].wf, L[2].kpf, n->p + L[2].boff, nullptr, nullptr, force, nullptr, L[2].co, 8,
                              nx, ny, nz, nrm, force_on);
    if (e == hipSuccess)
        e = conv<32, 1, 0>(s, n->a2, L[2].wf, L[2].kpf, n->p + L[2].boff, nullptr, nullptr, n->y, nullptr, L[2].co, 8,
                           nx, ny, nz);
    return e;
}

// Workgroups of k_dw for a volume: a share of the row pairs each.
static int dw_blocks(int nx, int ny, int nz) {
    return (int)std::min<long long>(DBLK, (long long)nz * ((nx + DSEG - 1) / DSEG) * ((ny + 1) / 2));
}

// Partials of layer l in n->partial: DBLK blocks of weights, then of biases;
// l = 3: the length.
static size_t partial_offset(const mhd_net_t *n, int l) {
    size_t off = 0;
    for (int i = 0; i < l; ++i) off += (size_t)DBLK * (27 * n->L[i].co_pad * n->L[i].ci_pad + 32);
    return off;
}
static float *dw_weights(const mhd_net_t *n, int l) { return n->partial + partial_offset(n, l); }
static float *dw_biases(const mhd_net_t *n, int l) {
    return dw_weights(n, l) + (size_t)DBLK * 27 * n->L[l].co_pad * n->L[l].ci_pad;
}

template <int CI, int CO>
static hipError_t dw(mhd_net_t *n, const bf16 *x, int l, const bf16 *g, int nx, int ny, int nz) {
    const Layer &L = n->L[l];
    if (L.ci_pad != CI || L.co_pad != CO) return hipErrorInvalidValue;
    constexpr int lds = dw_lds_bytes<CI, CO>();
    static_assert(lds <= 160 * 1024, "the LDS of a CU");
    static std::atomic<unsigned long long> attr{0};
    hipError_t e = rmhd::lds_limit_once(attr, reinterpret_cast<const void *>(&k_dw<CI, CO>), lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_dw<CI, CO>), dim3(dw_blocks(nx, ny, nz)), dim3(768), lds, n->stream, x, L.cis, g, L.cos_, L.co,
                       nx, ny, nz, dw_weights(n, l), dw_biases(n, l));
    return hipGetLastError();
}

// backward from the input x and g3 (both BF16, stride 8): the layers' gradient
// partials; with want_dx the input gradient (FP32, stride 8) into dx32.
static hipError_t backward(mhd_net_t *n, const bf16 *x, int nx, int ny, int nz, bool want_dx) {
    const Layer *L = n->L;
    hipError_t e = dw<32, 16>(n, n->a2, 2, n->g3, nx, ny, nz);
    if (e == hipSuccess)
        e = conv<8, 2, 2>(n->stream, n->g3, L[2].wb, L[2].kpb, nullptr, n->z2, n->g2, nullptr, nullptr, L[2].ci,
                          L[2].cis, nx, ny, nz);
    if (e == hipSuccess) e = dw<32, 32>(n, n->a1, 1, n->g2, nx, ny, nz);
    if (e == hipSuccess)
        e = conv<32, 2, 2>(n->stream, n->g2, L[1].wb, L[1].kpb, nullptr, n->z1, n->g1, nullptr, nullptr, L[1].ci,
                           L[1].cis, nx, ny, nz);
    if (e == hipSuccess) e = dw<16, 32>(n, x, 0, n->g1, nx, ny, nz);
    if (e == hipSuccess && want_dx)
        e = conv<32, 1, 3>(n->stream, n->g1, L[0].wb, L[0].kpb, nullptr, nullptr, nullptr, n->dx32, nullptr, L[0].ci,
                           8, nx, ny, nz);
    return e;
}

// Gradients from the partials of backward() into n->grad; with train the Adam
// step number n->adam_t and the new weight panels.
static hipError_t update(mhd_net_t *n, int nx, int ny, int nz, bool train, float lr) {
    UpdateArgs a;
    for (int l = 0; l < 3; ++l) {
        const Layer &L = n->L[l];
        a.l[l] = LayerDev{L.woff, L.boff, L.co, L.ci, L.co_pad, L.ci_pad, L.cis, L.cos_, L.kpf, L.kpb,
                          dw_weights(n, l), dw_biases(n, l), L.wf, L.wb};
    }
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - powf(b1, (float)n->adam_t), c2 = 1.f - powf(b2, (float)n->adam_t);
    hipLaunchKernelGGL(k_update, dim3((unsigned)((n->nparam + UPD_OUT - 1) / UPD_OUT)), dim3(UPD_OUT * UPD_GRP), 0,
                       n->stream, a, dw_blocks(nx, ny, nz), n->nparam, n->grad, train ? 1 : 0, n->p, n->am, n->av, lr, b1,
                       b2, 1e-8f, c1, c2);
    return hipGetLastError();
}

static int upload_input(mhd_net_t *n, const float *x, long long nvox, bf16 *dst) {
    NHIP(n, hipMemcpyAsync(n->tmp32, x, nvox * n->cin * sizeof(float), hipMemcpyHostToDevice, n->stream));
    hipLaunchKernelGGL(k_f32_to_bf16, dim3((unsigned)((nvox * 8 + 255) / 256)), dim3(256), 0, n->stream, n->tmp32, dst,
                       nvox, n->cin, 8);
    NHIP(n, hipGetLastError());
    return MHD_OK;
}

static int check_dims(mhd_net_t *n, int nx, int ny, int nz, const char *who) {
    if (!n) return nfail(nullptr, MHD_ERR_ARG, "%s: null handle", who);
    if (nx < 1 || ny < 1 || nz < 1) return nfail(n, MHD_ERR_ARG, "%s: volume %dx%dx%d", who, nx, ny, nz);
    return MHD_OK;
}

extern "C" int mhd_net_create(int cin, int width, int cout, mhd_net_t **out) {
    if (!out) return nfail(nullptr, MHD_ERR_ARG, "mhd_net_create: null argument");
    *out = nullptr;
    if (cin != 8 || width != 32 || cout < 1 || cout > 8)
        return nfail(nullptr, MHD_ERR_SCOPE, "mhd_net_create: built for cin=8, width=32, cout<=8 (got %d, %d, %d)",
                     cin, width, cout);
    mhd_net_t *n = new (std::nothrow) mhd_net();
    if (!n) return nfail(nullptr, MHD_ERR_ARG, "mhd_net_create: out of host memory");
    n->cin = cin;
    n->width = width;
    n->cout = cout;
    const int ci[3] = {cin, width, width}, co[3] = {width, width, cout};
    const int cis[3] = {8, width, width}, cos_[3] = {width, width, 8};
    long long off = 0;
    for (int l = 0; l < 3; ++l) {
        Layer &L = n->L[l];
        L.ci = ci[l];
        L.co = co[l];
        L.cis = cis[l];
        L.cos_ = cos_[l];
        L.co_pad = (co[l] + 15) / 16 * 16;
        L.ci_pad = (ci[l] + 15) / 16 * 16;
        L.kpf = (27 * L.cis + 31) / 32 * 32;
        L.kpb = (27 * L.cos_ + 31) / 32 * 32;
        L.woff = off;
        off += (long long)L.co * 27 * L.ci;
        L.boff = off;
        off += L.co;
    }
    n->nparam = off;
    hipError_t e = hipGetDevice(&n->dev);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking);
    for (float **b : {&n->p, &n->grad, &n->am, &n->av})
        if (e == hipSuccess) e = hipMalloc(b, off * sizeof(float));
    for (int l = 0; l < 3 && e == hipSuccess; ++l) {
        Layer &L = n->L[l];
        e = hipMalloc(&L.wf, (size_t)L.co_pad * L.kpf * sizeof(bf16));
        if (e == hipSuccess) e = hipMalloc(&L.wb, (size_t)L.ci_pad * L.kpb * sizeof(bf16));
    }
    if (e == hipSuccess) e = hipMalloc(&n->partial, partial_offset(n, 3) * sizeof(float));
    if (e == hipSuccess) e = hipMalloc(&n->lpart, 1024 * sizeof(double));
    if (e == hipSuccess) e = hipMemset(n->p, 0, off * sizeof(float));
    if (e == hipSuccess) e = hipMemset(n->am, 0, off * sizeof(float));
    if (e == hipSuccess) e = hipMemset(n->av, 0, off * sizeof(float));
    if (e != hipSuccess) {
        const int rc = nfail(nullptr, MHD_ERR_HIP, "mhd_net_create: %s", hipGetErrorString(e));
        mhd_net_destroy(n);
        return rc;
    }
    *out = n;
    return MHD_OK;
}

extern "C" long long mhd_net_num_params(const mhd_net_t *n) { return n ? n->nparam : 0; }

extern "C" int mhd_net_set_params(mhd_net_t *n, const float *params) {
    if (!n || !params) return nfail(n, MHD_ERR_ARG, "mhd_net_set_params: null argument");
    NHIP(n, hipSetDevice(n->dev));
    NHIP(n, hipMemcpyAsync(n->p, params, n->nparam * sizeof(float), hipMemcpyHostToDevice, n->stream));
    NHIP(n, hipMemsetAsync(n->am, 0, n->nparam * sizeof(float), n->stream));
    NHIP(n, hipMemsetAsync(n->av, 0, n->nparam * sizeof(float), n->stream));
    n->adam_t = 0;
    NHIP(n, pack_weights(n));
    NHIP(n, hipStreamSynchronize(n->stream));
    return MHD_OK;
}

extern "C" int mhd_net_get_params(mhd_net_t *n, float *params) {
    if (!n || !params) return nfail(n, MHD_ERR_ARG, "mhd_net_get_params: null argument");
    NHIP(n, hipSetDevice(n->dev));
    NHIP(n, hipMemcpyAsync(params, n->p, n->nparam * sizeof(float), hipMemcpyDeviceToHost, n->stream));
    NHIP(n, hipStreamSynchronize(n->stream));
    return MHD_OK;
}

extern "C" int mhd_net_forward(mhd_net_t *n, int nx, int ny, int nz, const float *x, float *y) {
    int rc = check_dims(n, nx, ny, nz, "mhd_net_forward");
    if (rc) return rc;
    if (!x || !y) return nfail(n, MHD_ERR_ARG, "mhd_net_forward: null array");
    const long long nvox = (long long)nx * ny * nz;
    NHIP(n, hipSetDevice(n->dev));
    rc = ensure_workspace(n, nvox);
    if (rc) return rc;
    rc = upload_input(n, x, nvox, n->a0);
    if (rc) return rc;
    NHIP(n, forward_on(n, n->stream, n->a0, nx, ny, nz, false));
    // y (stride 8) -> host (stride cout)
    std::vector<float> tmp((size_t)nvox * 8);
    NHIP(n, hipMemcpyAsync(tmp.data(), n->y, nvox * 8 * sizeof(float), hipMemcpyDeviceToHost, n->stream));
    NHIP(n, hipStreamSynchronize(n->stream));
    for (long long v = 0; v < nvox; ++v)
        for (int c = 0; c < n->cout; ++c) y[v * n->cout + c] = tmp[(size_t)v * 8 + c];
    return MHD_OK;
}

extern "C" int mhd_net_gradient(mhd_net_t *n, int nx, int ny, int nz, const float *x, const float *dy,
                                float *dparams, float *dx) {
    int rc = check_dims(n, nx, ny, nz, "mhd_net_gradient");
    if (rc) return rc;
    if (!x || !dy || !dparams) return nfail(n, MHD_ERR_ARG, "mhd_net_gradient: null array");
    const long long nvox = (long long)nx * ny * nz;
    NHIP(n, hipSetDevice(n->dev));
    rc = ensure_workspace(n, nvox);
    if (rc) return rc;
    rc = upload_input(n, x, nvox, n->a0);
    if (rc) return rc;
    NHIP(n, forward_on(n, n->stream, n->a0, nx, ny, nz, true));
    std::vector<float> g8((size_t)nvox * 8, 0.f);
    for (long long v = 0; v < nvox; ++v)
        for (int c = 0; c < n->cout; ++c) g8[(size_t)v * 8 + c] = dy[v * n->cout + c];
    NHIP(n, hipMemcpyAsync(n->tmp32, g8.data(), g8.size() * sizeof(float), hipMemcpyHostToDevice, n->stream));
    hipLaunchKernelGGL(k_f32_to_bf16, dim3((unsigned)((nvox * 8 + 255) / 256)), dim3(256), 0, n->stream, n->tmp32,
                       n->g3, nvox, 8, 8);
    NHIP(n, hipGetLastError());
    NHIP(n, backward(n, n->a0, nx, ny, nz, dx != nullptr));
    NHIP(n, update(n, nx, ny, nz, false, 0.f));
    NHIP(n, hipMemcpyAsync(dparams, n->grad, n->nparam * sizeof(float), hipMemcpyDeviceToHost, n->stream));
    if (dx) {
        NHIP(n, hipMemcpyAsync(g8.data(), n->dx32, nvox * 8 * sizeof(float), hipMemcpyDeviceToHost, n->stream));
    }
    NHIP(n, hipStreamSynchronize(n->stream));
    if (dx)
        for (long long v = 0; v < nvox; ++v)
            for (int c = 0; c < n->cin; ++c) dx[v * n->cin + c] = g8[(size_t)v * 8 + c];
    return MHD_OK;
}

extern "C" int mhd_net_add_sample(mhd_net_t *n, int nx, int ny, int nz, const float *x, const float *t) {
    int rc = check_dims(n, nx, ny, nz, "mhd_net_add_sample");
    if (rc) return rc;
    if (!x || !t) return nfail(n, MHD_ERR_ARG, "mhd_net_add_sample: null array");
    const long long nvox = (long long)nx * ny * nz;
    NHIP(n, hipSetDevice(n->dev));
    rc = ensure_workspace(n, nvox);
    if (rc) return rc;
    Sample s{nx, ny, nz, nullptr, nullptr};
    NHIP(n, hipMalloc(&s.x, nvox * 8 * sizeof(bf16)));
    hipError_t e = hipMalloc(&s.t, nvox * 8 * sizeof(float));
    if (e != hipSuccess) {
        (void)hipFree(s.x);
        return nfail(n, MHD_ERR_HIP, "mhd_net_add_sample: %s", hipGetErrorString(e));
    }
    n->samples.push_back(s);
    rc = upload_input(n, x, nvox, s.x);
    if (rc) return rc;
    std::vector<float> t8((size_t)nvox * 8, 0.f);
    for (long long v = 0; v < nvox; ++v)
        for (int c = 0; c < n->cout; ++c) t8[(size_t)v * 8 + c] = t[v * n->cout + c];
    NHIP(n, hipMemcpyAsync(s.t, t8.data(), t8.size() * sizeof(float), hipMemcpyHostToDevice, n->stream));
    NHIP(n, hipStreamSynchronize(n->stream));
    return MHD_OK;
}

extern "C" int mhd_net_num_samples(const mhd_net_t *n) { return n ? (int)n->samples.size() : 0; }

extern "C" int mhd_net_clear_samples(mhd_net_t *n) {
    if (!n) return nfail(nullptr, MHD_ERR_ARG, "mhd_net_clear_samples: null handle");
    NHIP(n, hipSetDevice(n->dev));
    NHIP(n, hipStreamSynchronize(n->stream));
    for (auto &s : n->samples) {
        (void)hipFree(s.x);
        (void)hipFree(s.t);
    }
    n->samples.clear();
    return MHD_OK;
}

// loss of the current parameters on sample s (forward only); with train,
// one Adam step on it.
static int sample_step(mhd_net_t *n, int s, bool train, float lr, double *loss) {
    const Sample &S = n->samples[s];
    const long long nvox = (long long)S.nx * S.ny * S.nz;
    const int rc = ensure_workspace(n, nvox);
    if (rc) return rc;
    NHIP(n, forward_on(n, n->stream, S.x, S.nx, S.ny, S.nz, train));
    const int nb = (int)std::min<long long>(1024, (nvox * 8 + 255) / 256);
    const float gscale = (float)(2.0 / ((double)nvox * n->cout));
    hipLaunchKernelGGL(k_loss, dim3(nb), dim3(256), 0, n->stream, n->y, S.t, n->cout, nvox, gscale,
                       train ? n->g3 : nullptr, n->lpart);
    NHIP(n, hipGetLastError());
    if (train) {
        NHIP(n, backward(n, S.x, S.nx, S.ny, S.nz, false));
        ++n->adam_t;
        NHIP(n, update(n, S.nx, S.ny, S.nz, true, lr));
    }
    if (loss) {
        std::vector<double> lp(nb);
        NHIP(n, hipMemcpyAsync(lp.data(), n->lpart, nb * sizeof(double), hipMemcpyDeviceToHost, n->stream));
        NHIP(n, hipStreamSynchronize(n->stream));
        double s2 = 0;
        for (double v : lp) s2 += v;
        *loss = s2 / ((double)nvox * n->cout);
    }
    return MHD_OK;
}

extern "C" int mhd_net_train(mhd_net_t *n, int iters, float lr, double *loss_first, double *loss_last) {
    if (!n) return nfail(nullptr, MHD_ERR_ARG, "mhd_net_train: null handle");
    if (n->samples.empty()) return nfail(n, MHD_ERR_STATE, "mhd_net_train: no samples");
    if (iters < 1 || !(lr > 0.f)) return nfail(n, MHD_ERR_ARG, "mhd_net_train: iters %d, lr %g", iters, lr);
    NHIP(n, hipSetDevice(n->dev));
    for (int it = 0; it < iters; ++it) {
        double *lp = (it == 0) ? loss_first : (it == iters - 1 ? loss_last : nullptr);
        const int rc = sample_step(n, it % (int)n->samples.size(), true, lr, lp);
        if (rc) return rc;
    }
    if (iters == 1 && loss_last && loss_first) *loss_last = *loss_first;
    NHIP(n, hipStreamSynchronize(n->stream));
    return MHD_OK;
}

extern "C" int mhd_net_loss(mhd_net_t *n, int s, double *loss) {
    if (!n) return nfail(nullptr, MHD_ERR_ARG, "mhd_net_loss: null handle");
    if (s < 0 || s >= (int)n->samples.size()) return nfail(n, MHD_ERR_ARG, "mhd_net_loss: sample %d", s);
    NHIP(n, hipSetDevice(n->dev));
    return sample_step(n, s, false, 0.f, loss);
}

extern "C" int mhd_net_time_forward(mhd_net_t *n, int nx, int ny, int nz, int reps, double *ms) {
    int rc = check_dims(n, nx, ny, nz, "mhd_net_time_forward");
    if (rc) return rc;
    if (reps < 1) return nfail(n, MHD_ERR_ARG, "mhd_net_time_forward: reps %d", reps);
    NHIP(n, hipSetDevice(n->dev));
    rc = ensure_workspace(n, (long long)nx * ny * nz);
    if (rc) return rc;
    NHIP(n, forward_on(n, n->stream, n->a0, nx, ny, nz, false));  // warm-up (also sets kernel attributes)
    hipEvent_t a, b;
    NHIP(n, hipEventCreate(&a));
    NHIP(n, hipEventCreate(&b));
    NHIP(n, hipEventRecord(a, n->stream));
    for (int r = 0; r < reps; ++r) NHIP(n, forward_on(n, n->stream, n->a0, nx, ny, nz, false));
    NHIP(n, hipEventRecord(b, n->stream));
    NHIP(n, hipEventSynchronize(b));
    float t = 0;
    NHIP(n, hipEventElapsedTime(&t, a, b));
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    if (ms) *ms = t / reps;
    return MHD_OK;
}

extern "C" const char *mhd_net_last_error(const mhd_net_t *n) { return n ? n->err : g_net_err; }

extern "C" void mhd_net_destroy(mhd_net_t *n) {
    if (!n) return;
    (void)hipSetDevice(n->dev);
    if (n->stream) (void)hipStreamSynchronize(n->stream);
    for (auto &s : n->samples) {
        (void)hipFree(s.x);
        (void)hipFree(s.t);
    }
    void *bufs[] = {n->p, n->grad, n->am, n->av, n->a0, n->a1, n->a2, n->g1, n->g2, n->g3, n->z1, n->z2,
                    n->y, n->tmp32, n->dx32, n->partial, n->lpart, n->L[0].wf, n->L[0].wb, n->L[1].wf,
                    n->L[1].wb, n->L[2].wf, n->L[2].wb};
    for (void *b : bufs)
        if (b) (void)hipFree(b);
    if (n->stream) (void)hipStreamDestroy(n->stream);
    delete n;
}

// Device-side entry points for the closure-corrected step (mhd_capi.hip).
namespace rmhd {

int net_shape(const mhd_net_t *n, int *cin, int *cout) {
    if (!n) return MHD_ERR_ARG;
    *cin = n->cin;
    *cout = n->cout;
    return MHD_OK;
}

// Workspace for volumes of nvox points and the device the network lives on.
int net_prepare(mhd_net_t *n, long long nvox, int *dev) {
    *dev = n->dev;
    const int rc = ensure_workspace(n, nvox);
    if (rc) return rc;
    return hipStreamSynchronize(n->stream) == hipSuccess ? MHD_OK : MHD_ERR_HIP;
}

// force = net(x) * std + mean (FP32, stride 8; nrm: mean[7][nz], std[7]) for a
// BF16 input (stride 8) resident on the device, queued on stream s; *force_on is
// cleared if a value is not finite.
hipError_t net_force(mhd_net_t *n, hipStream_t s, int nx, int ny, int nz, const __bf16 *x, const float *nrm,
                     float *force, int *force_on) {
    if (ensure_workspace(n, (long long)nx * ny * nz) != MHD_OK) return hipErrorOutOfMemory;
    return forward_on(n, s, x, nx, ny, nz, false, nrm, force, force_on);
}

}  // namespace rmhd
