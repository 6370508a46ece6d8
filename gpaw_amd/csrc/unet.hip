// Learned preconditioner: the layers of a small 3D U-Net on gfx950 matrix
// cores.  It replaces the multigrid V-cycle of the eigensolver
// (gpaw/preconditioner.py:9-93, called from gpaw/eigensolvers/rmmdiis.py:
// 138-143): d = f(R, v), a correction from the residual R and the local
// potential v.
//
// Activations are BF16, channel-last: act[b][x][y][z][C] (C = 8, 16 or 32)
// on a periodic grid.  Weights are BF16; every product is summed in FP32
// (v_mfma_f32_16x16x16bf16_1k).  A 3x3x3 convolution is a GEMM of
// (points) x (27 taps * C_in) against (27 taps * C_in) x (C_out): a
// wavefront owns 16 points (flattened (y, z) of one x-plane) and all output
// channels; for each k-chunk of 16 (tap, channel) pairs each lane gathers
// the 4 channels of one neighbour of its point (8 bytes) and the matching
// 4 x 16 weights, pre-packed on the host in the lane order of the
// instruction.  Periodic neighbours wrap by index.  Epilogue: bias, ReLU,
// BF16 store.
//
// Input modes of the convolution:
//   FIRST  channel 0 = s_b R[b][p], channel 1 = v_scale v[p] (FP32 or FP64
//          inputs, band-major grids), no other channels (C_in = 2);
//   PLAIN  act_in[b][p][:];
//   UPADD  act_in[b][p / 2][:] + skip[b][p][:] (nearest upsampling of a
//          coarse tensor plus a skip connection, summed in FP32).
// The remaining layers (2x2x2 average pooling, 1x1 channel maps, the final
// 1x1 map to the FP32 / FP64 correction with the per-band scale) are
// memory-bound element kernels.
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "common.h"
#include "internal.h"

namespace gh {

namespace {

typedef short bf4 __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(unsigned short h) {
    return __uint_as_float((unsigned)h << 16);
}
// round to nearest even
__device__ __forceinline__ unsigned short f2bf(float f) {
    unsigned u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (unsigned short)(u >> 16);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

// two values, round to nearest even, in one instruction (low half: a)
typedef float f2v __attribute__((ext_vector_type(2)));
typedef __bf16 b2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned f2bf2(float a, float b) {
    const b2v r = __builtin_convertvector((f2v{a, b}), b2v);
    unsigned u;
    __builtin_memcpy(&u, &r, 4);
    return u;
}
__device__ __forceinline__ float bf_lo(unsigned u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf_hi(unsigned u) { return __uint_as_float(u & 0xffff0000u); }

enum { kFirst = 0, kPlain = 1, kUpAdd = 2 };

struct ConvGeom {
    int nx, ny, nz;      // output (and input, except the coarse UPADD input) grid
    int nbands;
};

template <typename T>
struct FirstIn {
    const T* R;          // (nbands, nx, ny, nz)
    const T* v;          // (nx, ny, nz)
    const float* scale;  // per band
    float vscale;
};

// 3x3x3 periodic convolution, C_in -> C_out (C_out multiple of 8, <= 32).
// Grid: (ceil(ny * nz / 64), nx, nbands); block 256 (4 waves x 16 points).
// W: packed bf16 [ct][kc][lane][4], NK = ceil(27 C_in / 16) chunks,
// NCT = ceil(C_out / 16) column tiles.
template <int CIN, int COUT, int MODE, typename T>
__global__ void __launch_bounds__(256)
conv3_kernel(ConvGeom g, const unsigned short* __restrict__ in,
             const unsigned short* __restrict__ skip, FirstIn<T> fin,
             const unsigned short* __restrict__ W, const float* __restrict__ bias,
             int relu, unsigned short* __restrict__ out) {
    constexpr int NK = (27 * CIN + 15) / 16;
    constexpr int NCT = (COUT + 15) / 16;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int grp = lane >> 4, row = lane & 15;
    const int b = blockIdx.z, x = blockIdx.y;
    const int nyz = g.ny * g.nz;
    const int p0 = (blockIdx.x * 4 + wave) * 16;          // first point of the wave
    if (p0 >= nyz) return;                                  // whole wave idle
    const int p = p0 + row;                                 // this lane's A row
    const bool pv = p < nyz;
    const int y = pv ? p / g.nz : 0, z = pv ? p - (p / g.nz) * g.nz : 0;
    const int64_t plane = (int64_t)nyz;
    const int cnx = g.nx / 2, cny = g.ny / 2, cnz = g.nz / 2;   // UPADD coarse grid

    f4v acc[NCT];
#pragma unroll
    for (int t = 0; t < NCT; t++) acc[t] = f4v{0.f, 0.f, 0.f, 0.f};

    for (int kc = 0; kc < NK; kc++) {
        bf4 a = bf4{0, 0, 0, 0};
        const int k0 = 16 * kc + 4 * grp;
        if (MODE == kFirst) {
            // C_in = 2: the 4 k of a lane span two taps
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int k = k0 + e;
                const int tap = k >> 1, ci = k & 1;
                float v = 0.f;
                if (pv && tap < 27) {
                    const int dx = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dz = tap % 3 - 1;
                    int xx = x + dx, yy = y + dy, zz = z + dz;
                    xx += xx < 0 ? g.nx : (xx >= g.nx ? -g.nx : 0);
                    yy += yy < 0 ? g.ny : (yy >= g.ny ? -g.ny : 0);
                    zz += zz < 0 ? g.nz : (zz >= g.nz ? -g.nz : 0);
                    const int64_t q = ((int64_t)xx * g.ny + yy) * g.nz + zz;
                    v = ci == 0 ? (float)fin.R[(int64_t)b * g.nx * plane + q] * fin.scale[b]
                                : (float)fin.v[q] * fin.vscale;
                }
                a[e] = (short)f2bf(v);
            }
        } else {
            const int tap = k0 / CIN, ci = k0 - tap * CIN;
            if (pv && tap < 27) {
                const int dx = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dz = tap % 3 - 1;
                int xx = x + dx, yy = y + dy, zz = z + dz;
                xx += xx < 0 ? g.nx : (xx >= g.nx ? -g.nx : 0);
                yy += yy < 0 ? g.ny : (yy >= g.ny ? -g.ny : 0);
                zz += zz < 0 ? g.nz : (zz >= g.nz ? -g.nz : 0);
                if (MODE == kPlain) {
                    const int64_t q = (((int64_t)b * g.nx + xx) * g.ny + yy) * g.nz + zz;
                    a = *reinterpret_cast<const bf4*>(in + q * CIN + ci);
                } else {
                    const int64_t q = (((int64_t)b * g.nx + xx) * g.ny + yy) * g.nz + zz;
                    const int64_t qc =
                        (((int64_t)b * cnx + (xx >> 1)) * cny + (yy >> 1)) * cnz + (zz >> 1);
                    const bf4 s = *reinterpret_cast<const bf4*>(skip + q * CIN + ci);
                    const bf4 c = *reinterpret_cast<const bf4*>(in + qc * CIN + ci);
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        a[e] = (short)f2bf(bf2f((unsigned short)s[e]) +
                                           bf2f((unsigned short)c[e]));
                }
            }
        }
#pragma unroll
        for (int t = 0; t < NCT; t++) {
            const bf4 w = *reinterpret_cast<const bf4*>(W + (((int64_t)t * NK + kc) * 64 + lane) * 4);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, w, acc[t], 0, 0, 0);
        }
    }
    // D[i][j]: point p0 + 4 grp + r, channel t * 16 + row
#pragma unroll
    for (int t = 0; t < NCT; t++) {
        const int co = t * 16 + row;
        if (co >= COUT) continue;
        const float bb = bias[co];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int pp = p0 + 4 * grp + r;
            if (pp >= nyz) continue;
            float v = acc[t][r] + bb;
            if (relu) v = fmaxf(v, 0.f);
            out[(((int64_t)b * g.nx + x) * plane + pp) * COUT + co] = f2bf(v);
        }
    }
}

// The same convolution with the input slab staged in LDS: a block owns
// TY full rows (all z) of one x-plane and stages the 3 x-planes x (TY + 2)
// rows x (nz + 2) points (periodic wrap applied while staging) of its
// input once -- for UPADD the upsampled sum and for FIRST the scaled R and
// v (as 4 channels: R, v, 0, 0) are formed there, once per input point
// instead of once per use -- then every wave walks its 16-point tiles of
// the block reading the A operand from LDS.  CL: staged channels (CIN, or
// 4 for FIRST).
template <int CIN, int COUT, int MODE, typename T>
__global__ void __launch_bounds__(256)
conv3_lds_kernel(ConvGeom g, int ty, const unsigned short* __restrict__ in,
                 const unsigned short* __restrict__ skip, FirstIn<T> fin,
                 const unsigned short* __restrict__ W, const float* __restrict__ bias,
                 int relu, unsigned short* __restrict__ out) {
    constexpr int CL = MODE == kFirst ? 4 : CIN;
    constexpr int NK = (27 * CL + 15) / 16;
    constexpr int NCT = (COUT + 15) / 16;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    unsigned short* sIn = reinterpret_cast<unsigned short*>(smem_raw);
    const int b = blockIdx.z, x = blockIdx.y;
    const int y0 = blockIdx.x * ty;
    const int tye = min(ty, g.ny - y0);
    const int nz = g.nz, nzp = nz + 2, rows = tye + 2;
    const int64_t plane = (int64_t)g.ny * nz;
    const int cnx = g.nx / 2, cny = g.ny / 2, cnz = g.nz / 2;
    // ---- stage: (3, rows, nzp) points x CL channels, 4 channels per item
    const int nitem = 3 * rows * nzp * (CL / 4);
    for (int it = threadIdx.x; it < nitem; it += blockDim.x) {
        const int c4 = it % (CL / 4);
        int q = it / (CL / 4);
        const int zl = q % nzp; q /= nzp;
        const int yl = q % rows;
        const int dx = q / rows;
        int xx = x + dx - 1, yy = y0 + yl - 1, zz = zl - 1;
        xx += xx < 0 ? g.nx : (xx >= g.nx ? -g.nx : 0);
        yy += yy < 0 ? g.ny : (yy >= g.ny ? -g.ny : 0);
        zz += zz < 0 ? g.nz : (zz >= g.nz ? -g.nz : 0);
        const int64_t pt = ((int64_t)xx * g.ny + yy) * nz + zz;   // in the band
        bf4 a;
        if (MODE == kFirst) {
            const float r = (float)fin.R[(int64_t)b * g.nx * plane + pt] * fin.scale[b];
            const float v = (float)fin.v[pt] * fin.vscale;
            a = bf4{(short)f2bf(r), (short)f2bf(v), 0, 0};
        } else if (MODE == kPlain) {
            a = *reinterpret_cast<const bf4*>(in + ((int64_t)b * g.nx * plane + pt) * CIN +
                                              4 * c4);
        } else {
            const int64_t qc =
                (((int64_t)b * cnx + (xx >> 1)) * cny + (yy >> 1)) * cnz + (zz >> 1);
            const bf4 sv = *reinterpret_cast<const bf4*>(
                skip + ((int64_t)b * g.nx * plane + pt) * CIN + 4 * c4);
            const bf4 cv = *reinterpret_cast<const bf4*>(in + qc * CIN + 4 * c4);
#pragma unroll
            for (int e = 0; e < 4; e++)
                a[e] = (short)f2bf(bf2f((unsigned short)sv[e]) + bf2f((unsigned short)cv[e]));
        }
        *reinterpret_cast<bf4*>(sIn + (((dx * rows + yl) * nzp + zl) * CL + 4 * c4)) = a;
    }
    __syncthreads();
    // ---- products: 16-point tiles of the block's rows x nz points
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int grp = lane >> 4, row = lane & 15;
    const int npts = tye * nz;
    // small layers keep their B operands in registers for all the wave's
    // tiles (the fine levels, where the tiles are many)
    constexpr bool WREG = NK * NCT <= 28;
    bf4 wr[WREG ? NK * NCT : 1];
    if constexpr (WREG) {
#pragma unroll
        for (int i = 0; i < NK * NCT; i++)
            wr[i] = *reinterpret_cast<const bf4*>(W + ((int64_t)i * 64 + lane) * 4);
    }
    for (int p0 = wave * 16; p0 < npts; p0 += 64) {
        const int p = p0 + row;
        const bool pv = p < npts;
        const int yl = pv ? p / nz : 0, z = pv ? p - (p / nz) * nz : 0;
        f4v acc[NCT];
#pragma unroll
        for (int t = 0; t < NCT; t++) acc[t] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kc = 0; kc < NK; kc++) {
            const int k0 = 16 * kc + 4 * grp;
            const int tap = k0 / CL, ci = k0 - tap * CL;
            bf4 a = bf4{0, 0, 0, 0};
            if (pv && tap < 27) {
                const int dx = tap / 9, dy = (tap / 3) % 3, dz = tap % 3;
                a = *reinterpret_cast<const bf4*>(
                    sIn + (((dx * rows + yl + dy) * nzp + z + dz) * CL + ci));
            }
#pragma unroll
            for (int t = 0; t < NCT; t++) {
                bf4 w;
                if constexpr (WREG) w = wr[t * NK + kc];
                else w = *reinterpret_cast<const bf4*>(W + (((int64_t)t * NK + kc) * 64 + lane) * 4);
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, w, acc[t], 0, 0, 0);
            }
        }
#pragma unroll
        for (int t = 0; t < NCT; t++) {
            const int co = t * 16 + row;
            if (co >= COUT) continue;
            const float bb = bias[co];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int pp = p0 + 4 * grp + r;
                if (pp >= npts) continue;
                float v = acc[t][r] + bb;
                if (relu) v = fmaxf(v, 0.f);
                out[(((int64_t)b * g.nx + x) * plane + (int64_t)y0 * nz + pp) * COUT + co] =
                    f2bf(v);
            }
        }
    }
}

// The convolution of the two fine levels (C_in <= 16, C_out <= 16), marching
// along x.  A block owns one band, ty full rows and lx planes; a ring of
// four planes (its rows and halo, periodic images included) is in LDS, every
// plane is loaded into registers one iteration ahead and staged once (the
// per-plane kernel above stages three planes for every plane it computes),
// and there is one barrier per plane.
//   * The products are formed as W^T A^T: a lane ends with four channels of
//     one point, so results leave in 8-byte stores, and what follows the
//     layer can work on them in registers: kHead, the final 1x1 map to the
//     correction, and kMap, the 1x1 map 16 -> 8 that precedes the upsampling.
//   * The taps' LDS offsets are uniform, so a product costs a selection and
//     an add, one 8-byte LDS read and the matrix instruction.  Two 16-point
//     tiles per wave interleave their chains.
// The order of the products and sums of a result is that of the kernel above
// (same k-chunks, same instruction), so are its bits.
// Bounds: staging and epilogue instructions and LDS reads; activations move
// 16 to 40 bytes per point.  64 bands of 96^3 (48^3 on the coarse level), us,
// the per-plane kernel and the map's own pass -> here:
//   2 -> 8 first layer             2609        -> 519  (bytes: 270)
//   8 -> 16 coarse                  435        -> 118
//   16 -> 16 upsampled + 16 -> 8    905 + 203  -> 382
//   8 -> 8 upsampled + correction  4528 + 220  -> 860  (bytes: 290)
enum { kStore = 0, kHead = 1, kMap = 2 };

template <typename T>
struct MarchOut {
    unsigned short* act;      // kStore: channel-last result; kMap: 8 channels
    T* corr;                  // kHead: the correction
    const float* W;           // kHead: W[c]; kMap: W[ci][8]
    const float* bias;        // kMap: 8 values
    const float* scale;       // kHead: per band
    float bias0;              // kHead
};

constexpr int kMarchThreads = 512;
// staged items per thread and plane (each up to 8 registers)
template <int CL> struct MarchItems { static constexpr int value = CL == 4 ? 4 : 2; };

template <int CIN, int COUT, int MODE, int EPI, typename T>
__global__ void __launch_bounds__(kMarchThreads, CIN == 16 ? 2 : 4)
conv3_march_kernel(ConvGeom g, int ty, int lx, int nyt, int nxc, unsigned zmagic,
                   const unsigned short* __restrict__ in,
                   const unsigned short* __restrict__ skip, FirstIn<T> fin,
                   const unsigned short* __restrict__ W, const float* __restrict__ bias,
                   int relu, MarchOut<T> o) {
    constexpr int CL = MODE == kFirst ? 4 : CIN;
    // Staged points are PB bytes apart; 16 channels are two halves of 8 in
    // planes of their own (32 bytes apart, the 16 points of a read would meet
    // in the same LDS banks twice).
    constexpr int PB = CL >= 8 ? 16 : 8;
    constexpr int IPP = 2 * CL / PB;                  // items of PB bytes per point
    constexpr int NK = (27 * CL + 15) / 16;
    constexpr int NI = MarchItems<CL>::value;
    static_assert(COUT <= 16 && CL <= 16, "one column tile");
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = lane >> 4, row = lane & 15;
    int L = xcd_swizzle(blockIdx.x, gridDim.x);
    const int yt = L % nyt;
    L /= nyt;
    const int xc = L % nxc, b = L / nxc;
    const int y0 = yt * ty, tye = min(ty, g.ny - y0);
    const int x0 = xc * lx, x1 = min(x0 + lx, g.nx);
    const int nz = g.nz, nzp = nz + 2;
    const int half = (ty + 2) * nzp * PB, slab = half * IPP;
    const int64_t plane = (int64_t)g.ny * nz;
    const int cny = g.ny / 2, cnz = g.nz / 2;
    const int64_t cplane = (int64_t)cny * cnz;
    const int nitem = (tye + 2) * nzp * IPP;
    const int npts = tye * nz;

    // staged items of this thread: offset in the plane (and coarse plane),
    // in elements
    int goff[NI], coff[NI];
#pragma unroll
    for (int u = 0; u < NI; u++) {
        const int it = min(tid + u * kMarchThreads, nitem - 1);
        const int q = it / IPP, c = (it - q * IPP) * (PB / 2);
        const int yl = q / nzp, zl = q - yl * nzp;
        int yy = y0 + yl - 1, zz = zl - 1;
        yy += yy < 0 ? g.ny : (yy >= g.ny ? -g.ny : 0);
        zz += zz < 0 ? nz : (zz >= nz ? -nz : 0);
        goff[u] = MODE == kFirst ? yy * nz + zz : (yy * nz + zz) * CIN + c;
        coff[u] = MODE == kUpAdd ? ((yy >> 1) * cnz + (zz >> 1)) * CIN + c : 0;
    }
    struct Raw { u4 a, c; T r, v; };
    Raw raw[NI];
    const float sc = MODE == kFirst ? fin.scale[b] : 0.f;
    auto load = [&](int xp) {
        const int xx = xp < 0 ? xp + g.nx : (xp >= g.nx ? xp - g.nx : xp);
        if constexpr (MODE == kFirst) {
            const T* R = fin.R + ((int64_t)b * g.nx + xx) * plane;
            const T* v = fin.v + xx * plane;
#pragma unroll
            for (int u = 0; u < NI; u++)
                if (tid + u * kMarchThreads < nitem) {
                    raw[u].r = R[goff[u]];
                    raw[u].v = v[goff[u]];
                }
        } else {
            const unsigned short* f =
                (MODE == kPlain ? in : skip) + ((int64_t)b * g.nx + xx) * plane * CIN;
            const unsigned short* c =
                MODE == kUpAdd ? in + ((int64_t)b * (g.nx / 2) + (xx >> 1)) * cplane * CIN : in;
#pragma unroll
            for (int u = 0; u < NI; u++)
                if (tid + u * kMarchThreads < nitem) {
                    raw[u].a = *reinterpret_cast<const u4*>(f + goff[u]);
                    if (MODE == kUpAdd) raw[u].c = *reinterpret_cast<const u4*>(c + coff[u]);
                }
        }
    };
    auto stage = [&](int slot) {
        unsigned char* ring = smem_raw + slot * slab;
#pragma unroll
        for (int u = 0; u < NI; u++) {
            const int it = tid + u * kMarchThreads;
            if (it >= nitem) continue;
            unsigned char* d = ring + (it % IPP) * half + (it / IPP) * PB;
            if constexpr (MODE == kFirst) {
                const float r = (float)raw[u].r * sc, v = (float)raw[u].v * fin.vscale;
                *reinterpret_cast<u2*>(d) = u2{f2bf2(r, v), 0u};
            } else if constexpr (MODE == kPlain) {
                *reinterpret_cast<u4*>(d) = raw[u].a;
            } else {
                u4 s;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const unsigned p = raw[u].a[e], q = raw[u].c[e];
                    s[e] = f2bf2(bf_lo(p) + bf_lo(q), bf_hi(p) + bf_hi(q));
                }
                *reinterpret_cast<u4*>(d) = s;
            }
        }
    };

    // A k-chunk of 16 covers 16 / CL taps; this lane's is tap
    // kc 16 / CL + 4 grp / CL, its channels 4 grp % CL ...  The taps' offsets
    // in the ring are uniform (sb: slots of the planes x - 1, x, x + 1), so
    // only the selection between a chunk's taps is the lane's own.  A tap
    // beyond the last reads tap 26 and counts as zero.
    constexpr int TPC = 16 / CL;
    int sb[3] = {0, 0, 0};
    const int own = IPP == 2 ? (grp >> 1) * half + 8 * (grp & 1) : 2 * (4 * grp % CL);
    const int sub = 4 * grp / CL;
    auto tap_off = [&](int tap) {
        tap = tap < 27 ? tap : 26;
        return sb[tap / 9] + (((tap / 3) % 3) * nzp + tap % 3) * PB;
    };
    auto chunk_off = [&](int kc) {
        int v = tap_off(kc * TPC);
#pragma unroll
        for (int t = 1; t < TPC; t++) v = sub == t ? tap_off(kc * TPC + t) : v;
        return v;
    };
    const bool tail = 16 * (NK - 1) + 4 * grp >= 27 * CL;
    bf4 wr[NK];
#pragma unroll
    for (int kc = 0; kc < NK; kc++)
        wr[kc] = *reinterpret_cast<const bf4*>(W + ((int64_t)kc * 64 + lane) * 4);
    float bv[4];
#pragma unroll
    for (int r = 0; r < 4; r++) bv[r] = 4 * grp + r < COUT ? bias[4 * grp + r] : 0.f;
    float mw[EPI == kMap ? 32 : 1];       // kMap: the weights of this lane's two results
    if constexpr (EPI == kMap) {
#pragma unroll
        for (int c = 0; c < 16; c++) {
            mw[2 * c] = o.W[c * 8 + 2 * grp];
            mw[2 * c + 1] = o.W[c * 8 + 2 * grp + 1];
        }
    }
    float hw[4];
    float inv_scale = 1.f;
    if constexpr (EPI == kHead) {
#pragma unroll
        for (int r = 0; r < 4; r++) hw[r] = o.W[(4 * grp + r) & 7];
        inv_scale = o.scale[b];
    }

    // one result tile: channels 4 grp .. of point p
    unsigned short* oact = nullptr;      // this lane's channels of the plane's first point
    T* ocorr = nullptr;
    const float mb0 = EPI == kMap ? o.bias[2 * grp] : 0.f;
    const float mb1 = EPI == kMap ? o.bias[2 * grp + 1] : 0.f;
    auto finish = [&](f4v acc, int p) {
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            v[r] = acc[r] + bv[r];
            if (relu) v[r] = fmaxf(v[r], 0.f);
        }
        const u2 h = u2{f2bf2(v[0], v[1]), f2bf2(v[2], v[3])};
        if constexpr (EPI == kStore) {
            if (p < npts && 4 * grp < COUT) *reinterpret_cast<u2*>(oact + p * COUT) = h;
        } else if constexpr (EPI == kHead) {
            // the sum over channels in order: lane group 0, then group 1
            const float f[4] = {bf_lo(h.x), bf_hi(h.x), bf_lo(h.y), bf_hi(h.y)};
            float s = o.bias0;
#pragma unroll
            for (int r = 0; r < 4; r++) s += hw[r] * f[r];
            s = __shfl(s, row);
#pragma unroll
            for (int r = 0; r < 4; r++) s += hw[r] * f[r];
            if (grp == 1 && p < npts) ocorr[p] = (T)(s / inv_scale);
        } else {
            // every lane gathers the point's 16 channels and forms two of
            // the 8 results
            float s0 = mb0, s1 = mb1;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const unsigned p0 = (unsigned)__shfl((int)h.x, 16 * q + row);
                const unsigned p1 = (unsigned)__shfl((int)h.y, 16 * q + row);
                const float f[4] = {bf_lo(p0), bf_hi(p0), bf_lo(p1), bf_hi(p1)};
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    s0 += mw[2 * (4 * q + r)] * f[r];
                    s1 += mw[2 * (4 * q + r) + 1] * f[r];
                }
            }
            if (p < npts) *reinterpret_cast<unsigned*>(oact + p * 8) = f2bf2(s0, s1);
        }
    };

    // slot of plane xp: (xp - x0 + 1) mod 4
    load(x0 - 1);
    stage(0);
    load(x0);
    stage(1);
    load(x0 + 1);
    stage(2);
    __syncthreads();
    constexpr int NW = kMarchThreads / 64;
    for (int x = x0; x < x1; x++) {
        const bool more = x + 1 < x1;
        if (more) load(x + 2);                 // in flight during this plane
#pragma unroll
        for (int d = 0; d < 3; d++) sb[d] = ((x - x0 + d) & 3) * slab;
        const int64_t pt0 = ((int64_t)b * g.nx + x) * plane + (int64_t)y0 * nz;
        if constexpr (EPI == kHead) ocorr = o.corr + pt0;
        else oact = o.act + pt0 * (EPI == kMap ? 8 : COUT) + (EPI == kMap ? 2 : 4) * grp;
        for (int p0 = wave * 16; p0 < npts; p0 += 2 * NW * 16) {
            const int pa = p0 + row, pb = pa + NW * 16;
            const unsigned ca = min(pa, npts - 1), cb = min(pb, npts - 1);
            const int ya = (int)__umulhi(ca, zmagic), yb = (int)__umulhi(cb, zmagic);
            // ca / nz by the magic factor; slab offset of the point
            const int ba = (ya * nzp + (int)ca - ya * nz) * PB + own;
            const int bb = (yb * nzp + (int)cb - yb * nz) * PB + own;
            f4v acca = f4v{0.f, 0.f, 0.f, 0.f}, accb = acca;
            const bool two = p0 + NW * 16 < npts;      // wave-uniform
            auto chain = [&](auto both) {
#pragma unroll
                for (int kc = 0; kc < NK; kc++) {
                    const int off = chunk_off(kc);
                    const bool zero = kc == NK - 1 && (27 * CL) % 16 != 0 && tail;
                    bf4 a = *reinterpret_cast<const bf4*>(smem_raw + ba + off);
                    if (zero) a = bf4{0, 0, 0, 0};
                    acca = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(wr[kc], a, acca, 0, 0, 0);
                    if constexpr (decltype(both)::value) {
                        bf4 c = *reinterpret_cast<const bf4*>(smem_raw + bb + off);
                        if (zero) c = bf4{0, 0, 0, 0};
                        accb = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(wr[kc], c, accb, 0, 0, 0);
                    }
                }
            };
            if (two) chain(std::true_type{});
            else chain(std::false_type{});
            finish(acca, pa);
            if (two) finish(accb, pb);
        }
        if (more) stage((x - x0 + 3) & 3);
        __syncthreads();
    }
}

// Launch of the marching form; GH_ERR_UNSUPPORTED when a row does not fit.
template <int CIN, int COUT, int MODE, int EPI, typename T>
int launch_march(const ConvGeom& g, const void* in, const void* skip, const FirstIn<T>& fin,
                 const void* W, const float* bias, int relu, const MarchOut<T>& o,
                 hipStream_t st) {
    constexpr int CL = MODE == kFirst ? 4 : CIN;
    constexpr int PB = 2 * CL, IPP = PB < 16 ? 1 : PB / 16;
    const int nzp = g.nz + 2;
    // rows: 80 KB of LDS (two blocks per CU) and MarchItems items per thread
    const int64_t lds_row = 4LL * nzp * PB;
    int ty = (int)std::min<int64_t>(g.ny, std::min<int64_t>(80 * 1024 / lds_row,
                                        (int64_t)MarchItems<CL>::value * kMarchThreads / (nzp * IPP)) - 2);
    if (ty < 1 || g.nz < 2 || (int64_t)g.ny * g.nz * CIN >= (1ll << 31)) return GH_ERR_UNSUPPORTED;
    const int nyt = (g.ny + ty - 1) / ty;
    ty = (g.ny + nyt - 1) / nyt;
    // x-runs: two blocks per CU four times over where the grid allows it
    // (each run stages two planes more), at least 8 planes
    const int64_t base = (int64_t)g.nbands * nyt;
    int nxc = (int)std::min<int64_t>(std::max(1, g.nx / 8), std::max<int64_t>(1, 2048 / base));
    const int lx = (g.nx + nxc - 1) / nxc;
    nxc = (g.nx + lx - 1) / lx;
    const int64_t nblk = base * nxc;
    GH_REQUIRE(nblk < (1ll << 31), GH_ERR_SHAPE, "unet_conv3: too many blocks");
    const size_t lds = (size_t)lds_row * (ty + 2);
    auto kfn = conv3_march_kernel<CIN, COUT, MODE, EPI, T>;
    const int rc = ensure_max_lds((const void*)kfn, 160 * 1024);
    if (rc != GH_OK) return rc;
    const unsigned magic = (unsigned)(((1ull << 32) + g.nz - 1) / g.nz);
    hipLaunchKernelGGL(kfn, dim3((unsigned)nblk), dim3(kMarchThreads), lds, st, g, ty, lx, nyt,
                       nxc, magic, (const unsigned short*)in, (const unsigned short*)skip, fin,
                       (const unsigned short*)W, bias, relu, o);
    GH_CHECK_LAUNCH();
    return GH_OK;
}

// 2x2x2 average of a channel-last BF16 tensor (fine grid nx, ny, nz even),
// 8 channels (16 bytes) per thread.  HBM bound; with one channel per thread
// the 2-byte loads bound it: 64 bands of 96^3, 8 channels (1.02 GB), 243 ->
// 214 us, of 48^3, 16 channels, 62 -> 39.
typedef unsigned u4any __attribute__((ext_vector_type(4), aligned(2)));

template <int C>
__global__ void __launch_bounds__(256)
pool2_kernel(const unsigned short* __restrict__ in, unsigned short* __restrict__ out,
             int nx, int ny, int nz, int64_t total) {
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= total) return;
    const int c = (int)(t % (C / 8)) * 8;
    int64_t q = t / (C / 8);
    const int cz = nz / 2, cy = ny / 2, cx = nx / 2;
    const int Z = (int)(q % cz); q /= cz;
    const int Y = (int)(q % cy); q /= cy;
    const int X = (int)(q % cx);
    const int64_t b = q / cx;
    u4any v[8];
#pragma unroll
    for (int d = 0; d < 8; d++) {
        const int xx = 2 * X + (d >> 2), yy = 2 * Y + ((d >> 1) & 1), zz = 2 * Z + (d & 1);
        v[d] = *reinterpret_cast<const u4any*>(
            in + (((b * nx + xx) * ny + yy) * nz + zz) * C + c);
    }
    u4any o;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        float lo = 0.f, hi = 0.f;
#pragma unroll
        for (int d = 0; d < 8; d++) {
            lo += bf_lo(v[d][e]);
            hi += bf_hi(v[d][e]);
        }
        o[e] = f2bf2(0.125f * lo, 0.125f * hi);
    }
    *reinterpret_cast<u4any*>(out + t * 8) = o;
}

// 1x1 channel map C_in -> C_out (FP32 weights W[ci][co], bias), BF16 in/out,
// a point per thread; the weights are uniform.  64 bands of 24^3, 32 -> 16:
// one result per thread 82 us, 21 here.
template <int CIN, int COUT>
__global__ void __launch_bounds__(256)
map1_kernel(const unsigned short* __restrict__ in, const float* __restrict__ W,
            const float* __restrict__ bias, unsigned short* __restrict__ out, int64_t npts) {
    const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (p >= npts) return;
    u4any v[CIN / 8];
#pragma unroll
    for (int k = 0; k < CIN / 8; k++)
        v[k] = *reinterpret_cast<const u4any*>(in + p * CIN + 8 * k);
    float s[COUT];
#pragma unroll
    for (int co = 0; co < COUT; co++) s[co] = bias[co];
#pragma unroll
    for (int ci = 0; ci < CIN; ci++) {
        const unsigned w = v[ci / 8][ci % 8 / 2];
        const float x = ci & 1 ? bf_hi(w) : bf_lo(w);
#pragma unroll
        for (int co = 0; co < COUT; co++) s[co] += W[ci * COUT + co] * x;
    }
#pragma unroll
    for (int k = 0; k < COUT / 8; k++) {
        u4any o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = f2bf2(s[8 * k + 2 * e], s[8 * k + 2 * e + 1]);
        *reinterpret_cast<u4any*>(out + p * COUT + 8 * k) = o;
    }
}

// final 1x1 map C -> 1 into the correction, times the inverse band scale
template <int C, typename T>
__global__ void __launch_bounds__(256)
head_kernel(const unsigned short* __restrict__ in, const float* __restrict__ W, float bias,
            const float* __restrict__ scale, int64_t npb, int64_t total, T* __restrict__ out) {
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= total) return;
    const int64_t b = t / npb;
    float s = bias;
#pragma unroll
    for (int ci = 0; ci < C; ci++) s += W[ci] * bf2f(in[t * C + ci]);
    out[t] = (T)(s / scale[b]);
}

constexpr int kConvLds = 60 * 1024;   // LDS budget of the staged slab

template <int CIN, int COUT, int MODE, typename T>
int launch_conv3(const ConvGeom& g, const void* in, const void* skip, const FirstIn<T>& fin,
                 const void* W, const float* bias, int relu, void* out, hipStream_t st) {
    constexpr int CL = MODE == kFirst ? 4 : CIN;
    if constexpr (CIN <= 16 && COUT <= 16) {
        MarchOut<T> o{};
        o.act = (unsigned short*)out;
        const int rc = launch_march<CIN, COUT, MODE, kStore, T>(g, in, skip, fin, W, bias, relu,
                                                                o, st);
        if (rc != GH_ERR_UNSUPPORTED) return rc;
    }
    const int64_t per_row = 3LL * (g.nz + 2) * CL * 2;
    const int ty = (int)std::min<int64_t>(g.ny, kConvLds / per_row - 2);
    if (ty >= 1) {
        const size_t lds = (size_t)per_row * (ty + 2);
        dim3 grid((unsigned)((g.ny + ty - 1) / ty), (unsigned)g.nx, (unsigned)g.nbands);
        hipLaunchKernelGGL((conv3_lds_kernel<CIN, COUT, MODE, T>), grid, dim3(256), lds, st,
                           g, ty, (const unsigned short*)in, (const unsigned short*)skip, fin,
                           (const unsigned short*)W, bias, relu, (unsigned short*)out);
        GH_CHECK_LAUNCH();
        return GH_OK;
    }
    if (MODE == kFirst) {
        set_error("unet_conv3: rows of %d points do not fit the LDS slab", g.nz);
        return GH_ERR_UNSUPPORTED;
    }
    const int nyz = g.ny * g.nz;
    dim3 grid((unsigned)((nyz + 63) / 64), (unsigned)g.nx, (unsigned)g.nbands);
    hipLaunchKernelGGL((conv3_kernel<CIN, COUT, MODE, T>), grid, dim3(256), 0, st, g,
                       (const unsigned short*)in, (const unsigned short*)skip, fin,
                       (const unsigned short*)W, bias, relu, (unsigned short*)out);
    GH_CHECK_LAUNCH();
    return GH_OK;
}

}  // namespace

}  // namespace gh

using namespace gh;

extern "C" {

int64_t gh_unet_conv3_weight_elems(int cin, int cout) {
    if (cin < 1 || cout < 1) return -1;
    const int64_t nk = (27 * cin + 15) / 16, nct = (cout + 15) / 16;
    return nct * nk * 64 * 4;
}

// Pack W[co][ci][kx][ky][kz] (float, torch's conv3d layout) into the lane
// order of the matrix-core instruction (bf16 bits), k = tap * cin + ci with
// tap = (kx * 3 + ky) * 3 + kz.
int gh_unet_pack_conv3(int cin, int cout, const float* W, uint16_t* packed) {
    GH_REQUIRE(W && packed && cin >= 1 && cout >= 1, GH_ERR_ARG, "unet_pack: bad argument");
    const int nk = (27 * cin + 15) / 16, nct = (cout + 15) / 16;
    for (int t = 0; t < nct; t++)
        for (int kc = 0; kc < nk; kc++)
            for (int lane = 0; lane < 64; lane++)
                for (int e = 0; e < 4; e++) {
                    const int k = 16 * kc + 4 * (lane >> 4) + e;
                    const int co = t * 16 + (lane & 15);
                    float v = 0.f;
                    if (k < 27 * cin && co < cout) {
                        const int tap = k / cin, ci = k % cin;
                        v = W[((int64_t)co * cin + ci) * 27 + tap];
                    }
                    uint32_t u;
                    std::memcpy(&u, &v, 4);
                    if ((u & 0x7f800000u) != 0x7f800000u) u += 0x7fffu + ((u >> 16) & 1u);
                    packed[(((int64_t)t * nk + kc) * 64 + lane) * 4 + e] = (uint16_t)(u >> 16);
                }
    return GH_OK;
}

int gh_unet_conv3(int cin, int cout, int mode, int dtype, int nbands, const int64_t* n_c,
                  const void* in_dev, const void* skip_dev, const void* R_dev,
                  const void* v_dev, const float* scale_dev, double vscale,
                  const void* W_dev, const float* bias_dev, int relu, void* out_dev,
                  void* stream) {
    GH_REQUIRE(n_c && W_dev && bias_dev && out_dev && nbands >= 0, GH_ERR_ARG,
               "unet_conv3: null argument");
    ConvGeom g;
    g.nx = (int)n_c[0]; g.ny = (int)n_c[1]; g.nz = (int)n_c[2];
    g.nbands = nbands;
    GH_REQUIRE(g.nx >= 1 && g.ny >= 1 && g.nz >= 1 && (int64_t)g.ny * g.nz < (1 << 30),
               GH_ERR_SHAPE, "unet_conv3: bad grid");
    if (nbands == 0) return GH_OK;
    if (mode == kUpAdd)
        GH_REQUIRE(g.nx % 2 == 0 && g.ny % 2 == 0 && g.nz % 2 == 0 && skip_dev && in_dev,
                   GH_ERR_SHAPE, "unet_conv3: upsampling needs an even grid and a skip");
    hipStream_t st = (hipStream_t)stream;
    FirstIn<float> f32{};
    FirstIn<double> f64{};
    if (mode == kFirst) {
        GH_REQUIRE(R_dev && v_dev && scale_dev && cin == 2, GH_ERR_ARG,
                   "unet_conv3: the first layer takes R, v and the band scales "
                   "(weights packed for 4 input channels, the last two zero)");
        GH_REQUIRE(dtype == GH_F32 || dtype == GH_F64, GH_ERR_UNSUPPORTED,
                   "unet_conv3: real residuals only");
        f32 = FirstIn<float>{(const float*)R_dev, (const float*)v_dev, scale_dev, (float)vscale};
        f64 = FirstIn<double>{(const double*)R_dev, (const double*)v_dev, scale_dev,
                              (float)vscale};
    } else {
        GH_REQUIRE(in_dev, GH_ERR_ARG, "unet_conv3: null input");
    }
#define GH_CONV(CI, CO, MD)                                                          \
    if (cin == CI && cout == CO && mode == MD) {                                     \
        if (MD == kFirst && dtype == GH_F64)                                         \
            return launch_conv3<CI, CO, MD, double>(g, in_dev, skip_dev, f64, W_dev, \
                                                    bias_dev, relu, out_dev, st);    \
        return launch_conv3<CI, CO, MD, float>(g, in_dev, skip_dev, f32, W_dev,      \
                                               bias_dev, relu, out_dev, st);         \
    }
    GH_CONV(2, 8, kFirst)
    GH_CONV(8, 16, kPlain)
    GH_CONV(16, 32, kPlain)
    GH_CONV(32, 32, kPlain)
    GH_CONV(16, 16, kUpAdd)
    GH_CONV(8, 8, kUpAdd)
    GH_CONV(8, 8, kPlain)
    GH_CONV(16, 16, kPlain)
#undef GH_CONV
    set_error("unet_conv3: layer %d -> %d (mode %d) not built", cin, cout, mode);
    return GH_ERR_UNSUPPORTED;
}

int gh_unet_conv3_map1(int nbands, const int64_t* n_c, const void* in_dev, const void* skip_dev,
                       const void* W_dev, const float* bias_dev, const float* Wm_dev,
                       const float* bm_dev, void* out_dev, void* stream) {
    GH_REQUIRE(n_c && W_dev && bias_dev && Wm_dev && bm_dev && nbands >= 0, GH_ERR_ARG,
               "unet_conv3_map1: null argument");
    if (nbands == 0) return GH_OK;
    ConvGeom g{(int)n_c[0], (int)n_c[1], (int)n_c[2], nbands};
    GH_REQUIRE(g.nx >= 2 && g.ny >= 2 && g.nz >= 2 && g.nx % 2 == 0 && g.ny % 2 == 0 &&
                   g.nz % 2 == 0 && in_dev && skip_dev && out_dev,
               GH_ERR_SHAPE, "unet_conv3_map1: upsampling needs an even grid and a skip");
    MarchOut<float> o{};
    o.act = (unsigned short*)out_dev;
    o.W = Wm_dev;
    o.bias = bm_dev;
    const int rc = launch_march<16, 16, kUpAdd, kMap, float>(
        g, in_dev, skip_dev, FirstIn<float>{}, W_dev, bias_dev, 1, o, (hipStream_t)stream);
    if (rc == GH_ERR_UNSUPPORTED) set_error("unet_conv3_map1: rows of %d points", g.nz);
    return rc;
}

int gh_unet_conv3_head(int dtype, int nbands, const int64_t* n_c, const void* in_dev,
                       const void* skip_dev, const void* W_dev, const float* bias_dev,
                       const float* Wh_dev, double bias, const float* scale_dev, void* out_dev,
                       void* stream) {
    GH_REQUIRE(n_c && W_dev && bias_dev && Wh_dev && nbands >= 0, GH_ERR_ARG,
               "unet_conv3_head: null argument");
    GH_REQUIRE(dtype == GH_F32 || dtype == GH_F64, GH_ERR_UNSUPPORTED,
               "unet_conv3_head: real outputs only");
    if (nbands == 0) return GH_OK;
    ConvGeom g{(int)n_c[0], (int)n_c[1], (int)n_c[2], nbands};
    GH_REQUIRE(g.nx >= 2 && g.ny >= 2 && g.nz >= 2 && g.nx % 2 == 0 && g.ny % 2 == 0 &&
                   g.nz % 2 == 0 && in_dev && skip_dev && out_dev && scale_dev,
               GH_ERR_SHAPE, "unet_conv3_head: upsampling needs an even grid and a skip");
    int rc;
    if (dtype == GH_F32) {
        MarchOut<float> o{};
        o.corr = (float*)out_dev;
        o.W = Wh_dev;
        o.scale = scale_dev;
        o.bias0 = (float)bias;
        rc = launch_march<8, 8, kUpAdd, kHead, float>(g, in_dev, skip_dev, FirstIn<float>{},
                                                      W_dev, bias_dev, 1, o, (hipStream_t)stream);
    } else {
        MarchOut<double> o{};
        o.corr = (double*)out_dev;
        o.W = Wh_dev;
        o.scale = scale_dev;
        o.bias0 = (float)bias;
        rc = launch_march<8, 8, kUpAdd, kHead, double>(g, in_dev, skip_dev, FirstIn<double>{},
                                                       W_dev, bias_dev, 1, o,
                                                       (hipStream_t)stream);
    }
    if (rc == GH_ERR_UNSUPPORTED) set_error("unet_conv3_head: rows of %d points", g.nz);
    return rc;
}

int gh_unet_pool2(int c, int nbands, const int64_t* n_c, const void* in_dev, void* out_dev,
                  void* stream) {
    GH_REQUIRE(n_c && in_dev && out_dev, GH_ERR_ARG, "unet_pool2: null argument");
    const int nx = (int)n_c[0], ny = (int)n_c[1], nz = (int)n_c[2];
    GH_REQUIRE(nx % 2 == 0 && ny % 2 == 0 && nz % 2 == 0, GH_ERR_SHAPE,
               "unet_pool2: odd grid");
    const int64_t points = (int64_t)nbands * (nx / 2) * (ny / 2) * (nz / 2);
    if (points * c == 0) return GH_OK;
    const int64_t total = points * (c / 8);
    hipStream_t st = (hipStream_t)stream;
    const unsigned nblk = (unsigned)((total + 255) / 256);
    switch (c) {
        case 8: hipLaunchKernelGGL((pool2_kernel<8>), dim3(nblk), dim3(256), 0, st, (const unsigned short*)in_dev, (unsigned short*)out_dev, nx, ny, nz, total); break;
        case 16: hipLaunchKernelGGL((pool2_kernel<16>), dim3(nblk), dim3(256), 0, st, (const unsigned short*)in_dev, (unsigned short*)out_dev, nx, ny, nz, total); break;
        case 32: hipLaunchKernelGGL((pool2_kernel<32>), dim3(nblk), dim3(256), 0, st, (const unsigned short*)in_dev, (unsigned short*)out_dev, nx, ny, nz, total); break;
        default: set_error("unet_pool2: %d channels", c); return GH_ERR_UNSUPPORTED;
    }
    GH_CHECK_LAUNCH();
    return GH_OK;
}

int gh_unet_map1(int cin, int cout, int64_t npts, const void* in_dev, const float* W_dev,
                 const float* bias_dev, void* out_dev, void* stream) {
    GH_REQUIRE(in_dev && W_dev && bias_dev && out_dev && npts >= 0, GH_ERR_ARG,
               "unet_map1: bad argument");
    if (npts == 0) return GH_OK;
    hipStream_t st = (hipStream_t)stream;
    const unsigned nblk = (unsigned)((npts + 255) / 256);
    const unsigned short* in = (const unsigned short*)in_dev;
    unsigned short* out = (unsigned short*)out_dev;
    if (cin == 32 && cout == 16)
        hipLaunchKernelGGL((map1_kernel<32, 16>), dim3(nblk), dim3(256), 0, st, in, W_dev, bias_dev, out, npts);
    else if (cin == 16 && cout == 8)
        hipLaunchKernelGGL((map1_kernel<16, 8>), dim3(nblk), dim3(256), 0, st, in, W_dev, bias_dev, out, npts);
    else {
        set_error("unet_map1: %d -> %d not built", cin, cout);
        return GH_ERR_UNSUPPORTED;
    }
    GH_CHECK_LAUNCH();
    return GH_OK;
}

int gh_unet_head(int cin, int dtype, int nbands, int64_t npts_per_band, const void* in_dev,
                 const float* W_dev, double bias, const float* scale_dev, void* out_dev,
                 void* stream) {
    GH_REQUIRE(in_dev && W_dev && scale_dev && out_dev && nbands >= 0, GH_ERR_ARG,
               "unet_head: bad argument");
    GH_REQUIRE(cin == 8, GH_ERR_UNSUPPORTED, "unet_head: %d channels not built", cin);
    const int64_t total = (int64_t)nbands * npts_per_band;
    if (total == 0) return GH_OK;
    hipStream_t st = (hipStream_t)stream;
    const unsigned nblk = (unsigned)((total + 255) / 256);
    const unsigned short* in = (const unsigned short*)in_dev;
    if (dtype == GH_F32)
        hipLaunchKernelGGL((head_kernel<8, float>), dim3(nblk), dim3(256), 0, st, in, W_dev,
                           (float)bias, scale_dev, npts_per_band, total, (float*)out_dev);
    else if (dtype == GH_F64)
        hipLaunchKernelGGL((head_kernel<8, double>), dim3(nblk), dim3(256), 0, st, in, W_dev,
                           (float)bias, scale_dev, npts_per_band, total, (double*)out_dev);
    else {
        set_error("unet_head: real outputs only");
        return GH_ERR_UNSUPPORTED;
    }
    GH_CHECK_LAUNCH();
    return GH_OK;
}

}  // extern "C"
