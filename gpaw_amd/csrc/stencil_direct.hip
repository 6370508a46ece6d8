// Finite-difference stencils along the grid axes without LDS: the form for
// grids that the LDS ring (stencil_rows.hip) cannot fill the GPU with, one or
// a few small ones, and for rows too long for its tiles.
//
// A thread owns PT z-adjacent points (16 bytes) of one row and marches along
// x with a register queue of the 2R + 1 planes; the y and z neighbours come
// straight from global memory, where the tile's rows have just been brought
// into L1 / L2 by the threads that own them.  No barrier and no wave roles:
// any tile, any x-run and as many waves as the registers allow, so the
// launch is split along z, y and x until the GPU is full.  What bounds it is
// the L1 rate for many bands (R = 3: 13 vector loads of 16 bytes per thread
// and plane) and the load latency of one short x-run for small grids.
// Rows need no alignment: vector loads of 16 bytes at element alignment.
// When PT does not divide n2 the last thread of a row is moved down to end
// at the row's end and stores only the points that no other thread owns.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "internal.h"

namespace gh {

namespace {

template <typename S, int R>
struct DirectArgs {
    int n0, n1, n2;
    int pbc0, pbc1, pbc2;
    int tz, ty, lx;        // vectors and rows per tile, planes per block
    int nzt, nyt, nxc;
    int phases;            // complex data with a y or z Bloch phase
    S c0;
    S cm[3][R], cp[3][R];
    S re[3][2], im[3][2];
    const double* eps;
};

// N contiguous elements at element alignment
template <int N, typename V>
__device__ __forceinline__ void load_n(const V* __restrict__ p, V* v) {
    __builtin_memcpy(v, p, N * sizeof(V));
}

// SYM: equal coefficients at +j and -j; the sums then have the order of the
// ring kernels, so a grid gives the same bits whichever kernel takes it.
template <typename V, typename S, int R, int PT, bool SYM, bool HAS_V, bool HAS_SRC>
__global__ void __launch_bounds__(512)
stencil_direct_kernel(const V* __restrict__ in, V* __restrict__ out, const S* __restrict__ vt,
                      const V* src, S beta, DirectArgs<S, R> g) {
    constexpr bool CPLX = is_complex<V>::value;
    const int n2 = g.n2;
    // block -> (band, x chunk, y tile, z tile), z fastest
    int L = xcd_swizzle(blockIdx.x, gridDim.x);
    const int zt = L % g.nzt;
    L /= g.nzt;
    const int yt = L % g.nyt;
    L /= g.nyt;
    const int xc = L % g.nxc;
    const int band = L / g.nxc;
    const int r = threadIdx.x / g.tz;
    const int zv = (zt * g.tz + (int)threadIdx.x - r * g.tz) * PT;
    const int y = yt * g.ty + r;
    if (r >= g.ty || y >= g.n1 || zv >= n2) return;
    const int z = min(zv, n2 - PT);
    const int x0 = xc * g.lx, x1 = min(x0 + g.lx, g.n0);
    const size_t plane = (size_t)g.n1 * n2;
    const V* __restrict__ inb = in + band * plane * g.n0;
    const V* srcb = HAS_SRC ? src + band * plane * g.n0 : nullptr;
    V* __restrict__ outb = out + band * plane * g.n0;
    const S c0b = g.eps ? g.c0 - (S)g.eps[band] : g.c0;
    const int yz = y * n2 + z;

    // rows y -+ (j + 1): offset of the row (wrapped; own row when beyond a
    // zero boundary) and, for the lanes whose rows leave the grid, why
    int yo[2 * R];
    unsigned ylow = 0, yhigh = 0;      // bit j: row j lies below / above the grid
#pragma unroll
    for (int j = 0; j < 2 * R; j++) {
        int yy = j < R ? y - 1 - j : y + 1 + (j - R);
        if (yy < 0) ylow |= 1u << j;
        if (yy >= g.n1) yhigh |= 1u << j;
        if (yy < 0 || yy >= g.n1) yy = g.pbc1 ? (yy < 0 ? yy + g.n1 : yy - g.n1) : y;
        yo[j] = yy * n2 + z;
    }
    const unsigned yout = ylow | yhigh;
    const bool yfix = __any((int)yout) && (!g.pbc1 || (CPLX && g.phases));
    const bool zedge = z - R < 0 || z + PT - 1 + R >= n2;

    // element at any z of the plane's row (edge lanes only)
    auto at_z = [&](const V* __restrict__ row, int zz) -> V {
        if (zz >= 0 && zz < n2) return row[zz];
        if (!g.pbc2) return vzero<V>();
        const int d = zz < 0 ? 1 : 0;
        return mul_phase(row[zz < 0 ? zz + n2 : zz - n2], g.re[2][d], g.im[2][d]);
    };
    struct Pt { V v[PT]; };
    // own points of plane x in [-n0, 2 n0)
    auto own = [&](int x) {
        Pt p;
        int xx = x;
        if (x < 0 || x >= g.n0) {
            if (!g.pbc0) {
#pragma unroll
                for (int i = 0; i < PT; i++) p.v[i] = vzero<V>();
                return p;
            }
            xx = x < 0 ? x + g.n0 : x - g.n0;
        }
        load_n<PT>(inb + xx * plane + yz, p.v);
        if (CPLX && xx != x) {
            const int d = x < 0 ? 1 : 0;
#pragma unroll
            for (int i = 0; i < PT; i++) p.v[i] = mul_phase(p.v[i], g.re[0][d], g.im[0][d]);
        }
        return p;
    };

    Pt q[2 * R + 1];
#pragma unroll
    for (int j = 0; j < 2 * R; j++) q[j] = own(x0 - R + j);
    Pt nxt = own(x0 + R);
    for (int x = x0; x < x1; x++) {
        q[2 * R] = nxt;
        if (x + 1 < x1) nxt = own(x + 1 + R);      // in flight during this plane
        const V* __restrict__ pl = inb + x * plane;
        Pt yv[2 * R];
#pragma unroll
        for (int j = 0; j < 2 * R; j++) load_n<PT>(pl + yo[j], yv[j].v);
        V w[2 * R];                                 // z - R .. z - 1, z + PT ..
        if (!zedge) {
            load_n<R>(pl + yz - R, w);
            load_n<R>(pl + yz + PT, w + R);
        } else {
            const V* __restrict__ row = pl + (yz - z);
#pragma unroll
            for (int j = 0; j < R; j++) {
                w[j] = at_z(row, z - R + j);
                w[R + j] = at_z(row, z + PT + j);
            }
        }
        S vv[PT];
        Pt sv;
        if (HAS_V) load_n<PT>(vt + x * plane + yz, vv);
        if (HAS_SRC) load_n<PT>(srcb + x * plane + yz, sv.v);
        if (yfix) {
#pragma unroll
            for (int j = 0; j < 2 * R; j++) {
                if (!g.pbc1) {
#pragma unroll
                    for (int i = 0; i < PT; i++)
                        yv[j].v[i] = (yout >> j) & 1 ? vzero<V>() : yv[j].v[i];
                } else if (CPLX) {
                    const int d = (ylow >> j) & 1;
                    const bool wr = (yout >> j) & 1;
                    const S pr = wr ? g.re[1][d] : (S)1, pi = wr ? g.im[1][d] : (S)0;
#pragma unroll
                    for (int i = 0; i < PT; i++) yv[j].v[i] = mul_phase_of(wr, yv[j].v[i], pr, pi);
                }
            }
        }
        Pt acc;
#pragma unroll
        for (int i = 0; i < PT; i++) {
            V a = vscale(q[R].v[i], c0b);
            auto add_pair = [&](int c, int j, V m, V p) {
                if constexpr (SYM) a = fma_rs(g.cm[c][j], vadd(m, p), a);
                else a = fma_rs(g.cp[c][j], p, fma_rs(g.cm[c][j], m, a));
            };
#pragma unroll
            for (int j = 0; j < R; j++) add_pair(0, j, q[R - 1 - j].v[i], q[R + 1 + j].v[i]);
#pragma unroll
            for (int j = 0; j < R; j++) add_pair(1, j, yv[j].v[i], yv[R + j].v[i]);
            // element e of the window z - R .. z + PT - 1 + R
            auto we = [&](int e) {
                return e < R ? w[e] : e < R + PT ? q[R].v[e - R] : w[e - PT];
            };
#pragma unroll
            for (int j = 0; j < R; j++) add_pair(2, j, we(R + i - 1 - j), we(R + i + 1 + j));
            if (HAS_V) a = fma_rs(vv[i], q[R].v[i], a);
            if (HAS_SRC) a = fma_rs(beta, sv.v[i], a);
            acc.v[i] = a;
        }
        V* __restrict__ o = outb + x * plane + yz;
        if (z == zv) {
            __builtin_memcpy(o, acc.v, PT * sizeof(V));
        } else {
#pragma unroll
            for (int i = 1; i < PT; i++)
                if (z + i >= zv) o[i] = acc.v[i];
        }
#pragma unroll
        for (int j = 0; j < 2 * R; j++) q[j] = q[j + 1];
    }
}

// Threads per block, threads at which the GPU counts as full (half of the
// 2048 per CU), shortest x-run.  191 x 191 x 223 FP64, R = 3 with a source:
// 57.8 us (256, 2^18, 4); 58.8 with 512 threads per block, 57.3 at 2^19
// threads, 65.8 at 2^17 and runs of 8.
constexpr int kThreads = 256;
constexpr int64_t kFill = 262144;
constexpr int kMinPlanes = 4;

template <typename V, typename S, int R, int PT>
int launch_r(const DirectStencil& h, const void* in, void* out, int64_t nbands,
             const double* phase_cd, const void* vt, const void* src, double beta, double alpha,
             double gamma, const double* eps, hipStream_t st) {
    DirectArgs<S, R> g;
    g.n0 = h.n[0]; g.n1 = h.n[1]; g.n2 = h.n[2];
    g.pbc0 = h.pbc[0]; g.pbc1 = h.pbc[1]; g.pbc2 = h.pbc[2];
    g.c0 = (S)(alpha * h.c0 + gamma);
    g.eps = eps;
    for (int c = 0; c < 3; c++)
        for (int j = 0; j < R; j++) {
            g.cm[c][j] = (S)(alpha * h.cm[c][j]);
            g.cp[c][j] = (S)(alpha * h.cp[c][j]);
        }
    const Phases ph = make_phases(phase_cd);
    g.phases = 0;
    for (int c = 0; c < 3; c++)
        for (int d = 0; d < 2; d++) {
            g.re[c][d] = (S)ph.re[c][d];
            g.im[c][d] = (S)ph.im[c][d];
            if (c > 0 && (g.re[c][d] != (S)1 || g.im[c][d] != (S)0)) g.phases = 1;
        }
    // Tile: rows of about equal z pieces of at most 64 vectors, and rows
    // until the block has kThreads threads (their 2R ghost rows come from
    // the neighbouring tiles' lines in L2).
    const int nv = (g.n2 + PT - 1) / PT;
    g.nzt = (nv + 63) / 64;
    g.tz = (nv + g.nzt - 1) / g.nzt;
    int ty = h.rows > 0 ? h.rows : std::max(1, kThreads / g.tz);
    ty = std::min(std::min(ty, g.n1), std::max(1, 512 / g.tz));
    g.nyt = (g.n1 + ty - 1) / ty;
    g.ty = h.rows > 0 ? ty : (g.n1 + g.nyt - 1) / g.nyt;
    const int threads = (g.tz * g.ty + 63) / 64 * 64;
    // x chunks: each re-reads 2R planes (from L2 / MALL), so only until
    // kFill threads run, and not below kMinPlanes planes
    if (h.planes > 0) {
        g.lx = std::min(h.planes, g.n0);
    } else {
        const int64_t base = nbands * (int64_t)g.nyt * g.nzt * threads;
        int nxc = (int)std::min<int64_t>(g.n0, std::max<int64_t>(1, kFill / std::max<int64_t>(base, 1)));
        g.lx = std::max((g.n0 + nxc - 1) / nxc, std::min(kMinPlanes, g.n0));
    }
    g.nxc = (g.n0 + g.lx - 1) / g.lx;
    const int64_t nblocks = nbands * (int64_t)g.nyt * g.nzt * g.nxc;
    GH_REQUIRE(nblocks < (1ll << 31), GH_ERR_SHAPE, "stencil: too many blocks");
    bool sym = true;
    for (int c = 0; c < 3; c++)
        for (int j = 0; j < R; j++) sym = sym && h.cm[c][j] == h.cp[c][j];
    auto go = [&](auto symmetric) {
        constexpr bool SY = decltype(symmetric)::value;
#define GH_DIRECT(HV, HS)                                                                     \
    hipLaunchKernelGGL((stencil_direct_kernel<V, S, R, PT, SY, HV, HS>),                      \
                       dim3((unsigned)nblocks), dim3(threads), 0, st, (const V*)in, (V*)out,  \
                       (const S*)vt, (const V*)src, (S)beta, g)
        if (vt && src) GH_DIRECT(true, true);
        else if (vt) GH_DIRECT(true, false);
        else if (src) GH_DIRECT(false, true);
        else GH_DIRECT(false, false);
#undef GH_DIRECT
    };
    if (sym) go(std::true_type{});
    else go(std::false_type{});
    GH_CHECK_LAUNCH();
    return GH_OK;
}

template <typename V, typename S, int PT>
int launch(const DirectStencil& h, const void* in, void* out, int64_t nb, const double* ph,
           const void* vt, const void* src, double beta, double al, double ga,
           const double* eps, hipStream_t st) {
    if constexpr (PT > 1)   // rows shorter than a vector
        if (h.n[2] < PT)
            return launch<V, S, 1>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, st);
    switch (h.R) {
        case 1: return launch_r<V, S, 1, PT>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, st);
        case 2: return launch_r<V, S, 2, PT>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, st);
        case 3: return launch_r<V, S, 3, PT>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, st);
        case 4: return launch_r<V, S, 4, PT>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, st);
        case 5: return launch_r<V, S, 5, PT>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, st);
        case 6: return launch_r<V, S, 6, PT>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, st);
    }
    set_error("stencil: radius %d unsupported", h.R);
    return GH_ERR_UNSUPPORTED;
}

}  // namespace

int stencil_direct(int dtype, const DirectStencil& h, const void* in, void* out, int64_t nb,
                   const double* ph, const void* vt, const void* src, double beta, double al,
                   double ga, const double* eps, hipStream_t st) {
    switch (dtype) {
        case GH_F64: return launch<double, double, 2>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, st);
        case GH_C128: return launch<cplx<double>, double, 1>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, st);
        case GH_F32: return launch<float, float, 4>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, st);
        case GH_C64: return launch<cplx<float>, float, 2>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, st);
    }
    return GH_ERR_ARG;
}

}  // namespace gh
