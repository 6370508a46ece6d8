// Stencil of an interpolated function, out = S(I(u)) + sum_s beta_s src_s,
// in one pass: u lies on the coarse grid, I is the linear (nn = 1)
// interpolation to the grid of twice the spacing's half, S a symmetric
// stencil along the axes of radius 1 to 3.  The interpolated function is
// never stored.
//
// The last half of a V-cycle level is this: correct by the interpolated
// coarse solution, then smooth.  As two kernels it writes and reads the
// fine function once more than needed.  HBM bound here: sources read, result
// written, the coarse function an eighth of that.
//
// I is linear along x, so with F_i the coarse plane i interpolated along z
// and y, the fine plane 2 i is F_i and 2 i + 1 is (F_i + F_i+1) / 2.  The
// y and z parts of S are applied to the F_i alone and averaged, which halves
// their work and keeps one plane of LDS per coarse plane; the x part reads
// the thread's own points of F_i-2 .. F_i+2 from registers.
//
// A block owns one band, ty full fine rows and a run of coarse planes.  Per
// step its compute threads (16 bytes of z each) make their points of
// F_i+2 from coarse values loaded one step ahead and put them into one of two
// LDS planes, apply the stencil to F_i+1 in the other, and finish the fine
// planes 2 i and 2 i + 1.  A few more waves make the tile's ghost rows and
// ghost columns, images and Bloch phases included, so that the stencil has
// no boundary cases.  One barrier per step.
//
// A whole V-cycle, us, with the interpolations and smoothers apart and with
// this kernel:
//   256 x 112^3 float64                  4159 -> 2341
//   32 x 95 x 99 x 103 float64, zero bc   439 ->  297
//   16 x 48^3 float32                      52 ->   41
//   64 x 64 x 72 x 80 float32             156 ->  109
//   40 x 64 x 72 x 80 complex64, general k  246 -> 182
//   40 x 64 x 72 x 80 complex128, k along x  334 -> 265, general k 384 -> 337
// At 256 x 112^3 the radius 3 pass alone takes 1249 us for 6.1 GB, the rate
// of a copy (5.1 TB/s at most: 1200 us).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "internal.h"
#include "linear_interp.h"

namespace gh {

namespace {

constexpr int kMaxThreads = 1024;
constexpr size_t kLdsBytes = 64 * 1024;
// ghost vectors per thread of a ghost wave (complex128: registers)
template <typename V> constexpr int kGhostItems = sizeof(V) > 8 ? 2 : 4;

template <typename S, int R>
struct InterpArgs {
    LinGrid<S> u;                 // coarse grid
    int n0, n1, n2;               // fine grid
    int odd0;                     // fine planes 2 i - odd0, + 1 belong to F_i
    int ty, lx, nyt, nxc;         // rows and coarse planes of a block
    int ncomp;                    // compute waves
    int pitch, slot;              // elements per LDS row, plane
    S c0, k[3][R];
    S beta[2];
};

template <typename V, typename S, int R, int PT, bool ALIGNED, int NS>
__global__ void __launch_bounds__(kMaxThreads)
stencil_interp_kernel(const V* __restrict__ coarse, V* __restrict__ out,
                      const V* __restrict__ src0, const V* __restrict__ src1,
                      InterpArgs<S, R> g) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    V* lds = reinterpret_cast<V*>(smem_raw);
    typedef LinPoints<V, S, PT> Points;
    typedef typename Points::Raw Raw;
    typedef typename Points::Vec Vec;
    typedef Vec UVec __attribute__((aligned(sizeof(V))));
    constexpr int E = 16 / (int)sizeof(S), C = E / PT;
    static_assert(C * sizeof(S) == sizeof(V), "points per vector");
    constexpr int NW = (R + PT - 1) / PT;            // ghost vectors per side

    const int tiles = g.nyt * g.nxc;
    const int L = xcd_swizzle(blockIdx.x, gridDim.x);
    const int band = L / tiles, tile = L - band * tiles;
    const int xc = tile / g.nyt, yt = tile - xc * g.nyt;
    const int y0 = yt * g.ty, tye = min(g.ty, g.n1 - y0);
    const int ni = g.n0 / 2 + g.odd0;                // pairs of fine planes
    const int i0 = xc * g.lx, i1 = min(i0 + g.lx, ni);
    const V* __restrict__ cb = coarse + (size_t)band * g.u.n[0] * g.u.n[1] * g.u.n[2];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nv = (g.n2 + PT - 1) / PT;

    auto put = [&](int pos, int i, Vec v) {
        *reinterpret_cast<Vec*>(lds + (i & 1) * g.slot + pos) = v;
    };

    if (wave >= g.ncomp) {
        // ---------------------------------------------------- ghosts --
        const int nt = blockDim.x - g.ncomp * 64, t = threadIdx.x - g.ncomp * 64;
        const int rowvec = nv + 2 * NW;                       // vectors per LDS row
        const int nrow = 2 * R * rowvec, n = nrow + tye * 2 * NW;
        constexpr int GI = kGhostItems<V>;
        Points it[GI];
        int pos[GI];
        Raw raw[GI];
#pragma unroll
        for (int a = 0; a < GI; a++) {
            const int p = min(t + a * nt, n - 1);
            int r, c;
            if (p < nrow) {                                   // a ghost row
                r = p / rowvec;
                c = p - r * rowvec;
                if (r >= R) r += tye;
            } else {                                          // a row's ghost columns
                r = (p - nrow) / (2 * NW);
                c = p - nrow - r * 2 * NW;
                if (c >= NW) c += nv;
                r += R;
            }
            it[a].set(y0 - R + r, (c - NW) * PT, g.u);
            pos[a] = r * g.pitch + c * PT;
        }
        auto all = [&](int i) {
#pragma unroll
            for (int a = 0; a < GI; a++) it[a].load(cb, i, g.u, raw[a]);
        };
        auto store = [&](int i) {
#pragma unroll
            for (int a = 0; a < GI; a++) put(pos[a], i, it[a].make(raw[a], i, g.u));
        };
        all(i0);
        store(i0);
        all(i0 + 1);
        store(i0 + 1);
        all(i0 + 2);
        __syncthreads();
        for (int i = i0; i < i1; i++) {
            __syncthreads();
            store(i + 2);
            all(i + 3);
        }
        return;
    }

    // ------------------------------------------------------ compute --
    // threads beyond the tile repeat its last vector (the same values to the
    // same places), so that no access is conditional
    const int pp = min((int)threadIdx.x, tye * nv - 1);
    const int yl = pp / nv, z = (pp - yl * nv) * PT;
    Points it;
    it.set(y0 + yl, z, g.u);
    const int pos = (yl + R) * g.pitch + (NW * PT + z);
    const bool part = !ALIGNED && z + PT > g.n2;
    const int short_by = ALIGNED ? 0 : nv * PT - g.n2;
    const int down = part ? short_by : 0;
    const size_t plane = (size_t)g.n1 * g.n2;
    const int yz = (y0 + yl) * g.n2 + z;
    const size_t b0 = (size_t)band * plane * g.n0;
    auto src_at = [&](const V* s, int x) {
        x = min(max(x, 0), g.n0 - 1);
        return (Vec)*reinterpret_cast<const UVec*>(s + b0 + (size_t)x * plane + (yz - down));
    };
    auto shifted = [&](Vec v) {
        if constexpr (!ALIGNED) {
            Vec o = v;
#pragma unroll
            for (int t = 1; t < PT; t++)
#pragma unroll
                for (int e = 0; e < E; e++)
                    if (short_by == t) o[e] = e + t * C < E ? v[e + t * C] : (S)0;
#pragma unroll
            for (int e = 0; e < E; e++) v[e] = part ? o[e] : v[e];
        }
        return v;
    };
    // y and z parts and the centre on the plane of F_i (f: its own points)
    auto yz_part = [&](int i, Vec f) {
        const V* p = lds + (i & 1) * g.slot + pos;
        Vec acc = f * g.c0;
#pragma unroll
        for (int j = 0; j < R; j++)
            acc = (*reinterpret_cast<const Vec*>(p - (j + 1) * g.pitch) +
                   *reinterpret_cast<const Vec*>(p + (j + 1) * g.pitch)) * g.k[1][j] + acc;
        struct { S v[(2 * NW + 1) * E]; } w;
#pragma unroll
        for (int a = 0; a <= 2 * NW; a++) {
            const Vec t = a == NW ? f : *reinterpret_cast<const Vec*>(p + (a - NW) * PT);
#pragma unroll
            for (int e = 0; e < E; e++) w.v[a * E + e] = t[e];
        }
#pragma unroll
        for (int e = 0; e < E; e++)
#pragma unroll
            for (int j = 0; j < R; j++)
                acc[e] = fma_rs(g.k[2][j], w.v[NW * E + e - (j + 1) * C] +
                                               w.v[NW * E + e + (j + 1) * C], acc[e]);
        return acc;
    };
    auto finish = [&](int x, Vec acc, const Vec* s) {
#pragma unroll
        for (int q = 0; q < NS; q++) acc = s[q] * g.beta[q] + acc;
        V* o = out + b0 + (size_t)x * plane + yz;
        if (!part) {
            __builtin_nontemporal_store((UVec)acc, reinterpret_cast<UVec*>(o));
        } else {
#pragma unroll
            for (int e = 0; e < E; e++)
                if (z + e / C < g.n2) reinterpret_cast<S*>(o)[e] = acc[e];
        }
    };

    Vec f[5];                                        // F_i-2 .. F_i+2
    {
        Raw r[4];
#pragma unroll
        for (int a = 0; a < 4; a++) it.load(cb, i0 - 2 + a, g.u, r[a]);
#pragma unroll
        for (int a = 0; a < 4; a++) f[a] = it.make(r[a], i0 - 2 + a, g.u);
    }
    put(pos, i0, f[2]);
    put(pos, i0 + 1, f[3]);
    Raw raw;
    it.load(cb, i0 + 2, g.u, raw);
    Vec s[2][NS];
    auto load_src = [&](int i, Vec (&t)[2][NS]) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            t[h][0] = src_at(src0, 2 * i - g.odd0 + h);
            if constexpr (NS == 2) t[h][1] = src_at(src1, 2 * i - g.odd0 + h);
        }
    };
    // sources are loaded a step ahead, too, where registers are left
    constexpr bool kAhead = sizeof(V) < 16;
    if (kAhead) load_src(i0, s);
    __syncthreads();
    Vec w0 = yz_part(i0, f[2]);
    for (int i = i0; i < i1; i++) {
        __syncthreads();
        f[4] = it.make(raw, i + 2, g.u);
        put(pos, i + 2, f[4]);
        it.load(cb, i + 3, g.u, raw);
        Vec t[2][NS];
        if (kAhead) load_src(i + 1, t);
        else load_src(i, s);
        const Vec w1 = yz_part(i + 1, f[3]);
        // fine planes 2 i - 4 .. 2 i + 4 from F: even F, odd the means
        Vec h[4];
#pragma unroll
        for (int a = 0; a < 4; a++) h[a] = (f[a] + f[a + 1]) * (S)0.5;
        auto fine = [&](int d) { return d & 1 ? h[(d + 3) / 2] : f[(d + 4) / 2]; };   // plane 2 i + d
        const int x = 2 * i - g.odd0;
#pragma unroll
        for (int par = 0; par < 2; par++) {
            Vec acc = par ? (w0 + w1) * (S)0.5 : w0;
#pragma unroll
            for (int j = 0; j < R; j++)
                acc = (fine(par - 1 - j) + fine(par + 1 + j)) * g.k[0][j] + acc;
#pragma unroll
            for (int q = 0; q < NS; q++) s[par][q] = shifted(s[par][q]);
            if (x + par >= 0) finish(x + par, acc, s[par]);
        }
        w0 = w1;
#pragma unroll
        for (int a = 0; a < 4; a++) f[a] = f[a + 1];
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int q = 0; q < NS; q++)
                if (kAhead) s[a][q] = t[a][q];
    }
}

template <typename V, typename S, int R>
int launch_r(const DirectStencil& h, const LinearMap& ig, const void* coarse, void* out,
             int64_t nbands, const double* phase_cd, int ns, const void* const* src,
             const double* beta, double alpha, double gamma, hipStream_t st) {
    constexpr int PT = 16 / (int)sizeof(V), NW = (R + PT - 1) / PT;
    InterpArgs<S, R> g;
    g.n0 = h.n[0]; g.n1 = h.n[1]; g.n2 = h.n[2];
    g.odd0 = !h.pbc[0];
    for (int c = 0; c < 3; c++) {
        // the two grids of a V-cycle; an image is one period away at most
        const int odd = !h.pbc[c];
        if (ig.pbc[c] != h.pbc[c] || ig.plo[c] != odd || ig.skip[c] != odd ||
            h.n[c] != 2 * ig.n[c] + odd || ig.n[c] < 4)
            return GH_ERR_UNSUPPORTED;
        g.u.n[c] = ig.n[c];
        g.u.pbc[c] = ig.pbc[c];
        g.u.plo[c] = g.u.skip[c] = odd;
        for (int j = 0; j < R; j++) {
            if (h.cm[c][j] != h.cp[c][j]) return GH_ERR_UNSUPPORTED;
            g.k[c][j] = (S)(alpha * h.cm[c][j]);
        }
    }
    // two sources: the 7-point Laplacians of the coarse levels
    if (ns == 2 && R != 1) return GH_ERR_UNSUPPORTED;
    // a vector that straddles the end of a periodic row has no place here
    if (h.pbc[2] && g.n2 % PT) return GH_ERR_UNSUPPORTED;
    uintptr_t bits = (uintptr_t)coarse | (uintptr_t)out;
    for (int q = 0; q < ns; q++) bits |= (uintptr_t)src[q];
    if (bits & (sizeof(S) - 1)) return GH_ERR_UNSUPPORTED;
    g.c0 = (S)(alpha * h.c0 + gamma);
    g.beta[0] = (S)beta[0];
    g.beta[1] = ns > 1 ? (S)beta[1] : (S)0;
    set_phases(g.u, phase_cd);
    const int nv = (g.n2 + PT - 1) / PT, ni = g.n0 / 2 + g.odd0;
    g.pitch = (nv + 2 * NW) * PT;
    auto lds_of = [&](int ty) { return 2 * (size_t)(ty + 2 * R) * g.pitch * sizeof(V); };
    auto comp_of = [&](int ty) { return (ty * nv + 63) / 64; };
    auto ghost_of = [&](int ty) {
        const int items = 2 * R * (nv + 2 * NW) + ty * 2 * NW;
        return (items + 64 * kGhostItems<V> - 1) / (64 * kGhostItems<V>);
    };
    int ncu = 0;
    const int crc = device_cu_count(&ncu);
    if (crc != GH_OK) return crc;
    // Rows and run: the pair with the least estimated time.  A block takes
    // lx + 4 steps of a fixed cost (latency and barrier, about the time of
    // 8 KB at a CU's share of the HBM rate) plus the bytes of two planes of
    // every block beside it on the CU.
    double best = 0;
    g.ty = 0;
    for (int ty = 1; ty <= g.n1; ty++) {
        const int threads = (comp_of(ty) + ghost_of(ty)) * 64;
        if (lds_of(ty) > kLdsBytes || threads > kMaxThreads) break;
        const int nyt = (g.n1 + ty - 1) / ty;
        const double fit = std::max(1, 1024 / threads), room = fit * ncu;
        const double bytes = (2.0 * (1 + ns) * ty + 0.5 * (ty + 2 * R)) * g.n2 * sizeof(V);
        for (int nxc = 1; nxc <= std::max(1, ni / 2); nxc += 1 + nxc / 8) {
            const int lx = (ni + nxc - 1) / nxc;
            const double blocks = (double)nbands * nyt * ((ni + lx - 1) / lx);
            const double rounds = std::ceil(blocks / room);
            const double t = rounds * (lx + 4) *
                             (std::min(fit, std::ceil(blocks / ncu)) * bytes + 8192.0);
            if (g.ty == 0 || t < best) {
                best = t;
                g.ty = ty;
                g.lx = lx;
            }
            if (rounds > 8) break;
        }
    }
    if (g.ty == 0) return GH_ERR_UNSUPPORTED;
    g.nyt = (g.n1 + g.ty - 1) / g.ty;
    g.nxc = (ni + g.lx - 1) / g.lx;
    g.ncomp = comp_of(g.ty);
    g.slot = (g.ty + 2 * R) * g.pitch;
    const int64_t nblocks = nbands * (int64_t)g.nyt * g.nxc;
    if (nblocks >= (1ll << 31)) return GH_ERR_UNSUPPORTED;
    const dim3 grid((unsigned)nblocks), block((g.ncomp + ghost_of(g.ty)) * 64);
    const size_t lds = lds_of(g.ty);
#define GH_GO(AL, NSRC)                                                                       \
    hipLaunchKernelGGL((stencil_interp_kernel<V, S, R, PT, AL, NSRC>), grid, block, lds, st,  \
                       (const V*)coarse, (V*)out, (const V*)src[0],                           \
                       (const V*)src[NSRC - 1], g)
    if (PT == 1 || g.n2 % PT == 0) {
        if (ns == 1) GH_GO(true, 1);
        else if constexpr (R == 1) GH_GO(true, 2);
    } else if constexpr (PT > 1) {
        if (ns == 1) GH_GO(false, 1);
        else if constexpr (R == 1) GH_GO(false, 2);
    }
#undef GH_GO
    GH_CHECK_LAUNCH();
    return GH_OK;
}

template <typename V, typename S>
int launch(const DirectStencil& h, const LinearMap& ig, const void* u, void* out, int64_t nb,
           const double* ph, int ns, const void* const* src, const double* beta, double al,
           double ga, hipStream_t st) {
    switch (h.R) {
        case 1: return launch_r<V, S, 1>(h, ig, u, out, nb, ph, ns, src, beta, al, ga, st);
        case 2: return launch_r<V, S, 2>(h, ig, u, out, nb, ph, ns, src, beta, al, ga, st);
        case 3: return launch_r<V, S, 3>(h, ig, u, out, nb, ph, ns, src, beta, al, ga, st);
    }
    return GH_ERR_UNSUPPORTED;
}

}  // namespace

int stencil_interp(const gh_stencil* h, const gh_transformer* intp, const void* u, void* out,
                   int64_t nb, const double* ph, int ns, const void* const* src,
                   const double* beta, double al, double ga, hipStream_t st) {
    DirectStencil d;
    LinearMap ig;
    const int dtype = stencil_dtype(h);
    if (!stencil_axes(h, &d) || !transformer_linear(intp, dtype, &ig) || !ig.interp) return GH_ERR_UNSUPPORTED;
    switch (dtype) {
        case GH_F64: return launch<double, double>(d, ig, u, out, nb, ph, ns, src, beta, al, ga, st);
        case GH_C128: return launch<cplx<double>, double>(d, ig, u, out, nb, ph, ns, src, beta, al, ga, st);
        case GH_F32: return launch<float, float>(d, ig, u, out, nb, ph, ns, src, beta, al, ga, st);
        case GH_C64: return launch<cplx<float>, float>(d, ig, u, out, nb, ph, ns, src, beta, al, ga, st);
    }
    return GH_ERR_UNSUPPORTED;
}

}  // namespace gh
