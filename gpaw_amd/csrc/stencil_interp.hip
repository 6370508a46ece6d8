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

namespace gh {

namespace {

constexpr int kMaxThreads = 1024;
constexpr size_t kLdsBytes = 64 * 1024;
// ghost vectors per thread of a ghost wave (complex128: registers)
template <typename V> constexpr int kGhostItems = sizeof(V) > 8 ? 2 : 4;

template <typename S, int R>
struct InterpArgs {
    int nc0, nc1, nc2;            // coarse grid
    int n0, n1, n2;               // fine grid
    int pbc0, pbc1, pbc2;
    int odd0, odd1, odd2;         // zero boundaries: fine point 0 is odd
    int ty, lx, nyt, nxc;         // rows and coarse planes of a block
    int ncomp;                    // compute waves
    int pitch, slot;              // elements per LDS row, plane
    int yzphase;
    S c0, k[3][R];
    S beta[2];
    S re[3][2], im[3][2];
};

// One vector of PT fine points: where its coarse values are.
template <int NC>
struct Item {
    int row[2], z[NC];            // coarse row starts, coarse z
    unsigned flags;               // see below
    int lds;
};
// flag bits: 0 fine row between two coarse rows, 1 fine z likewise (PT = 1);
// 2, 3 row r lies beyond a zero boundary; 4.. the same for z; from 8 on two
// bits (below, above) for each row and z that is a periodic image
constexpr unsigned kOddY = 1, kOddZ = 2;
constexpr unsigned zero_bits(int nc) { return 0xCu | (((1u << nc) - 1) << 4); }

template <typename V, typename S, int R, int PT, bool ALIGNED, int NS>
__global__ void __launch_bounds__(kMaxThreads)
stencil_interp_kernel(const V* __restrict__ coarse, V* __restrict__ out,
                      const V* __restrict__ src0, const V* __restrict__ src1,
                      InterpArgs<S, R> g) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    V* lds = reinterpret_cast<V*>(smem_raw);
    constexpr bool CPLX = is_complex<V>::value;
    typedef S Vec __attribute__((ext_vector_type(16 / sizeof(S))));
    typedef Vec UVec __attribute__((aligned(sizeof(V))));
    constexpr int E = 16 / (int)sizeof(S), C = E / PT;
    static_assert(C * sizeof(S) == sizeof(V), "points per vector");
    constexpr int NC = PT == 1 ? 2 : PT / 2 + 1;     // coarse values per row
    constexpr int NW = (R + PT - 1) / PT;            // ghost vectors per side
    typedef Item<NC> It;
    struct Raw { V v[2][NC]; };

    const int tiles = g.nyt * g.nxc;
    const int L = xcd_swizzle(blockIdx.x, gridDim.x);
    const int band = L / tiles, tile = L - band * tiles;
    const int xc = tile / g.nyt, yt = tile - xc * g.nyt;
    const int y0 = yt * g.ty, tye = min(g.ty, g.n1 - y0);
    const int ni = g.n0 / 2 + g.odd0;                // pairs of fine planes
    const int i0 = xc * g.lx, i1 = min(i0 + g.lx, ni);
    const int cplane = g.nc1 * g.nc2;
    const V* __restrict__ cb = coarse + (size_t)band * g.nc0 * cplane;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nv = (g.n2 + PT - 1) / PT;

    // coarse index of a periodic image or beyond a zero boundary
    auto wrap = [](int& c, int n, int pbc, bool& low, bool& high, bool& zero) {
        low = c < 0;
        high = c >= n;
        zero = (low || high) && !pbc;
        if (pbc) c += low ? n : high ? -n : 0;
        else c = min(max(c, 0), n - 1);
    };
    auto make_item = [&](int y, int z, int ldspos) {
        It it;
        it.flags = 0;
        it.lds = ldspos;
        const int qy = y + g.odd1, cy = (qy >> 1) - g.odd1;
        if (qy & 1) it.flags |= kOddY;
#pragma unroll
        for (int r = 0; r < 2; r++) {
            int c = cy + ((qy & 1) ? r : 0);
            bool low, high, zero;
            wrap(c, g.nc1, g.pbc1, low, high, zero);
            it.row[r] = c * g.nc2;
            if (zero) it.flags |= 4u << r;
            it.flags |= (unsigned)low << (8 + 2 * r) | (unsigned)high << (9 + 2 * r);
        }
        const int qz = z + g.odd2, cz = (qz >> 1) - g.odd2;
        if (PT == 1 && (qz & 1)) it.flags |= kOddZ;
#pragma unroll
        for (int k = 0; k < NC; k++) {
            int c = cz + (PT == 1 && !(qz & 1) ? 0 : k);
            bool low, high, zero;
            wrap(c, g.nc2, g.pbc2, low, high, zero);
            it.z[k] = c;
            if (zero) it.flags |= 16u << k;
            it.flags |= (unsigned)low << (12 + 2 * k) | (unsigned)high << (13 + 2 * k);
        }
        return it;
    };
    // coarse plane of F_i: its image inside the grid
    auto plane_ptr = [&](int i) {
        int c = i - g.odd0;
        if (g.pbc0) c += c < 0 ? g.nc0 : c >= g.nc0 ? -g.nc0 : 0;
        else c = min(max(c, 0), g.nc0 - 1);
        return cb + (size_t)c * cplane;
    };
    auto load = [&](const It& it, int i, Raw& raw) {
        const V* p = plane_ptr(i);
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int k = 0; k < NC; k++) raw.v[r][k] = p[it.row[r] + it.z[k]];
    };
    const bool zeros = !(g.pbc1 && g.pbc2);
    auto half = [](V a, V b) { return vscale(vadd(a, b), (S)0.5); };
    // F_i at the item's points
    auto make = [&](const It& it, int i, Raw raw) {
        if (zeros && __any((int)(it.flags & zero_bits(NC)))) {
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int k = 0; k < NC; k++)
                    if (it.flags & (4u << r | 16u << k)) raw.v[r][k] = vzero<V>();
        }
        if constexpr (CPLX) {
            if (g.yzphase && __any((int)(it.flags >> 8))) {
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    const bool l = it.flags >> (8 + 2 * r) & 1, h = it.flags >> (9 + 2 * r) & 1;
                    const S pr = l ? g.re[1][1] : h ? g.re[1][0] : (S)1;
                    const S pi = l ? g.im[1][1] : h ? g.im[1][0] : (S)0;
#pragma unroll
                    for (int k = 0; k < NC; k++) {
                        const bool zl = it.flags >> (12 + 2 * k) & 1,
                                   zh = it.flags >> (13 + 2 * k) & 1;
                        raw.v[r][k] = mul_phase(raw.v[r][k], pr, pi);
                        raw.v[r][k] = mul_phase(raw.v[r][k],
                                                zl ? g.re[2][1] : zh ? g.re[2][0] : (S)1,
                                                zl ? g.im[2][1] : zh ? g.im[2][0] : (S)0);
                    }
                }
            }
        }
        V f[2][PT];
#pragma unroll
        for (int r = 0; r < 2; r++) {
            if constexpr (PT == 1) {
                f[r][0] = it.flags & kOddZ ? half(raw.v[r][0], raw.v[r][1]) : raw.v[r][0];
            } else {
#pragma unroll
                for (int e = 0; e < PT; e += 2) {
                    const V m = half(raw.v[r][e / 2], raw.v[r][e / 2 + 1]);
                    f[r][e] = g.odd2 ? m : raw.v[r][e / 2];
                    f[r][e + 1] = g.odd2 ? raw.v[r][e / 2 + 1] : m;
                }
            }
        }
        V o[PT];
        const int c = i - g.odd0;
        const bool xlow = c < 0, xhigh = c >= g.nc0;
#pragma unroll
        for (int e = 0; e < PT; e++) {
            o[e] = it.flags & kOddY ? half(f[0][e], f[1][e]) : f[0][e];
            if (!g.pbc0 && (xlow || xhigh)) o[e] = vzero<V>();
            if constexpr (CPLX)
                if (xlow || xhigh) o[e] = mul_phase(o[e], g.re[0][xlow], g.im[0][xlow]);
        }
        Vec v;
        __builtin_memcpy(&v, o, sizeof(v));
        return v;
    };
    auto put = [&](const It& it, int i, Vec v) {
        *reinterpret_cast<Vec*>(lds + (i & 1) * g.slot + it.lds) = v;
    };

    if (wave >= g.ncomp) {
        // ---------------------------------------------------- ghosts --
        const int nt = blockDim.x - g.ncomp * 64, t = threadIdx.x - g.ncomp * 64;
        const int rowvec = nv + 2 * NW;                       // vectors per LDS row
        const int nrow = 2 * R * rowvec, n = nrow + tye * 2 * NW;
        constexpr int GI = kGhostItems<V>;
        It it[GI];
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
            it[a] = make_item(y0 - R + r, (c - NW) * PT, r * g.pitch + c * PT);
        }
        auto all = [&](int i) {
#pragma unroll
            for (int a = 0; a < GI; a++) load(it[a], i, raw[a]);
        };
        auto store = [&](int i) {
#pragma unroll
            for (int a = 0; a < GI; a++) put(it[a], i, make(it[a], i, raw[a]));
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
    const It it = make_item(y0 + yl, z, (yl + R) * g.pitch + (NW * PT + z));
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
        const V* p = lds + (i & 1) * g.slot + it.lds;
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
        for (int a = 0; a < 4; a++) load(it, i0 - 2 + a, r[a]);
#pragma unroll
        for (int a = 0; a < 4; a++) f[a] = make(it, i0 - 2 + a, r[a]);
    }
    put(it, i0, f[2]);
    put(it, i0 + 1, f[3]);
    Raw raw;
    load(it, i0 + 2, raw);
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
        f[4] = make(it, i + 2, raw);
        put(it, i + 2, f[4]);
        load(it, i + 3, raw);
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
int launch_r(const DirectStencil& h, const InterpGrid& ig, const void* coarse, void* out,
             int64_t nbands, const double* phase_cd, int ns, const void* const* src,
             const double* beta, double alpha, double gamma, hipStream_t st) {
    constexpr int PT = 16 / (int)sizeof(V), NW = (R + PT - 1) / PT;
    InterpArgs<S, R> g;
    g.nc0 = ig.n[0]; g.nc1 = ig.n[1]; g.nc2 = ig.n[2];
    g.n0 = h.n[0]; g.n1 = h.n[1]; g.n2 = h.n[2];
    g.pbc0 = h.pbc[0]; g.pbc1 = h.pbc[1]; g.pbc2 = h.pbc[2];
    g.odd0 = !g.pbc0; g.odd1 = !g.pbc1; g.odd2 = !g.pbc2;
    for (int c = 0; c < 3; c++) {
        // the two grids of a V-cycle; an image is one period away at most
        const int odd = !h.pbc[c];
        if (ig.pbc[c] != h.pbc[c] || ig.plo[c] != odd || ig.skip[c] != odd ||
            h.n[c] != 2 * ig.n[c] + odd || ig.n[c] < 4)
            return GH_ERR_UNSUPPORTED;
        for (int j = 0; j < R; j++) {
            if (h.cm[c][j] != h.cp[c][j]) return GH_ERR_UNSUPPORTED;
            g.k[c][j] = (S)(alpha * h.cm[c][j]);
        }
    }
    // two sources: the 7-point Laplacians of the coarse levels
    if (ns == 2 && R != 1) return GH_ERR_UNSUPPORTED;
    // a vector that straddles the end of a periodic row has no place here
    if (g.pbc2 && g.n2 % PT) return GH_ERR_UNSUPPORTED;
    uintptr_t bits = (uintptr_t)coarse | (uintptr_t)out;
    for (int q = 0; q < ns; q++) bits |= (uintptr_t)src[q];
    if (bits & (sizeof(S) - 1)) return GH_ERR_UNSUPPORTED;
    g.c0 = (S)(alpha * h.c0 + gamma);
    g.beta[0] = (S)beta[0];
    g.beta[1] = ns > 1 ? (S)beta[1] : (S)0;
    const Phases ph = make_phases(phase_cd);
    g.yzphase = 0;
    for (int c = 0; c < 3; c++)
        for (int d = 0; d < 2; d++) {
            g.re[c][d] = (S)ph.re[c][d];
            g.im[c][d] = (S)ph.im[c][d];
            if (c > 0 && (g.re[c][d] != (S)1 || g.im[c][d] != (S)0)) g.yzphase = 1;
        }
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
int launch(const DirectStencil& h, const InterpGrid& ig, const void* u, void* out, int64_t nb,
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
    InterpGrid ig;
    const int dtype = stencil_dtype(h);
    if (!stencil_axes(h, &d) || !transformer_interp(intp, dtype, &ig)) return GH_ERR_UNSUPPORTED;
    switch (dtype) {
        case GH_F64: return launch<double, double>(d, ig, u, out, nb, ph, ns, src, beta, al, ga, st);
        case GH_C128: return launch<cplx<double>, double>(d, ig, u, out, nb, ph, ns, src, beta, al, ga, st);
        case GH_F32: return launch<float, float>(d, ig, u, out, nb, ph, ns, src, beta, al, ga, st);
        case GH_C64: return launch<cplx<float>, float>(d, ig, u, out, nb, ph, ns, src, beta, al, ga, st);
    }
    return GH_ERR_UNSUPPORTED;
}

}  // namespace gh
