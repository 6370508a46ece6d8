// Restriction and interpolation with the short filter (nn = 1): every thread
// reads what its own points need and marches along x, no LDS, no barriers.
//
// The filters take 3 (restriction) or 2 points per axis, so that a block's
// threads share almost all of their reads through L1: 27 and 8 inputs per
// point cost less than staging.  Staged in LDS planes, as the long filters
// are (transformers.hip), each plane pays two barriers and an exposed load,
// 1.5 us, which small grids cannot hide.  us, staged and here (FP64, restriction
// r to or interpolation i from the given grid):
//   191 x 191 x 223 r 30.4 -> 14.0    95 x 95 x 111 i 26.9 -> 16.7
//   95 x 95 x 111 r   17.4 ->  5.1    47 x 47 x 55 i   9.3 ->  5.0
//   16 x 48^3 FP32 r   8.4 ->  7.3    16 x 24^3 FP32 i 8.5 ->  5.5
//   40 x 72 x 66 x 68 complex128 r 60 -> 35, i back 50 -> 46
//   64 x 56^3 i        227 -> 206     100 x 40 x 44 x 48 FP32 i 117 -> 94
// Some large calls stay staged (staged() in transformers.hip).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "internal.h"
#include "linear_interp.h"

namespace gh {

namespace {

constexpr int kMaxThreads = 256;

template <typename S>
struct LinArgs {
    LinGrid<S> g;                 // input grid
    int m[3];                     // output grid
    int lx, nxc, nblk;            // run along x, runs, blocks of a plane
    S alpha;
};

// Input values of one restricted point: 3 x 3 of a plane.
template <typename V> struct Nine { V v[3][3]; };

template <typename V, typename S>
__global__ void __launch_bounds__(kMaxThreads)
restrict_linear_kernel(const V* __restrict__ in, V* __restrict__ out, LinArgs<S> a) {
    constexpr bool CPLX = is_complex<V>::value;
    const LinGrid<S>& g = a.g;
    const int L = xcd_swizzle(blockIdx.x, gridDim.x);
    const int per = a.nblk * a.nxc, band = L / per, rem = L - band * per;
    const int xc = rem / a.nblk;
    const int npts = a.m[1] * a.m[2];
    // threads beyond the plane repeat its last point
    const int p = min((rem - xc * a.nblk) * (int)blockDim.x + (int)threadIdx.x, npts - 1);
    const int y = p / a.m[2], z = p - y * a.m[2];
    const size_t plane = (size_t)g.n[1] * g.n[2];
    const V* __restrict__ inb = in + (size_t)band * g.n[0] * plane;
    V* __restrict__ outb = out + (size_t)band * a.m[0] * npts;

    int row[3], col[3];
    unsigned zeros = 0, image = 0;   // bits r, 3 + k: zero; pairs (below, above): image
#pragma unroll
    for (int r = 0; r < 3; r++) {
        bool low, high, zero;
        row[r] = lin_wrap(2 * y - g.plo[1] + r, g.n[1], g.pbc[1], low, high, zero) * g.n[2];
        if (zero) zeros |= 1u << r;
        image |= (unsigned)low << (2 * r) | (unsigned)high << (2 * r + 1);
        col[r] = lin_wrap(2 * z - g.plo[2] + r, g.n[2], g.pbc[2], low, high, zero);
        if (zero) zeros |= 8u << r;
        image |= (unsigned)low << (2 * r + 6) | (unsigned)high << (2 * r + 7);
    }
    const bool zfix = !(g.pbc[1] && g.pbc[2]) && __any((int)zeros);
    const bool pfix = CPLX && g.yzphase && __any((int)image);
    auto filter = [](V lo, V mid, V hi) {
        return vscale(fma_rs((S)0.5, vadd(hi, lo), mid), (S)0.5);
    };
    auto load = [&](int c, Nine<V>& t) {
        bool low, high, zero;
        const V* pl = inb + lin_wrap(c, g.n[0], g.pbc[0], low, high, zero) * plane;
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
            for (int k = 0; k < 3; k++) t.v[r][k] = pl[row[r] + col[k]];
    };
    // plane c filtered along y and z
    auto make = [&](int c, Nine<V> t) {
        bool xlow, xhigh, xzero;
        lin_wrap(c, g.n[0], g.pbc[0], xlow, xhigh, xzero);
        if (zfix) {
#pragma unroll
            for (int r = 0; r < 3; r++)
#pragma unroll
                for (int k = 0; k < 3; k++)
                    if (zeros & (1u << r | 8u << k)) t.v[r][k] = vzero<V>();
        }
        if constexpr (CPLX) {
            if (pfix) {
#pragma unroll
                for (int r = 0; r < 3; r++) {
                    const bool l = image >> (2 * r) & 1, h = image >> (2 * r + 1) & 1;
                    const S pr = l ? g.re[1][1] : h ? g.re[1][0] : (S)1;
                    const S pi = l ? g.im[1][1] : h ? g.im[1][0] : (S)0;
#pragma unroll
                    for (int k = 0; k < 3; k++) {
                        const bool zl = image >> (2 * k + 6) & 1, zh = image >> (2 * k + 7) & 1;
                        t.v[r][k] = mul_phase(t.v[r][k], pr, pi);
                        t.v[r][k] = mul_phase(t.v[r][k], zl ? g.re[2][1] : zh ? g.re[2][0] : (S)1,
                                              zl ? g.im[2][1] : zh ? g.im[2][0] : (S)0);
                    }
                }
            }
        }
        V f[3];
#pragma unroll
        for (int k = 0; k < 3; k++) f[k] = filter(t.v[0][k], t.v[1][k], t.v[2][k]);
        V v = filter(f[0], f[1], f[2]);
        if (xzero) v = vzero<V>();
        if constexpr (CPLX)
            if (xlow || xhigh) v = mul_phase(v, g.re[0][xlow], g.im[0][xlow]);
        return v;
    };
    const int I0 = xc * a.lx, I1 = min(I0 + a.lx, a.m[0]);
    int c = 2 * I0 - g.plo[0];
    V* o = outb + (size_t)I0 * npts + p;
    Nine<V> t0, t1;
    load(c, t0);
    V f0 = make(c, t0);
    for (int I = I0; I < I1; I++, c += 2, o += npts) {
        load(c + 1, t0);
        load(c + 2, t1);
        const V f1 = make(c + 1, t0), f2 = make(c + 2, t1);
        *o = vscale(filter(f0, f1, f2), a.alpha);
        f0 = f2;
    }
}

// out = alpha I(in) or, with BASE, base + alpha I(in) (base may be out)
template <typename V, typename S, bool BASE>
__global__ void __launch_bounds__(kMaxThreads)
interpolate_linear_kernel(const V* __restrict__ in, V* out, const V* base, LinArgs<S> a) {
    constexpr int PT = 16 / (int)sizeof(V);
    typedef LinPoints<V, S, PT> Points;
    typedef typename Points::Vec Vec;
    typedef typename Points::Raw Raw;
    typedef Vec UVec __attribute__((aligned(sizeof(V))));
    constexpr int E = 16 / (int)sizeof(S), C = E / PT;
    const LinGrid<S>& g = a.g;
    const int L = xcd_swizzle(blockIdx.x, gridDim.x);
    const int per = a.nblk * a.nxc, band = L / per, rem = L - band * per;
    const int xc = rem / a.nblk;
    const int nv = (a.m[2] + PT - 1) / PT;
    const int p = (rem - xc * a.nblk) * (int)blockDim.x + (int)threadIdx.x;
    if (p >= a.m[1] * nv) return;
    const int y = p / nv, z = (p - y * nv) * PT;
    const bool part = z + PT > a.m[2];               // the row ends inside the vector
    const size_t plane = (size_t)a.m[1] * a.m[2];
    const V* __restrict__ inb = in + (size_t)band * g.n[0] * g.n[1] * g.n[2];
    const size_t off = (size_t)band * a.m[0] * plane + (size_t)y * a.m[2] + z;
    Points pts;
    pts.set(y, z, g);

    auto finish = [&](int x, Vec v) {
        if (x < 0 || x >= a.m[0]) return;
        const size_t gi = off + (size_t)x * plane;
        v *= a.alpha;
        if (!part) {
            if (BASE) v += (Vec)*reinterpret_cast<const UVec*>(base + gi);
            *reinterpret_cast<UVec*>(out + gi) = (UVec)v;
        } else {
#pragma unroll
            for (int e = 0; e < E; e++)
                if (z + e / C < a.m[2]) {
                    S s = v[e];
                    if (BASE) s += reinterpret_cast<const S*>(base + gi)[e];
                    reinterpret_cast<S*>(out + gi)[e] = s;
                }
        }
    };
    // fine planes 2 i - skip and the next belong to F_i
    const int first = g.skip[0] >> 1, last = (a.m[0] - 1 + g.skip[0]) >> 1;
    const int i0 = first + xc * a.lx, i1 = min(i0 + a.lx, last + 1);
    Raw r0, raw;
    pts.load(inb, i0, g, r0);
    pts.load(inb, i0 + 1, g, raw);
    Vec f = pts.make(r0, i0, g);
    for (int i = i0; i < i1; i++) {
        const Vec h = pts.make(raw, i + 1, g);
        if (i + 1 < i1) pts.load(inb, i + 2, g, raw);
        const int x = 2 * i - g.skip[0];
        finish(x, f);
        finish(x + 1, (f + h) * (S)0.5);
        f = h;
    }
}

template <typename V, typename S>
int launch(const LinearMap& h, const void* in, void* out, const void* base, int64_t nbands,
           const double* phase_cd, double alpha, hipStream_t st) {
    constexpr int PT = 16 / (int)sizeof(V);
    LinArgs<S> a;
    for (int c = 0; c < 3; c++) {
        a.g.n[c] = h.n[c];
        a.g.pbc[c] = h.pbc[c];
        a.g.plo[c] = h.plo[c];
        a.g.skip[c] = h.skip[c];
        a.m[c] = h.m[c];
    }
    set_phases(a.g, phase_cd);
    a.alpha = (S)alpha;
    int ncu = 0;
    const int crc = device_cu_count(&ncu);
    if (crc != GH_OK) return crc;
    const int64_t threads = (int64_t)h.m[1] * (h.interp ? (h.m[2] + PT - 1) / PT : h.m[2]);
    const int steps = h.interp ? ((h.m[0] - 1 + h.skip[0]) >> 1) - (h.skip[0] >> 1) + 1 : h.m[0];
    // Threads of a block: what leaves the fewest idle ones on a plane (8 x 8
    // points kept three waves of four idle); every halving counts 6 %, since
    // smaller blocks share fewer rows (us with 256 threads, with the fewest idle
    // ones at any price, and here: complex128, 5 x 112 x 92 x 112 with a general k
    // restricted 20, 26, 21; float64, 200 x 16^3 restricted 6.9, 3.7, 3.7).
    int tb = kMaxThreads;
    double least = 0;
    for (int t = kMaxThreads; t >= 64; t -= 64) {
        const double padded = (double)((threads + t - 1) / t * t) * (1.0 + 0.06 * std::log2((double)kMaxThreads / t));
        if (t == kMaxThreads || padded < least) {
            least = padded;
            tb = t;
        }
    }
    a.nblk = (int)((threads + tb - 1) / tb);
    // The run along x with the least estimated time.  A step takes the longer of
    // its latency and, at 0.18 of that for every wave beside it, the CU's
    // instructions and loads, and a tenth of the other; a run starts with half a
    // step; a CU holds 28 waves.  Constants that choose best among the measured
    // runs of 700 calls: 2 to 3 % above the fastest on average (3 and 7 % for a
    // full step at the start, six blocks per CU and latency alone).
    double best = 0;
    const double waves = tb / 64, fit = std::floor(28 / waves);
    const double per_room = 1.0 / (ncu * fit), per_cu = 1.0 / ncu;
    for (int nxc = 1; nxc <= steps; nxc += 1 + nxc / 8) {
        const int lx = (steps + nxc - 1) / nxc;
        const double blocks = (double)nbands * a.nblk * ((steps + lx - 1) / lx);
        const double rounds = std::ceil(blocks * per_room - 1e-9);
        const double busy = 0.18 * waves * std::min(fit, std::ceil(blocks * per_cu - 1e-9));
        // (blocks of later rounds start as those of earlier ones end)
        const double t = (0.6 * std::max(1.0, blocks * per_room) + 0.4 * rounds) * (lx + 0.5) *
                         (std::max(busy, 1.0) + 0.1 * std::min(busy, 1.0));
        if (nxc == 1 || t < best) {
            best = t;
            a.lx = lx;
        }
        if (rounds > 16) break;
    }
    a.nxc = (steps + a.lx - 1) / a.lx;
    const int64_t nblocks = nbands * (int64_t)a.nblk * a.nxc;
    GH_REQUIRE(nblocks < (1ll << 31), GH_ERR_SHAPE, "transformer: too many blocks");
    const dim3 grid((unsigned)nblocks), block(tb);
    if (!h.interp)
        hipLaunchKernelGGL((restrict_linear_kernel<V, S>), grid, block, 0, st, (const V*)in,
                           (V*)out, a);
    else if (base)
        hipLaunchKernelGGL((interpolate_linear_kernel<V, S, true>), grid, block, 0, st,
                           (const V*)in, (V*)out, (const V*)base, a);
    else
        hipLaunchKernelGGL((interpolate_linear_kernel<V, S, false>), grid, block, 0, st,
                           (const V*)in, (V*)out, (const V*)nullptr, a);
    GH_CHECK_LAUNCH();
    return GH_OK;
}

}  // namespace

int linear_map(int dtype, const LinearMap& h, const void* in, void* out, const void* base,
               int64_t nb, const double* ph, double al, hipStream_t st) {
    switch (dtype) {
        case GH_F64: return launch<double, double>(h, in, out, base, nb, ph, al, st);
        case GH_C128: return launch<cplx<double>, double>(h, in, out, base, nb, ph, al, st);
        case GH_F32: return launch<float, float>(h, in, out, base, nb, ph, al, st);
        case GH_C64: return launch<cplx<float>, float>(h, in, out, base, nb, ph, al, st);
    }
    set_error("transformer: bad dtype");
    return GH_ERR_ARG;
}

}  // namespace gh
