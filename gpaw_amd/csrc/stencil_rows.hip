// Finite-difference stencils along the grid axes: an LDS ring of x-planes, for
// rows of any length and alignment, every element type, boundary and Bloch
// phase (radius 1 to 6).
//
// A block owns one band, a tile of ty full (y, z) rows and a run of
// x-planes.  Loader wavefronts stream the tile's rows and its 2R ghost rows
// HBM -> LDS by DMA as contiguous runs, D planes ahead in a ring of R + D + 1
// slots: 16 bytes per lane where the rows are 16-byte aligned, else 4.  The
// instruction issue of these few waves is what limits a tile, so their loop
// is one address and four instructions per 4 x 64 lanes (rows with padding,
// one address and mask per row, took 1.7 to 3 times as long), and they run
// at a raised priority.  A compute thread owns PT z-adjacent points (16
// bytes), keeps the x queue in registers and reads its y and z neighbours
// from LDS.  The march has no divergent branch: z neighbours beyond the row
// are read at wrapped offsets worked out once, or selected away at zero
// boundaries, and phases are multiplied in where a wave has such lanes (with
// a separate path for edge lanes every wave ran both: complex64 at 96^3
// 567 -> 382 us for this alone).
//
// HBM bound for many bands (psi read, result written; ghost rows from L2).
// T + v, R = 3, us, against the ring with one point per thread for complex
// phases, its register-queue fallback for odd rows and fixed 16-row tiles:
//   256 x 112^3 float64           1355 -> 1262  (copy of the bytes: 1128; 1390 -> 1297
//                                 between the other kernels of an H psi)
//   64 x 96^3 float64              295 ->  195  (178)
//   48 x 95 x 95 x 103, zero bc    418 ->  194  (140)
//   128 x 96^3 complex64, k along x  580 -> 382, general k 1046 -> 411 (355)
//   64 x 72 x 80 x 90 complex128, general k   465 -> 272  (208)
//   256 x 112^3 float32            712 ->  632  (564)
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "internal.h"

namespace gh {

namespace {

// Radii above 3 need up to 235 registers: half the threads, without scratch.
// T + v, R = 4 and 6, us, the kernel without LDS and here: 64 x 96^3 float64 554
// -> 391, 758 -> 334; 32 x 96^3 complex128, general k 1011 -> 386, 1436 -> 1434;
// 64 x 64^3 complex128, k along x 587 -> 252, 737 -> 370.
template <int R> constexpr int kMaxThreads = R > 3 ? 512 : 1024;
constexpr size_t kLdsBytes = 160 * 1024;
constexpr int kDepth = 2;         // planes in flight

template <typename S, int R>
struct RowsArgs {
    int n0, n1, n2;
    int pbc0, pbc1, pbc2;
    int ty, lx, nyt, nxc;
    int ncomp, lw;         // compute waves; loader waves per plane in flight
    int slot;              // elements per ring slot
    int nv_points;         // points of the row's vectors: n2 rounded up
    int wide;              // 16-byte DMA
    int yphase, zphase;    // complex data with a y / z Bloch phase
    int bgroup, nbands;
    S c0;
    S km[3][R], kp[3][R];  // coefficients of the offsets -(j + 1), +(j + 1)
    S re[3][2], im[3][2];
    const double* eps;
};

__device__ __forceinline__ void barrier_only() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}
__device__ __forceinline__ void wait_vm0() {
    __builtin_amdgcn_s_waitcnt(0x0F70);          // vmcnt(0)
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}
// One DMA instruction per lane of BYTES bytes; OFF counts on both sides.
template <int BYTES, int OFF>
__device__ __forceinline__ void dma(const char* s, char* d) {
    auto* l = (__attribute__((address_space(3))) void*)d;
    if constexpr (BYTES == 16) __builtin_amdgcn_global_load_lds((const void*)s, l, 16, OFF, 0);
    else __builtin_amdgcn_global_load_lds((const void*)s, l, 4, OFF, 0);
}

// nbytes HBM -> LDS; all but the lane's own offset is wave-uniform
template <int BYTES>
__device__ __forceinline__ void dma_run(const char* s, char* d, int nbytes, int lane) {
    constexpr int STEP = 64 * BYTES;
    s += lane * BYTES;
    int left = nbytes;
    for (; left >= 4 * STEP; left -= 4 * STEP) {
        dma<BYTES, 0>(s, d);
        dma<BYTES, STEP>(s, d);
        dma<BYTES, 2 * STEP>(s, d);
        dma<BYTES, 3 * STEP>(s, d);
        s += 4 * STEP;
        d += 4 * STEP;
    }
    for (left -= lane * BYTES; left > 0; left -= STEP) {
        dma<BYTES, 0>(s, d);
        s += STEP;
        d += STEP;
    }
}

// N contiguous elements at element alignment
template <int N, typename V>
__device__ __forceinline__ void load_n(const V* p, V* v) {
    __builtin_memcpy(v, p, N * sizeof(V));
}

// ALIGNED: n2 is a multiple of PT, so every vector of a slot is 16-byte
// aligned (FP32 gains most: one 16-byte LDS read instead of two of 8 bytes).
// SYM: the coefficients of +j and -j are equal along every axis (every
// Laplacian), so half of them are live.
template <typename V, typename S, int R, int PT, bool ALIGNED, bool SYM, bool HAS_V,
          bool HAS_SRC>
__global__ void __launch_bounds__(kMaxThreads<R>)
stencil_rows_kernel(const V* __restrict__ in, V* __restrict__ out, const S* __restrict__ vt,
                    const V* src, S beta, RowsArgs<S, R> g) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    V* ring = reinterpret_cast<V*>(smem_raw);
    constexpr bool CPLX = is_complex<V>::value;
    constexpr int D = kDepth, P = R + D + 1;
    const int n2 = g.n2;
    // logical tiles of one XCD are contiguous, all tiles of a few bands
    // running together (shared ghost rows and potential in its L2)
    int band, xc, yt;
    {
        const int L = xcd_swizzle(blockIdx.x, gridDim.x);
        const int tiles = g.nyt * g.nxc, per = g.bgroup * tiles;
        const int grp = L / per;
        const int bg = min(g.bgroup, g.nbands - grp * g.bgroup);
        const int rem = L - grp * per, tile = rem / bg;
        band = grp * g.bgroup + rem - tile * bg;
        xc = tile / g.nyt;
        yt = tile - xc * g.nyt;
    }
    const int y0 = yt * g.ty, tye = min(g.ty, g.n1 - y0);
    const int x0 = xc * g.lx, x1 = min(x0 + g.lx, g.n0);
    const int rows = tye + 2 * R;
    const int slot = g.slot;
    const size_t plane = (size_t)g.n1 * n2;
    const V* __restrict__ inb = in + band * plane * g.n0;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;

    // rows beyond a zero y boundary: zero once, in every slot (nothing writes
    // there afterwards)
    if (!g.pbc1 && (y0 < R || y0 + tye + R > g.n1)) {
        for (int sl = 0; sl < P; sl++)
            for (int r = wave; r < rows; r += blockDim.x >> 6) {
                const int y = y0 - R + r;
                if (y >= 0 && y < g.n1) continue;
                for (int c = lane; c < n2; c += 64) ring[sl * slot + r * n2 + c] = vzero<V>();
            }
        __syncthreads();
    }

    if (wave >= g.ncomp) {
        // ---------------------------------------------------- loader --
        __builtin_amdgcn_s_setprio(3);
        const int w = (wave - g.ncomp) / g.lw, l = (wave - g.ncomp) % g.lw;
        // up to three runs of rows: beyond y = 0 (periodic image), inside,
        // beyond n1 - 1; this wave's share of each, in 16-byte steps
        const int ylo = y0 - R, rbytes = n2 * (int)sizeof(V);
        const int in0 = max(0, -ylo), in1 = min(rows, g.n1 - ylo);
        auto run = [&](const char* pl, char* dst, int r0, int r1, int yshift) {
            const int bytes = (r1 - r0) * rbytes;
            const int per = (bytes / g.lw + 15) & ~15;
            const int b0 = min(bytes, l * per), b1 = l + 1 == g.lw ? bytes : min(bytes, b0 + per);
            const char* s = pl + (int64_t)(ylo + r0 + yshift) * rbytes + b0;
            char* d = dst + r0 * rbytes + b0;
            if (g.wide) dma_run<16>(s, d, b1 - b0, lane);
            else dma_run<4>(s, d, b1 - b0, lane);
        };
        auto issue = [&](int xp) {
            int xs = xp;
            if (xs >= g.n0) {
                if (!g.pbc0) return;
                xs -= g.n0;
            }
            const char* pl = reinterpret_cast<const char*>(inb + xs * plane);
            char* dst = reinterpret_cast<char*>(ring + ((xp - x0) % P) * slot);
            if (g.pbc1 && in0 > 0) run(pl, dst, 0, in0, g.n1);
            run(pl, dst, in0, in1, 0);
            if (g.pbc1 && rows > in1) run(pl, dst, in1, rows, -g.n1);
        };
        const int xend = x1 + R;                  // planes [x0, xend)
        for (int xp = x0 + w; xp <= x0 + R; xp += D) issue(xp);
        wait_vm0();
        // one plane per loader in flight from here on
        for (int xp = x0 + R + 1; xp < x0 + R + D; xp++)
            if (xp < xend && (xp - x0) % D == w) issue(xp);
        for (int x = x0; x < x1; x++) {
            const bool mine = (x + R - x0) % D == w;
            if (mine && x > x0) wait_vm0();
            barrier_only();
            if (mine && x + R + D < xend) issue(x + R + D);
        }
        return;
    }

    // ------------------------------------------------------ compute --
    typedef S Vec __attribute__((ext_vector_type(16 / sizeof(S))));   // PT points
    typedef Vec UVec __attribute__((aligned(sizeof(V))));              // any row
    constexpr int E = 16 / (int)sizeof(S), C = E / PT;   // scalars per vector, point
    static_assert(C * sizeof(S) == sizeof(V), "points per vector");
    const int nv = (n2 + PT - 1) / PT;
    const bool act = (int)threadIdx.x < tye * nv;
    const int pp = act ? threadIdx.x : 0;
    const int yl = pp / nv, z = (pp - yl * nv) * PT;
    // a row that ends inside its last vector: loads move down to end at the
    // row's end and the values are shifted back (`short_by` points)
    const bool part = !ALIGNED && z + PT > n2;
    const int short_by = ALIGNED ? 0 : g.nv_points - n2;
    const int yz = (y0 + yl) * n2 + z;
    const S c0b = g.eps ? g.c0 - (S)g.eps[band] : g.c0;
    V* __restrict__ outb = out + band * plane * g.n0;
    const V* srcb = HAS_SRC ? src + band * plane * g.n0 : nullptr;

    const int down = part ? short_by : 0;
    auto load_points = [&](const V* p) {          // own points, any alignment
        return (Vec)*reinterpret_cast<const UVec*>(p - down);
    };
    auto shifted = [&](Vec v) {
        if constexpr (!ALIGNED) {
            if (short_by == 0) return v;
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
    auto x_phase = [&](Vec v, int d) {
        if constexpr (CPLX) {
            const S pr = g.re[0][d], pi = g.im[0][d];
#pragma unroll
            for (int i = 0; i < PT; i++) {
                const S a = v[2 * i], b = v[2 * i + 1];
                v[2 * i] = a * pr - b * pi;
                v[2 * i + 1] = a * pi + b * pr;
            }
        }
        return v;
    };
    auto plane_points = [&](int x) {              // x in [-n0, n0)
        if (x >= 0) return shifted(load_points(inb + x * plane + yz));
        if (!g.pbc0) return Vec(0);
        return x_phase(shifted(load_points(inb + (x + g.n0) * plane + yz)), 1);
    };
    Vec q[2 * R + 1];
#pragma unroll
    for (int j = 0; j < R; j++) q[j] = plane_points(x0 - R + j);
    // the coefficients live in VGPRs (uniform, but the scalar file is full
    // here); complex128 and two sets have none to spare for them
    constexpr bool kPin = sizeof(V) < 16 && SYM;
    S k0 = c0b, km[3][R], kp[3][R];
    if (kPin) asm volatile("" : "+v"(k0));
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
        for (int j = 0; j < R; j++) {
            km[c][j] = g.km[c][j];
            if (kPin) asm volatile("" : "+v"(km[c][j]));
            kp[c][j] = SYM ? km[c][j] : g.kp[c][j];
        }
    const V* own = ring + (yl + R) * n2 + z;
    auto slot_of = [&](int xp) { return own + ((xp - x0) % P) * slot; };
    auto read_own = [&](const V* p) {
        Vec v;
        if constexpr (ALIGNED) v = *reinterpret_cast<const Vec*>(p);
        else __builtin_memcpy(&v, p, sizeof(v));
        return v;
    };
    // rows y -+ (j + 1) beyond a periodic y face (bit j, R + j) need a phase
    unsigned ylow = 0, yhigh = 0;
#pragma unroll
    for (int j = 0; j < R; j++) {
        if (y0 + yl - 1 - j < 0) ylow |= 1u << j;
        if (y0 + yl + 1 + j >= g.n1) yhigh |= 1u << j;
    }
    const bool yfix = CPLX && g.yphase && __any((int)(ylow | yhigh));
    auto phase = [&](Vec v, int c, bool low, bool high) {
        if constexpr (CPLX) {
            const S pr = low ? g.re[c][1] : high ? g.re[c][0] : (S)1;
            const S pi = low ? g.im[c][1] : high ? g.im[c][0] : (S)0;
            const bool image = low || high;      // see mul_phase_of
#pragma unroll
            for (int i = 0; i < PT; i++) {
                const S a = v[2 * i], b = v[2 * i + 1];
                v[2 * i] = a * pr - (image ? b : (S)0) * pi;
                v[2 * i + 1] = (image ? a : (S)0) * pi + b * pr;
            }
        }
        return v;
    };
    // aligned rows: the NW vectors below and above, wrapped, and which of
    // them lie beyond the row
    constexpr int NW = (R + PT - 1) / PT;
    int zo[2 * NW];
    unsigned zout = 0;
#pragma unroll
    for (int i = 0; i < 2 * NW; i++) {
        zo[i] = (i < NW ? i - NW : i - NW + 1) * PT;
        if (z + zo[i] < 0 || z + zo[i] >= n2) {
            zout |= 1u << i;
            zo[i] += i < NW ? n2 : -n2;
        }
    }
    const bool zfix = (!g.pbc2 || (CPLX && g.zphase)) && __any((int)zout);
    // other periodic rows: every point of the window and the thread's own
    // points from the second on, wrapped singly
    int eo[2 * R + PT];
#pragma unroll
    for (int j = 0; j < 2 * R + PT - 1; j++) {
        eo[j] = j < R ? j - R : j < 2 * R ? PT + j - R : j - 2 * R + 1;
        if (z + eo[j] < 0) eo[j] += n2;
        else if (z + eo[j] >= n2) eo[j] = min(eo[j] - n2, n2 - 1 - z);
    }
    auto z_ghost = [&](V v, int zz) {
        if (!CPLX || !g.zphase) return v;
        const bool low = zz < 0, high = zz >= n2;
        return mul_phase_of(low || high, v, low ? g.re[2][1] : high ? g.re[2][0] : (S)1,
                            low ? g.im[2][1] : high ? g.im[2][0] : (S)0);
    };
    barrier_only();
#pragma unroll
    for (int j = 0; j < R; j++) {                 // the first planes of the run
        const int xp = x0 + j;
        Vec v = read_own(slot_of(xp));
        if (xp >= g.n0) v = g.pbc0 ? x_phase(v, 0) : Vec(0);
        q[R + j] = v;
    }
    for (int x = x0; x < x1; x++) {
        if (x > x0) barrier_only();
        {
            const int xp = x + R;
            Vec v = read_own(slot_of(xp));
            if (xp >= g.n0) v = g.pbc0 ? x_phase(v, 0) : Vec(0);
            q[2 * R] = v;
        }
        const size_t gi = (size_t)x * plane + yz;
        struct Pot { S v[PT]; } pot;
        Vec ss;
        if (HAS_V) __builtin_memcpy(&pot, vt + gi - down, sizeof(pot));
        if (HAS_SRC) ss = load_points(srcb + gi);
        const V* sl = slot_of(x);
        Vec acc = q[R] * k0;
        auto add_pair = [&](int c, int j, Vec a, Vec b) {   // offsets -+(j + 1) along c
            if constexpr (SYM) acc = (a + b) * km[c][j] + acc;
            else acc = b * kp[c][j] + (a * km[c][j] + acc);
        };
#pragma unroll
        for (int j = 0; j < R; j++) add_pair(0, j, q[R - 1 - j], q[R + 1 + j]);
        if (!yfix) {
#pragma unroll
            for (int j = 0; j < R; j++)
                add_pair(1, j, read_own(sl - (1 + j) * n2), read_own(sl + (1 + j) * n2));
        } else {
#pragma unroll
            for (int j = 0; j < R; j++)
                add_pair(1, j, phase(read_own(sl - (1 + j) * n2), 1, (ylow >> j) & 1, false),
                         phase(read_own(sl + (1 + j) * n2), 1, false, (yhigh >> j) & 1));
        }
        // z: each branch adds its own terms, so that only the sums live on
        auto add_z = [&](const V* lo, const V* mid, const V* hi) {
            // scalar e of z - R .. z + PT - 1 + R
            struct { S v[R * C]; } l, h;
            struct { S v[E]; } m;
            __builtin_memcpy(&l, lo, sizeof(l));
            __builtin_memcpy(&m, mid, sizeof(m));
            __builtin_memcpy(&h, hi, sizeof(h));
            auto we = [&](int e) {
                return e < R * C ? l.v[e] : e < R * C + E ? m.v[e - R * C] : h.v[e - E - R * C];
            };
#pragma unroll
            for (int e = 0; e < E; e++)
#pragma unroll
                for (int j = 0; j < R; j++) {
                    const S a = we(R * C + e - (j + 1) * C), b = we(R * C + e + (j + 1) * C);
                    if constexpr (SYM) acc[e] = fma_rs(km[2][j], a + b, acc[e]);
                    else acc[e] = fma_rs(kp[2][j], b, fma_rs(km[2][j], a, acc[e]));
                }
        };
        V mid[PT];
        __builtin_memcpy(mid, &q[R], sizeof(mid));
        if constexpr (ALIGNED) {
            // whole vectors on both sides, wrapped into the row
            Vec t[2 * NW];
#pragma unroll
            for (int i = 0; i < 2 * NW; i++) t[i] = read_own(sl + zo[i]);
            if (zfix) {
#pragma unroll
                for (int i = 0; i < 2 * NW; i++) {
                    const bool out = (zout >> i) & 1;
                    if (!g.pbc2) t[i] = out ? Vec(0) : t[i];
                    else t[i] = phase(t[i], 2, out && i < NW, out && i >= NW);
                }
            }
            struct { V v[NW * PT]; } l, h;
            __builtin_memcpy(&l, t, sizeof(l));
            __builtin_memcpy(&h, t + NW, sizeof(h));
            add_z(l.v + NW * PT - R, mid, h.v);
        } else {
            // lo: z - R .. z - 1, hi: z + PT ..; mid's points beyond the row's
            // end are ghosts as well
            V lo[R], hi[R];
            if (!g.pbc2) {
                load_n<R>(sl - R, lo);
                load_n<R>(sl + PT, hi);
#pragma unroll
                for (int j = 0; j < R; j++) {
                    lo[j] = z - R + j < 0 ? vzero<V>() : lo[j];
                    hi[j] = z + PT + j >= n2 ? vzero<V>() : hi[j];
                }
#pragma unroll
                for (int i = 1; i < PT; i++) mid[i] = z + i >= n2 ? vzero<V>() : mid[i];
            } else {
#pragma unroll
                for (int j = 0; j < R; j++) {
                    lo[j] = z_ghost(sl[eo[j]], z - R + j);
                    hi[j] = z_ghost(sl[eo[R + j]], z + PT + j);
                }
                if (short_by > 0) {
#pragma unroll
                    for (int i = 1; i < PT; i++) {
                        const V v = z_ghost(sl[eo[2 * R + i - 1]], z + i);
                        mid[i] = z + i >= n2 ? v : mid[i];
                    }
                }
            }
            add_z(lo, mid, hi);
        }
        S vv[PT];
        if (HAS_V) {
#pragma unroll
            for (int i = 0; i < PT; i++) vv[i] = pot.v[i];
            if (!ALIGNED && short_by > 0) {
#pragma unroll
                for (int t = 1; t < PT; t++)
#pragma unroll
                    for (int i = 0; i + t < PT; i++)
                        if (short_by == t) vv[i] = part ? pot.v[i + t] : vv[i];
            }
        }
        if (HAS_SRC) ss = shifted(ss);
#pragma unroll
        for (int e = 0; e < E; e++) {
            S a = acc[e];
            if (HAS_V) a = fma_rs(vv[e / C], q[R][e], a);
            if (HAS_SRC) a = fma_rs(beta, ss[e], a);
            acc[e] = a;
        }
        if (act) {
            V* o = outb + gi;
            if (!part) {
                __builtin_nontemporal_store((UVec)acc, reinterpret_cast<UVec*>(o));
            } else {
#pragma unroll
                for (int e = 0; e < E; e++)
                    if (z + e / C < n2) reinterpret_cast<S*>(o)[e] = acc[e];
            }
        }
#pragma unroll
        for (int j = 0; j < 2 * R; j++) q[j] = q[j + 1];
    }
}

template <typename V, typename S, int R>
int launch_r(const DirectStencil& h, const void* in, void* out, int64_t nbands,
             const double* phase_cd, const void* vt, const void* src, double beta, double alpha,
             double gamma, const double* eps, int ncu, hipStream_t st) {
    constexpr int PT = 16 / (int)sizeof(V);
    RowsArgs<S, R> g;
    g.n0 = h.n[0]; g.n1 = h.n[1]; g.n2 = h.n[2];
    g.pbc0 = h.pbc[0]; g.pbc1 = h.pbc[1]; g.pbc2 = h.pbc[2];
    g.c0 = (S)(alpha * h.c0 + gamma);
    g.eps = eps;
    bool sym = true;
    for (int c = 0; c < 3; c++)
        for (int j = 0; j < R; j++) {
            sym = sym && h.cm[c][j] == h.cp[c][j];
            g.km[c][j] = (S)(alpha * h.cm[c][j]);
            g.kp[c][j] = (S)(alpha * h.cp[c][j]);
        }
    const Phases ph = make_phases(phase_cd);
    g.yphase = g.zphase = 0;
    for (int c = 0; c < 3; c++)
        for (int d = 0; d < 2; d++) {
            g.re[c][d] = (S)ph.re[c][d];
            g.im[c][d] = (S)ph.im[c][d];
            const bool one = g.re[c][d] == (S)1 && g.im[c][d] == (S)0;
            if (c == 1 && !one) g.yphase = 1;
            if (c == 2 && !one) g.zphase = 1;
        }
    g.wide = (g.n2 * sizeof(V)) % 16 == 0 && ((uintptr_t)in & 15u) == 0;
    if (((uintptr_t)in & (sizeof(S) - 1)) || ((uintptr_t)out & (sizeof(S) - 1)))
        return GH_ERR_UNSUPPORTED;
    const int nv = (g.n2 + PT - 1) / PT;
    if (g.n2 < PT) return GH_ERR_UNSUPPORTED;
    g.nv_points = nv * PT;
    g.lw = g.wide ? 1 : 2;
    auto lds_of = [&](int ty) {
        // slots are 16-byte multiples; a vector may read past the last row
        const size_t slot = ((size_t)(ty + 2 * R) * g.n2 * sizeof(V) + 15) / 16 * 16;
        return (R + kDepth + 1) * slot + 16;
    };
    auto comp_of = [&](int ty) { return (ty * nv + 63) / 64; };
    // Tile and x-run: the pair with the least estimated time.  A block takes
    // lx + R + 2 iterations of a fixed cost (latency and barrier, the time of
    // about 6 KB at a CU's share of the HBM rate) plus the bytes of a plane
    // (ghost rows come from L2 and count half) of every block that its CU
    // runs beside it; blocks beyond what the CUs hold go into further rounds.
    // One row count for each number of tiles and one run length for each number
    // of runs: the choice of all pairs, at 4 to 20 % of the host time (1 us
    // per call at 16 x 48^3, 6 at 2 x 256 x 256 x 24).
    struct Run { int lx, nxc; };
    Run runs[192];
    int nruns = 0;
    if (h.planes > 0) {
        const int lx = std::min(h.planes, g.n0);
        runs[nruns++] = Run{lx, (g.n0 + lx - 1) / lx};
    } else {
        for (int nxc = 1; nxc <= std::max(1, g.n0 / (2 * R)) && nruns < 192;) {
            const int lx = (g.n0 + nxc - 1) / nxc;
            runs[nruns++] = Run{lx, (g.n0 + lx - 1) / lx};
            if (lx == 1) break;
            nxc = std::max(nxc + nxc / 16, (g.n0 + lx - 2) / (lx - 1));
        }
    }
    auto fits = [&](int ty) {
        return lds_of(ty) <= kLdsBytes - 1024 && (comp_of(ty) + kDepth * g.lw) * 64 <= kMaxThreads<R>;
    };
    double best = 0;
    int nyt_last = 0;
    g.ty = 0;
    for (int ty = 1; ty <= g.n1 && fits(ty); ty++) {
        // rows that were asked for: as many of them as fit
        if (h.rows > 0 && ty < std::min(h.rows, g.n1) && ty < g.n1 && fits(ty + 1)) continue;
        const int nyt = (g.n1 + ty - 1) / ty;
        if (nyt == nyt_last) continue;
        nyt_last = nyt;
        const int threads = (comp_of(ty) + kDepth * g.lw) * 64;
        const double fit = std::max(1, std::min(1024 / threads, (int)(kLdsBytes / lds_of(ty))));
        const double tiles = (double)nbands * nyt, bytes = (2.0 * ty + R) * g.n2 * sizeof(V);
        // (the small number keeps whole quotients whole)
        const double per_room = 1.0 / (ncu * fit), per_cu = 1.0 / ncu;
        for (int k = 0; k < nruns; k++) {
            const double blocks = tiles * runs[k].nxc;
            const double rounds = std::ceil(blocks * per_room - 1e-9);
            const double beside = std::min(fit, std::ceil(blocks * per_cu - 1e-9));
            const double t = rounds * (runs[k].lx + R + 2) * (beside * bytes + 6144.0);
            if (g.ty == 0 || t < best) {
                best = t;
                g.ty = ty;
                g.lx = runs[k].lx;
            }
            if (rounds > 8) break;
        }
        if (h.rows > 0) break;
    }
    // (long complex128 rows leave a tile so few rows beside its 2R ghost rows
    // that the kernel without LDS is faster: 115^3, R = 5, one row 73 us, 44)
    if (g.ty == 0 || (R > 3 && h.rows == 0 && g.ty < std::min(R / 2, g.n1))) return GH_ERR_UNSUPPORTED;
    g.nyt = (g.n1 + g.ty - 1) / g.ty;
    g.nxc = (g.n0 + g.lx - 1) / g.lx;
    g.ncomp = comp_of(g.ty);
    g.nbands = (int)nbands;
    g.bgroup = std::min<int>(std::max(1, ncu / kNumXCD / (g.nyt * g.nxc)), (int)nbands);
    const int64_t nblocks = nbands * (int64_t)g.nyt * g.nxc;
    GH_REQUIRE(nblocks < (1ll << 31), GH_ERR_SHAPE, "stencil: too many blocks");
    const size_t lds = lds_of(g.ty);
    g.slot = (int)((lds - 16) / (R + kDepth + 1) / sizeof(V));
    const dim3 grid((unsigned)nblocks), block((g.ncomp + kDepth * g.lw) * 64);
    auto go = [&](auto aligned, auto symmetric) {
        constexpr bool AL = decltype(aligned)::value, SY = decltype(symmetric)::value;
#define GH_ROWS(HV, HS)                                                                    \
    do {                                                                                   \
        auto kfn = stencil_rows_kernel<V, S, R, PT, AL, SY, HV, HS>;                       \
        int rc = ensure_max_lds((const void*)kfn, (int)kLdsBytes);                         \
        if (rc != GH_OK) return rc;                                                        \
        hipLaunchKernelGGL(kfn, grid, block, lds, st, (const V*)in, (V*)out, (const S*)vt, \
                           (const V*)src, (S)beta, g);                                     \
    } while (0)
        if (vt && src) GH_ROWS(true, true);
        else if (vt) GH_ROWS(true, false);
        else if (src) GH_ROWS(false, true);
        else GH_ROWS(false, false);
#undef GH_ROWS
        return (int)GH_OK;
    };
    int rc;
    if (!sym) rc = go(std::false_type{}, std::false_type{});
    else if constexpr (PT == 1) rc = go(std::true_type{}, std::true_type{});
    else rc = g.n2 % PT == 0 ? go(std::true_type{}, std::true_type{})
                             : go(std::false_type{}, std::true_type{});
    if (rc != GH_OK) return rc;
    GH_CHECK_LAUNCH();
    return GH_OK;
}

template <typename V, typename S>
int launch(const DirectStencil& h, const void* in, void* out, int64_t nb, const double* ph,
           const void* vt, const void* src, double beta, double al, double ga,
           const double* eps, int ncu, hipStream_t st) {
    switch (h.R) {
        case 1: return launch_r<V, S, 1>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, ncu, st);
        case 2: return launch_r<V, S, 2>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, ncu, st);
        case 3: return launch_r<V, S, 3>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, ncu, st);
        case 4: return launch_r<V, S, 4>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, ncu, st);
        case 5: return launch_r<V, S, 5>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, ncu, st);
        case 6: return launch_r<V, S, 6>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, ncu, st);
    }
    return GH_ERR_UNSUPPORTED;
}

}  // namespace

int stencil_rows(int dtype, const DirectStencil& h, const void* in, void* out, int64_t nb,
                 const double* ph, const void* vt, const void* src, double beta, double al,
                 double ga, const double* eps, int ncu, hipStream_t st) {
    switch (dtype) {
        case GH_F64: return launch<double, double>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, ncu, st);
        case GH_C128: return launch<cplx<double>, double>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, ncu, st);
        case GH_F32: return launch<float, float>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, ncu, st);
        case GH_C64: return launch<cplx<float>, float>(h, in, out, nb, ph, vt, src, beta, al, ga, eps, ncu, st);
    }
    return GH_ERR_ARG;
}

}  // namespace gh
