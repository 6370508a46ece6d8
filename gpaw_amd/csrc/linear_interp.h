// Linear (nn = 1) interpolation to the grid of half the spacing, a vector of
// fine points per thread: where its coarse values are, and its values on the
// plane of F_i, the coarse plane i - plo interpolated along z and y.
#pragma once

#include "common.h"

namespace gh {

// Coarse grid n, ghosts below (plo), fine points left out below (skip): fine
// point o lies on coarse point (o + skip) / 2 - plo or half way to the next.
template <typename S>
struct LinGrid {
    int n[3], pbc[3], plo[3], skip[3];
    int yzphase;                  // complex data with a y or z Bloch phase
    S re[3][2], im[3][2];
};

template <typename S>
inline void set_phases(LinGrid<S>& g, const double* phase_cd) {
    const Phases ph = make_phases(phase_cd);
    g.yzphase = 0;
    for (int c = 0; c < 3; c++)
        for (int d = 0; d < 2; d++) {
            g.re[c][d] = (S)ph.re[c][d];
            g.im[c][d] = (S)ph.im[c][d];
            if (c > 0 && (g.re[c][d] != (S)1 || g.im[c][d] != (S)0)) g.yzphase = 1;
        }
}

// Interior index of coarse point c: its image one period away, or clamped
// with `zero` set.
__device__ __forceinline__ int lin_wrap(int c, int n, int pbc, bool& low, bool& high,
                                        bool& zero) {
    low = c < 0;
    high = c >= n;
    if (pbc) c += low ? n : high ? -n : 0;
    zero = c < 0 || c >= n;
    return min(max(c, 0), n - 1);
}

template <typename V, typename S, int PT>
struct LinPoints {
    static constexpr bool CPLX = is_complex<V>::value;
    static constexpr int NC = PT == 1 ? 2 : PT / 2 + 1;   // coarse values per row
    typedef S Vec __attribute__((ext_vector_type(16 / sizeof(S))));
    struct Raw { V v[2][NC]; };

    int row[2], z[NC];            // coarse row starts, coarse z
    // bits: 0 fine row between two coarse rows, 1 fine z likewise (PT = 1);
    // 2, 3 row r lies beyond a zero boundary; 4.. the same for z; from 8 on
    // two bits (below, above) for each row and z that is a periodic image
    unsigned flags;
    static constexpr unsigned kOddY = 1, kOddZ = 2;
    static constexpr unsigned kZero = 0xCu | (((1u << NC) - 1) << 4);

    // fine row y, fine points z0 .. z0 + PT - 1 (z0 a multiple of PT)
    __device__ __forceinline__ void set(int y, int z0, const LinGrid<S>& g) {
        flags = 0;
        const int qy = y + g.skip[1];
        if (qy & 1) flags |= kOddY;
#pragma unroll
        for (int r = 0; r < 2; r++) {
            bool low, high, zero;
            const int c = lin_wrap((qy >> 1) - g.plo[1] + ((qy & 1) ? r : 0), g.n[1], g.pbc[1],
                                   low, high, zero);
            row[r] = c * g.n[2];
            if (zero) flags |= 4u << r;
            flags |= (unsigned)low << (8 + 2 * r) | (unsigned)high << (9 + 2 * r);
        }
        const int qz = z0 + g.skip[2];
        if (PT == 1 && (qz & 1)) flags |= kOddZ;
#pragma unroll
        for (int k = 0; k < NC; k++) {
            bool low, high, zero;
            z[k] = lin_wrap((qz >> 1) - g.plo[2] + (PT == 1 && !(qz & 1) ? 0 : k), g.n[2],
                            g.pbc[2], low, high, zero);
            if (zero) flags |= 16u << k;
            flags |= (unsigned)low << (12 + 2 * k) | (unsigned)high << (13 + 2 * k);
        }
    }
    // coarse values of F_i (for planes beyond the grid: of the image, or some)
    __device__ __forceinline__ void load(const V* __restrict__ band, int i, const LinGrid<S>& g,
                                         Raw& raw) const {
        bool low, high, zero;
        const int c = lin_wrap(i - g.plo[0], g.n[0], g.pbc[0], low, high, zero);
        const V* p = band + (size_t)c * g.n[1] * g.n[2];
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int k = 0; k < NC; k++) raw.v[r][k] = p[row[r] + z[k]];
    }
    // F_i at the points
    __device__ __forceinline__ Vec make(Raw raw, int i, const LinGrid<S>& g) const {
        auto half = [](V a, V b) { return vscale(vadd(a, b), (S)0.5); };
        if (!(g.pbc[1] && g.pbc[2]) && __any((int)(flags & kZero))) {
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int k = 0; k < NC; k++)
                    if (flags & (4u << r | 16u << k)) raw.v[r][k] = vzero<V>();
        }
        if constexpr (CPLX) {
            if (g.yzphase && __any((int)(flags >> 8))) {
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    const bool l = flags >> (8 + 2 * r) & 1, h = flags >> (9 + 2 * r) & 1;
                    const S pr = l ? g.re[1][1] : h ? g.re[1][0] : (S)1;
                    const S pi = l ? g.im[1][1] : h ? g.im[1][0] : (S)0;
#pragma unroll
                    for (int k = 0; k < NC; k++) {
                        const bool zl = flags >> (12 + 2 * k) & 1,
                                   zh = flags >> (13 + 2 * k) & 1;
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
                f[r][0] = flags & kOddZ ? half(raw.v[r][0], raw.v[r][1]) : raw.v[r][0];
            } else {
#pragma unroll
                for (int e = 0; e < PT; e += 2) {
                    const V m = half(raw.v[r][e / 2], raw.v[r][e / 2 + 1]);
                    f[r][e] = g.skip[2] & 1 ? m : raw.v[r][e / 2];
                    f[r][e + 1] = g.skip[2] & 1 ? raw.v[r][e / 2 + 1] : m;
                }
            }
        }
        bool xlow, xhigh, xzero;
        lin_wrap(i - g.plo[0], g.n[0], g.pbc[0], xlow, xhigh, xzero);
        V o[PT];
#pragma unroll
        for (int e = 0; e < PT; e++) {
            o[e] = flags & kOddY ? half(f[0][e], f[1][e]) : f[0][e];
            if (xzero) o[e] = vzero<V>();
            if constexpr (CPLX)
                if (xlow || xhigh) o[e] = mul_phase(o[e], g.re[0][xlow], g.im[0][xlow]);
        }
        Vec v;
        __builtin_memcpy(&v, o, sizeof(v));
        return v;
    }
};

}  // namespace gh
