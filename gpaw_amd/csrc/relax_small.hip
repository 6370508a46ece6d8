// Jacobi sweeps of a small grid in one launch: one workgroup keeps the
// function in LDS and its points' sources in registers.
//
// The coarsest levels of a multigrid solve relax grids of a hundred to a few
// thousand points four to eight times; with one launch per sweep each sweep
// costs 4.2 to 4.6 us, nearly all of it the launch.  Here it costs two
// barriers and the instructions of its points on one CU.  us, radius 1, FP64,
// a launch per sweep and one launch:
//   5 x 5 x 6, zero boundaries, 8 sweeps   33.3 -> 3.8
//   11 x 11 x 13, 4 sweeps                 18.8 -> 5.8
//   16^3, 4 sweeps                         17.9 -> 8.7  (1 sweep 6.4 -> 5.8)
// Up to 4 points per thread: at 14 (23 x 23 x 27) a sweep takes about 4.2 us
// on one CU, as long as a launch over many.
#include <algorithm>

#include "common.h"
#include "internal.h"

namespace gh {

namespace {

constexpr int kThreads = 1024, kPoints = 4;

template <typename S>
struct RelaxArgs {
    int n0, n1, n2, pbc0, pbc1, pbc2, sweeps;
    S c0, k[3], beta;
};

template <typename S>
__global__ void __launch_bounds__(kThreads)
relax_small_kernel(const S* f, S* out, const S* __restrict__ s, RelaxArgs<S> g) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    S* lds = reinterpret_cast<S*>(smem_raw);
    const int n = g.n0 * g.n1 * g.n2, nt = blockDim.x, t = threadIdx.x;
    int pos[kPoints];                 // x, y, z of the thread's points, 10 bits each
    S sv[kPoints], nw[kPoints];
#pragma unroll
    for (int k = 0; k < kPoints; k++) {
        const int p = t + k * nt;
        pos[k] = 0;
        sv[k] = nw[k] = 0;
        if (k * nt < n) {
            const int q = min(p, n - 1), xy = q / g.n2, x = xy / g.n1;
            pos[k] = x << 20 | (xy - x * g.n1) << 10 | (q - xy * g.n2);
            sv[k] = s[q];
            if (p < n) lds[p] = f[p];
        }
    }
    const int strx = g.n1 * g.n2, stry = g.n2;
    for (int w = 0; w < g.sweeps; w++) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kPoints; k++) {
            if (k * nt >= n) continue;
            const int x = pos[k] >> 20, y = pos[k] >> 10 & 1023, z = pos[k] & 1023;
            const int q = x * strx + y * stry + z;
            // both neighbours along an axis, wrapped or zero
            auto pair = [&](int i, int len, int str, int pbc) {
                const bool low = i == 0, high = i == len - 1;
                S m = lds[q + (low ? (pbc ? (len - 1) * str : 0) : -str)];
                S p = lds[q + (high ? (pbc ? (1 - len) * str : 0) : str)];
                if (low && !pbc) m = 0;
                if (high && !pbc) p = 0;
                return m + p;
            };
            S a = lds[q] * g.c0;
            a = fma_rs(g.k[0], pair(x, g.n0, strx, g.pbc0), a);
            a = fma_rs(g.k[1], pair(y, g.n1, stry, g.pbc1), a);
            a = fma_rs(g.k[2], pair(z, g.n2, 1, g.pbc2), a);
            nw[k] = fma_rs(g.beta, sv[k], a);
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kPoints; k++) {
            if (t + k * nt < n) lds[t + k * nt] = nw[k];
        }
    }
#pragma unroll
    for (int k = 0; k < kPoints; k++) {
        const int p = t + k * nt;
        if (p < n) out[p] = nw[k];
    }
}

template <typename S>
int launch(const DirectStencil& h, const void* f, void* out, const void* s, int sweeps,
             double beta, double alpha, double gamma, hipStream_t st) {
    const int64_t n = (int64_t)h.n[0] * h.n[1] * h.n[2];
    RelaxArgs<S> g;
    for (int c = 0; c < 3; c++) {
        // a neighbour lies one period away at most; 10 bits per coordinate
        if (h.n[c] > 1023 || h.cm[c][0] != h.cp[c][0]) return GH_ERR_UNSUPPORTED;
        g.k[c] = (S)(alpha * h.cm[c][0]);
    }
    if (h.R != 1 || n > kThreads * kPoints) return GH_ERR_UNSUPPORTED;
    g.n0 = h.n[0]; g.n1 = h.n[1]; g.n2 = h.n[2];
    g.pbc0 = h.pbc[0]; g.pbc1 = h.pbc[1]; g.pbc2 = h.pbc[2];
    g.sweeps = sweeps;
    g.c0 = (S)(alpha * h.c0 + gamma);
    g.beta = (S)beta;
    const int threads = (int)std::min<int64_t>(kThreads, (n + 63) / 64 * 64);
    hipLaunchKernelGGL((relax_small_kernel<S>), dim3(1), dim3(threads), n * sizeof(S), st, (const S*)f, (S*)out,
                       (const S*)s, g);
    GH_CHECK_LAUNCH();
    return GH_OK;
}

}  // namespace

int relax_small(const gh_stencil* h, const void* f, void* out, const void* s, int sweeps,
                double beta, double al, double ga, hipStream_t st) {
    DirectStencil d;
    if (!stencil_axes(h, &d)) return GH_ERR_UNSUPPORTED;
    if (stencil_dtype(h) == GH_F64) return launch<double>(d, f, out, s, sweeps, beta, al, ga, st);
    if (stencil_dtype(h) == GH_F32) return launch<float>(d, f, out, s, sweeps, beta, al, ga, st);
    return GH_ERR_UNSUPPORTED;
}

}  // namespace gh
