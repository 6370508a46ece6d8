// Rotation of up to 64 real wave functions, out = U psi, on the matrix cores
// (v_mfma_f64_16x16x4f64): U is a small matrix, psi a tall one.
//
// HBM bound: psi is read and out written once (64 functions of 64^3 points: 268
// MB, 53 us at a copy's rate); the products, 2.1 GFLOP, take 27 us at the
// FP64 matrix rate.  A wave keeps all of U in registers (64 x 64
// values: 128 VGPRs) and walks over tiles of 16 grid points; the whole column
// of a tile (16 loads of 4 rows x 128 bytes) is in flight while the one
// before it is multiplied.  No LDS, no barriers.  The library's product tiles
// both operands through LDS and reads at under half the rate of a copy:
// 64 functions of 64^3 points (268 MB) 146 -> 70 us.
#include <algorithm>

#include "common.h"
#include "internal.h"

namespace gh {

namespace {

constexpr int kThreads = 256, kMax = 64;
typedef double d4 __attribute__((ext_vector_type(4)));

// MT tiles of 16 results, KS steps of 4 functions
template <int MT, int KS>
__global__ void __launch_bounds__(kThreads, 2)
rotate_kernel(const double* __restrict__ U, int m, int k, const double* __restrict__ psi,
              double* __restrict__ out, int64_t n) {
    const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
    double a[MT][KS];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int s = 0; s < KS; s++) {
            const int i = t * 16 + col, j = 4 * s + grp;
            a[t][s] = i < m && j < k ? U[i * k + j] : 0.0;
        }
    const int64_t tiles = (n + 15) / 16;
    const int64_t step = (int64_t)gridDim.x * (kThreads / 64);
    int64_t tile = blockIdx.x * (int64_t)(kThreads / 64) + (threadIdx.x >> 6);
    // uniform row pointers and 32-bit offsets of the lane's group and point
    // (with 64-bit addresses per row U no longer fits the registers)
    const unsigned gn = (unsigned)(grp * n);
    const int ke = k / 4, kr = k - 4 * ke;
    const unsigned gpart = (unsigned)(min(grp, max(kr, 1) - 1) * n);
    auto load = [&](int s, unsigned p) {
        const char* r = reinterpret_cast<const char*>(psi + (int64_t)(4 * s) * n);
        if (s < ke) return *reinterpret_cast<const double*>(r + (gn + p) * 8u);
        if (s == ke && kr > 0) {
            const double v = *reinterpret_cast<const double*>(r + (gpart + p) * 8u);
            return grp < kr ? v : 0.0;
        }
        return 0.0;
    };
    auto point = [&](int64_t t) { return (unsigned)min(t * 16 + col, n - 1); };
    double b[KS];
    if (tile < tiles) {
        const unsigned p = point(tile);
#pragma unroll
        for (int s = 0; s < KS; s++) b[s] = load(s, p);
    }
    for (; tile < tiles; tile += step) {
        const unsigned pn = point(min(tile + step, tiles - 1));
        d4 acc[MT];
#pragma unroll
        for (int t = 0; t < MT; t++) acc[t] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < KS; s++) {
#pragma unroll
            for (int t = 0; t < MT; t++)
                acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t][s], b[s], acc[t], 0, 0, 0);
            b[s] = load(s, pn);
        }
        if (tile * 16 + col < n) {
            const unsigned p = (gn + (unsigned)(tile * 16 + col)) * 8u;
#pragma unroll
            for (int t = 0; t < MT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    char* o = reinterpret_cast<char*>(out + (int64_t)(t * 16 + 4 * r) * n);
                    if (t * 16 + 4 * r + grp < m) *reinterpret_cast<double*>(o + p) = acc[t][r];
                }
        }
    }
}

}  // namespace

}  // namespace gh

using namespace gh;

extern "C" int gh_rotate(int m, int k, int64_t n, const double* U_dev, const double* psi_dev,
                         double* out_dev, void* stream) {
    GH_REQUIRE(m >= 1 && k >= 1 && n >= 0, GH_ERR_ARG, "rotate: bad sizes");
    GH_REQUIRE(m <= kMax && k <= kMax, GH_ERR_UNSUPPORTED, "rotate: %d x %d, at most %d", m, k,
               kMax);
    GH_REQUIRE(n < (1ll << 27), GH_ERR_UNSUPPORTED, "rotate: %lld points", (long long)n);
    if (n == 0) return GH_OK;  // empty arrays may carry null pointers
    GH_REQUIRE(U_dev && psi_dev && out_dev, GH_ERR_ARG, "rotate: null argument");
    GH_REQUIRE(psi_dev != out_dev, GH_ERR_ARG, "rotate: psi and out must differ");
    int ncu = 0;
    const int rc = device_cu_count(&ncu);
    if (rc != GH_OK) return rc;
    // two blocks per CU (registers), each wave with many tiles; a few
    // functions leave so little in flight per wave that eight are needed
    // (2 x 2, 1.4 M points: 37 us with two, 21 with eight)
    const int64_t tiles = (n + 15) / 16;
    const unsigned blocks =
        (unsigned)std::min<int64_t>((tiles + 3) / 4, (m + k <= 16 ? 8 : 2) * ncu);
    const int ks = (k + 15) / 16, mt = (m + 15) / 16;
    hipStream_t st = (hipStream_t)stream;
#define GH_ROT(MT, KB)                                                                  \
    hipLaunchKernelGGL((rotate_kernel<MT, 4 * KB>), dim3(blocks), dim3(kThreads), 0, st, \
                       U_dev, m, k, psi_dev, out_dev, n)
#define GH_ROTM(MT)                                   \
    do {                                              \
        if (ks == 1) GH_ROT(MT, 1);                   \
        else if (ks == 2) GH_ROT(MT, 2);              \
        else if (ks == 3) GH_ROT(MT, 3);              \
        else GH_ROT(MT, 4);                           \
    } while (0)
    if (mt == 1) GH_ROTM(1);
    else if (mt == 2) GH_ROTM(2);
    else if (mt == 3) GH_ROTM(3);
    else GH_ROTM(4);
#undef GH_ROTM
#undef GH_ROT
    GH_CHECK_LAUNCH();
    return GH_OK;
}
