// Band overlap matrices on the matrix cores: C = alpha * A B^H for
// band-major arrays A (m rows) and B (n rows) of length k -- the subspace
// matrices S = <psi|psi> and H = <psi|H|psi> of the eigensolvers (the
// reference forms them with rk / r2k / gemm, gpaw/utilities/blas.py:39,273,
// 314 -> c/blas.c:48,101,140, called from gpaw/matrix.py and
// gpaw/wavefunctions/arrays.py:262-340).
//
// The shape is tall-skinny: m, n are band counts (a few hundred) and k is a
// grid (10^5 .. 10^7 points), so the work is split along k.  A workgroup
// owns one block pair (BM rows of A x BN rows of B) and one k-chunk; it
// streams 128-byte row segments of both blocks through LDS and multiplies
// them on the MFMA units:
//   float / complex64   v_mfma_f32_32x32x2f32  (FP32 products and sums)
//   double / complex128 v_mfma_f64_16x16x4f64
// Each chunk's partial block is written to a workspace in the element
// precision, and a second kernel adds the chunks in FP64 in a fixed order
// (deterministic; FP32 sums never run over more than one chunk).
//
// Complex data: with A = a + ib and B = a' + ib' interleaved,
//   Re C = sum (a a' + b b')      -- the real product of the interleaved rows
//   Im C = sum (b a' - a b')      -- the same A operand against (-b', a')
// so each B value feeds two MFMAs (one per part) and no conjugate copy of B
// is formed.
//
// Hermitian mode (m == n, the product known to be Hermitian, e.g. S or H):
// only blocks holding some element i >= j are computed and the upper
// triangle is the conjugate of the lower one (what rk / r2k's "lower
// triangle" contract gives the reference's callers).
//
// k-order inside a 128-byte segment: lane group g of an MFMA supplies
// elements [g W, (g + 1) W) of the segment (W = elements per segment / K of
// the instruction), the same permutation for A and B, so each lane reads W
// contiguous elements with 16-byte LDS reads.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace gh {

namespace {

template <typename T> struct Mfma;

template <> struct Mfma<float> {
    static constexpr int TILE = 32;  // output tile TILE x TILE
    static constexpr int KOP = 2;    // k per instruction
    static constexpr int NACC = 16;  // accumulators per lane
    typedef float acc_t __attribute__((ext_vector_type(16)));
    static __device__ __forceinline__ acc_t op(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
    }
    // output row of accumulator r in lane group g (column = lane % TILE)
    static __device__ __forceinline__ int row(int r, int g) {
        return 8 * (r / 4) + 4 * g + (r % 4);
    }
};

template <> struct Mfma<double> {
    static constexpr int TILE = 16;
    static constexpr int KOP = 4;
    static constexpr int NACC = 4;
    typedef double acc_t __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ acc_t op(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int r, int g) { return g + 4 * r; }
};

constexpr int kSeg = 128;          // bytes of a row per stage
constexpr int kRowPitch = 144;     // LDS bytes per row (16-byte pad: no bank conflicts)
constexpr int kBM = 128;           // rows of A per block
constexpr int kThreads = 256;      // 4 waves: 2 x 2 over the block

// Block pairs in Hermitian mode: (I, J) with some i >= j, i.e.
// J <= q (I + 1) - 1 for q = BM / BN; row I holds q (I + 1) of them.
__host__ __device__ inline int herm_pair_index(int I, int J, int q) {
    return q * I * (I + 1) / 2 + J;
}

__device__ inline void herm_pair_of(int p, int q, int& I, int& J) {
    int i = 0;
    while (p >= q * (i + 1)) {
        p -= q * (i + 1);
        i++;
    }
    I = i;
    J = p;
}

template <typename T, bool CPLX, int WN>
__global__ void __launch_bounds__(kThreads)
gram_mfma_kernel(const char* __restrict__ A, const char* __restrict__ B,
                 int64_t lda, int64_t ldb,          // row pitch in bytes
                 int m, int n, int64_t nseg,        // segments of kSeg bytes per row
                 int64_t kbytes,                    // valid bytes per row
                 int herm, int npairs, int nJ, int nchunks,
                 T* __restrict__ work) {
    using M = Mfma<T>;
    constexpr int TILE = M::TILE, KOP = M::KOP, NACC = M::NACC;
    constexpr int BN = 2 * WN;
    constexpr int MT = 64 / TILE;            // row tiles per wave
    constexpr int NT = WN / TILE;            // column tiles per wave
    constexpr int EL = kSeg / sizeof(T);     // elements per segment
    constexpr int W = EL / KOP;              // elements per lane group
    constexpr int NC = CPLX ? 2 : 1;
    constexpr int AV = kBM * (kSeg / 16) / kThreads;   // 16-byte loads per thread
    constexpr int BV = BN * (kSeg / 16) / kThreads;
    static_assert(W % 2 == 0 && (W * sizeof(T)) % 16 == 0, "lane run");
    static_assert(AV >= 1 && BV >= 1, "loader");

    __shared__ __align__(16) char sA[kBM * kRowPitch];
    __shared__ __align__(16) char sB[BN * kRowPitch];

    // block id -> (chunk, pair); ids are dealt round-robin to the 8 XCDs,
    // so the pairs of one chunk (which read the same rows) are placed on
    // one XCD
    const int nblk = npairs * nchunks;
    const int lin = xcd_swizzle(blockIdx.x, nblk);
    const int pair = lin % npairs;
    const int chunk = lin / npairs;
    int I, J;
    if (herm) herm_pair_of(pair, kBM / BN, I, J);
    else { I = pair / nJ; J = pair % nJ; }
    const int row0 = I * kBM, col0 = J * BN;
    const bool sameAB = (A == B) && (lda == ldb) && row0 == col0 && BN == kBM;

    const int64_t s_beg = nseg * chunk / nchunks;
    const int64_t s_end = nseg * (chunk + 1) / nchunks;

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wr = wave >> 1, wc = wave & 1;
    const int lg = lane / TILE, lr = lane % TILE;

    typedef float f4 __attribute__((ext_vector_type(4)));
    f4 ra[AV], rb[BV];

    auto load = [&](int64_t s) {
        const int64_t kb0 = s * kSeg;
#pragma unroll
        for (int v = 0; v < AV; v++) {
            const int idx = tid + v * kThreads;
            const int r = idx / (kSeg / 16), c = idx % (kSeg / 16);
            const int64_t kb = kb0 + c * 16;
            f4 x = {0.f, 0.f, 0.f, 0.f};
            if (row0 + r < m && kb < kbytes)
                x = *(const f4*)(A + (int64_t)(row0 + r) * lda + kb);
            ra[v] = x;
        }
        if (!sameAB) {
#pragma unroll
            for (int v = 0; v < BV; v++) {
                const int idx = tid + v * kThreads;
                const int r = idx / (kSeg / 16), c = idx % (kSeg / 16);
                const int64_t kb = kb0 + c * 16;
                f4 x = {0.f, 0.f, 0.f, 0.f};
                if (col0 + r < n && kb < kbytes)
                    x = *(const f4*)(B + (int64_t)(col0 + r) * ldb + kb);
                rb[v] = x;
            }
        }
    };
    auto stash = [&]() {
#pragma unroll
        for (int v = 0; v < AV; v++) {
            const int idx = tid + v * kThreads;
            const int r = idx / (kSeg / 16), c = idx % (kSeg / 16);
            *(f4*)(sA + r * kRowPitch + c * 16) = ra[v];
        }
        if (!sameAB) {
#pragma unroll
            for (int v = 0; v < BV; v++) {
                const int idx = tid + v * kThreads;
                const int r = idx / (kSeg / 16), c = idx % (kSeg / 16);
                *(f4*)(sB + r * kRowPitch + c * 16) = rb[v];
            }
        }
    };

    typename M::acc_t acc[NC][MT][NT];
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int r = 0; r < NACC; r++) acc[c][i][j][r] = T(0);

    const char* sBr = sameAB ? sA : sB;
    if (s_beg < s_end) load(s_beg);
    for (int64_t s = s_beg; s < s_end; s++) {
        __syncthreads();          // the previous stage's LDS reads are done
        stash();
        __syncthreads();
        if (s + 1 < s_end) load(s + 1);   // in flight during the products
        T a[MT][W], b[NT][W];
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const char* p = sA + (wr * 64 + i * TILE + lr) * kRowPitch + lg * W * sizeof(T);
#pragma unroll
            for (int q = 0; q < W * (int)sizeof(T) / 16; q++) {
                f4 x = *(const f4*)(p + 16 * q);
                __builtin_memcpy(&a[i][q * 16 / sizeof(T)], &x, 16);
            }
        }
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const char* p = sBr + (wc * WN + j * TILE + lr) * kRowPitch + lg * W * sizeof(T);
#pragma unroll
            for (int q = 0; q < W * (int)sizeof(T) / 16; q++) {
                f4 x = *(const f4*)(p + 16 * q);
                __builtin_memcpy(&b[j][q * 16 / sizeof(T)], &x, 16);
            }
        }
#pragma unroll
        for (int e = 0; e < W; e++) {
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    acc[0][i][j] = M::op(a[i][e], b[j][e], acc[0][i][j]);
                    if constexpr (CPLX) {
                        // (re, im) of B at e even / odd -> (-im, re)
                        const T y = (e & 1) ? b[j][e - 1] : -b[j][e + 1];
                        acc[NC - 1][i][j] = M::op(a[i][e], y, acc[NC - 1][i][j]);
                    }
                }
        }
    }

    // partial block -> work[(pair, chunk)][part][BM][BN]
    T* out = work + ((int64_t)pair * nchunks + chunk) * NC * kBM * BN;
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int r = 0; r < NACC; r++) {
                    const int row = wr * 64 + i * TILE + M::row(r, lg);
                    const int col = wc * WN + j * TILE + lr;
                    out[(int64_t)c * kBM * BN + row * BN + col] = acc[c][i][j][r];
                }
}

// Band counts up to 64 (both operands): the 128 x 128 block above would
// spend three of its four waves on rows that do not exist, so here every
// wave owns the whole 64 x 64 product of a k-slice (complex128: two waves
// share a slice, 32 columns each, to fit the registers).  A 128-byte segment
// of 64 + 64 rows is 64 instructions for 16 KB, more time on the matrix cores
// than its loads take, so the registers go to one wave per SIMD with the next
// segment's loads in flight.  At the size below it reaches 37 % of the matrix
// rate, and its bytes would take 26 us (one operand) to 53 (two) at a copy's
// rate: neither limits it; with one wave per SIMD, latency likely does.  The
// waves share no data and each lane's 16-byte loads of a row use whole 128-byte
// lines, so there is no LDS stage and no barrier in the loop.  In Hermitian mode tiles above the diagonal are
// skipped.  The block's slices are added in FP64 through LDS and one partial
// block per workgroup (always FP64) goes to the workspace.  64 FP64 bands of
// 64^3 points: 182 us with the 128-row blocks, 73 us here (29 TFLOP/s of the
// full product).
constexpr int kSB = 64;

template <typename T, bool CPLX> struct SmallWN { static constexpr int value = 64; };
template <> struct SmallWN<double, true> { static constexpr int value = 32; };

template <typename T, bool CPLX>
__global__ void __launch_bounds__(kThreads)
gram_small_kernel(const char* __restrict__ A, const char* __restrict__ B, int64_t lda,
                  int64_t ldb, int m, int n, int64_t nseg, int64_t kbytes, int herm,
                  double* __restrict__ work) {
    using M = Mfma<T>;
    constexpr int TILE = M::TILE, KOP = M::KOP, NACC = M::NACC;
    constexpr int WN = SmallWN<T, CPLX>::value;
    constexpr int WC = kSB / WN, KS = 4 / WC;   // waves along columns, slices per block
    constexpr int MT = kSB / TILE, NT = WN / TILE;
    constexpr int W = kSeg / (int)sizeof(T) / KOP;      // elements per lane and row
    constexpr int Q = W * (int)sizeof(T) / 16;          // 16-byte loads per lane and row
    constexpr int NC = CPLX ? 2 : 1;
    typedef float f4 __attribute__((ext_vector_type(4)));
    __shared__ double red[NC][kSB][kSB];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ks = wave / WC, cg = wave % WC;
    const int lg = lane / TILE, lr = lane % TILE;
    const int64_t slice = (int64_t)blockIdx.x * KS + ks, nslice = (int64_t)gridDim.x * KS;
    const int64_t s_beg = nseg * slice / nslice, s_end = nseg * (slice + 1) / nslice;

    // rows beyond the operand repeat its last row: they only feed results
    // that are not read
    const char* pa[MT];
    const char* pb[NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
        pa[i] = A + (int64_t)min(i * TILE + lr, m - 1) * lda + lg * W * (int)sizeof(T);
#pragma unroll
    for (int j = 0; j < NT; j++)
        pb[j] = B + (int64_t)min(cg * WN + j * TILE + lr, n - 1) * ldb + lg * W * (int)sizeof(T);
    f4 ra[MT][Q], rb[NT][Q];
    auto load = [&](int64_t s) {
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const int64_t kb = s * kSeg + 16 * q;
            const bool in = kb + lg * W * (int)sizeof(T) < kbytes;
#pragma unroll
            for (int i = 0; i < MT; i++) ra[i][q] = in ? *(const f4*)(pa[i] + kb) : f4{0, 0, 0, 0};
#pragma unroll
            for (int j = 0; j < NT; j++) rb[j][q] = in ? *(const f4*)(pb[j] + kb) : f4{0, 0, 0, 0};
        }
    };
    typename M::acc_t acc[NC][MT][NT];
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int r = 0; r < NACC; r++) acc[c][i][j][r] = T(0);
    if (s_beg < s_end) load(s_beg);
    for (int64_t s = s_beg; s < s_end; s++) {
        T a[MT][W], b[NT][W];
        __builtin_memcpy(a, ra, sizeof(a));
        __builtin_memcpy(b, rb, sizeof(b));
        if (s + 1 < s_end) load(s + 1);
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++) {
                if (herm && i * TILE + TILE <= cg * WN + j * TILE) continue;
#pragma unroll
                for (int e = 0; e < W; e++) {
                    acc[0][i][j] = M::op(a[i][e], b[j][e], acc[0][i][j]);
                    if constexpr (CPLX) {
                        const T y = (e & 1) ? b[j][e - 1] : -b[j][e + 1];
                        acc[NC - 1][i][j] = M::op(a[i][e], y, acc[NC - 1][i][j]);
                    }
                }
            }
    }
    for (int k = 0; k < KS; k++) {
        if (ks == k) {
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < NT; j++)
#pragma unroll
                        for (int r = 0; r < NACC; r++) {
                            double* p = &red[c][i * TILE + M::row(r, lg)]
                                            [cg * WN + j * TILE + lr];
                            *p = (k ? *p : 0.0) + (double)acc[c][i][j][r];
                        }
        }
        __syncthreads();
    }
    double* out = work + (int64_t)blockIdx.x * NC * kSB * kSB;
    for (int i = tid; i < NC * kSB * kSB; i += kThreads) out[i] = (&red[0][0][0])[i];
}

// C[i][j] = alpha * sum over chunks (FP64, a fixed order) of the partial
// blocks; Hermitian mode forms i >= j and writes its mirror image too;
// conj_out conjugates.  A block sums NO neighbouring outputs, 256 / NO chunks
// at a time, 16 outputs where there are many chunks: at 64 bands a thread per
// output left 16 blocks to walk about 1000 chunks one after the other (339
// us; with the 64-row form's 256 chunks now under 17 us).  Many bands have few
// chunks, and 16 outputs would leave threads without one (1000 x 1000 float32
// over 1728 points, 3 chunks, product and sum: 73 us with 16, 52 with 256).
template <typename T, bool CPLX, int BM, int BN, int NO>
__global__ void __launch_bounds__(256)
gram_reduce_kernel(const T* __restrict__ work, int m, int n, int herm, int nJ,
                   int nchunks, double alpha, int conj_out, int i0,
                   double* __restrict__ C) {
    constexpr int NC = CPLX ? 2 : 1;
    constexpr int NG = 256 / NO;
    __shared__ double red[NC][NG][NO + 1];
    const int jl = threadIdx.x % NO, grp = threadIdx.x / NO;
    const int i = i0 + (int)blockIdx.y, j = blockIdx.x * NO + jl;
    if (herm && i < (int)blockIdx.x * NO) return;   // the whole block is above
    const bool live = j < n && (!herm || j <= i);
    double re = 0.0, im = 0.0;
    if (live) {
        const int I = i / BM, J = j / BN;
        const int pair = herm ? herm_pair_index(I, J, BM / BN) : I * nJ + J;
        const T* p = work + (int64_t)pair * nchunks * NC * BM * BN + (i % BM) * BN + j % BN;
#pragma unroll 4
        for (int c = grp; c < nchunks; c += NG) {
            re += (double)p[(int64_t)c * NC * BM * BN];
            if (CPLX) im += (double)p[(int64_t)c * NC * BM * BN + BM * BN];
        }
    }
    red[0][grp][jl] = re;
    if (CPLX) red[NC - 1][grp][jl] = im;
    __syncthreads();
    if (grp > 0 || !live) return;
    re = im = 0.0;
    for (int g = 0; g < NG; g++) {
        re += red[0][g][jl];
        if (CPLX) im += red[NC - 1][g][jl];
    }
    if (conj_out) im = -im;
    if (herm && i == j) im = 0.0;   // a Hermitian matrix has a real diagonal
    const int64_t t = (int64_t)i * n + j, u = (int64_t)j * n + i;
    if (CPLX) {
        C[2 * t] = alpha * re;
        C[2 * t + 1] = alpha * im;
        if (herm) {
            C[2 * u] = alpha * re;
            C[2 * u + 1] = i == j ? alpha * im : -(alpha * im);
        }
    } else {
        C[t] = alpha * re;
        if (herm) C[u] = alpha * re;
    }
}

struct GramPlan {
    int BN, npairs, nI, nJ, nchunks;
    bool small;
    int64_t nseg, work_bytes;
};

GramPlan gram_plan(int dtype, int64_t m, int64_t n, int64_t kbytes, int herm) {
    GramPlan p;
    const int es = dtype_size(dtype);   // complex: two parts of half size
    p.nseg = (kbytes + kSeg - 1) / kSeg;
    p.small = m <= kSB && n <= kSB;
    if (p.small) {
        // up to 256 workgroups (one wave per SIMD, what the registers allow)
        // of 4 (complex128: 2) slices, at least 4 segments per slice
        const int ks = dtype == GH_C128 ? 2 : 4;
        p.BN = kSB;
        p.nI = p.nJ = p.npairs = 1;
        p.nchunks = (int)std::max<int64_t>(1, std::min<int64_t>(256, p.nseg / (4 * ks)));
        const int nc = dtype == GH_C128 || dtype == GH_C64 ? 2 : 1;
        p.work_bytes = (int64_t)p.nchunks * nc * kSB * kSB * (int64_t)sizeof(double);
        return p;
    }
    p.BN = dtype == GH_C128 ? 64 : 128;
    p.nI = (int)((m + kBM - 1) / kBM);
    p.nJ = (int)((n + p.BN - 1) / p.BN);
    const int q = kBM / p.BN;
    p.npairs = herm ? q * p.nI * (p.nI + 1) / 2 : p.nI * p.nJ;
    // about 1024 workgroups (4 per CU), a multiple of the XCD count, and
    // at least 16 segments per chunk
    int64_t nc = std::max<int64_t>(1, 1024 / std::max(p.npairs, 1));
    nc = std::min<int64_t>(nc, std::max<int64_t>(1, p.nseg / 16));
    while (nc > 1 && (p.npairs * nc) % kNumXCD) nc--;
    p.nchunks = (int)nc;
    p.work_bytes = (int64_t)p.npairs * p.nchunks * kBM * p.BN * es;
    return p;
}

template <typename T, bool CPLX, int BM, int BN>
int launch_gram_reduce(const GramPlan& pl, int m, int n, double alpha, int herm, int conj_out,
                       double* C, const void* work, hipStream_t st) {
    const int nchunks = pl.nseg > 0 ? pl.nchunks : 0;
    for (int i0 = 0; i0 < m; i0 += (int)kBandSlice) {   // one grid row per output row
        const int mi = std::min<int>((int)kBandSlice, m - i0);
        auto go = [&](auto outputs) {
            constexpr int NO = decltype(outputs)::value;
            hipLaunchKernelGGL((gram_reduce_kernel<T, CPLX, BM, BN, NO>),
                               dim3((unsigned)((n + NO - 1) / NO), (unsigned)mi), dim3(256), 0,
                               st, (const T*)work, m, n, herm, pl.nJ, nchunks, alpha, conj_out, i0,
                               C);
        };
        if (nchunks > 16 || n <= 16) go(std::integral_constant<int, 16>{});
        else if (nchunks > 4 || n <= 64) go(std::integral_constant<int, 64>{});
        else go(std::integral_constant<int, 256>{});
        GH_CHECK_LAUNCH();
    }
    return GH_OK;
}

template <typename T, bool CPLX, int WN>
int launch_gram_mfma(const GramPlan& pl, int m, int n, int64_t kbytes,
                     const void* A, int64_t lda, const void* B, int64_t ldb,
                     double alpha, int herm, int conj_out, double* C, void* work,
                     hipStream_t st) {
    if (pl.small) {
        if (pl.nseg > 0) {
            hipLaunchKernelGGL((gram_small_kernel<T, CPLX>), dim3(pl.nchunks), dim3(kThreads), 0,
                               st, (const char*)A, (const char*)B, lda, ldb, m, n, pl.nseg,
                               kbytes, herm, (double*)work);
            GH_CHECK_LAUNCH();
        }
        return launch_gram_reduce<double, CPLX, kSB, kSB>(pl, m, n, alpha, herm, conj_out, C,
                                                          work, st);
    }
    const int nblk = pl.npairs * pl.nchunks;
    if (nblk > 0 && pl.nseg > 0) {
        hipLaunchKernelGGL((gram_mfma_kernel<T, CPLX, WN>), dim3(nblk), dim3(kThreads), 0, st,
                           (const char*)A, (const char*)B, lda, ldb, m, n, pl.nseg, kbytes,
                           herm, pl.npairs, pl.nJ, pl.nchunks, (T*)work);
        GH_CHECK_LAUNCH();
    }
    return launch_gram_reduce<T, CPLX, kBM, 2 * WN>(pl, m, n, alpha, herm, conj_out, C, work,
                                                    st);
}

}  // namespace

}  // namespace gh

using namespace gh;

extern "C" {

int64_t gh_gram_work_bytes(int dtype, int64_t m, int64_t n, int64_t k, int hermitian) {
    if (dtype < GH_F64 || dtype > GH_C64 || m < 0 || n < 0 || k < 0) return -1;
    return gram_plan(dtype, m, n, k * dtype_size(dtype), hermitian).work_bytes;
}

int gh_gram(int dtype, int64_t m, int64_t n, int64_t k, const void* A_dev,
            int64_t lda, const void* B_dev, int64_t ldb, double alpha,
            int hermitian, int conj_out, double* C_dev, void* work_dev,
            int64_t work_bytes, void* stream) {
    GH_REQUIRE(dtype >= GH_F64 && dtype <= GH_C64, GH_ERR_ARG, "gram: bad dtype");
    GH_REQUIRE(m >= 0 && n >= 0 && k >= 0 && m < (1 << 20) && n < (1 << 20), GH_ERR_ARG,
               "gram: bad sizes m=%lld n=%lld k=%lld", (long long)m, (long long)n,
               (long long)k);
    GH_REQUIRE(!hermitian || m == n, GH_ERR_SHAPE, "gram: Hermitian mode needs m == n");
    if (m == 0 || n == 0) return GH_OK;
    GH_REQUIRE(A_dev && B_dev && C_dev, GH_ERR_ARG, "gram: null argument");
    GH_REQUIRE(lda >= k && ldb >= k, GH_ERR_ARG, "gram: row pitch below k");
    const int es = dtype_size(dtype);
    const int64_t kbytes = k * es;
    GH_REQUIRE(kbytes % 16 == 0 && (lda * es) % 16 == 0 && (ldb * es) % 16 == 0,
               GH_ERR_UNSUPPORTED, "gram: rows must be multiples of 16 bytes");
    GH_REQUIRE(((uintptr_t)A_dev & 15) == 0 && ((uintptr_t)B_dev & 15) == 0,
               GH_ERR_UNSUPPORTED, "gram: A and B must be 16-byte aligned");
    const GramPlan pl = gram_plan(dtype, m, n, kbytes, hermitian);
    GH_REQUIRE(work_dev || pl.work_bytes == 0, GH_ERR_ARG, "gram: null workspace");
    GH_REQUIRE(work_bytes >= pl.work_bytes, GH_ERR_ARG,
               "gram: workspace of %lld bytes, %lld needed", (long long)work_bytes,
               (long long)pl.work_bytes);
    hipStream_t st = (hipStream_t)stream;
    const int mi = (int)m, ni = (int)n;
    const int64_t la = lda * es, lb = ldb * es;
    switch (dtype) {
        case GH_F32:
            return launch_gram_mfma<float, false, 64>(pl, mi, ni, kbytes, A_dev, la, B_dev, lb,
                                                      alpha, hermitian, conj_out, C_dev,
                                                      work_dev, st);
        case GH_C64:
            return launch_gram_mfma<float, true, 64>(pl, mi, ni, kbytes, A_dev, la, B_dev, lb,
                                                     alpha, hermitian, conj_out, C_dev,
                                                     work_dev, st);
        case GH_F64:
            return launch_gram_mfma<double, false, 64>(pl, mi, ni, kbytes, A_dev, la, B_dev,
                                                       lb, alpha, hermitian, conj_out, C_dev,
                                                       work_dev, st);
        case GH_C128:
            return launch_gram_mfma<double, true, 32>(pl, mi, ni, kbytes, A_dev, la, B_dev,
                                                      lb, alpha, hermitian, conj_out, C_dev,
                                                      work_dev, st);
    }
    return GH_ERR_ARG;
}

}  // extern "C"
