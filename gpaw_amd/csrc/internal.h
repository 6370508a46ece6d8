// Library-internal entry points shared between translation units.
#pragma once

#include "common.h"

namespace gh {

// out = alpha * (L in) + gamma * in [+ vt .* in] [+ beta * src]
int stencil_apply_scaled(const gh_stencil* h, const void* in, void* out,
                         int64_t nbands, const double* phase_cd,
                         const void* vt, const void* src, double beta,
                         double alpha, double gamma, hipStream_t st);

// as stencil_apply_scaled, with the centre coefficient alpha c0 + gamma -
// eps[band] per band (eps: nbands device doubles or null); orthogonal
// stencils only
int stencil_apply_full(const gh_stencil* h, const void* in, void* out,
                       int64_t nbands, const double* phase_cd,
                       const void* vt, const void* src, double beta,
                       double alpha, double gamma, const double* eps,
                       hipStream_t st);

// A stencil along the grid axes for the LDS-free kernel (stencil_direct.hip):
// grid, boundaries, radius and coefficients; rows / planes: tile (0: chosen)
constexpr int kDirectMaxR = 6;
struct DirectStencil {
    int n[3], pbc[3], R;
    double c0, cm[3][kDirectMaxR], cp[3][kDirectMaxR];
    int rows, planes;
};
int stencil_direct(int dtype, const DirectStencil& h, const void* in, void* out,
                   int64_t nbands, const double* phase_cd, const void* vt,
                   const void* src, double beta, double alpha, double gamma,
                   const double* eps, hipStream_t st);

// The LDS ring (stencil_rows.hip): stencils of radius 1..6, rows of any length and alignment, any Bloch phases;
// GH_ERR_UNSUPPORTED where no tile fits
int stencil_rows(int dtype, const DirectStencil& h, const void* in, void* out,
                 int64_t nbands, const double* phase_cd, const void* vt,
                 const void* src, double beta, double alpha, double gamma,
                 const double* eps, int ncu, hipStream_t st);

// The stencil as axis coefficients; false for another form, or where
// GPAW_AMD_STENCIL names a kernel
bool stencil_axes(const gh_stencil* h, DirectStencil* out);

// A transformer with nn = 1: input and output grid, ghosts below the input,
// fine points skipped below (interpolation), boundaries
struct LinearMap {
    int n[3], m[3], plo[3], skip[3], pbc[3];
    bool interp;
};
bool transformer_linear(const gh_transformer* h, int dtype, LinearMap* out);

// out = [base +] al * T(in) (transformers_linear.hip); base only with
// interpolation, may be out
int linear_map(int dtype, const LinearMap& h, const void* in, void* out, const void* base,
               int64_t nb, const double* phase_cd, double al, hipStream_t st);

// out = al * (L I u) + ga * I u + sum_q beta[q] src[q] (1 or 2 sources), I the
// interpolation (stencil_interp.hip); GH_ERR_UNSUPPORTED where that kernel
// has no path
int stencil_interp(const gh_stencil* h, const gh_transformer* intp, const void* u, void* out,
                   int64_t nb, const double* phase_cd, int ns, const void* const* src,
                   const double* beta, double al, double ga, hipStream_t st);

// Jacobi sweeps of a small real grid in one launch (relax_small.hip), the
// function from f to out (may be f); out' = al * L f + ga * f + beta * s;
// GH_ERR_UNSUPPORTED for larger grids and other stencils
int relax_small(const gh_stencil* h, const void* f, void* out, const void* s, int sweeps,
                double beta, double al, double ga, hipStream_t st);

int device_cu_count(int* out);
int ensure_max_lds(const void* kernel, int bytes);

// out = alpha * T(in)
int transformer_apply_scaled(const gh_transformer* h, const void* in,
                             void* out, int64_t nbands,
                             const double* phase_cd, double alpha,
                             hipStream_t st);

int64_t stencil_points(const gh_stencil* h);
int stencil_dtype(const gh_stencil* h);
int64_t transformer_in_points(const gh_transformer* h);
int64_t transformer_out_points(const gh_transformer* h);

}  // namespace gh
