// ref_fft.hpp -- compiled transforms and the right-hand side on the reference
// layout (one field = cI x ny complex, x fastest), for the lengths that have
// a lane-group FFT (fft_wave.hpp). The other lengths run on the runtime plans
// of kernels_ref.hpp. Implemented in ref_fft.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "fft_block.hpp"

namespace s2d {

// A grid as these kernels see it. kx = i, ky = j (or j - ny above ny / 2).
struct RefGrid {
    int cI, ny;             // complex row length (nx / 2 + 1), rows
    int h;                  // nx / 2, the length of the rows' complex transforms
    const void *tw_col;     // exp(-2 pi i e / ny)
    const void *tw_h;       // exp(-2 pi i e / h)
    const void *tw_x;       // exp(-2 pi i e / nx)
    double norm;            // nx * ny
    int x_mask, y_mask;     // Nyquist column and row (-1: none)
    long long kc2;          // kept modes: kx^2 + ky^2 <= kc2
};

// Lengths with compiled kernels: columns (ny) and rows (h).
bool ref_col_ok(int ny);
bool ref_row_ok(int h);

// np planes ps elements apart, in place. dir -1 forward, +1 inverse;
// normalize: the result divided by norm (TransformR2C).
template <typename T>
void ref_col(hipStream_t st, const RefGrid &g, cpx<T> *data, int dir, bool normalize, int np,
             long long ps);
template <typename T>
void ref_row(hipStream_t st, const RefGrid &g, cpx<T> *data, bool r2c, int np, long long ps);

// ComputeRHS in three launches (src/Spectral.F90:396-482), with the results of
// the routines one by one: u, v from psi_in and the inverse column transforms
// of u, v, w; the rows to physical space, the products u w and v w, the rows
// back; the forward columns, Truncate, DuDx, DuDy and the sum.
// stage 0: u, v, w and dW receive what ComputeRHS leaves in them. Stages 1,
// 2, 3: the Shu-Osher update as well (src/TimeIntegration.F90:156-209), with
// w0 the step's W, then ComputePsi and Truncate; out, psi: the new stage and
// its streamfunction. Stage 1 also leaves the round-tripped W in w, stage 3
// u, v, w (WS) and dW. What the next stage overwrites or never reads (the
// columns past the kept ones, zero by Truncate) is not stored.
template <typename T>
void ref_rhs(hipStream_t st, const RefGrid &g, const cpx<T> *psi_in, cpx<T> *u, cpx<T> *v,
             cpx<T> *w, cpx<T> *dW, double nu, int stage, double dt, const cpx<T> *w0, cpx<T> *out,
             cpx<T> *psi);

} // namespace s2d
