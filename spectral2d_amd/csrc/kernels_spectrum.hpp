// kernels_spectrum.hpp -- the shell energy spectrum of ComputeSpectrum
// (src/Analysis.F90:267-460) on the device, in FP64.
//
// Shell b holds the modes with floor(|k| + 1/2) = b (the reference's edges
// 0, 0.5, 1.5, ..., with a binary search; |k| is never a half-integer for
// integer wavenumbers, so the two agree): kx^2 + ky^2 = 0 for b = 0 and
// b^2 - b + 1 <= kx^2 + ky^2 <= b^2 + b for b >= 1. One block per shell
// walks its annulus in a fixed order and reduces in a fixed tree, so the
// result does not depend on scheduling.
//
// The walk goes along kx where |ky| >= kx and along ky where |ky| < kx: a
// step then meets one or two modes on either side of zero. (Along kx alone,
// the thread at kx = b has sqrt(2 b) of them on a side, one read behind the
// other.)
#pragma once

#include "fft_block.hpp"

namespace s2d {

// integer square root: the largest r with r*r <= m
template <typename U>
__device__ __forceinline__ U isqrt_floor(U m)
{
    U r = (U)sqrt((double)m);
    while (r * r > m) --r;
    while ((r + 1) * (r + 1) <= m) ++r;
    return r;
}

// Energy density Ehat = |u_hat|^2 + |v_hat|^2 of one mode from psi_hat,
// with u = DuDy(psi) (ky = kyMG row masked) and v = -DuDx(psi) (kx = kxMG
// column masked), src/Spectral.F90:576-610, the products of
// src/Analysis.F90:380-386.
template <typename T>
__device__ __forceinline__ double mode_energy(cpx<T> p, int kx, int ky, bool mx, bool my)
{
    const double a = (double)p.re, b = (double)p.im;
    const double fy = my ? 0.0 : (double)ky, fx = mx ? 0.0 : (double)kx;
    const double ur = -(fy * b), ui = fy * a;
    const double vr = -1.0 * (-(fx * b)), vi = -1.0 * (fx * a);
    return (ur * ur + ui * ui) + (vr * vr + vi * vi);
}

// Ehat of one mode from the velocity spectra themselves, as
// ComputeSpectrum forms it from its uC, vC arguments (src/Analysis.F90:384).
template <typename T>
__device__ __forceinline__ double mode_energy_uv(cpx<T> u, cpx<T> v)
{
    const double ur = (double)u.re, ui = (double)u.im, vr = (double)v.re, vi = (double)v.im;
    return (ur * ur + ui * ui) + (vr * vr + vi * vi);
}

// ek[b] for b in [0, nbins), in the reference layout (cISize, nyG) with
// FFTW-order rows: from psi (UV false; v unused) or from the velocity
// spectra u, v (UV true). kxMG / kyMG: the Nyquist wavenumbers (masked and
// weight 1/2 at kx = 0 and kx = kxMG, src/Analysis.F90:389-395). cnt[b]: the
// shell's modes of the full spectrum (weights 1 / 2, src/Analysis.F90:389-395),
// counted on the walk. Bound by the latency of the annuli's strided reads:
// eight neighbouring shells, which share their cache lines, go to one XCD.
// Np = 1536 FP64: 14 us (36 along kx alone). U: unsigned where (nb + 1)^2
// fits, else 64 bits.
template <typename T, bool UV, typename U>
__global__ __launch_bounds__(256) void k_spectrum(const cpx<T> *__restrict__ psi,
                                                  const cpx<T> *__restrict__ v, int cISize,
                                                  int nyG, int kxMG, int kyMG, int maskX,
                                                  int maskY, int nb, double *__restrict__ ek,
                                                  int *__restrict__ cnt)
{
    __shared__ double red[256];
    __shared__ int redc[256];
    // 64 consecutive blocks hold 64 shells, eight to an XCD (blocks go round the XCDs)
    const int bl = (int)blockIdx.x, in = bl & 63;
    const int shell = (bl - in) + (in & 7) * 8 + (in >> 3);
    if (shell >= nb) return; // (the grid is rounded up to 64)
    const U b = (U)shell;
    const U lo = b == 0 ? 0 : b * b - b + 1, hi = b * b + b * (b != 0);
    const int diag = (int)isqrt_floor<U>(hi / 2); // the last kx with |ky| >= kx in the shell
    const int kyMin = nyG / 2 - nyG + 1, kyLow = -(nyG / 2) + 1;
    double acc = 0.0;
    int n = 0;
    // steps 0..diag: kx = step, |ky| >= kx; then ky = step - diag - 1, kx > |ky|
    for (int st = threadIdx.x; st <= 2 * diag + 1; st += blockDim.x) {
        const bool alongx = st <= diag;
        const U f = (U)(alongx ? st : st - diag - 1), f2 = f * f;
        if (f2 > hi) continue;
        const U r_hi = isqrt_floor<U>(hi - f2);
        U r_lo = lo <= f2 ? 0 : isqrt_floor<U>(lo - f2 - 1) + 1;
        const U first = alongx ? f : f + 1;
        if (r_lo < first) r_lo = first;
        for (U r = r_lo; r <= r_hi; ++r) {
            const int kx = (int)(alongx ? f : r), ka = (int)(alongx ? r : f);
            if (kx >= cISize) break;
            const double wt = (kx == 0 || kx == kxMG) ? 0.5 : 1.0;
            const bool mx = maskX && kx == kxMG;
            // ky = ka and, for ka > 0, -ka (FFTW rows: ky >= 0 at j = ky, ky < 0 at nyG + ky)
#pragma unroll
            for (int sgn = 0; sgn < 2; ++sgn) {
                const int ky = sgn == 0 ? ka : -ka;
                if (ky > nyG / 2 || ky < kyMin || (sgn == 1 && ka == 0)) continue;
                n += (kx == 0 || kx == kxMG) ? 1 : 2;
                if (ky < kyLow) continue; // (the lowest row of an odd nyG: counted only)
                const int j = ky >= 0 ? ky : nyG + ky;
                const bool my = maskY && ky == kyMG;
                const size_t o = (size_t)kx + (size_t)j * cISize;
                if constexpr (UV)
                    acc += wt * mode_energy_uv(psi[o], v[o]);
                else
                    acc += wt * mode_energy(psi[o], kx, ky, mx, my);
            }
        }
    }
    red[threadIdx.x] = acc;
    redc[threadIdx.x] = n;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            red[threadIdx.x] += red[threadIdx.x + s];
            redc[threadIdx.x] += redc[threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        ek[b] = red[0];
        cnt[b] = redc[0];
    }
}

} // namespace s2d
