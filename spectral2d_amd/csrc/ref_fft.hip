// ref_fft.hip -- the reference-layout transforms and ComputeRHS on lane-group
// FFTs (declared in ref_fft.hpp).
//
// Columns. A block takes LPB adjacent columns; thread = column + LPB * t, so
// that the load or store of an element covers LPB adjacent elements of each
// row; the transforms exchange through LDS behind workgroup barriers (wave
// fences when the block is one wave). Blocks are XCD-major: those that share
// the lines of adjacent columns run on one XCD. Wider tiles (64-byte segments
// at Np = 1536 FP64, 32 at 3072 FP32) measured the same: the column kernels
// move 2 to 3 TB/s whatever the width, bound by the 12 KB row stride. Storing
// the fields between the launches tile by tile instead took 20 % off the
// column kernels and doubled the row kernel's time.
// Rows. A lane group per row (length nx / 2, the even/odd packing of a real
// row), several rows per block; the mirrored elements of the packing come
// through LDS, its twiddles from one loaded value each and constants.
//
// ComputeRHS on these is three launches where the routines one by one are
// seventeen: every field crosses memory once each way per launch, and the
// physical-space fields never do. Measured, 1536^2 padded FP64 (18.9 MB a
// field), us: columns of one field 38 -> 14 forward or inverse, rows 16 -> 10
// to 13; ComputeRHS 370 -> 105 (velocity 25, rows 36, columns 47 moving 94,
// 113 and 132 MB); IntegrateOneStep 1291 -> 337.
#include <hip/hip_runtime.h>

#include "kernels_fused_v2.hpp"
#include "ref_fft.hpp"

namespace s2d {
namespace {

// Elements per lane and lanes of a compiled length, 3 2^k or 9 2^k (the
// lengths the 3/2 rule gives).
template <int N>
struct CtLen {
    static constexpr int E = 12, TG = N / E;
};

// The twiddles, all from the table: in one batch ahead of the transform, in
// FP64 the early passes' only (the others as the final pass uses them, from
// L1). Products of three of them in the final pass's place took 4 % less
// time, but left a larger error than the runtime plans (4.8e-16 against
// 4.1e-16 of a 1024^2 IntegrateOneStep). Butterflies take sqrt(3)/2 in two
// terms (TW_ACC), with which every length is at least as accurate as its
// runtime plan.
template <typename T, int N>
constexpr int ct_tw()
{
    return TW_ACC | (sizeof(T) == 8 ? TW_EARLY : TW_ALL);
}

constexpr int round_up(int a, int b) { return (a + b - 1) / b * b; }

// ------------------------------------------------------------- columns

template <typename T, int NY>
struct ColCfg {
    static constexpr int E = CtLen<NY>::E, TG = CtLen<NY>::TG;
    // columns per block: segments of 64 to 128 bytes while a block stays at
    // 256 threads (FP32: 512), at least two
    static constexpr int WANT = (sizeof(T) == 8 ? 256 : 512) / TG;
    static constexpr int CAP = sizeof(T) == 8 ? 8 : 16;
    static constexpr int P2 = WANT >= 16 ? 16 : WANT >= 8 ? 8 : WANT >= 4 ? 4 : 2;
    static constexpr int LPB = P2 < CAP ? P2 : CAP;
    static constexpr int THR = LPB * TG;
    static constexpr bool BLK = THR > 64;
    // slices spaced so that LPB columns x consecutive elements spread evenly
    // over the banks (PH elements cover them)
    static constexpr int PH = 256 / (int)sizeof(cpx<T>);
    static constexpr int SL = round_up(LdsMap<TG>::size(NY), PH) + PH / LPB;
    static_assert(THR <= 1024, "column block too large");
    static constexpr int WPE = sizeof(T) == 8 ? (THR > 384 ? 2 : 3) : 4; // waves per SIMD
};

// v / norm of TransformR2C (src/Spectral.F90:761-762); FP32: div_real's
// product with 1 / norm.
template <typename T, int E>
__device__ __forceinline__ void normalized(cpx<T> (&v)[E], double norm)
{
#pragma clang fp contract(off)
    if constexpr (sizeof(T) == 8) {
        const double r = 1.0 / norm;
        bool odd = false;
        cpx<T> y[E];
#pragma unroll
        for (int s = 0; s < E; ++s)
            y[s] = mk<T>(div_by(v[s].re, norm, r, &odd), div_by(v[s].im, norm, r, &odd));
        if (odd) {
#pragma unroll
            for (int s = 0; s < E; ++s) y[s] = div_real(v[s], norm);
        }
#pragma unroll
        for (int s = 0; s < E; ++s) v[s] = y[s];
    } else {
#pragma unroll
        for (int s = 0; s < E; ++s) v[s] = div_real(v[s], norm);
    }
}

// The block's place: column i of element rows t + TG s.
struct ColPlace {
    int g, t, i;
    bool active, any;
};
template <typename T, int NY>
__device__ __forceinline__ ColPlace col_place(int cI, int tile)
{
    using C = ColCfg<T, NY>;
    ColPlace p;
    p.g = threadIdx.x % C::LPB;
    p.t = threadIdx.x / C::LPB;
    const int i0 = tile * C::LPB;
    p.any = i0 < cI; // block-uniform
    p.i = i0 + p.g;
    p.active = p.i < cI;
    return p;
}
template <typename T, int NY>
dim3 col_blocks(int cI, int np, int fields = 1)
{
    constexpr int LPB = ColCfg<T, NY>::LPB;
    return dim3(round_up(fields * ((cI + LPB - 1) / LPB), 8), np);
}

// A column's elements t + TG s (inactive columns read the last one).
template <typename T, int NY>
__device__ __forceinline__ void col_load(cpx<T> (&v)[CtLen<NY>::E], const cpx<T> *__restrict__ f,
                                         const ColPlace &p, int cI)
{
    const cpx<T> *c = f + (p.active ? p.i : cI - 1) + (size_t)p.t * cI;
#pragma unroll
    for (int s = 0; s < CtLen<NY>::E; ++s) v[s] = c[(size_t)(CtLen<NY>::TG * s) * cI];
}
template <typename T, int NY>
__device__ __forceinline__ void col_store(const cpx<T> (&v)[CtLen<NY>::E], cpx<T> *f,
                                          const ColPlace &p, int cI)
{
    if (!p.active) return;
    cpx<T> *c = f + p.i + (size_t)p.t * cI;
#pragma unroll
    for (int s = 0; s < CtLen<NY>::E; ++s) c[(size_t)(CtLen<NY>::TG * s) * cI] = v[s];
}

template <typename T, int NY, int D>
__device__ __forceinline__ void col_fft(cpx<T> (&v)[CtLen<NY>::E], cpx<T> *slice, int t,
                                        const GroupTw<T, CtLen<NY>::E, CtLen<NY>::TG, ct_tw<T, NY>()> &gt)
{
    using C = ColCfg<T, NY>;
    group_fft<T, C::E, C::TG, D, ct_tw<T, NY>(), C::BLK>(v, slice, t, gt);
}

template <typename T, int NY, int D>
__global__ __launch_bounds__((ColCfg<T, NY>::THR))
__attribute__((amdgpu_waves_per_eu(ColCfg<T, NY>::WPE))) void
k_ct_col(cpx<T> *data, int cI, const cpx<T> *__restrict__ tw, int normalize, double norm,
         long long ps)
{
    using C = ColCfg<T, NY>;
    __shared__ cpx<T> lds[C::LPB * C::SL];
    const ColPlace p = col_place<T, NY>(cI, xcd_major(blockIdx.x, gridDim.x));
    if (!p.any) return;
    data += (size_t)blockIdx.y * ps;
    cpx<T> v[C::E];
    col_load<T, NY>(v, data, p, cI);
    GroupTw<T, C::E, C::TG, ct_tw<T, NY>()> gt;
    gt.load(tw, p.t);
    col_fft<T, NY, D>(v, lds + p.g * C::SL, p.t, gt);
    if (normalize) normalized<T, C::E>(v, norm);
    col_store<T, NY>(v, data, p, cI);
}

// Signed wavenumber of row j.
__device__ __forceinline__ int ky_of(int j, int ny) { return j > ny / 2 ? j - ny : j; }

// u = II ky psi, v = -(II kx psi) (ComputeVelocity, src/Spectral.F90:591-603)
// and w: the inverse transforms of their first ncol columns, u and v written,
// w in place. A block per field and column tile, the field fastest, so that the blocks that
// read one tile of psi run together on one XCD.
template <typename T, int NY>
__global__ __launch_bounds__((ColCfg<T, NY>::THR))
__attribute__((amdgpu_waves_per_eu(ColCfg<T, NY>::WPE))) void
k_rhs_velocity(const cpx<T> *__restrict__ psi, cpx<T> *__restrict__ u, cpx<T> *__restrict__ v,
               cpx<T> *w, int cI, int ncol, const cpx<T> *__restrict__ tw, int x_mask, int y_mask)
{
#pragma clang fp contract(off)
    using C = ColCfg<T, NY>;
    __shared__ cpx<T> lds[C::LPB * C::SL];
    const int job = xcd_major(blockIdx.x, gridDim.x), f = job % 3;
    const ColPlace p = col_place<T, NY>(ncol, job / 3);
    if (!p.any) return;
    cpx<T> x[C::E];
    col_load<T, NY>(x, f == 2 ? w : psi, p, cI);
    GroupTw<T, C::E, C::TG, ct_tw<T, NY>()> gt;
    gt.load(tw, p.t);
    const cpx<T> zero = mk<T>((T)0, (T)0);
    const T qx = (T)p.i;
    if (f < 2) { // block-uniform
#pragma unroll
        for (int s = 0; s < C::E; ++s) {
            const int j = p.t + C::TG * s;
            const T q = f == 0 ? (T)ky_of(j, NY) : qx;
            const bool off = f == 0 ? j == y_mask : p.i == x_mask;
            const cpx<T> r = sel(off, zero, mk<T>(-(q * x[s].im), q * x[s].re));
            x[s] = f == 0 ? r : mk<T>((T)-1 * r.re, (T)-1 * r.im);
        }
    }
    col_fft<T, NY, 1>(x, lds + p.g * C::SL, p.t, gt);
    col_store<T, NY>(x, f == 0 ? u : f == 1 ? v : w, p, cI);
}

// The arguments of k_rhs_columns.
template <typename T>
struct RhsArgs {
    cpx<T> *u, *v, *w, *dW;
    const cpx<T> *w0;
    cpx<T> *out, *psi;
    int cI, ncol, x_mask, y_mask;
    long long kc2;
    double norm, nu, dt;
    const cpx<T> *tw;
};

// The forward column transforms of u w, v w and w, then per mode
// TransformR2C's division, Truncate, DuDx / DuDy and dW = -u - v - nu k^2 w
// (src/Spectral.F90:451-481), and with STAGE 1-3 the Shu-Osher update,
// ComputePsi and Truncate (see ref_rhs_columns), in the routines' own
// expression order. One field's column is in flight at a time next to the sum
// (FP64: at the lengths 3 2^k stages 0 and 3 keep 2 to 16 registers in scratch;
// with a second column loaded ahead they took 10 % longer).
template <typename T, int NY, int STAGE>
__global__ __launch_bounds__((ColCfg<T, NY>::THR))
__attribute__((amdgpu_waves_per_eu(2))) void
k_rhs_columns(RhsArgs<T> A)
{
#pragma clang fp contract(off)
    using C = ColCfg<T, NY>;
    __shared__ cpx<T> lds[C::LPB * C::SL];
    const int cI = A.cI;
    const cpx<T> zero = mk<T>((T)0, (T)0);
    constexpr bool ALL = STAGE == 0 || STAGE == 3; // u, v, w, dW stay
    const ColPlace p = col_place<T, NY>(cI, xcd_major(blockIdx.x, gridDim.x));
    if (!p.any) return;
    cpx<T> x[C::E], r[C::E];
    // stages 1 and 2: the columns past the kept ones hold zeros, which only
    // the streamfunction of stage 2 is left with (PSIS)
    if (p.i - p.g >= A.ncol) { // block-uniform
        if constexpr (STAGE == 2) {
#pragma unroll
            for (int s = 0; s < C::E; ++s) x[s] = zero;
            col_store<T, NY>(x, A.psi, p, cI);
        }
        return;
    }
    col_load<T, NY>(x, A.u, p, cI);
    GroupTw<T, C::E, C::TG, ct_tw<T, NY>()> gt;
    gt.load(A.tw, p.t);
    cpx<T> *slice = lds + p.g * C::SL;
    const T qx = (T)p.i;
    auto cut = [&](int s) { // Truncate
        const int ky = ky_of(p.t + C::TG * s, NY);
        return (long long)p.i * p.i + (long long)ky * ky > A.kc2;
    };
    // u w: DuDx
    col_fft<T, NY, -1>(x, slice, p.t, gt);
    normalized<T, C::E>(x, A.norm);
#pragma unroll
    for (int s = 0; s < C::E; ++s) {
        const cpx<T> a = sel(cut(s), zero, x[s]);
        x[s] = sel(p.i == A.x_mask, zero, mk<T>(-(qx * a.im), qx * a.re));
        r[s] = mk<T>(-x[s].re, -x[s].im);
    }
    if constexpr (ALL) col_store<T, NY>(x, A.u, p, cI);
    // v w: DuDy
    col_load<T, NY>(x, A.v, p, cI);
    col_fft<T, NY, -1>(x, slice, p.t, gt);
    normalized<T, C::E>(x, A.norm);
#pragma unroll
    for (int s = 0; s < C::E; ++s) {
        const int j = p.t + C::TG * s;
        const T q = (T)ky_of(j, NY);
        const cpx<T> a = sel(cut(s), zero, x[s]);
        x[s] = sel(j == A.y_mask, zero, mk<T>(-(q * a.im), q * a.re));
        r[s] = sub(r[s], x[s]);
    }
    if constexpr (ALL) col_store<T, NY>(x, A.v, p, cI);
    // w
    col_load<T, NY>(x, A.w, p, cI);
    col_fft<T, NY, -1>(x, slice, p.t, gt);
    normalized<T, C::E>(x, A.norm);
#pragma unroll
    for (int s = 0; s < C::E; ++s) {
        const T q = (T)ky_of(p.t + C::TG * s, NY);
        const T k2 = (T)A.nu * (qx * qx + q * q);
        r[s] = mk<T>(r[s].re - k2 * x[s].re, r[s].im - k2 * x[s].im);
    }
    cpx<T> a[C::E];
    if constexpr (STAGE > 1) col_load<T, NY>(a, A.w0, p, cI);
    if constexpr (ALL || STAGE == 1) col_store<T, NY>(x, A.w, p, cI);
    if constexpr (ALL) col_store<T, NY>(r, A.dW, p, cI);
    if constexpr (STAGE > 0) {
        const T dt = (T)A.dt;
#pragma unroll
        for (int s = 0; s < C::E; ++s) {
            const cpx<T> b = x[s], d = r[s];
            cpx<T> o;
            if constexpr (STAGE == 1) {
                o = mk<T>(b.re + dt * d.re, b.im + dt * d.im);
            } else if constexpr (STAGE == 2) {
                const T c = (T)0.25 * dt;
                o = mk<T>(((T)0.75 * a[s].re + (T)0.25 * b.re) + c * d.re,
                          ((T)0.75 * a[s].im + (T)0.25 * b.im) + c * d.im);
            } else {
                const T c = dt * (T)2;
                o = mk<T>((div3_any(a[s].re) + div3_any((T)2 * b.re)) + div3_any(c * d.re),
                          (div3_any(a[s].im) + div3_any((T)2 * b.im)) + div3_any(c * d.im));
            }
            // ComputePsi, then Truncate of both
            const int j = p.t + C::TG * s;
            const T q = (T)ky_of(j, NY);
            const T dd = p.i == 0 ? q * q : j == 0 ? qx * qx : qx * qx + q * q;
            const bool off = cut(s);
            r[s] = sel(off, zero, o);
            x[s] = sel(off || (p.i == 0 && j == 0), zero, mk<T>(o.re / dd, o.im / dd));
        }
        col_store<T, NY>(r, A.out, p, cI);
        col_store<T, NY>(x, A.psi, p, cI);
    }
}

// ---------------------------------------------------------------- rows

template <typename T, int H>
struct RowCfg {
    static constexpr int E = CtLen<H>::E, TG = CtLen<H>::TG;
    // rows per block: 128 threads (whole waves for 3 2^k lanes: 192)
    static constexpr bool P2 = (TG & (TG - 1)) == 0;
    static constexpr int RB = P2 ? (TG >= 128 ? 1 : 128 / TG) : 192 / TG;
    static constexpr int THR = RB * TG;
    static constexpr int PH = 256 / (int)sizeof(cpx<T>);
    static constexpr int SL = round_up(LdsMap<TG>::size(H), PH) + (TG < PH ? TG : 0);
};

template <typename T, int H, int PRE = ct_tw<T, H>()>
using RowTw = GroupTw<T, CtLen<H>::E, CtLen<H>::TG, PRE>;

// twx[t + TG s] = exp(-2 pi i (t + TG s) / (2 H)) from w0 = twx[t]: the step
// TG s is a multiple of 15 degrees, a compile-time constant.
template <typename T, int S>
__device__ __forceinline__ cpx<T> tw_of(cpx<T> w0)
{
    return twiddle_const<T, -1, 24, S>(w0);
}

// The real row of a half spectrum v (x[t + TG s]; last: X_h), as (even, odd)
// pairs: k_row_c2r's arithmetic (only Re of X_0 and X_h is read). The
// mirrored elements come through LDS.
template <typename T, int H, int PRE>
__device__ __forceinline__ void row_c2r(cpx<T> (&v)[CtLen<H>::E], cpx<T> last, int t, cpx<T> w0,
                                        cpx<T> *slice,
                                        const RowTw<T, H, PRE> &gt)
{
    constexpr int E = CtLen<H>::E, TG = CtLen<H>::TG;
    using M = LdsMap<TG>;
    const int it = M::idx(t);
#pragma unroll
    for (int s = 0; s < E; ++s) slice[M::idx_sum(it, TG * s)] = v[s];
    group_sync<TG>();
    static_for<0, E>([&](auto sI) {
        constexpr int s = decltype(sI)::value;
        const int k = t + TG * s;
        cpx<T> a = v[s], b = slice[M::idx(s == 0 && k == 0 ? 0 : H - k)];
        if constexpr (s == 0) {
            b = sel(k == 0, last, b);
            a.im = k == 0 ? (T)0 : a.im;
            b.im = k == 0 ? (T)0 : b.im;
        }
        b.im = -b.im;
        const cpx<T> sm = add(a, b), df = sub(a, b);
        const cpx<T> tt = mulc(df, tw_of<T, s>(w0));
        v[s] = mk<T>(sm.re - tt.im, sm.im + tt.re);
    });
    group_sync<TG>(); // every mirrored element has been read
    group_fft<T, E, TG, 1>(v, slice, t, gt);
}

// The half spectrum of (even, odd) pairs, its first n elements written to the
// row: k_row_r2c's arithmetic.
template <typename T, int H, int PRE>
__device__ __forceinline__ void row_r2c(cpx<T> (&v)[CtLen<H>::E], cpx<T> *row, int t, int n,
                                        cpx<T> w0, cpx<T> *slice,
                                        const RowTw<T, H, PRE> &gt)
{
    constexpr int E = CtLen<H>::E, TG = CtLen<H>::TG;
    using M = LdsMap<TG>;
    group_fft<T, E, TG, -1>(v, slice, t, gt);
    const int it = M::idx(t);
#pragma unroll
    for (int s = 0; s < E; ++s) slice[M::idx_sum(it, TG * s)] = v[s];
    group_sync<TG>();
    auto split = [&](cpx<T> zk, cpx<T> zc, cpx<T> w) {
        zc.im = -zc.im;
        const cpx<T> ev = mk<T>((T)0.5 * (zk.re + zc.re), (T)0.5 * (zk.im + zc.im));
        const cpx<T> od = mk<T>((T)0.5 * (zk.im - zc.im), (T)-0.5 * (zk.re - zc.re));
        const cpx<T> tt = mul(w, od);
        return mk<T>(ev.re + tt.re, ev.im + tt.im);
    };
    static_for<0, E>([&](auto sI) {
        constexpr int s = decltype(sI)::value;
        const int k = t + TG * s;
        const cpx<T> zc = slice[M::idx(s == 0 && k == 0 ? 0 : H - k)];
        const cpx<T> o = split(v[s], zc, tw_of<T, s>(w0));
        if (k < n) row[k] = o;
    });
    if (H < n && t == 0) row[H] = split(v[0], v[0], mk<T>((T)-1, (T)0)); // twx[H]
    group_sync<TG>(); // (the slice's next writer waits for these reads)
}

// A row's elements t + TG s, zeros from the n-th on.
template <typename T, int H>
__device__ __forceinline__ void row_load(cpx<T> (&v)[CtLen<H>::E], const cpx<T> *row, int t, int n)
{
#pragma unroll
    for (int s = 0; s < CtLen<H>::E; ++s) {
        const int k = t + CtLen<H>::TG * s;
        v[s] = mk<T>((T)0, (T)0);
        if (k < n) v[s] = row[k];
    }
}

// The block's row (rows past the end repeat the last one, unstored).
template <typename T, int H>
__device__ __forceinline__ int row_place(int ny, bool *active)
{
    const int j = blockIdx.x * RowCfg<T, H>::RB + (int)threadIdx.x / RowCfg<T, H>::TG;
    *active = j < ny;
    return *active ? j : ny - 1;
}

template <typename T, int H, bool R2C>
__global__ __launch_bounds__((RowCfg<T, H>::THR))
__attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 3 : 4))) void
k_ct_row(cpx<T> *data, int cI, int ny, const cpx<T> *__restrict__ tw,
         const cpx<T> *__restrict__ twx, long long ps)
{
    using C = RowCfg<T, H>;
    __shared__ cpx<T> lds[C::RB * C::SL];
    bool active;
    const int j = row_place<T, H>(ny, &active), t = threadIdx.x % C::TG;
    cpx<T> *row = data + (size_t)blockIdx.y * ps + (size_t)j * cI;
    cpx<T> *slice = lds + threadIdx.x / C::TG * C::SL;
    RowTw<T, H> gt;
    cpx<T> v[C::E];
    row_load<T, H>(v, row, t, H);
    if constexpr (R2C) {
        const cpx<T> w0 = twx[t];
        gt.load(tw, t);
        row_r2c<T, H>(v, row, t, active ? H + 1 : 0, w0, slice, gt);
    } else {
        const cpx<T> last = row[H], w0 = twx[t];
        gt.load(tw, t);
        row_c2r<T, H>(v, last, t, w0, slice, gt);
        if (active) {
#pragma unroll
            for (int s = 0; s < C::E; ++s) row[t + C::TG * s] = v[s];
            if (t == 0) row[H] = mk<T>((T)0, (T)0); // the two padding reals
        }
    }
}

// ComputeRHS's rows (src/Spectral.F90:433-453): u, v, w to physical space, the
// products u w and v w, and all three back, w by the same round trip. nin:
// the columns from there on are zeros (not read); nout: those from there on
// are not needed (not written).
template <typename T, int H>
__global__ __launch_bounds__((RowCfg<T, H>::THR))
__attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 2 : 3))) void
k_rhs_rows(cpx<T> *u, cpx<T> *v, cpx<T> *w, int cI, int nin, int nout, int ny,
           const cpx<T> *__restrict__ tw, const cpx<T> *__restrict__ twx)
{
#pragma clang fp contract(off)
    using C = RowCfg<T, H>;
    __shared__ cpx<T> lds[C::RB * C::SL];
    bool active;
    const int j = row_place<T, H>(ny, &active), t = threadIdx.x % C::TG;
    const size_t at = (size_t)j * cI;
    const int no = active ? nout : 0;
    cpx<T> *slice = lds + threadIdx.x / C::TG * C::SL;
    auto last = [&](const cpx<T> *f) { return nin > H ? f[H] : mk<T>((T)0, (T)0); };
    cpx<T> ww[C::E], x[C::E];
    row_load<T, H>(ww, w + at, t, nin);
    const cpx<T> lw = last(w + at), w0 = twx[t];
    RowTw<T, H> gt;
    gt.load(tw, t);
    row_c2r<T, H>(ww, lw, t, w0, slice, gt);
#pragma unroll 1 // (FP64 puts 6 / 10 / 22 / 34 registers in scratch at H = 192 / 384 / 768 /
                 // 1536; unrolled, holding both fields' tables, 21 / 39 / 70 / 83)
    for (int i = 0; i < 2; ++i) {
        cpx<T> *f = (i == 0 ? u : v) + at;
        row_load<T, H>(x, f, t, nin);
        row_c2r<T, H>(x, last(f), t, w0, slice, gt);
#pragma unroll
        for (int s = 0; s < C::E; ++s) x[s] = mk<T>(x[s].re * ww[s].re, x[s].im * ww[s].im);
        row_r2c<T, H>(x, f, t, no, w0, slice, gt);
    }
    row_r2c<T, H>(ww, w + at, t, no, w0, slice, gt);
}

// The same rows with a lane group to a field: u w, v w and w's round trip run
// beside each other, each group transforming w itself, so that a row's chain
// is three transforms instead of six for half as much work again. For grids
// whose k_rhs_rows blocks leave CUs idle, where that chain is the time
// (rhs_rows_split; the same arithmetic, to the bit).
template <typename T, int H>
struct RowSplitCfg {
    using C = RowCfg<T, H>;
    static constexpr int RB = C::P2 ? (C::TG >= 64 ? 1 : 64 / C::TG) : C::TG >= 96 ? 1 : 96 / C::TG;
    static constexpr int THR = 3 * RB * C::TG;
};

template <typename T, int H>
__global__ __launch_bounds__((RowSplitCfg<T, H>::THR)) void
k_rhs_rows_split(cpx<T> *u, cpx<T> *v, cpx<T> *w, int cI, int nin, int nout, int ny,
                 const cpx<T> *__restrict__ tw, const cpx<T> *__restrict__ twx)
{
#pragma clang fp contract(off)
    using C = RowCfg<T, H>;
    constexpr int RB = RowSplitCfg<T, H>::RB;
    __shared__ cpx<T> lds[3 * RB * C::SL];
    const int gr = (int)threadIdx.x / C::TG, t = threadIdx.x % C::TG;
    const int j0 = blockIdx.x * RB + gr % RB, field = gr / RB;
    const int j = j0 < ny ? j0 : ny - 1; // (rows past the end repeat the last one, unstored)
    const size_t at = (size_t)j * cI;
    cpx<T> *slice = lds + gr * C::SL;
    auto last = [&](const cpx<T> *f) { return nin > H ? f[H] : mk<T>((T)0, (T)0); };
    cpx<T> *f = (field == 0 ? u : field == 1 ? v : w) + at;
    cpx<T> ww[C::E], x[C::E];
    row_load<T, H>(ww, w + at, t, nin);
    row_load<T, H>(x, f, t, nin);
    const cpx<T> lw = last(w + at), lf = last(f), w0 = twx[t];
    RowTw<T, H> gt;
    gt.load(tw, t);
    row_c2r<T, H>(ww, lw, t, w0, slice, gt);
    row_c2r<T, H>(x, lf, t, w0, slice, gt);
#pragma unroll
    for (int s = 0; s < C::E; ++s)
        x[s] = field == 2 ? ww[s] : mk<T>(x[s].re * ww[s].re, x[s].im * ww[s].im);
    __syncthreads(); // (every group has its w: the third may write it)
    row_r2c<T, H>(x, f, t, j0 < ny ? nout : 0, w0, slice, gt);
}

// Rows by k_rhs_rows_split: while k_rhs_rows has no more than 128 blocks in FP64
// and 384 in FP32. Past that the chip is full and the work added
// costs more than the shorter chain gives. ComputeRHS, us, one group to a row /
// one to a field, FP64: 64^2 35.3 / 32.6, 256^2 51.1 / 45.9, 384^2 (72 blocks)
// 58.3 / 55.3, 512 x 256 (96) 57.3 / 51.6, 512^2 (192) 67.7 / 69.9, 256 x 1024
// (192) 72.0 / 74.5; FP32: 64^2 31.8 / 27.9, 512^2 57.4 / 54.8, 512 x 1024 (384)
// 74.2 / 72.2.
template <typename T, int H>
constexpr bool row_split_len()
{
    return H <= 384;
}
template <typename T, int H>
bool rhs_rows_split(int ny)
{
    constexpr int RB = RowCfg<T, H>::RB;
    return row_split_len<T, H>() && (ny + RB - 1) / RB <= (sizeof(T) == 8 ? 128 : 384);
}

// f(std::integral_constant<int, n>) for a compiled length.
template <typename F>
bool with_length(int n, F &&f)
{
#define S2D_LEN(N) case N: f(std::integral_constant<int, N>{}); return true;
    switch (n) {
        S2D_LEN(48) S2D_LEN(96) S2D_LEN(192) S2D_LEN(384) S2D_LEN(768) S2D_LEN(1536) S2D_LEN(3072)
        S2D_LEN(72) S2D_LEN(144) S2D_LEN(288) S2D_LEN(576) S2D_LEN(1152) S2D_LEN(2304)
    }
#undef S2D_LEN
    return false;
}

} // namespace

bool ref_col_ok(int ny) { return with_length(ny, [](auto) {}); }
bool ref_row_ok(int h) { return h <= 1536 && with_length(h, [](auto) {}); }

template <typename T>
void ref_col(hipStream_t st, const RefGrid &g, cpx<T> *data, int dir, bool normalize, int np,
             long long ps)
{
    with_length(g.ny, [&](auto n) {
        constexpr int NY = decltype(n)::value;
        {
            const dim3 grid = col_blocks<T, NY>(g.cI, np), blk(ColCfg<T, NY>::THR);
            const cpx<T> *tw = static_cast<const cpx<T> *>(g.tw_col);
            if (dir < 0)
                hipLaunchKernelGGL((k_ct_col<T, NY, -1>), grid, blk, 0, st, data, g.cI, tw,
                                   normalize ? 1 : 0, g.norm, ps);
            else
                hipLaunchKernelGGL((k_ct_col<T, NY, 1>), grid, blk, 0, st, data, g.cI, tw,
                                   normalize ? 1 : 0, g.norm, ps);
        }
    });
}

template <typename T>
void ref_row(hipStream_t st, const RefGrid &g, cpx<T> *data, bool r2c, int np, long long ps)
{
    with_length(g.h, [&](auto n) {
        constexpr int H = decltype(n)::value;
        if constexpr (H <= 1536) {
            constexpr int RB = RowCfg<T, H>::RB;
            const dim3 grid((g.ny + RB - 1) / RB, np), blk(RowCfg<T, H>::THR);
            const cpx<T> *tw = static_cast<const cpx<T> *>(g.tw_h),
                         *twx = static_cast<const cpx<T> *>(g.tw_x);
            if (r2c)
                hipLaunchKernelGGL((k_ct_row<T, H, true>), grid, blk, 0, st, data, g.cI, g.ny, tw,
                                   twx, ps);
            else
                hipLaunchKernelGGL((k_ct_row<T, H, false>), grid, blk, 0, st, data, g.cI, g.ny,
                                   tw, twx, ps);
        }
    });
}

template <typename T>
void ref_rhs(hipStream_t st, const RefGrid &g, const cpx<T> *psi_in, cpx<T> *u, cpx<T> *v,
             cpx<T> *w, cpx<T> *dW, double nu, int stage, double dt, const cpx<T> *w0, cpx<T> *out,
             cpx<T> *psi)
{
    const cpx<T> *twc = static_cast<const cpx<T> *>(g.tw_col);
    // columns that can hold something: stages 2 and 3 start from truncated
    // fields, stages 1 and 2 end in them
    int kept = 0;
    while (kept < g.cI && (long long)kept * kept <= g.kc2) ++kept;
    const int nin = stage == 2 || stage == 3 ? kept : g.cI;
    const int nout = stage == 1 || stage == 2 ? kept : g.cI;
    with_length(g.ny, [&](auto n) {
        constexpr int NY = decltype(n)::value;
        hipLaunchKernelGGL((k_rhs_velocity<T, NY>), (col_blocks<T, NY>(nin, 1, 3)),
                               dim3(ColCfg<T, NY>::THR), 0, st, psi_in, u, v, w, g.cI, nin, twc,
                               g.x_mask, g.y_mask);
    });
    with_length(g.h, [&](auto n) {
        constexpr int H = decltype(n)::value;
        if constexpr (H <= 1536) {
            const cpx<T> *th = static_cast<const cpx<T> *>(g.tw_h);
            const cpx<T> *tx = static_cast<const cpx<T> *>(g.tw_x);
            if constexpr (row_split_len<T, H>()) {
                if (rhs_rows_split<T, H>(g.ny)) {
                    constexpr int RS = RowSplitCfg<T, H>::RB;
                    hipLaunchKernelGGL((k_rhs_rows_split<T, H>), dim3((g.ny + RS - 1) / RS),
                                       dim3(RowSplitCfg<T, H>::THR), 0, st, u, v, w, g.cI, nin,
                                       nout, g.ny, th, tx);
                    return;
                }
            }
            constexpr int RB = RowCfg<T, H>::RB;
            hipLaunchKernelGGL((k_rhs_rows<T, H>), dim3((g.ny + RB - 1) / RB),
                               dim3(RowCfg<T, H>::THR), 0, st, u, v, w, g.cI, nin, nout, g.ny, th,
                               tx);
        }
    });
    const RhsArgs<T> a = {u,    v,    w,        dW,       w0,    out,    psi, g.cI,
                          nout, g.x_mask, g.y_mask, g.kc2, g.norm, nu,  dt,   twc};
    with_length(g.ny, [&](auto n) {
        constexpr int NY = decltype(n)::value;
        {
            const dim3 grid = col_blocks<T, NY>(stage == 1 ? nout : g.cI, 1),
                       blk(ColCfg<T, NY>::THR);
            switch (stage) {
            case 1: hipLaunchKernelGGL((k_rhs_columns<T, NY, 1>), grid, blk, 0, st, a); break;
            case 2: hipLaunchKernelGGL((k_rhs_columns<T, NY, 2>), grid, blk, 0, st, a); break;
            case 3: hipLaunchKernelGGL((k_rhs_columns<T, NY, 3>), grid, blk, 0, st, a); break;
            default: hipLaunchKernelGGL((k_rhs_columns<T, NY, 0>), grid, blk, 0, st, a); break;
            }
        }
    });
}

#define S2D_INST(T)                                                                              \
    template void ref_col<T>(hipStream_t, const RefGrid &, cpx<T> *, int, bool, int, long long); \
    template void ref_row<T>(hipStream_t, const RefGrid &, cpx<T> *, bool, int, long long);      \
    template void ref_rhs<T>(hipStream_t, const RefGrid &, const cpx<T> *, cpx<T> *, cpx<T> *,   \
                             cpx<T> *, cpx<T> *, double, int, double, const cpx<T> *, cpx<T> *,  \
                             cpx<T> *);
S2D_INST(double)
S2D_INST(float)

} // namespace s2d
