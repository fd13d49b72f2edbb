// fft_wave.hpp -- compile-time Stockham FFT on a lane group.
//
// A length n = E*TG transform (n = 2^a 3^b) is carried by a group of TG
// lanes, TG a power of two (2..256) or, with E = 12, 3*2^k (6..192). Groups
// that divide a wave live inside one (64/TG groups per wave); the others
// (TG > 64, or 3*2^k lanes, whose groups straddle waves) span waves of one
// workgroup. Lane t of the group holds x[t + TG*s], s < E. The early passes
// are radix-R Stockham passes (R in {12, 8, 6, 4, 2}, R | E, the radices
// multiply to TG) that exchange through the group's LDS slice; the final
// pass is one radix-E butterfly per lane, in registers, whose outputs
// X[t + TG*m] are again the lane's own elements.
//
// LDS slots are spread over the banks (LdsMap): for a power of two by a
// permutation inside aligned blocks of 16 elements, without padding; for
// 3*2^k by one pad element in 12. Groups inside one wave synchronise with
// wave-scope fences; the others use workgroup barriers, which every thread
// of the workgroup must reach the same number of times.
//
// Per-lane twiddles come from the FP64-generated table tw[e] =
// exp(-2 pi i e / n) of the transform length (rounded to T); the twiddles
// inside the in-register DFTs are compile-time constants.
#pragma once

#include <type_traits>

#include "fft_block.hpp"

namespace s2d {

__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// BLK: the group's lanes span waves (or share them in another order than
// TG consecutive lanes per group)
template <int TG, bool BLK = (64 % TG != 0)>
__device__ __forceinline__ void group_sync()
{
    if constexpr (BLK)
        __syncthreads();
    else
        wave_sync();
}

// LDS slot of element i of a TG-lane group.
//
// TG a power of two: bits 0-3 XORed with bits 3-6, a permutation inside each
// aligned block of 16 elements (n is a multiple of 16 for every size used).
// It keeps the strided Stockham writes and the contiguous reads within
// 1.25-1.5x of conflict-free for both 32- and 64-bank LDS, with no padding.
// Every exchange addresses slot b + c, with b from the lane and c a
// compile-time constant that shares no set bit with b, so that idx_sum takes
// one XOR with a constant, and the addition folds into the LDS instruction's
// offset.
//
// TG = 3*2^k: i + i/12. The first pass (radix 12, or 6 for TG = 6) writes R
// consecutive elements per lane, 13 slots apart (a stride of 12 would put
// every fourth lane of an FP64 write, every eighth of an FP32 one, on the
// same banks), and every later offset is a multiple of 12: idx(b + c) is
// idx(b) + idx(c), all of it in the instruction's offset.
template <int TG>
struct LdsMap {
    static constexpr bool P2 = (TG & (TG - 1)) == 0;
    static __host__ __device__ constexpr int idx(int i)
    {
        return P2 ? i ^ ((i >> 3) & 15) : i + i / 12;
    }
    // idx(b + c) from ib = idx(b), for the b and c of the exchanges
    static __host__ __device__ constexpr int idx_sum(int ib, int c)
    {
        return P2 ? (ib ^ (idx(c) & 15)) + (c & ~15) : ib + idx(c);
    }
    static constexpr int size(int n) { return P2 ? n : n / 12 * 13; }
};

// idx_sum against idx over every pair of disjoint 8-bit values (idx reads
// bits 0-6 only, so higher bits just add).
constexpr bool lds_idx_sum_exact()
{
    for (int b = 0; b < 256; ++b)
        for (int c = 0; c < 256; ++c)
            if ((b & c) == 0 && LdsMap<1>::idx_sum(LdsMap<1>::idx(b), c) != LdsMap<1>::idx(b + c))
                return false;
    return true;
}
static_assert(lds_idx_sum_exact(), "idx_sum differs from idx");

// Largest early radix in {12, 6, 8, 4, 2} dividing both E and the remaining
// product rem of the group size (12 and 6 only serve TG = 3*2^k: they take
// its factor 3 in the first pass).
constexpr int early_radix(int E, int rem)
{
    return (E % 12 == 0 && rem % 12 == 0) ? 12
           : (E % 6 == 0 && rem % 6 == 0) ? 6
           : (E % 8 == 0 && rem % 8 == 0) ? 8
           : (E % 4 == 0 && rem % 4 == 0) ? 4
                                          : 2;
}

// The same for TG = 3*2^k and E = 12, over every address of its transform:
// the reads t + TG s and each early pass's writes (t - k) R + k + TG q R + m Ls.
template <int TG>
constexpr bool lds_idx_sum_exact3()
{
    using M = LdsMap<TG>;
    constexpr int E = 12;
    for (int t = 0; t < TG; ++t) {
        for (int s = 0; s < E; ++s)
            if (M::idx_sum(M::idx(t), TG * s) != M::idx(t + TG * s)) return false;
        for (int Ls = 1; Ls < TG;) {
            const int R = early_radix(E, TG / Ls), k = t % Ls, b = (t - k) * R + k;
            for (int q = 0; q < E / R; ++q)
                for (int m = 0; m < R; ++m)
                    if (M::idx_sum(M::idx(b), TG * q * R + m * Ls) !=
                        M::idx(b + TG * q * R + m * Ls))
                        return false;
            Ls *= R;
        }
    }
    return true;
}
static_assert(lds_idx_sum_exact3<6>() && lds_idx_sum_exact3<12>() && lds_idx_sum_exact3<24>() &&
                  lds_idx_sum_exact3<48>() && lds_idx_sum_exact3<96>() && lds_idx_sum_exact3<192>(),
              "idx_sum differs from idx");

// t % Ls for a lane index t >= 0.
template <int Ls>
__device__ __forceinline__ int lane_mod(int t)
{
    if constexpr ((Ls & (Ls - 1)) == 0) return t & (Ls - 1);
    else return (int)((unsigned)t % (unsigned)Ls);
}

// Compile-time loop: f(std::integral_constant<int, I>) for I in [B, N).
template <int B, int N, typename F>
__device__ __forceinline__ void static_for(F &&f)
{
    if constexpr (B < N) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, N>(f);
    }
}

// cos(15 a degrees), a in 0..6: the constant twiddles of sizes dividing 24.
constexpr double kCos15[7] = {1.0,
                              0.96592582628906828674974319972890,
                              0.86602540378443864676372317075294,
                              0.70710678118654752440084436210485,
                              0.5,
                              0.25881904510252076234889883762405,
                              0.0};
constexpr double cos15(int a)
{
    a = ((a % 24) + 24) % 24;
    return a <= 6 ? kCos15[a] : a <= 12 ? -kCos15[12 - a] : a <= 18 ? -kCos15[a - 12] : kCos15[24 - a];
}
constexpr double sin15(int a) { return cos15(a - 6); }

// What cos(15 a degrees) has beyond its value in T where that is +-sqrt(3)/2,
// else 0: the one constant of radix 12 that is not exact. FP64 rounds it by
// 0.45 of its last place, FP32 by 0.26. (long double is double on the device.)
template <typename T>
constexpr double cos15_low(int a)
{
    constexpr double low = sizeof(T) == 8 ? 5.01754211090345140e-17 : kCos15[2] - (double)(float)kCos15[2];
    const double c = cos15(a);
    return c == kCos15[2] ? low : c == -kCos15[2] ? -low : 0.0;
}

// x * exp(D i 2 pi e / N) for compile-time e and N | 24 (D = -1 forward,
// +1 inverse): multiples of a quarter turn are exact swaps and negations,
// the rest one complex product with constants.
// ACC: sqrt(3)/2 in two terms, one FMA more. As a single constant in every
// pass its rounding adds up: FP64 error of a transform of length 144 / 1152
// and back 2.83e-16 / 3.07e-16, in two terms here and in radix 3 2.36e-16 /
// 2.70e-16 (the runtime plans, whose table twiddles all round differently,
// 2.57e-16 / 2.86e-16); an FP32 IntegrateOneStep at 48 / 192 2.18e-7 / 2.63e-7
// and 1.88e-7 / 1.98e-7 (plans 2.10e-7 / 2.78e-7). FP64 IntegrateOneStep at
// 96 / 768 / 1024 97 -> 101, 238 -> 242 and 334 -> 336 us, FP32 at 1024
// 219 -> 221.
template <typename T, int D, int N, int e, bool ACC = false>
__device__ __forceinline__ cpx<T> twiddle_const(cpx<T> x)
{
    static_assert(24 % N == 0, "constant twiddles cover sizes dividing 24");
    constexpr int a = (((24 / N) * e) % 24 + 24) % 24; // the angle in 15-degree units
    if constexpr (a == 0) {
        return x;
    } else if constexpr (a == 12) {
        return mk<T>(-x.re, -x.im);
    } else if constexpr (a == 6 || a == 18) { // W = (0, D) or (0, -D)
        constexpr int sg = a == 6 ? D : -D;
        return sg > 0 ? mk<T>(-x.im, x.re) : mk<T>(x.im, -x.re);
    } else {
        constexpr T c = (T)cos15(a), sn = (T)(D * sin15(a));
        if constexpr (ACC && cos15_low<T>(a) != 0.0) {
            constexpr T cl = (T)cos15_low<T>(a);
            return mk<T>(fma(x.re, c, fma(x.re, cl, -(x.im * sn))),
                         fma(x.im, c, fma(x.im, cl, x.re * sn)));
        } else if constexpr (ACC && cos15_low<T>(a - 6) != 0.0) {
            constexpr T sl = (T)(D * cos15_low<T>(a - 6));
            return mk<T>(fma(-x.im, sn, fma(-x.im, sl, x.re * c)),
                         fma(x.re, sn, fma(x.re, sl, x.im * c)));
        } else {
            return mul(x, mk<T>(c, sn));
        }
    }
}

// Radix 3 with sqrt(3)/2 in two terms (see twiddle_const).
template <typename T, int D>
__device__ __forceinline__ void dft3_acc(cpx<T> *a)
{
    constexpr T h = (T)(-D * cos15(2)), l = (T)(-D * cos15_low<T>(2));
    const cpx<T> t1 = add(a[1], a[2]), q = sub(a[1], a[2]);
    const cpx<T> t2 = mk<T>(a[0].re - (T)0.5 * t1.re, a[0].im - (T)0.5 * t1.im);
    const cpx<T> t3 = mk<T>(fma(q.re, h, q.re * l), fma(q.im, h, q.im * l));
    a[0] = add(a[0], t1);
    a[1] = mk<T>(t2.re + t3.im, t2.im - t3.re);
    a[2] = mk<T>(t2.re - t3.im, t2.im + t3.re);
}

// In-register DFT of compile-time size N on a[0..N-1] (natural order in and
// out). Base radices 2, 3, 4, 8; composite N = N1*N2 by Cooley-Tukey with
// N1 the largest base radix dividing N, and compile-time twiddles.
template <typename T, int N, int D, bool ACC = false>
__device__ __forceinline__ void dft_ct(cpx<T> *a)
{
    if constexpr (ACC && N == 3) {
        dft3_acc<T, D>(a);
    } else if constexpr (N == 2 || N == 3 || N == 4 || N == 8) {
        dft<T, N, D>(a);
    } else {
        constexpr int N1 = (N % 8 == 0) ? 8 : (N % 4 == 0) ? 4 : (N % 3 == 0) ? 3 : 2;
        constexpr int N2 = N / N1;
        cpx<T> y[N];
        static_for<0, N2>([&](auto n2I) {
            constexpr int n2 = decltype(n2I)::value;
            cpx<T> b[N1];
#pragma unroll
            for (int n1 = 0; n1 < N1; ++n1) b[n1] = a[N2 * n1 + n2];
            dft<T, N1, D>(b);
            static_for<0, N1>([&](auto k1I) {
                constexpr int k1 = decltype(k1I)::value;
                y[n2 * N1 + k1] = twiddle_const<T, D, N, n2 * k1, ACC>(b[k1]);
            });
        });
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) {
            cpx<T> c[N2];
#pragma unroll
            for (int n2 = 0; n2 < N2; ++n2) c[n2] = y[n2 * N1 + k1];
            dft_ct<T, N2, D, ACC>(c);
#pragma unroll
            for (int k2 = 0; k2 < N2; ++k2) a[k1 + N1 * k2] = c[k2];
        }
    }
}

// Number of per-lane twiddles of the early passes before the one at Ls
// (the first pass, Ls = 1, needs none).
template <int E, int TG, int Ls, int L = 1>
constexpr int early_tw_offset()
{
    if constexpr (L >= Ls || L >= TG) {
        return 0;
    } else {
        constexpr int R = early_radix(E, TG / L);
        return (L > 1 ? R - 1 : 0) + early_tw_offset<E, TG, Ls, L * R>();
    }
}

// The per-lane twiddles of one lane-group transform: R - 1 per early pass
// and E - 1 for the final pass, as forward values (an inverse transform
// multiplies by their conjugates). PRE selects which are loaded in one
// batch ahead of the transform's LDS exchanges (bit 0: the early passes',
// bit 1: the final pass's); the others are loaded by their pass. A load
// issued after an exchange's fence cannot be moved above it, so per-pass
// loads wait once per pass; batched ones hold registers for the whole
// transform.
constexpr int TW_EARLY = 1, TW_FINAL = 2, TW_ALL = 3, TW_FINAL_POW = 4;
// bit 3: the constants inside the butterflies to more than T (twiddle_const's
// ACC)
constexpr int TW_ACC = 8;

template <typename T, int E, int TG, int PRE = TW_ALL>
struct GroupTw {
    static constexpr int n = E * TG;
    static constexpr int NE = early_tw_offset<E, TG, TG>();
    static constexpr bool PE = (PRE & TW_EARLY) != 0, PF = (PRE & TW_FINAL) != 0;
    // bit 2: the final pass's twiddles W^(m t) as powers of W^t, one complex
    // multiplication each instead of a load (at most about E ulps apart
    // from the table's values)
    static constexpr bool PP = (PRE & TW_FINAL_POW) != 0;
    static constexpr bool ACC = (PRE & TW_ACC) != 0;
    cpx<T> e[PE && NE > 0 ? NE : 1];
    cpx<T> f[PF ? E : 1];
    cpx<T> w1; // W^t (PP)
    const cpx<T> *tw;
    int t;

    __device__ __forceinline__ void load(const cpx<T> *__restrict__ tw_, int t_)
    {
        tw = tw_;
        t = t_;
        if constexpr (PE) load_early<1>();
        if constexpr (PP) w1 = tw[t];
        if constexpr (PF) {
#pragma unroll
            for (int m = 1; m < E; ++m) f[m] = tw[m * t];
        }
    }
    // twiddle m (1 <= m < R) of the radix-R early pass at Ls
    template <int Ls, int R>
    __device__ __forceinline__ cpx<T> early(int m) const
    {
        if constexpr (PE) return e[early_tw_offset<E, TG, Ls>() + m - 1];
        else return tw[m * lane_mod<Ls>(t) * (n / (Ls * R))];
    }
    // twiddle m (1 <= m < E) of the final pass
    __device__ __forceinline__ cpx<T> final(int m) const
    {
        if constexpr (PF) return f[m];
        else return tw[m * t];
    }

  private:
    template <int Ls>
    __device__ __forceinline__ void load_early()
    {
        if constexpr (Ls < TG) {
            constexpr int R = early_radix(E, TG / Ls);
            if constexpr (Ls > 1) {
                constexpr int o = early_tw_offset<E, TG, Ls>(), ts = n / (Ls * R);
                const int k = lane_mod<Ls>(t);
#pragma unroll
                for (int m = 1; m < R; ++m) e[o + m - 1] = tw[m * k * ts];
            }
            load_early<Ls * R>();
        }
    }
};

// w for the forward direction, conj(w) for the inverse.
template <typename T, int D>
__device__ __forceinline__ cpx<T> dir(cpx<T> w)
{
    if constexpr (D > 0) w.im = -w.im;
    return w;
}

// One early radix-R pass with Ls = product of the previous radices (Ls
// divides TG, so k = j % Ls = t % Ls for every butterfly of the lane).
template <typename T, int E, int TG, int R, int Ls, int D, class G>
__device__ __forceinline__ void group_pass(cpx<T> (&v)[E], cpx<T> *lds, int t, const G &g)
{
    constexpr int Q = E / R;
    const int k = lane_mod<Ls>(t);
    // slot of output m of butterfly q: (t - k) R + k, the lane's part, plus
    // TG q R + m Ls, which shares no bit with it
    const int ib = LdsMap<TG>::idx((t - k) * R + k);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        cpx<T> a[R];
#pragma unroll
        for (int m = 0; m < R; ++m) a[m] = v[q + m * Q];
        if constexpr (Ls > 1) {
#pragma unroll
            for (int m = 1; m < R; ++m) a[m] = mul(a[m], dir<T, D>(g.template early<Ls, R>(m)));
        }
        dft_ct<T, R, D, G::ACC>(a);
#pragma unroll
        for (int m = 0; m < R; ++m) lds[LdsMap<TG>::idx_sum(ib, TG * q * R + m * Ls)] = a[m];
    }
}

template <typename T, int E, int TG, int D, int Ls, bool BLK, class G>
__device__ __forceinline__ void early_passes(cpx<T> (&v)[E], cpx<T> *lds, int t, const G &g)
{
    if constexpr (Ls < TG) {
        constexpr int R = early_radix(E, TG / Ls);
        static_assert(E % R == 0 && (TG / Ls) % R == 0, "no early radix");
        group_pass<T, E, TG, R, Ls, D, G>(v, lds, t, g);
        group_sync<TG, BLK>();
        const int it = LdsMap<TG>::idx(t);
#pragma unroll
        for (int s = 0; s < E; ++s) v[s] = lds[LdsMap<TG>::idx_sum(it, TG * s)];
        group_sync<TG, BLK>();
        early_passes<T, E, TG, D, Ls * R, BLK, G>(v, lds, t, g);
    }
}

// Final radix-E pass of lane t (Ls = TG, k = t): X[t + TG*k] = sum_m
// v[m] W_n^{m t} W_E^{m k}: the E - 1 per-lane twiddles W_n^{m t}, then an
// in-register E-point DFT whose own twiddles are compile-time constants.
template <typename T, int E, int TG, int D, class G>
__device__ __forceinline__ void final_pass(cpx<T> (&v)[E], const G &g)
{
    if constexpr (G::PP) {
        cpx<T> p = g.w1;
        v[1] = mul(v[1], dir<T, D>(p));
#pragma unroll
        for (int m = 2; m < E; ++m) {
            p = mul(p, g.w1);
            v[m] = mul(v[m], dir<T, D>(p));
        }
    } else {
#pragma unroll
        for (int m = 1; m < E; ++m) v[m] = mul(v[m], dir<T, D>(g.final(m)));
    }
    dft_ct<T, E, D, G::ACC>(v);
}

// Full transform of the group: on entry v[s] = x[t + TG*s], on exit
// v[s] = X[t + TG*s]. lds is the group's slice (LdsMap<TG>::size(n)); g holds
// the lane's twiddles (GroupTw::load with the table of length n).
template <typename T, int E, int TG, int D, int PRE, bool BLK = (64 % TG != 0)>
__device__ __forceinline__ void group_fft(cpx<T> (&v)[E], cpx<T> *lds, int t,
                                          const GroupTw<T, E, TG, PRE> &g)
{
    early_passes<T, E, TG, D, 1, BLK>(v, lds, t, g);
    final_pass<T, E, TG, D>(v, g);
}

} // namespace s2d
