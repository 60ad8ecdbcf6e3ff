// fft.hpp -- complex FFT of one line of N = 2^n points, n <= 13, in the registers
// of T = N/E threads (R = double: complex128, R = float: complex64).
//
// Stockham autosort formulation.  Thread t holds the points x = t + T*e, e < E,
// before and after the transform.  A pass of radix Q takes Q points at stride
// N/Q, which are the thread's own (e = q + r*E/Q, r < Q, for its E/Q
// butterflies q), twiddles them, does a Q-point DFT in registers and puts the
// results in natural order.  Only between two passes do the points change
// threads, through LDS: two exchanges for the three passes of 512 points and
// more, one from 64, none below (a thread does the whole line).  Lines of up to
// 1024 points stay within one wave, whose exchanges need no barrier.
//
// The exchanges pad one value after every 16, which puts the strided stores of
// the first passes (stride 16 or 32) on distinct banks.  Complex128 lines and
// complex64 lines of 8192 points exchange the real and the imaginary parts one
// after the other, so that two or three lines of 8192 points share a CU
// (complex64, 6144 lines: 380 us with one exchange of both parts and two lines
// on a CU, 305 us so).
//
// Twiddles are read from a table built on the host in long double and rounded
// to R, stored in the order in which the threads read it (coalesced): for each
// pass after the first, W^(k r N/(Ns Q)) at [r - 1][k], W = exp(-2 pi i/N).  Only
// the forward transform (FFTW's sign, exp(-2 pi i jk/N)) is coded; the backward
// one conjugates before and after.  Both are unnormalised.
#pragma once

#include "common.hpp"

namespace chimera {

// Points per thread and the radices of the passes, by N.
template <int N> struct FftPlan { static constexpr int E = N, R0 = N, R1 = 1, R2 = 1; };     // N <= 32: one thread
template <> struct FftPlan<64> { static constexpr int E = 8, R0 = 8, R1 = 8, R2 = 1; };
template <> struct FftPlan<128> { static constexpr int E = 16, R0 = 16, R1 = 8, R2 = 1; };
template <> struct FftPlan<256> { static constexpr int E = 16, R0 = 16, R1 = 16, R2 = 1; };
template <> struct FftPlan<512> { static constexpr int E = 8, R0 = 8, R1 = 8, R2 = 8; };
template <> struct FftPlan<1024> { static constexpr int E = 16, R0 = 16, R1 = 8, R2 = 8; };
template <> struct FftPlan<2048> { static constexpr int E = 16, R0 = 16, R1 = 16, R2 = 8; };
template <> struct FftPlan<4096> { static constexpr int E = 16, R0 = 16, R1 = 16, R2 = 16; };
template <> struct FftPlan<8192> { static constexpr int E = 32, R0 = 32, R1 = 16, R2 = 16; };

// Whether real and imaginary parts are exchanged one after the other.
template <int N, typename C>
constexpr bool fft_parts() { return sizeof(C) == 16 || N == 8192; }

// Block shape of the line kernels: one line of T > 64 threads, or 64 / T lines in one wave.
template <int N, typename R>
struct FftShape {
    static constexpr int E = FftPlan<N>::E, T = N / E, TPB = T > 64 ? T : 64, LINES = TPB / T;
    static constexpr size_t LS = (N + N / 16) * (fft_parts<N, cplx_t<R>>() ? 1 : 2) * sizeof(R);    // LDS bytes of a line
    static constexpr size_t LDS = T > 1 ? LINES * LS : 0;
};

template <typename C> __device__ __forceinline__ C cmi(C a) { C r; r.x = a.y, r.y = -a.x; return r; }    // -i a

// Forward DFTs of Q points in registers, natural order in and out.
template <int Q, typename C>
struct Dft;
template <typename C>
struct Dft<1, C> { __device__ static __forceinline__ void go(C*) {} };
template <typename C>
struct Dft<2, C> {
    __device__ static __forceinline__ void go(C* v) {
        const C a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    }
};
template <typename C>
struct Dft<4, C> {
    __device__ static __forceinline__ void go(C* v) {
        const C s0 = cadd(v[0], v[2]), d0 = csub(v[0], v[2]), s1 = cadd(v[1], v[3]), d1 = cmi(csub(v[1], v[3]));
        v[0] = cadd(s0, s1);
        v[1] = cadd(d0, d1);
        v[2] = csub(s0, s1);
        v[3] = csub(d0, d1);
    }
};

// exp(-2 pi i k/32)
__device__ __forceinline__ constexpr double w32_cos(int k) {
    constexpr double c[9] = {1.0, 0.98078528040323044913, 0.92387953251128675613, 0.83146961230254523708,
                             0.70710678118654752440, 0.55557023301960222474, 0.38268343236508977173,
                             0.19509032201612826785, 0.0};
    k &= 31;
    return k <= 8 ? c[k] : k <= 16 ? -c[16 - k] : k <= 24 ? -c[k - 16] : c[32 - k];
}
// v times exp(-2 pi i k/32), k a constant
template <int K, typename C>
__device__ __forceinline__ C w32(C v) {
    typedef decltype(v.x) R;
    constexpr int k = K & 31;
    if constexpr (k == 0) return v;
    else if constexpr (k == 8) return cmi(v);
    else if constexpr (k == 4) {
        C r = cadd(v, cmi(v));
        r.x *= (R)0.70710678118654752440, r.y *= (R)0.70710678118654752440;
        return r;
    } else if constexpr (k == 12) {
        C r = csub(cmi(v), v);
        r.x *= (R)0.70710678118654752440, r.y *= (R)0.70710678118654752440;
        return r;
    } else {
        constexpr double c = w32_cos(k), s = -w32_cos(k - 8);       // sin of -2 pi k/32
        C w;
        w.x = (R)c, w.y = (R)s;
        return cmul(v, w);
    }
}

// Q = P * S points: S-strided P-point DFTs, twiddles, S-point DFTs (S = 2 or 4).
template <int P, int S, int J, int K, typename C>
__device__ __forceinline__ void dft_twiddle(C (&y)[S][P]) {
    if constexpr (J < S) {
        if constexpr (K < P) {
            y[J][K] = w32<J * K * 32 / (P * S)>(y[J][K]);
            dft_twiddle<P, S, J, K + 1>(y);
        } else {
            dft_twiddle<P, S, J + 1, 0>(y);
        }
    }
}
template <int P, int S, typename C>
__device__ __forceinline__ void dft_split(C* v) {
    C y[S][P];
#pragma unroll
    for (int j = 0; j < S; j++) {
#pragma unroll
        for (int n = 0; n < P; n++) y[j][n] = v[S * n + j];
        Dft<P, C>::go(y[j]);
    }
    dft_twiddle<P, S, 1, 1>(y);
#pragma unroll
    for (int k = 0; k < P; k++) {
        C z[S];
#pragma unroll
        for (int j = 0; j < S; j++) z[j] = y[j][k];
        Dft<S, C>::go(z);
#pragma unroll
        for (int j = 0; j < S; j++) v[k + P * j] = z[j];
    }
}
template <typename C> struct Dft<8, C> { __device__ static __forceinline__ void go(C* v) { dft_split<4, 2>(v); } };
template <typename C> struct Dft<16, C> { __device__ static __forceinline__ void go(C* v) { dft_split<4, 4>(v); } };
template <typename C> struct Dft<32, C> { __device__ static __forceinline__ void go(C* v) { dft_split<8, 4>(v); } };

// A pass of radix Q after passes of product NS: its twiddles (tw: the pass's
// table), read before the exchange that precedes it, and the pass with them.
template <int N, int Q, int NS, typename C>
__device__ __forceinline__ void fft_tw(C* w, int t, const C* __restrict__ tw) {
    constexpr int E = FftPlan<N>::E, T = N / E, B = E / Q;
#pragma unroll
    for (int q = 0; q < B; q++)
#pragma unroll
        for (int r = 1; r < Q; r++) w[q * Q + r] = tw[(r - 1) * NS + (t + T * q) % NS];
}
template <int N, int Q, int NS, typename C>
__device__ __forceinline__ void fft_pass(C (&v)[FftPlan<N>::E], int t, const C* __restrict__ tw) {
    constexpr int E = FftPlan<N>::E, T = N / E, B = E / Q;
#pragma unroll
    for (int q = 0; q < B; q++) {
        C z[Q];
        const int k = (t + T * q) % NS;
#pragma unroll
        for (int r = 0; r < Q; r++) {
            z[r] = v[q + r * B];
            if (NS > 1 && r > 0) z[r] = cmul(z[r], tw[q * Q + r]);
        }
        Dft<Q, C>::go(z);
#pragma unroll
        for (int r = 0; r < Q; r++) v[q + r * B] = z[r];
    }
}

template <int T>
__device__ __forceinline__ void fft_sync() {
    if constexpr (T > 64) __syncthreads();
    else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// The results of a pass of radix Q (after passes of product NS) to natural
// order: value j*Q-block ... of butterfly j goes to (j/NS)*NS*Q + j%NS + r*NS.
// lds: the line's FftShape::LS bytes.
template <int N, int Q, int NS, typename C>
__device__ __forceinline__ void fft_exchange(C (&v)[FftPlan<N>::E], int t, void* lds) {
    constexpr int E = FftPlan<N>::E, T = N / E, B = E / Q;
    // value r of butterfly t + T*q goes to place st + (r*NS + q*T*Q), value e
    // comes from t + T*e: the low four bits of the two terms do not carry, so
    // the padding splits into that of the thread and a constant
    static_assert(B == 1 || (T % NS == 0 && (T * Q) % 16 == 0), "places of a butterfly");
    constexpr auto pad = [](int p) { return p + (p >> 4); };
    const int st = pad((t / NS) * NS * Q + t % NS), ld = pad(t);
    constexpr auto so = [pad](int e) { return pad((e / B) * NS + (e % B) * T * Q); };
    constexpr auto lo = [pad](int e) { return pad(T * e); };
    if constexpr (!fft_parts<N, C>()) {
        C* const s = static_cast<C*>(lds);
#pragma unroll
        for (int e = 0; e < E; e++) s[st + so(e)] = v[e];
        fft_sync<T>();
#pragma unroll
        for (int e = 0; e < E; e++) v[e] = s[ld + lo(e)];
        fft_sync<T>();
    } else {
        auto* const s = static_cast<decltype(v[0].x)*>(lds);
#pragma unroll
        for (int e = 0; e < E; e++) s[st + so(e)] = v[e].x;
        fft_sync<T>();
#pragma unroll
        for (int e = 0; e < E; e++) v[e].x = s[ld + lo(e)];
        fft_sync<T>();
#pragma unroll
        for (int e = 0; e < E; e++) s[st + so(e)] = v[e].y;
        fft_sync<T>();
#pragma unroll
        for (int e = 0; e < E; e++) v[e].y = s[ld + lo(e)];
        fft_sync<T>();
    }
}

// Transform of the line held by threads t = 0..T-1, v[e] = point t + T*e; sign < 0 forward, > 0 backward.
template <int N, typename C>
__device__ __forceinline__ void fft_line(C (&v)[FftPlan<N>::E], int t, void* lds, int sign, const C* __restrict__ tw) {
    typedef FftPlan<N> P;
    if (sign > 0) {
#pragma unroll
        for (int e = 0; e < P::E; e++) v[e].y = -v[e].y;
    }
    C w[P::E];
    fft_pass<N, P::R0, 1>(v, t, w);
    if constexpr (P::R1 > 1) {
        fft_tw<N, P::R1, P::R0>(w, t, tw);
        fft_exchange<N, P::R0, 1>(v, t, lds);
        fft_pass<N, P::R1, P::R0>(v, t, w);
    }
    if constexpr (P::R2 > 1) {
        fft_tw<N, P::R2, P::R0 * P::R1>(w, t, tw + (P::R1 - 1) * P::R0);
        fft_exchange<N, P::R1, P::R0>(v, t, lds);
        fft_pass<N, P::R2, P::R0 * P::R1>(v, t, w);
    }
    if (sign > 0) {
#pragma unroll
        for (int e = 0; e < P::E; e++) v[e].y = -v[e].y;
    }
}

}  // namespace chimera
