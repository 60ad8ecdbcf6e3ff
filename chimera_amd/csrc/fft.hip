// fft.hip -- the x transforms of the Fourier-Bessel side: lines of power-of-two
// length (k_fft_lines) and of any other (k_fft_bluestein), with the per-x and
// per-point multipliers, mode normalisation and ghost row that surround them.
#include <atomic>
#include <cmath>
#include <complex>
#include <map>
#include <mutex>
#include <vector>

#include "common.hpp"
#include "fb_kernels.hpp"
#include "fft.hpp"

namespace chimera {

// The radices of the passes of N = 2^n points, n = 0..13 (FftPlan).
template <int N>
static void fft_plan_of(int* r) { r[0] = FftPlan<N>::R0, r[1] = FftPlan<N>::R1, r[2] = FftPlan<N>::R2; }
static void fft_plan(int N, int* r) {
    switch (N) {
        case 64: return fft_plan_of<64>(r);
        case 128: return fft_plan_of<128>(r);
        case 256: return fft_plan_of<256>(r);
        case 512: return fft_plan_of<512>(r);
        case 1024: return fft_plan_of<1024>(r);
        case 2048: return fft_plan_of<2048>(r);
        case 4096: return fft_plan_of<4096>(r);
        case 8192: return fft_plan_of<8192>(r);
        default: r[0] = N, r[1] = r[2] = 1;      // one thread, no table
    }
}

template <typename R>
static const cplx_t<R>* fft_twiddles(int N) {
    typedef cplx_t<R> C;
    static std::mutex mu;
    static std::map<int, const C*> cache;
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find(N);
    if (it != cache.end()) return it->second;
    int rad[3];
    fft_plan(N, rad);
    std::vector<C> h;
    long long ns = rad[0];
    for (int p = 1; p < 3; ns *= rad[p], p++) {
        for (long long r = 1; r < rad[p]; r++) {
            for (long long k = 0; k < ns; k++) {
                // the angle is below one turn: k r < ns rad[p]
                const long double ang =
                    -2.0L * 3.141592653589793238462643383279502884L * (long double)(k * r) / (long double)(ns * rad[p]);
                h.push_back(cmake<R>((R)cosl(ang), (R)sinl(ang)));
            }
        }
    }
    if (h.empty()) h.push_back(cmake<R>(1, 0));
    const C* d = static_cast<const C*>(shared_table(h.data(), h.size() * sizeof(C)));
    if (d) cache[N] = d;
    return d;
}

constexpr int64_t FFT_PHASE_POINTS = 1 << 18;
constexpr int FFT_PHASE_LINE = 2048;          // 32 KiB of complex128 phases
constexpr int FFT_LDS_MAX = 120 * 1024;

// One line of a transform: its points in memory and what happens to them there.
template <typename R>
struct FftLine {
    typedef cplx_t<R> C;
    const C* in;
    C* out;
    const R* scale;
    C* ghost;               // row below row 1, for its line only (r = 0)
    R gsc;                  // mode normalisation
    int neg;                // ghost = -row (1), +row (0), zero (2)
    __device__ __forceinline__ FftLine(const FftArgsT<R>& a, int64_t line) {
        const int64_t r = line % a.n_inner, q = line / a.n_inner;
        in = a.in + r * a.in_r + q * a.in_q;
        out = a.out + r * a.out_r + q * a.out_q;
        scale = a.scale ? a.scale + (int64_t)a.N * r : nullptr;
        ghost = a.ghost && r == 0 ? out - a.out_r : nullptr;
        const int m = a.ghost ? (int)(q % a.nmodes) : 0;
        gsc = a.ghost < 2 ? (R)1 : a.ghost == 2 && m == 0 ? (R)(0.5 / M_PI) : (R)(1.0 / M_PI);
        // ghost radial row below row 1: zero (fb_io.f90:199), +-row 1 by mode
        // (grid_deps.f90:248-265), or +row 1 (3) / -row 1 (4) for every mode of
        // the envelope grid (grid_deps_env.f90:240-283: + when nkO = 0)
        neg = a.ghost == 1 ? 2 : a.ghost == 2 ? (m != 0) : a.ghost == 4;
    }
    __device__ __forceinline__ void store(const FftArgsT<R>& a, int x, C v) const {
        if (scale) v = crs(scale[x], v);
        if (a.ghost >= 2) v = crs(gsc, v);
        out[x] = v;
        if (ghost) ghost[x] = neg == 2 ? cmake<R>(0, 0) : neg ? cneg(v) : v;
    }
};

// The table of k_phase, exp(ph_s i kx[x] leftX), formed by the block in its LDS.
template <int TPB, typename R>
__device__ __forceinline__ void fft_phase(const FftArgsT<R>& a, cplx_t<R>* ph) {
    const double lx = a.ph_leftX_dev ? *a.ph_leftX_dev : a.ph_leftX;
#pragma unroll 1
    for (int x = threadIdx.x; x < a.N; x += TPB) {
        double sn, cs;
        sincos(lx * a.ph_kx[x], &sn, &cs);
        ph[x] = cmake<R>((R)cs, (R)(a.ph_s * sn));
    }
    fft_sync<TPB>();
}

// Lines of N points, FftShape::LINES to a block, each in the registers of
// its threads from the load to the store.  Bound by memory: a point is read and
// written once.  Measured with the multipliers and stores of the inverse
// transform on 4608 complex128 lines and of the forward one on 6144 complex64
// lines, against passes of radix 8 that keep the line in LDS and read the
// twiddles when they need them:
//   complex128  512: 36 -> 15 us   2048: 108 -> 62   4096: 249 -> 126   8192: 665 -> 340
//   complex64  1024: 64 -> 30      2048: 158 -> 54   4096: 263 -> 120   8192: 712 -> 306
// (4096 complex128: 4.8 TB/s, the rate of a copy).  A complex128 line of 8192
// points is held to 256 registers, so that two share a CU: some spill, and
// still 340 us against 460 without; complex64 fits three without.
template <int N, typename R>
__global__ void __launch_bounds__((FftShape<N, R>::TPB), N == 8192 ? (sizeof(R) == 4 ? 3 : 2) : 1)
    k_fft_lines(FftArgsT<R> a) {
    typedef cplx_t<R> C;
    typedef FftShape<N, R> S;
    extern __shared__ __align__(16) unsigned char fft_smem[];
    // a block of one line: l = 0, its pointers are the same for all threads
    const int t = S::LINES == 1 ? threadIdx.x : threadIdx.x % S::T, l = S::LINES == 1 ? 0 : threadIdx.x / S::T;
    void* const lds = fft_smem + l * S::LS;
    C* const ph = reinterpret_cast<C*>(fft_smem + S::LDS);
    const int64_t line = (int64_t)blockIdx.x * S::LINES + l;
    const bool on = line < a.nlines;
    const FftLine<R> ln(a, on ? line : 0);
    C v[S::E];
#pragma unroll
    for (int e = 0; e < S::E; e++) v[e] = on ? ln.in[t + S::T * e] : cmake<R>(0, 0);
    if (a.ph_at) fft_phase<S::TPB>(a, ph);      // while the loads are in flight
    if (a.pre) {
#pragma unroll
        for (int e = 0; e < S::E; e++) v[e] = cmul(v[e], a.pre[t + S::T * e]);
    } else if (a.ph_at == 1) {
#pragma unroll
        for (int e = 0; e < S::E; e++) v[e] = cmul(v[e], ph[t + S::T * e]);
    }
    fft_line<N>(v, t, lds, a.sign, a.tw);
    if (a.filtr) {
        // fb_io.f90:263: multiply the first nxfilt points, transform back
#pragma unroll
        for (int e = 0; e < S::E; e++) {
            const int x = t + S::T * e;
            if (x < a.nxfilt) v[e] = crs(a.filtr[x], v[e]);
        }
        fft_line<N>(v, t, lds, -a.sign, a.tw);
    }
    if (!on) return;
    if (a.post) {
#pragma unroll
        for (int e = 0; e < S::E; e++) v[e] = cmul(v[e], a.post[t + S::T * e]);
    } else if (a.ph_at == 2) {
#pragma unroll
        for (int e = 0; e < S::E; e++) v[e] = cmul(v[e], ph[t + S::T * e]);
    }
#pragma unroll
    for (int e = 0; e < S::E; e++) ln.store(a, t + S::T * e, v[e]);
}

// ---- lengths that are not powers of two (Bluestein)
// A length-N DFT of sign s is X_k = c_k * sum_n (x_n c_n) conj(c_(k-n)) with the
// chirp c_n = exp(s i pi n^2 / N) (from nk = (n^2 + k^2 - (k-n)^2) / 2): a
// circular convolution, of power-of-two length L >= 2N - 1, of the chirped,
// zero-padded line with g, g[m] = conj(c_|m|) for |m| < N.  ghat = FFT_L(g) / L,
// so that IFFT_L(FFT_L(a) * ghat) (both unnormalised) is the convolution.  The
// tables are built in long double with the angle pi (n^2 mod 2N) / N reduced
// exactly, then rounded to R.
static void host_fft_ld(std::vector<std::complex<long double>>& v) {
    // iterative radix-2, forward (exp(-2 pi i jk / L)), in place
    const size_t L = v.size();
    for (size_t i = 1, j = 0; i < L; i++) {
        size_t bit = L >> 1;
        for (; j & bit; bit >>= 1) j ^= bit;
        j ^= bit;
        if (i < j) std::swap(v[i], v[j]);
    }
    const long double pi = 3.141592653589793238462643383279502884L;
    for (size_t len = 2; len <= L; len <<= 1) {
        for (size_t i = 0; i < L; i += len) {
            for (size_t k = 0; k < len / 2; k++) {
                const long double ang = -2.0L * pi * (long double)k / (long double)len;
                const std::complex<long double> w(cosl(ang), sinl(ang));
                const std::complex<long double> u = v[i + k], t = w * v[i + k + len / 2];
                v[i + k] = u + t;
                v[i + k + len / 2] = u - t;
            }
        }
    }
}

int bluestein_length(int N) {
    int L = 64;         // the shortest line that a whole wave takes
    while (L < 2 * N - 1) L <<= 1;
    return L;
}

template <typename R>
static int32_t bluestein_tables(int N, int sign, const cplx_t<R>** chirp, const cplx_t<R>** ghat) {
    typedef cplx_t<R> C;
    static std::mutex mu;
    static std::map<std::pair<int, int>, std::pair<const C*, const C*>> cache;
    std::lock_guard<std::mutex> lk(mu);
    const auto key = std::make_pair(N, sign);
    auto it = cache.find(key);
    if (it == cache.end()) {
        const int L = bluestein_length(N);
        const long double pi = 3.141592653589793238462643383279502884L;
        std::vector<std::complex<long double>> c(N), g(L, std::complex<long double>(0, 0));
        for (int n = 0; n < N; n++) {
            const long long n2 = ((long long)n * n) % (2LL * N);
            const long double ang = (long double)sign * pi * (long double)n2 / (long double)N;
            c[n] = std::complex<long double>(cosl(ang), sinl(ang));
        }
        g[0] = std::conj(c[0]);
        for (int m = 1; m < N; m++) g[m] = g[L - m] = std::conj(c[m]);
        host_fft_ld(g);
        std::vector<C> hc(N), hg(L);
        for (int n = 0; n < N; n++) hc[n] = cmake<R>((R)c[n].real(), (R)c[n].imag());
        for (int k = 0; k < L; k++) hg[k] = cmake<R>((R)(g[k].real() / L), (R)(g[k].imag() / L));
        const C* dc = static_cast<const C*>(shared_table(hc.data(), hc.size() * sizeof(C)));
        const C* dg = static_cast<const C*>(shared_table(hg.data(), hg.size() * sizeof(C)));
        if (!dc || !dg) return ST_ENOMEM;
        it = cache.emplace(key, std::make_pair(dc, dg)).first;
    }
    *chirp = it->second.first;
    *ghat = it->second.second;
    return ST_OK;
}

// Lines of length N (not a power of two, 2N - 1 <= 8192) through Bluestein, in
// the registers of the threads of an L-point line.  Same loads, pre/post
// multipliers, absorbing-layer pass and stores as k_fft_lines.
template <int L, typename R>
__global__ void __launch_bounds__((FftShape<L, R>::TPB)) k_fft_bluestein(FftArgsT<R> a) {
    typedef cplx_t<R> C;
    typedef FftShape<L, R> S;
    extern __shared__ __align__(16) unsigned char fft_smem[];
    const int t = S::LINES == 1 ? threadIdx.x : threadIdx.x % S::T, l = S::LINES == 1 ? 0 : threadIdx.x / S::T;
    C* const ph = reinterpret_cast<C*>(fft_smem + S::LDS);
    void* const lds = fft_smem + l * S::LS;
    const int N = a.N;
    const int64_t line = (int64_t)blockIdx.x * S::LINES + l;
    const bool on = line < a.nlines;
    const FftLine<R> ln(a, on ? line : 0);
    C v[S::E];
#pragma unroll
    for (int e = 0; e < S::E; e++) {
        const int x = t + S::T * e;
        v[e] = cmake<R>(0, 0);
        if (x < N && on) {
            v[e] = ln.in[x];
            if (a.pre) v[e] = cmul(v[e], a.pre[x]);
        }
    }
    if (a.ph_at) fft_phase<S::TPB>(a, ph);
    if (a.ph_at == 1) {
#pragma unroll
        for (int e = 0; e < S::E; e++)
            if (t + S::T * e < N) v[e] = cmul(v[e], ph[t + S::T * e]);
    }
    const C *chirp = a.bs_chirp, *ghat = a.bs_ghat;
    for (int pass = 0;; pass++) {
#pragma unroll
        for (int e = 0; e < S::E; e++)
            if (t + S::T * e < N) v[e] = cmul(v[e], chirp[t + S::T * e]);
        fft_line<L>(v, t, lds, -1, a.tw);
#pragma unroll
        for (int e = 0; e < S::E; e++) v[e] = cmul(v[e], ghat[t + S::T * e]);
        fft_line<L>(v, t, lds, +1, a.tw);
#pragma unroll
        for (int e = 0; e < S::E; e++) {
            const int x = t + S::T * e;
            v[e] = x < N ? cmul(v[e], chirp[x]) : cmake<R>(0, 0);
            // fb_io.f90:263: multiply the first nxfilt points, transform back
            if (a.filtr && pass == 0 && x < a.nxfilt) v[e] = crs(a.filtr[x], v[e]);
        }
        if (!a.filtr || pass == 1) break;
        chirp = a.bs_chirp2, ghat = a.bs_ghat2;
    }
    if (!on) return;
    if (a.ph_at == 2) {
#pragma unroll
        for (int e = 0; e < S::E; e++)
            if (t + S::T * e < N) v[e] = cmul(v[e], ph[t + S::T * e]);
    }
#pragma unroll
    for (int e = 0; e < S::E; e++) {
        const int x = t + S::T * e;
        if (x < N) ln.store(a, x, a.post ? cmul(v[e], a.post[x]) : v[e]);
    }
}

int32_t fft_length_check(int N) {
    if (N < 1 || N > 8192 || ((N & (N - 1)) != 0 && bluestein_length(N) > 8192))
        return fail(ST_EUNSUP,
                    "FFT length %d: this build transforms powers of two up to 8192 and other lengths up to 4096 "
                    "along x", N);
    return ST_OK;
}

template <int N, typename R, bool BLUESTEIN>
static int32_t launch_fft_n(const FftArgsT<R>& a) {
    typedef FftShape<N, R> S;
    const unsigned grid = (unsigned)((a.nlines + S::LINES - 1) / S::LINES);
    const auto kern = BLUESTEIN ? k_fft_bluestein<N < 64 ? 64 : N, R> : k_fft_lines<N, R>;
    const size_t lds = S::LDS + (a.ph_at ? (size_t)a.N * sizeof(cplx_t<R>) : 0);
    if constexpr (S::LDS + (size_t)N * sizeof(cplx_t<R>) > 64 * 1024) {
        static std::atomic<bool> attr_done{false};
        if (!attr_done.load(std::memory_order_acquire)) {
            CH_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, FFT_LDS_MAX));
            attr_done.store(true, std::memory_order_release);
        }
    }
    KTimer kt(KF_FFT);
    hipLaunchKernelGGL(kern, grid, S::TPB, lds, stream(), a);
    CH_LAUNCH_CHECK(BLUESTEIN ? "k_fft_bluestein" : "k_fft_lines");
    return ST_OK;
}
template <int N, typename R>
static int32_t launch_fft_len(const FftArgsT<R>& a, int len, bool bluestein) {
    if constexpr (N <= 8192) {
        if (len != N) return launch_fft_len<2 * N, R>(a, len, bluestein);
        if constexpr (N >= 64)
            if (bluestein) return launch_fft_n<N, R, true>(a);
        return launch_fft_n<N, R, false>(a);
    }
    return fail(ST_EUNSUP, "FFT length %d", a.N);
}

template <typename R>
int32_t launch_fft(FftArgsT<R> a) {
    if (a.nlines <= 0) return ST_OK;
    const int N = a.N;
    CH_TRY(fft_length_check(N));
    const bool bs = (N & (N - 1)) != 0;
    const int len = bs ? bluestein_length(N) : N;
    a.tw = fft_twiddles<R>(len);
    if (!a.tw) return ST_ENOMEM;
    if (bs) {
        CH_TRY(bluestein_tables<R>(N, a.sign, &a.bs_chirp, &a.bs_ghat));
        if (a.filtr) CH_TRY(bluestein_tables<R>(N, -a.sign, &a.bs_chirp2, &a.bs_ghat2));
    }
    // The phase costs a sine and a cosine in double (about 80 FP64 operations)
    // for each point of every block when it is formed in the transform, and a
    // launch when k_phase forms it once for all lines.  Whole steps, in the
    // transforms and in k_phase: 49 000 points 161 and 166 us; 390 000 points 225
    // and 224; 1.5 million 369 and 353
    if (a.ph_at && (N > FFT_PHASE_LINE || a.nlines * N > FFT_PHASE_POINTS)) {
        CH_TRY(make_phase<R>(a.ph_table, a.ph_kx, a.ph_leftX, a.ph_s, N, a.ph_leftX_dev));
        if (a.ph_at == 1) a.pre = a.ph_table;
        else a.post = a.ph_table;
        a.ph_at = 0;
    }
    return launch_fft_len<1, R>(a, len, bs);
}
template int32_t launch_fft<double>(FftArgsT<double>);
template int32_t launch_fft<float>(FftArgsT<float>);

}  // namespace chimera
