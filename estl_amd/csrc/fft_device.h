// fft_device.h -- device building blocks of the gfx950 FFT kernels.
//
// * complex helpers on float2 (interleaved complex64, the layout of the FFTW3 path,
//   FFT_FFTW3.h:24, and of ComplexArray(..., planar=false), Complex.h:156-192);
// * compile-time twiddle constants W_R^k = exp(DIR * 2 pi i k / R), evaluated in double
//   by constexpr series and rounded once to float (the reference printed them with six
//   significant digits, KernelGenerator.h:60-66; here they are correctly rounded);
// * register-resident DFTs of size 2..32 (natural order in and out), plain or with their
//   inputs' twiddles folded into the butterflies.  They
//   play the role of OpenCLFFTAlgorithm::generateLocalFFTKernel (OpenCLFFTAlgorithm.h:14-43)
//   and of the +-1/+-i shortcuts of KomplexConstMultiplication (KernelGenerator.h:100-142),
//   as C++ templates instead of generated OpenCL strings.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

namespace estl {

// ---------------------------------------------------------------- complex helpers
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }

// a * w
__device__ __forceinline__ float2 cmul(float2 a, float2 w) {
    return make_float2(fmaf(a.x, w.x, -a.y * w.y), fmaf(a.x, w.y, a.y * w.x));
}
// a * conj(w)
__device__ __forceinline__ float2 cmulc(float2 a, float2 w) {
    return make_float2(fmaf(a.x, w.x, a.y * w.y), fmaf(a.y, w.x, -a.x * w.y));
}
// a * w for DIR = -1 (w as tabulated, forward) or a * conj(w) for DIR = +1 (backward):
// tables hold the forward twiddles exp(-2 pi i m / M); the backward ones are their
// conjugates, which is exact.
template <int DIR>
__device__ __forceinline__ float2 ctw(float2 a, float2 w) {
    if constexpr (DIR < 0) return cmul(a, w);
    else return cmulc(a, w);
}

// Streaming (nontemporal) global accesses for data touched exactly once.
typedef float v2f_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float2 ld_stream(const float2 *p) {
    v2f_t v = __builtin_nontemporal_load(reinterpret_cast<const v2f_t *>(p));
    return make_float2(v.x, v.y);
}
__device__ __forceinline__ void st_stream(float2 *p, float2 x) {
    v2f_t v = {x.x, x.y};
    __builtin_nontemporal_store(v, reinterpret_cast<v2f_t *>(p));
}
__device__ __forceinline__ float ld_stream_f(const float *p) { return __builtin_nontemporal_load(p); }
__device__ __forceinline__ void st_stream_f(float *p, float x) { __builtin_nontemporal_store(x, p); }

// The reference's tile-planarized layout (PlannarizedComplexArray<5>, Complex.h:34-48,
// 97-130): in a float array, the real part of value e sits at ((e >> 5) << 6) | (e & 31)
// and its imaginary part 32 floats later -- 32 reals, then their 32 imaginaries.
__device__ __forceinline__ long planar_pos(long e) { return ((e >> 5) << 6) | (e & 31); }
__device__ __forceinline__ float2 ld_planar(const float2 *base, long e) {
    const float *f = reinterpret_cast<const float *>(base) + planar_pos(e);
    return make_float2(__builtin_nontemporal_load(f), __builtin_nontemporal_load(f + 32));
}
__device__ __forceinline__ void st_planar(float2 *base, long e, float2 v) {
    float *f = reinterpret_cast<float *>(base) + planar_pos(e);
    __builtin_nontemporal_store(v.x, f);
    __builtin_nontemporal_store(v.y, f + 32);
}

// FP16 storage of a complex value (re, im as IEEE binary16), computed on in FP32.
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float2 ld_elem(const float2 *p) { return ld_stream(p); }
__device__ __forceinline__ void st_elem(float2 *p, float2 x) { st_stream(p, x); }
__device__ __forceinline__ float2 ld_elem(const f16x2 *p) {
    const f16x2 h = __builtin_nontemporal_load(p);
    return make_float2((float)h.x, (float)h.y);
}
__device__ __forceinline__ void st_elem(f16x2 *p, float2 x) {
    const f16x2 h = {(_Float16)x.x, (_Float16)x.y};  // round to nearest even
    __builtin_nontemporal_store(h, p);
}

// p as a pointer to global memory, for pointers whose origin the compiler does not see (one
// read from a descriptor, or behind an asm): it would access generic ones with flat
// instructions, whose loads also count as LDS accesses and hold up the waits for those.
template <class T>
__device__ __forceinline__ T *global_ptr(T *p) {
    return (T *)(T __attribute__((address_space(1))) *)reinterpret_cast<uintptr_t>(p);
}

// Returns p unchanged, but hides from the optimiser that it is loop-invariant.  Used on
// twiddle-table pointers inside loops over rows/items: otherwise every twiddle load of a
// pass is hoisted out of the loop and ~30 float2 stay live for the whole kernel, which
// costs occupancy; re-issued per use they hit in L1/L2.
template <class T>
__device__ __forceinline__ const T *opaque(const T *p) {
    asm volatile("" : "+s"(p));
    return global_ptr(p);
}
// Same for a per-lane value (the thread index): in loops whose body dispatches on a
// size class, addresses derived from the thread index alone would otherwise be hoisted
// for every class at once and all stay live.
// Value e of a convolution filter of length n built from k real taps h: the taps folded
// modulo n (a filter longer than the signal wraps, the circular definition) and rotated
// by `shift` -- the sum of h[t] over t = e + shift (mod n), accumulated in FP64.
__device__ __forceinline__ float fold_tap(const float *__restrict__ h, long k, long n, long shift, long e) {
    double acc = 0.0;
    for (long t = (e + shift) % n; t < k; t += n) acc += (double)h[t];
    return (float)acc;
}

__device__ __forceinline__ int opaque_lane(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

// ---------------------------------------------------------------- compile-time trig
namespace ct {
constexpr double kPi = 3.141592653589793238462643383279502884;

constexpr double sin_series(double x) {  // |x| <= pi/4
    double x2 = x * x, term = x, sum = x;
    for (int i = 1; i < 16; ++i) {
        term *= -x2 / double((2 * i) * (2 * i + 1));
        sum += term;
    }
    return sum;
}
constexpr double cos_series(double x) {  // |x| <= pi/4
    double x2 = x * x, term = 1.0, sum = 1.0;
    for (int i = 1; i < 16; ++i) {
        term *= -x2 / double((2 * i - 1) * (2 * i));
        sum += term;
    }
    return sum;
}
// cos and sin of 2 pi k / n for n a power of two: exact quarter-turn reduction, then a
// series on [-pi/4, pi/4].
constexpr long long pmod(long long k, long long n) { return ((k % n) + n) % n; }
constexpr double cos2pi(long long k, long long n) {
    long long m = pmod(k, n);
    if (n < 4) return (m == 0) ? 1.0 : -1.0;
    long long q = (4 * m + n / 2) / n;        // nearest quarter turn
    long long r = 4 * m - q * n;              // remainder in units of (2 pi / 4n)
    double phi = 2.0 * kPi * double(r) / double(4 * n);
    double c = cos_series(phi), s = sin_series(phi);
    switch (q & 3) {
        case 0: return c;
        case 1: return -s;
        case 2: return -c;
        default: return s;
    }
}
constexpr double sin2pi(long long k, long long n) {
    long long m = pmod(k, n);
    if (n < 4) return 0.0;
    long long q = (4 * m + n / 2) / n;
    long long r = 4 * m - q * n;
    double phi = 2.0 * kPi * double(r) / double(4 * n);
    double c = cos_series(phi), s = sin_series(phi);
    switch (q & 3) {
        case 0: return s;
        case 1: return c;
        case 2: return -s;
        default: return -c;
    }
}
}  // namespace ct

// x * W_R^K with W_R = exp(DIR 2 pi i / R); trivial rotations become swaps and negations.
template <int K, int R, int DIR>
__device__ __forceinline__ float2 twc(float2 x) {
    constexpr int k = int(ct::pmod(K, R));
    if constexpr (k == 0) {
        return x;
    } else if constexpr ((4 * k) % R == 0) {
        constexpr int q = (4 * k) / R;           // quarter turns, 1..3
        constexpr int qd = (DIR < 0) ? (4 - q) % 4 : q;  // positive-direction turns
        if constexpr (qd == 1) return make_float2(-x.y, x.x);   // * i
        else if constexpr (qd == 2) return make_float2(-x.x, -x.y);
        else return make_float2(x.y, -x.x);                     // * -i
    } else if constexpr ((8 * k) % R == 0) {
        constexpr float h = 0.70710678118654752440f;
        constexpr float c = float(ct::cos2pi(k, R));
        constexpr float s = float(DIR) * float(ct::sin2pi(k, R));
        // c, s = +-h: two adds and two multiplies
        constexpr float sc = (c > 0) ? 1.0f : -1.0f;
        constexpr float ss = (s > 0) ? 1.0f : -1.0f;
        return make_float2(h * (sc * x.x - ss * x.y), h * (ss * x.x + sc * x.y));
    } else {
        constexpr float c = float(ct::cos2pi(k, R));
        constexpr float s = float(DIR) * float(ct::sin2pi(k, R));
        return make_float2(fmaf(x.x, c, -x.y * s), fmaf(x.x, s, x.y * c));
    }
}

// compile-time for loop: f(std::integral_constant<int, I>) for I in [B, E)
template <int B, int E>
struct StaticFor {
    template <class F>
    static __device__ __forceinline__ void run(F &&f) {
        if constexpr (B < E) {
            f(std::integral_constant<int, B>{});
            StaticFor<B + 1, E>::run(f);
        }
    }
};

// ---------------------------------------------------------------- register DFTs
// Transforms of R <= 32 values in registers, natural order in and out, unnormalised, as
// radix-2 decimation in time.  A butterfly with twiddle w is six fused multiply-adds,
// a' = a + w b (two per component) and 2 a - a': with 3 log2 R instructions per value,
// twiddles included, fewer than higher radices with their products apart (a twiddled
// 16-point transform: 217 instructions with its twiddles' generation; as radix 4 after
// 15 products by powers of w: 276).

// a + w b and a - w b (as 2 a less the sum: a sum that overflows, or is of infinities, takes the
// difference with it); w as tabulated for the forward direction (DIR > 0 takes its
// conjugate), a quarter turn further with ROT.
template <int DIR, bool ROT>
__device__ __forceinline__ void butterfly(float2 a, float2 b, float2 w, float2 &sum, float2 &diff) {
    // the twiddle's real part c, and s: w = c + i s
    const float c = ROT ? w.y : w.x;
    const float s = ROT ? (DIR < 0 ? -w.x : w.x) : (DIR < 0 ? w.y : -w.y);
    const float2 t = make_float2(fmaf(-s, b.y, fmaf(c, b.x, a.x)), fmaf(s, b.x, fmaf(c, b.y, a.y)));
    sum = t;
    diff = make_float2(fmaf(2.0f, a.x, -t.x), fmaf(2.0f, a.y, -t.y));
}

// The twiddles of a DFT of R values weighted by w^i: on the level that joins transforms of
// r / 2 to r, w^(R/r) W_r^k for k < r / 4 (the next r / 4 are a quarter turn further), at
// r / 4 + k; for r = 2 at 0.
template <int R>
struct LevelTw {
    static constexpr int count = R > 4 ? R / 2 : R == 4 ? 2 : 1;
    float2 t[count];
    // from p[l] = w^(2^l), l < log2 R
    __device__ __forceinline__ explicit LevelTw(const float2 *p) {
        constexpr int LR = __builtin_ctz(R);
        t[0] = p[LR - 1];
        StaticFor<2, LR + 1>::run([&](auto lc) {
            constexpr int l = decltype(lc)::value, r = 1 << l;
            StaticFor<0, r / 4>::run([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                t[r / 4 + k] = twc<k, r, -1>(p[LR - l]);
            });
        });
    }
};

template <int R, int DIR, bool TW>
__device__ __forceinline__ void dft_dit(float2 (&x)[R], const float2 *tw) {
    static_assert(R >= 1 && (R & (R - 1)) == 0, "radix must be a power of two");
    if constexpr (R > 1) {
        float2 e[R / 2], o[R / 2];
        StaticFor<0, R / 2>::run([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            e[i] = x[2 * i];
            o[i] = x[2 * i + 1];
        });
        dft_dit<R / 2, DIR, TW>(e, tw);
        dft_dit<R / 2, DIR, TW>(o, tw);
        StaticFor<0, R / 2>::run([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            if constexpr (TW) {
                constexpr bool rot = R >= 4 && k >= R / 4;
                butterfly<DIR, rot>(e[k], o[k], tw[R / 4 + (rot ? k - R / 4 : k)], x[k], x[k + R / 2]);
            } else if constexpr ((4 * k) % R == 0) {
                const float2 b = twc<k, R, DIR>(o[k]);
                x[k] = cadd(e[k], b);
                x[k + R / 2] = csub(e[k], b);
            } else {
                constexpr float c = float(ct::cos2pi(k, R)), s = -float(ct::sin2pi(k, R));
                butterfly<DIR, false>(e[k], o[k], make_float2(c, s), x[k], x[k + R / 2]);
            }
        });
    }
}

// In-place DFT of x[0..R), sign DIR.
template <int R, int DIR>
struct Dft {
    static __device__ __forceinline__ void run(float2 *x) {
        float2 y[R];
        StaticFor<0, R>::run([&](auto ic) { y[decltype(ic)::value] = x[decltype(ic)::value]; });
        dft_dit<R, DIR, false>(y, nullptr);
        StaticFor<0, R>::run([&](auto ic) { x[decltype(ic)::value] = y[decltype(ic)::value]; });
    }
};

// a + w b and a - w b, each by itself: 8 instructions instead of butterfly's 6.
template <int K, int R, int DIR>
__device__ __forceinline__ void butterfly_apart(float2 a, float2 b, float2 &sum, float2 &diff) {
    if constexpr ((4 * K) % R == 0) {
        const float2 t = twc<K, R, DIR>(b);
        sum = cadd(a, t);
        diff = csub(a, t);
    } else {
        constexpr float c = float(ct::cos2pi(K, R)), s = float(DIR) * float(ct::sin2pi(K, R));
        sum = make_float2(fmaf(-s, b.y, fmaf(c, b.x, a.x)), fmaf(s, b.x, fmaf(c, b.y, a.y)));
        diff = make_float2(fmaf(s, b.y, fmaf(-c, b.x, a.x)), fmaf(-s, b.x, fmaf(-c, b.y, a.y)));
    }
}

// The DFT of a whole transform of R <= 16 values: no sum takes another along when it overflows,
// and no value meets two rotations by other than quarter turns, so an infinite input gives
// infinities of the right signs and no NaN.  Such transforms are HBM-bound (16 values per
// thread, no exchange).
template <int R, int DIR>
struct DftApart {
    static_assert(R <= 16, "one register DFT");
    static __device__ __forceinline__ void run(float2 *x) {
        if constexpr (R < 8) {
            Dft<R, DIR>::run(x);
        } else {
            // R / 4 apart: S transforms of 4 or 2 x 4 values, joined with one rotation each
            constexpr int S = R / 4;
            float2 e[S][4];
            StaticFor<0, S>::run([&](auto sc) {
                constexpr int s = decltype(sc)::value;
                StaticFor<0, 4>::run([&](auto mc) { e[s][decltype(mc)::value] = x[S * decltype(mc)::value + s]; });
                Dft<4, DIR>::run(e[s]);
            });
            StaticFor<0, 4>::run([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                if constexpr (S == 2) {
                    butterfly_apart<k, R, DIR>(e[0][k], e[1][k], x[k], x[k + 4]);
                } else {
                    float2 a, b, c, d;
                    butterfly_apart<2 * k, R, DIR>(e[0][k], e[2][k], a, b);
                    butterfly_apart<3 * k, R, DIR>(twc<k, R, DIR>(e[1][k]), e[3][k], c, d);
                    const float2 t = twc<1, 4, DIR>(d);
                    x[k] = cadd(a, c);
                    x[k + 4] = cadd(b, t);
                    x[k + 8] = csub(a, c);
                    x[k + 12] = csub(b, t);
                }
            });
        }
    }
};

__device__ __forceinline__ float2 csquare(float2 a) {
    return make_float2(fmaf(a.x, a.x, -a.y * a.y), 2.0f * a.x * a.y);
}

// In-place DFT of x_i w^i (conj(w)^i for DIR > 0), R <= 16, with w^4 given too (read only
// for R >= 8): w^2 and w^8 are then one squaring away from a rounded value, and the
// twiddles' error stays below that of products of powers of w alone.
template <int R, int DIR>
__device__ __forceinline__ void dft_twiddled(float2 (&x)[R], const float2 *__restrict__ w1, const float2 *__restrict__ w4) {
    constexpr int LR = __builtin_ctz(R);
    static_assert(LR >= 1 && LR <= 4, "radix 2 to 16");
    float2 p[4];
    p[0] = *w1;
    if constexpr (LR > 1) p[1] = csquare(p[0]);
    if constexpr (LR > 2) p[2] = *w4;
    if constexpr (LR > 3) p[3] = csquare(p[2]);
    const LevelTw<R> tw(p);
    dft_dit<R, DIR, true>(x, tw.t);
}

// ---------------------------------------------------------------- synthetic data
__device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
    uint64_t z = x + 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

}  // namespace estl
