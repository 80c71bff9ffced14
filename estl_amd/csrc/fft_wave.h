// fft_wave.h -- transforms whose order of bins does not matter (the convolutions'), with
// one exchange across the workgroup and the rest inside waves.
//
// A transform of N = 2^LOG2N points (2^10 .. 2^14) is spread over T = N / 32 threads, 32
// values per thread, and runs decimation in frequency: with n = t + T i and
// k = k1 + 32 k',
//
//   X[k1 + 32 k'] = sum_t W_T^{t k'} ( W_N^{t k1} sum_i x[t + T i] W_32^{i k1} )
//
// the inner sum is a 32-point DFT in registers, and what is left are 32 independent
// transforms of T points, one per k1, each over Q = T / 32 neighbouring threads -- threads
// of one wave.  They run the same step again (t = t' + Q i', k' = k2 + 32 k3) and end in
// transforms of Q points in registers.  So only the hand-over of the first step crosses
// the workgroup (and nothing does up to N = 2^11); the second stays inside a wave and needs
// no barrier.  The inverse runs the steps backwards (decimation in time), from the order
// in which the forward left the bins: thread u = k1 Q + t' holds in register r = m Q + k3
// bin k1 + 32 (m + (32 / Q) t') + 1024 k3, stored at r T + u in a spectrum.
//
// The exchanges send real and imaginary parts one after the other through half the LDS:
// 66 KiB at 2^14 points, two workgroups per CU at four waves per SIMD, where the whole
// values need 139 KiB and leave one.
#pragma once

#include "fft_device.h"
#include "internal.h"

namespace estl {

template <int LOG2N>
struct WaveGeom {
    static_assert(LOG2N >= 10 && LOG2N <= 14, "32 values per thread, rows of Q <= 16 threads");
    static constexpr int N = 1 << LOG2N, E = 32;
    static constexpr int T = N / E;  // threads per transform
    static constexpr int Q = T / 32;  // threads per row (the T-point transform of one k1)
    static constexpr bool in_wave = T <= 64;
    // Floats from one row's LDS slice to the next.  A row holds its T values (first
    // exchange), or them with one float of padding after every 32 (second).  33 Q puts the
    // 32 / Q rows of 32 lanes on distinct groups of Q banks: no access of either exchange
    // has a bank conflict.
    static constexpr int RS = 33 * Q;
    static constexpr int lds_floats = 32 * RS;
};

// Orders this wave's LDS accesses (a wave's LDS operations execute in order; the
// compiler must not move them across).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <bool IN_WAVE>
__device__ __forceinline__ void exchange_sync() {
    if constexpr (IN_WAVE) wave_lds_fence();
    else __syncthreads();
}

// Twiddles go to the inputs of each step, as powers of one root per transform, which
// dft_dit folds into its butterflies: before the second step value i' of row k1 has
// W_N^{t k1} = W_N^{t' k1} (W_1024^{k1})^{i'}, and the first factor waits for the third,
// where value t' of (k1, k2) has (W_N^{k1 + 32 k2})^{t'}; backwards, the roots are W_T^{t'}
// (powers k2) and W_N^t (powers k1).  The roots' table (wave_table), each value correctly
// rounded, with the fourth and sixteenth powers beside the roots so that no power is
// squared twice:
//   row:   W_1024^{e k1}, k1 < 32, for e = 1, 4, 16
//   bin:   W_N^{e (k1 + 32 k2)} at (k2 mod 32 / Q) T + thread (wave_bin), for e = 1, 4
//   pos:   W_T^{e t'}, t' < Q, for e = 1, 4, 16
//   point: W_N^{e t}, t < T, for e = 1, 4, 16
template <int LOG2N>
struct WaveRoots {
    static constexpr WaveLayout at{LOG2N};
    static_assert(at.T == WaveGeom<LOG2N>::T && at.Q == WaveGeom<LOG2N>::Q, "the table's geometry is the kernel's");
    static constexpr int row = at.row, bin = at.bin, pos = at.pos, point = at.point;
};

// w, w^4, w^16 of a 32-point step: at roots[t], [STRIDE + t], [2 STRIDE + t].  A step's roots
// are loaded before the exchange ahead of it, which needs few registers, and arrive
// meanwhile: loaded where they are used, each step of a lone wave waited for the L2 (a call of
// one row of 2^14 values 11.1 -> 10.6 us, 1000 rows of 2^11 8.9 -> 8.25, 63 rows of 2^20 at 4097
// taps 154 -> 145).  At 2^10 values (Q = 1, no exchange but one inside the wave) they are
// loaded at their use: 30001 rows 46.2 us with them ahead, 45.5 so.
struct Roots32 {
    float2 w1, w4, w16;
};
template <int STRIDE>
__device__ __forceinline__ Roots32 load_roots(const float2 *__restrict__ roots, int t) {
    // read anew at each use: kept from one use to the next their powers would take
    // tens of registers
    const float2 *q = opaque(roots);
    return {q[t], q[STRIDE + t], q[2 * STRIDE + t]};
}

// In-place DFT of v[i] w^i (conjugated for DIR > 0), i < 32.
template <int DIR>
__device__ __forceinline__ void dft32_rooted(float2 (&v)[32], const Roots32 &w) {
    const float2 p[5] = {w.w1, csquare(w.w1), w.w4, csquare(w.w4), w.w16};
    const LevelTw<32> tw(p);
    dft_dit<32, DIR, true>(v, tw.t);
}

// w and w^4 (Q > 4 only) of a Q-point step, at roots[t] and [1024 + t].
struct RootsQ {
    float2 w1, w4;
};

// In-place DFT of x[i] w^i, i < Q <= 16.
template <int Q, int DIR>
__device__ __forceinline__ void dft_rooted(float2 *x, const RootsQ &w) {
    constexpr int LQ = __builtin_ctz(Q);
    float2 p[4], y[Q];
    p[0] = w.w1;
    p[1] = csquare(p[0]);
    if constexpr (LQ > 2) p[2] = w.w4;
    if constexpr (LQ > 3) p[3] = csquare(p[2]);
    const LevelTw<Q> tw(p);
    StaticFor<0, Q>::run([&](auto ic) { y[decltype(ic)::value] = x[decltype(ic)::value]; });
    dft_dit<Q, DIR, true>(y, tw.t);
    StaticFor<0, Q>::run([&](auto ic) { x[decltype(ic)::value] = y[decltype(ic)::value]; });
}

// v[i] = x[t + T i] on entry, bin k1 + 32 (m + (32 / Q) t') + 1024 k3 in v[m Q + k3] on exit.
// `lds` holds WaveGeom::lds_floats floats of this transform.  All threads of the
// workgroup call it together; `tw` is the table of WaveRoots.  With lds_busy, other threads may still be reading the slice.
template <int LOG2N>
__device__ __forceinline__ void wave_fft(float2 (&v)[32], float *lds, int t, const float2 *__restrict__ tw, bool lds_busy) {
    using G = WaveGeom<LOG2N>;
    constexpr int T = G::T, Q = G::Q, RS = G::RS;
    float *row = lds + (t / Q) * RS;
    const int tq = t % Q;
    using W = WaveRoots<LOG2N>;
    Dft<32, -1>::run(v);
    Roots32 wr;
    if constexpr (Q > 1) wr = load_roots<32>(tw + W::row, t / Q);
    if (lds_busy) exchange_sync<G::in_wave>();
#pragma unroll
    for (int k = 0; k < 32; ++k) lds[k * RS + t] = v[k].x;
    exchange_sync<G::in_wave>();
#pragma unroll
    for (int i = 0; i < 32; ++i) v[i].x = row[tq + Q * i];
    exchange_sync<G::in_wave>();
#pragma unroll
    for (int k = 0; k < 32; ++k) lds[k * RS + t] = v[k].y;
    exchange_sync<G::in_wave>();
#pragma unroll
    for (int i = 0; i < 32; ++i) v[i].y = row[tq + Q * i];
    if constexpr (Q == 1) wr = load_roots<32>(tw + W::row, t / Q);
    dft32_rooted<-1>(v, wr);
    if constexpr (Q > 1) {
        RootsQ wb[32 / Q];
        const float2 *bin = opaque(tw + W::bin);
#pragma unroll
        for (int m = 0; m < 32 / Q; ++m) {
            wb[m].w1 = bin[T * m + t];
            if constexpr (Q > 4) wb[m].w4 = bin[1024 + T * m + t];
        }
        wave_lds_fence();
#pragma unroll
        for (int k = 0; k < 32; ++k) row[k * Q + (k * Q >> 5) + tq] = v[k].x;
        wave_lds_fence();
#pragma unroll
        for (int r = 0; r < 32; ++r) v[r].x = row[33 * tq + r];
        wave_lds_fence();
#pragma unroll
        for (int k = 0; k < 32; ++k) row[k * Q + (k * Q >> 5) + tq] = v[k].y;
        wave_lds_fence();
#pragma unroll
        for (int r = 0; r < 32; ++r) v[r].y = row[33 * tq + r];
        StaticFor<0, 32 / Q>::run([&](auto mc) {
            constexpr int m = decltype(mc)::value;
            dft_rooted<Q, -1>(v + Q * m, wb[m]);
        });
    }
}

// The unnormalised inverse: bins in the order wave_fft leaves them to x[t + T i] in v[i].
// The caller's own wave was the last to read its rows of the slice (wave_fft's end state).
template <int LOG2N>
__device__ __forceinline__ void wave_ifft(float2 (&v)[32], float *lds, int t, const float2 *__restrict__ tw) {
    using G = WaveGeom<LOG2N>;
    using W = WaveRoots<LOG2N>;
    constexpr int T = G::T, Q = G::Q, RS = G::RS;
    float *row = lds + (t / Q) * RS;
    const int tq = t % Q;
    if constexpr (Q > 1) {
        const Roots32 wp = load_roots<Q>(tw + W::pos, tq);
        StaticFor<0, 32 / Q>::run([&](auto mc) { Dft<Q, +1>::run(v + Q * decltype(mc)::value); });
        wave_lds_fence();
#pragma unroll
        for (int r = 0; r < 32; ++r) row[33 * tq + r] = v[r].x;
        wave_lds_fence();
#pragma unroll
        for (int k = 0; k < 32; ++k) v[k].x = row[k * Q + (k * Q >> 5) + tq];
        wave_lds_fence();
#pragma unroll
        for (int r = 0; r < 32; ++r) row[33 * tq + r] = v[r].y;
        wave_lds_fence();
#pragma unroll
        for (int k = 0; k < 32; ++k) v[k].y = row[k * Q + (k * Q >> 5) + tq];
        dft32_rooted<+1>(v, wp);
    } else {
        Dft<32, +1>::run(v);
    }
    Roots32 wn;
    if constexpr (Q > 1) wn = load_roots<T>(tw + W::point, t);
    wave_lds_fence();
#pragma unroll
    for (int i = 0; i < 32; ++i) row[tq + Q * i] = v[i].x;
    exchange_sync<G::in_wave>();
#pragma unroll
    for (int k = 0; k < 32; ++k) v[k].x = lds[k * RS + t];
    exchange_sync<G::in_wave>();
#pragma unroll
    for (int i = 0; i < 32; ++i) row[tq + Q * i] = v[i].y;
    exchange_sync<G::in_wave>();
#pragma unroll
    for (int k = 0; k < 32; ++k) v[k].y = lds[k * RS + t];
    if constexpr (Q == 1) wn = load_roots<T>(tw + W::point, t);
    dft32_rooted<+1>(v, wn);
}

}  // namespace estl
