// pass_wide.h -- a global Stockham pass (pass_tile.h) with 32 values per thread, for passes
// over complex rows, interleaved or (a plan's first input, its last output) planarized.
//
// Column j of a pass of radix B = 32 P (g = j / S, z = j mod S) is
//
//   X[k1 + 32 k2] = sum_t W_P^{t k2} W_{AB}^{t (g + A k1)} sum_i x[t + P i] W_{AB}^{g P i} W_32^{i k1}
//
// with t < P, i < 32: a 32-point transform of inputs weighted by powers of W_{AB}^{g P},
// one exchange, and 32 transforms of P points of inputs weighted by powers of
// W_{AB}^{g + A k1} -- the pass's own twiddles W_{AB}^{g s} and the radix's inner ones in
// one, folded into the butterflies (dft_dit), from the roots' powers 1, 2, 4, ..., each read
// as one product of a two-level table (by squaring, the errors of 2^20 points were 8 %
// larger).
//
// (lds_busy: the slice may still be being read on entry.)
//
// A tile is T = 2^LOG2T adjacent columns over P T threads.  Lanes run over columns where
// the rows of a tile's input lie T values apart in memory (S >= T), and after the exchange
// always, so every store and these loads move T consecutive values; in a last pass (S = 1)
// a column's values are contiguous and lanes run over t, P consecutive values, before the
// exchange.  Real and imaginary parts go through the LDS one after the other: 35 KiB for
// 2^13 values, four workgroups per CU at four waves per SIMD, where k_fft_pass has two.
#pragma once

#include "fft_block.h"
#include "pass_tile.h"
#include "internal.h"

namespace estl {

enum { kWideFirst = 0, kWideMiddle = 1, kWideLast = 2 };  // A = 1; A > 1 and S >= T; S = 1

template <int LOG2B, int LOG2T, int MODE>
struct WideTile {
    static constexpr int B = 1 << LOG2B, T = 1 << LOG2T, P = B / 32, threads = P * T;
    // LDS position of value t of row k1 in column c: no two of 32 neighbouring lanes on one
    // bank (one pair in a last pass's writes with P = 16)
    static constexpr int SC = MODE == kWideLast ? P + 1 : 1;                // column to column
    static constexpr int ST = MODE == kWideLast ? 1 : T;                    // t to t
    static constexpr int RS = MODE == kWideLast ? T * (P + 1) : P * T + (T < 32 ? T : 0);  // row to row
    static constexpr int lds_floats = 32 * RS;
};

// W_{AB}^m from the pass's two-level table
__device__ __forceinline__ float2 pass_root(const PassArgs &a, unsigned m) {
    const unsigned lomask = (1u << a.lobits) - 1u;
    return cmul(a.tw_lo[m & lomask], a.tw_hi[m >> a.lobits]);
}

template <int LOG2B, int DIR, int LOG2T, int MODE, typename ST>
__device__ __forceinline__ void wide_tile(const ST *__restrict__ in, ST *__restrict__ out, const PassArgs &a, long tile,
                                          float *lds, bool lds_busy = false) {
    using G = WideTile<LOG2B, LOG2T, MODE>;
    constexpr int P = G::P, T = G::T, LOG2P = LOG2B - 5;
    const int th = opaque_lane(threadIdx.x);
    const int lcpr = a.log2n - LOG2B;  // columns per row = 2^lcpr
    const long row = tile >> (lcpr - LOG2T);
    const int j0 = int(tile - (row << (lcpr - LOG2T))) << LOG2T;
    const int ls = a.log2S;
    const unsigned ab_mask = ((unsigned)a.A << LOG2B) - 1u;
    const int c2 = th & (T - 1), u = th >> LOG2T;  // after the exchange: column, thread of it
    float2 v[32];
    {
        const int c = MODE == kWideLast ? th >> LOG2P : c2;
        const int t = MODE == kWideLast ? th & (P - 1) : u;
        // a scalar base per element, and one lane offset of at most P S T values
        const ST *src = in + (row << a.log2n);
        unsigned lane;
        if constexpr (MODE == kWideLast) {
            src += (long)j0 << LOG2B;
            lane = (unsigned)(c << LOG2B) + (unsigned)t;
        } else {
            src += ((long)(j0 >> ls) << (ls + LOG2B)) + (j0 & ((1 << ls) - 1));
            lane = ((unsigned)t << ls) + (unsigned)c;
        }
        constexpr bool F32 = __is_same(ST, float2);
        if (F32 && MODE == kWideFirst && a.planar_in) {
            // the same values from the tile-planarized layout, by element index
            const long e0 = (row << a.log2n) + j0 + (long)lane;
#pragma unroll
            for (int i = 0; i < 32; ++i)
                v[i] = ld_planar(reinterpret_cast<const float2 *>(in), e0 + ((long)(P * i) << ls));
        } else
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            const ST *p = src + (MODE == kWideLast ? (long)(P * i) : (long)(P * i) << ls);
            v[i] = ld_elem(reinterpret_cast<const ST *>(reinterpret_cast<const char *>(p) + lane * (unsigned)sizeof(ST)));
        }
        if constexpr (MODE == kWideFirst) {
            Dft<32, DIR>::run(v);
        } else {
            const unsigned g = MODE == kWideLast ? unsigned(j0 + c) : unsigned(j0 >> ls);
            const unsigned m = g << LOG2P;
            float2 p[5];
            StaticFor<0, 5>::run([&](auto ec) { p[ec] = pass_root(a, (m << ec) & ab_mask); });
            const LevelTw<32> tw(p);
            dft_dit<32, DIR, true>(v, tw.t);
        }
        const int at = c * G::SC + t * G::ST;
        if (lds_busy) __syncthreads();  // the previous tile's last reads
#pragma unroll
        for (int k = 0; k < 32; ++k) lds[k * G::RS + at] = v[k].x;
        __syncthreads();
        const int from = u * G::RS + c2 * G::SC;
#pragma unroll
        for (int r = 0; r < 32; ++r) v[r].x = lds[from + (r / P) * P * G::RS + (r % P) * G::ST];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 32; ++k) lds[k * G::RS + at] = v[k].y;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 32; ++r) v[r].y = lds[from + (r / P) * P * G::RS + (r % P) * G::ST];
    }
    // rows k1 = u + P m: the roots differ by W_B^{P m} = W_32^m
    {
        const unsigned g = MODE == kWideFirst ? 0u : MODE == kWideLast ? unsigned(j0 + c2) : unsigned(j0 >> ls);
        const unsigned m0 = g + (unsigned)a.A * (unsigned)u;
        float2 w[LOG2P];
        StaticFor<0, LOG2P>::run([&](auto ec) { w[ec] = pass_root(a, (m0 << ec) & ab_mask); });
        StaticFor<0, 32 / P>::run([&](auto mc) {
            constexpr int m = decltype(mc)::value;
            float2 p[LOG2P], x[P];
            StaticFor<0, LOG2P>::run([&](auto ec) {
                constexpr int e = decltype(ec)::value;
                p[e] = twc<(m << e) & 31, 32, -1>(w[e]);
            });
            const LevelTw<P> tw(p);
            StaticFor<0, P>::run([&](auto ic) { x[decltype(ic)::value] = v[P * m + decltype(ic)::value]; });
            dft_dit<P, DIR, true>(x, tw.t);
            StaticFor<0, P>::run([&](auto ic) { v[P * m + decltype(ic)::value] = x[decltype(ic)::value]; });
        });
    }
    // register r = P m + k2 holds bin u + P m + 32 k2
    ST *dst = out + (row << a.log2n) + j0;
    const unsigned lane = ((unsigned)u << lcpr) + (unsigned)c2;
    const float sc = a.scale;
    if (__is_same(ST, float2) && a.planar_out) {
        const long e0 = (row << a.log2n) + j0 + (long)lane;
#pragma unroll
        for (int r = 0; r < 32; ++r)
            st_planar(reinterpret_cast<float2 *>(out), e0 + ((long)((r / P) * P + 32 * (r % P)) << lcpr),
                      cscale(v[r], sc));
        return;
    }
#pragma unroll
    for (int r = 0; r < 32; ++r) {
        ST *p = dst + ((long)((r / P) * P + 32 * (r % P)) << lcpr);
        st_elem(reinterpret_cast<ST *>(reinterpret_cast<char *>(p) + lane * (unsigned)sizeof(ST)), cscale(v[r], sc));
    }
}

}  // namespace estl
