// fft_block.h -- workgroup-cooperative Stockham FFT held in registers, exchanged
// through LDS.
//
// A sequence of length N = 2^LOG2N is spread over TPT = N / E threads, E = 16 values
// per thread: thread tl holds element tl + TPT*i in v[i].  The plan is the reference's
// global radix list (FFT_OpenCL_Contiguous.h:55-60: radix-16 passes, the 2^(log2N mod 4)
// remainder last) and every pass follows its Stockham recurrence
// (FFT_OpenCL_Contiguous.h:167-180, docs/ImplementationStrategy.pdf eq. 7/12):
//
//   d_q[(N/N_q)(g + A_q h) + z] = sum_s d_{q-1}[(N/N_q)(B_q g + s) + z] W_{N_q}^{g s} W_{B_q}^{h s}
//
// but where the reference runs one kernel launch (one HBM round trip) per pass, here a
// pass is a register DFT and the hand-over between passes is an LDS exchange.  After
// every pass thread tl holds d_q[tl + TPT*i] in v[i] again, so the first pass needs no
// exchange (its inputs are exactly what a coalesced load gives) and the last pass
// leaves the result in the order a coalesced store wants.
#pragma once

#include "fft_device.h"
#include "internal.h"

namespace estl {

template <int LOG2N>
struct BlockGeom {
    static constexpr int N = 1 << LOG2N;
    static constexpr int E = (LOG2N >= 4) ? 16 : N;  // complex values per thread
    static constexpr int TPT = N / E;                // threads per sequence
    static constexpr int NFULL = LOG2N / 4;          // radix-16 passes
    static constexpr int REM = LOG2N % 4;
    static constexpr int P = NFULL + (REM ? 1 : 0);  // passes
    static constexpr int radix(int q) { return q < NFULL ? 16 : (1 << REM); }
    static constexpr long A(int q) {
        long a = 1;
        for (int p = 0; p < q; ++p) a *= radix(p);
        return a;
    }
    // the power table: W_{N_q}^g for g in [0, A_q) per pass q >= 1, at
    // powoff(q), and their fourth powers powsum further on
    static constexpr long powoff(int q) {
        long o = 0;
        for (int p = 1; p < q; ++p) o += A(p);
        return o;
    }
    static constexpr long powsum = powoff(P), powsize = 2 * powsum;
    static constexpr bool uses_lds = TPT > 1;
};

// Twiddles of block_fft's passes q >= 1 (a butterfly of pass q, group g, needs W_{N_q}^{g s}
// for s in [1, B_q)): w = W_{N_q}^g and w^4 read from the power table (twice the sum of the
// A_q, 68 KiB at 2^14, mostly cache-resident), w^2 and w^8 by squaring, the twiddles of
// each level of the DFT from them (dft_twiddled).  A table of every W_{N_q}^{g s} (128 KiB
// at 2^14, B_q - 1 reads per butterfly) held in registers across rows needed 167-206 VGPRs
// and was 6-9 % slower at 4096 and 8192 points, and read again for each row slower still.
// Rel-L2 against FP64 is 1.6e-7 at 4096 points (the bound is 1.2e-5): 3.0e-7 when every
// power came from w alone, 1.2e-7 with that table's rounded values.

// LDS layout of a sequence's exchange buffer: one float2 of padding after every 16 values;
// addresses stay base + constant, so the exchanges use immediate offsets.
struct Lds {
    static constexpr int size(int n) { return n + (n >> 4); }
    static __device__ __forceinline__ int idx(int i) { return i + (i >> 4); }
    // idx(i + off), given idx(i), where adding off to i carries nothing into bit 4 (off a
    // multiple of 16, or i + off within the 16 values of i): one add with a constant, which
    // the LDS instructions take as their offset.  Formed from i + off, each address cost two
    // to four instructions (the 4096-point rows kernel had 845 vector instructions; 619
    // with these and dft_dit's folded twiddles).
    static __device__ __forceinline__ constexpr int step(int at, int off) { return at + off + (off >> 4); }
};

// On entry v[i] = x[tl + TPT*i]; on exit v[i] = X[tl + TPT*i] (X = DFT of x, sign DIR).
// `lds` is this sequence's LDS slice (Lds::size(N) float2); `tw` the size-N power table.
// All threads of the workgroup must call it together (it holds workgroup barriers).
// If `lds_busy` is set, the slice is still being read on entry and a barrier is placed
// before the first LDS write.  Twiddles are read anew at each use (from L1/L2): callers that
// run many rows or sizes in one loop would otherwise have all of them live.
template <int LOG2N, int DIR>
__device__ __forceinline__ void block_fft(float2 (&v)[BlockGeom<LOG2N>::E], float2 *lds, int tl,
                                          const float2 *__restrict__ tw, bool lds_busy = false) {
    using G = BlockGeom<LOG2N>;
    constexpr int N = G::N, E = G::E, TPT = G::TPT;
    StaticFor<0, G::P>::run([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        constexpr int B = G::radix(q);
        constexpr int NB = E / B;  // butterflies per thread in this pass
        constexpr int Aq = int(G::A(q));
        constexpr int S = N / (Aq * B);
        if constexpr (q == 0) {
            StaticFor<0, NB>::run([&](auto bc) {
                constexpr int b = decltype(bc)::value;
                float2 u[B];
                StaticFor<0, B>::run([&](auto sc) { u[decltype(sc)::value] = v[b + NB * decltype(sc)::value]; });
                if constexpr (G::P == 1) DftApart<B, DIR>::run(u);
                else Dft<B, DIR>::run(u);
                StaticFor<0, B>::run([&](auto hc) { v[b + NB * decltype(hc)::value] = u[decltype(hc)::value]; });
            });
        } else {
            if (q > 1 || lds_busy) __syncthreads();
            const int at = Lds::idx(tl);
#pragma unroll
            for (int i = 0; i < E; ++i) {
                if constexpr (TPT % 16 == 0) lds[Lds::step(at, TPT * i)] = v[i];
                else lds[Lds::idx(tl + TPT * i)] = v[i];
            }
            __syncthreads();
            StaticFor<0, NB>::run([&](auto bc) {
                constexpr int b = decltype(bc)::value;
                const int j = tl + TPT * b;
                const int g = j / S, z = j % S;   // S is a power of two
                const int base = S * B * g + z;
                float2 u[B];
                const int from = Lds::idx(base);
                // base is a multiple of S B plus z < S: S s is a multiple of 16, or less
                // than 16 - z within the aligned 16 of S B >= 16 or S B < 16 values
#pragma unroll
                for (int s = 0; s < B; ++s) u[s] = lds[Lds::step(from, S * s)];
                const float2 *w = opaque(tw) + G::powoff(q) + g;
                dft_twiddled<B, DIR>(u, w, w + G::powsum);
#pragma unroll
                for (int h = 0; h < B; ++h) v[b + NB * h] = u[h];
            });
        }
    });
}

}  // namespace estl
