// workqueue.hip -- k_ubatch: a batch of transforms of uneven power-of-two sizes in one
// persistent launch driven by a work queue.
//
// The reference batches only transforms of one size (batchCount, FFT.h:25-27) and
// serves mixed sizes with one FFT object -- one plan, one program, one launch per pass --
// per size (tests/Test.cpp:48-53).  Here a descriptor list holds every transform of the
// batch and one launch computes them all:
//   * a work item is either a group of same-size rows (n <= 2^13: kUThreads/TPT rows computed
//     like k_fft_rows) or one whole large transform (2^14 <= n <= 2^20: both passes of a
//     two-pass plan, tile by tile, through a scratch region, with a workgroup barrier
//     between the passes -- no dependency crosses workgroups);
//   * items are ordered largest first and handed out by an atomic ticket, so workgroups
//     that drew small items keep drawing while others finish large ones;
//   * the last workgroup to leave resets the ticket counters, so the launch can be
//     replayed (and captured in a HIP graph) without a memset.
#include <utility>

#include "pass_tile.h"
#include "pass_wide.h"
#include "ubatch.h"

namespace estl {

// workgroup size 2^kUThreadsLog2: small items take 2^kUThreadsLog2 / TPT rows, large
// items tiles of 2^(kUThreadsLog2 + 4 - B) columns.  Measured on MI355X (8192 sizes
// 2^U{8..18}): 512 threads at four waves per SIMD 2.53 ms, 256 threads 3.42 ms (its
// 8-column tiles of radix 2^9 read 64-byte runs), 512 threads at three waves 2.97 ms.
constexpr int kUThreads = 1 << kUThreadsLog2;

template <int L>
struct USmall {
    using G = BlockGeom<L>;
    static constexpr int TPW = kUThreads / G::TPT;
    static constexpr int slice = G::uses_lds ? Lds::size(G::N) : 0;
    static constexpr int lds = TPW * slice;
};
// Transforms of 2^17 values and more keep 32 values per thread (wide_tile, tiles of 2^14
// values: twice the bytes in flight at the same four waves per SIMD): 500 of 2^17
// 476-520 -> 457-476 us, 60 of 2^20 2.08 -> 1.31 ms, 8192 of 2^8 .. 2^18 2.43 -> 2.31 ms.  With so
// few tiles a transform, 2^15 and 2^16 are 7 % slower that way (as 2^8 2^8 or with a
// second radix of 2^9).
template <int L>
struct ULarge {
    static constexpr bool wide = L >= kUWideLog2;
    static constexpr int B1 = ubatch_split(L), B2 = L - B1;
    static constexpr int per = kUThreadsLog2 + (wide ? 5 : 4);  // values of a tile
    static constexpr int T1 = per - B1, T2 = per - B2;
    static constexpr int floats() {
        if constexpr (wide) {
            const int f = WideTile<B1, T1, kWideFirst>::lds_floats, l = WideTile<B2, T2, kWideLast>::lds_floats;
            return f > l ? f : l;
        } else {
            const int f = PassTile<B1, T1>::lds_size, l = PassTile<B2, T2>::lds_size;
            return 2 * (f > l ? f : l);
        }
    }
    static constexpr int lds = (floats() + 1) / 2;
};

template <int... Ls>
constexpr int small_lds_max(std::integer_sequence<int, Ls...>) {
    int m = 0;
    for (int v : {USmall<Ls + 1>::lds...}) m = v > m ? v : m;
    return m;
}
template <int... Ls>
constexpr int large_lds_max(std::integer_sequence<int, Ls...>) {
    int m = 0;
    for (int v : {ULarge<Ls + kUMaxSmallLog2 + 1>::lds...}) m = v > m ? v : m;
    return m;
}
// LDS of the kernel: the largest need over every size class it dispatches
constexpr int kULdsSmall = small_lds_max(std::make_integer_sequence<int, kUMaxSmallLog2>{});
constexpr int kULdsLarge = large_lds_max(std::make_integer_sequence<int, kUMaxLog2 - kUMaxSmallLog2>{});
constexpr int kULds = kULdsSmall > kULdsLarge ? kULdsSmall : kULdsLarge;
static_assert(kULds * 8 <= 79 * 1024, "two workgroups per CU");

template <int L, int DIR>
__device__ __forceinline__ void small_item(const UArgs &a, const UTables &tw, const UItem &it, float2 *lds) {
    using G = BlockGeom<L>;
    constexpr int N = G::N, E = G::E, TPT = G::TPT, TPW = USmall<L>::TPW;
    const int t = opaque_lane(threadIdx.x), w = t / TPT, tl = t % TPT;
    const bool active = w < it.count;
    const long off = a.offs[it.first + (active ? w : 0)];
    float2 v[E];
    const float2 *src = a.in + off + tl;
#pragma unroll
    for (int i = 0; i < E; ++i) v[i] = ld_stream(src + TPT * i);
    block_fft<L, DIR>(v, lds + w * USmall<L>::slice, tl, tw.pow[L], true);
    if (active) {
        float2 *dst = a.out + off + tl;
#pragma unroll
        for (int i = 0; i < E; ++i) st_stream(dst + TPT * i, cscale(v[i], a.scale));
    }
    (void)N;
    (void)TPW;
}

template <int L, int DIR>
__device__ __forceinline__ void large_item(const UArgs &a, const UTables &tw, const UItem &it, float2 *lds) {
    constexpr int B1 = ULarge<L>::B1, B2 = ULarge<L>::B2, T1 = ULarge<L>::T1, T2 = ULarge<L>::T2;
    constexpr bool WIDE = ULarge<L>::wide;
    const long off = a.offs[it.first];
    PassArgs p1{};
    p1.batch = 1;
    p1.A = 1;
    p1.log2n = L;
    p1.log2S = L - B1;
    p1.scale = 1.0f;
    if constexpr (WIDE) {
        p1.lobits = B1;
        p1.tw_lo = tw.first[B1];
        p1.tw_hi = tw.one;
    } else {
        p1.tw_local = tw.pow[B1];
    }
#pragma unroll 1
    for (long tile = 0; tile < (1L << (L - B1 - T1)); ++tile) {
        if constexpr (WIDE)
            wide_tile<B1, DIR, T1, kWideFirst>(a.in + off, a.scratch + off, p1, tile, reinterpret_cast<float *>(lds), true);
        else pass_tile<B1, DIR, T1>(a.in + off, a.scratch + off, p1, tile, lds, true);
    }
    __syncthreads();  // this workgroup's scratch writes are visible to all its threads
    PassArgs p2{};
    p2.batch = 1;
    p2.A = 1L << B1;
    p2.log2n = L;
    p2.log2S = 0;
    p2.lobits = tw.lobits[L];
    p2.scale = a.scale;
    if constexpr (!WIDE) p2.tw_local = tw.pow[B2];
    p2.tw_lo = tw.lo[L];
    p2.tw_hi = tw.hi[L];
#pragma unroll 1
    for (long tile = 0; tile < (1L << (L - B2 - T2)); ++tile) {
        if constexpr (WIDE)
            wide_tile<B2, DIR, T2, kWideLast>(a.scratch + off, a.out + off, p2, tile, reinterpret_cast<float *>(lds), true);
        else pass_tile<B2, DIR, T2>(a.scratch + off, a.out + off, p2, tile, lds, true);
    }
}

// waves per SIMD the register budget is held to (0: the compiler's choice)
#ifndef ESTL_UBATCH_WAVES
#define ESTL_UBATCH_WAVES 4
#endif
template <int DIR>
__global__ void __launch_bounds__(kUThreads)
#if ESTL_UBATCH_WAVES
__attribute__((amdgpu_waves_per_eu(ESTL_UBATCH_WAVES, ESTL_UBATCH_WAVES)))
#endif
k_ubatch(UArgs a) {
    __shared__ float2 lds[kULds];
    __shared__ int s_item;
    // The tables' addresses are read where an item needs them, from the kernel's argument
    // block: read ahead of the loop, those of all size classes filled the scalar registers, and
    // each workgroup started with a dozen waits for them in a row (batches of a few hundred
    // transforms 7.2 -> 7.9 us a call).  The other arguments stay in registers (all of them read
    // for each item: 100000 transforms of 2^4 .. 2^6 82.2 us, so 80.7).
    using KernArgs = const __attribute__((address_space(4))) UArgs;
    auto *ap = (KernArgs *)__builtin_amdgcn_kernarg_segment_ptr();
#pragma unroll 1
    for (;;) {
        asm volatile("" : "+s"(ap));
        const UTables &tw = ((const UArgs *)ap)->tw;
        if (threadIdx.x == 0) s_item = atomicAdd(&a.counters[0], 1);
        __syncthreads();
        // the ticket and the descriptor are the same for the whole workgroup: say so, so
        // the size switch below is a scalar branch rather than predicated code whose
        // cases would all be live at once
        const int idx = __builtin_amdgcn_readfirstlane(s_item);
        __syncthreads();
        if (idx >= a.n_items) break;  // every workgroup reaches this exit
        const UItem raw = a.items[idx];
        UItem it;
        it.log2n = __builtin_amdgcn_readfirstlane(raw.log2n);
        it.count = __builtin_amdgcn_readfirstlane(raw.count);
        it.first = __builtin_amdgcn_readfirstlane(raw.first);
        it.pad = 0;
        switch (it.log2n) {
#define SMALL(L) \
    case L: small_item<L, DIR>(a, tw, it, lds); break;
#define LARGE(L) \
    case L: large_item<L, DIR>(a, tw, it, lds); break;
            SMALL(1) SMALL(2) SMALL(3) SMALL(4) SMALL(5) SMALL(6) SMALL(7) SMALL(8) SMALL(9) SMALL(10) SMALL(11)
            SMALL(12) SMALL(13) LARGE(14) LARGE(15) LARGE(16) LARGE(17) LARGE(18) LARGE(19) LARGE(20)
#undef SMALL
#undef LARGE
            default: break;
        }
    }
    if (threadIdx.x == 0) {
        __threadfence();
        if (atomicAdd(&a.counters[1], 1) == (int)gridDim.x - 1) {
            atomicExch(&a.counters[0], 0);
            atomicExch(&a.counters[1], 0);
        }
    }
}

long ubatch_resident_blocks() {
    int per_cu = 0, cus = 0, dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) dev = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_ubatch<-1>, kUThreads, 0) != hipSuccess || per_cu < 1)
        per_cu = 1;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) cus = 256;
    return (long)per_cu * cus;
}

int ubatch_small_rows_per_item(int log2n) {
    switch (log2n) {
#define TPWC(L) \
    case L: return USmall<L>::TPW;
        TPWC(1) TPWC(2) TPWC(3) TPWC(4) TPWC(5) TPWC(6) TPWC(7) TPWC(8) TPWC(9) TPWC(10) TPWC(11) TPWC(12)
        TPWC(13)
#undef TPWC
        default: return 1;
    }
}

hipError_t launch_ubatch(int dir, const UArgs &a, long blocks, hipStream_t st) {
    if (dir < 0)
        hipLaunchKernelGGL(k_ubatch<-1>, dim3((unsigned)blocks), dim3(kUThreads), 0, st, a);
    else
        hipLaunchKernelGGL(k_ubatch<+1>, dim3((unsigned)blocks), dim3(kUThreads), 0, st, a);
    return hipGetLastError();
}

}  // namespace estl
