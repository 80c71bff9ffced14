// ubatch.h -- descriptors of the uneven-size batch (work-queue kernel k_ubatch).
#pragma once

#include <hip/hip_runtime.h>

namespace estl {

// work-queue workgroup size 2^kUThreadsLog2 (see workqueue.hip)
constexpr int kUThreadsLog2 = 9;
constexpr int kUMaxLog2 = 20;  // largest transform of an uneven batch
// up to here a work item is a group of rows (16 values per thread)
constexpr int kUMaxSmallLog2 = kUThreadsLog2 + 4;

// First radix of the large sizes' two passes.  Measured on MI355X (1 GiB of one size per
// launch): the even split beats skewed ones -- a radix-16 first pass with 256-column tiles
// and a 2^10..2^12 second pass was 1.7x (L = 14) to 6x (L = 16) slower, a 2^9 second pass
// 2-20 % slower.
#if defined(__HIPCC__)
__host__ __device__
#endif
constexpr int ubatch_split(int L) { return L / 2; }
constexpr int kUWideLog2 = 17;  // from here both passes keep 32 values per thread (workqueue.hip)

// One work item: `count` transforms of size 2^log2n, the `first`-th.. of the
// size-sorted offset list (count = 1 for large sizes).
struct UItem {
    int log2n;
    int count;
    int first;
    int pad;
};

// Device tables of every size class.
struct UTables {
    // power tables of BlockGeom<log2>, log2 0..kUMaxSmallLog2: the
    // small transforms and the radices of the large ones' passes
    const float2 *pow[kUMaxSmallLog2 + 1];
    // W_B^m, m < B = 2^log2, of the first passes in k_pass_wide's form, and the one entry
    // (1) of their second level
    const float2 *first[kUMaxLog2 / 2 + 1];
    const float2 *one;
    const float2 *lo[kUMaxLog2 + 1];          // pre-twiddle tables of the second pass
    const float2 *hi[kUMaxLog2 + 1];
    int lobits[kUMaxLog2 + 1];
};

struct UArgs {
    const UItem *items;
    int n_items;
    const long *offs;     // element offset of each transform, size-sorted
    const float2 *in;
    float2 *out;
    float2 *scratch;      // pass-1 output of large transforms (same offsets)
    int *counters;        // [0] ticket, [1] workgroups done (both zero between launches)
    float scale;
    UTables tw;
};

hipError_t launch_ubatch(int dir, const UArgs &a, long blocks, hipStream_t st);
long ubatch_resident_blocks();
int ubatch_small_rows_per_item(int log2n);

}  // namespace estl
