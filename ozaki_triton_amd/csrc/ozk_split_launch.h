#pragma once
// ozk_split_launch.h -- what the split planner (ozk_split.hip) and the units
// that hold the split kernels (one per slice dtype, ozk_split_{i8,f16,bf16,
// f32}.hip) share: the geometry of the cooperative kernels and the launches.
#include "ozk_internal.h"

namespace ozk {

constexpr int kCoopNT = 256;
constexpr int kCoopMaxP = 32;
constexpr int64_t kCoopMinColumnBytes = 64 * 1024;
// rows kernel shared by workgroups: 256 lanes, 64 (fp32) or 32 (fp64) values
// per lane, for rows longer than 16384 elements, at most 64 chunks by its own
// layout (one polling lane each) and 56 by the residency limit on MI355X
constexpr int kRowsCoopVariant = 100;
constexpr int64_t kRowsCoopMinK = 16384;
constexpr int kRowsCoopMaxP = 64;
constexpr uint64_t kCoopTickLimit = 200000000ull;   // 2 s of the 100 MHz counter
constexpr uint64_t kCoopTag = 1ull << 32;               // high word of a published maximum

constexpr int kFusedClasses = 6;   // classes of K of split_fused_kernel, up to 8192

// rows per lane of split_coop_kernel (64 values per lane: 32 rows of fp64,
// 16 of fp32), the members (K chunks of 32 * rpl rows) of a column group, and
// the exchange words of an operand (groups * L * members * columns; none for
// P = 1)
inline int coop_rpl(int xsz) { return 64 / (16 / xsz); }
inline int64_t coop_members(int64_t K, int xsz, int seg) {
    const int64_t ch = (int64_t)kCoopNT / seg * coop_rpl(xsz);
    return K <= 0 ? 1 : (K + ch - 1) / ch;
}
inline int64_t coop_slots(const SplitParams &p, int xsz, int seg) {
    const int64_t P = coop_members(p.K, xsz, seg);
    if (P <= 1) return 0;
    const int64_t sw = seg * (16 / xsz);
    const int64_t groups = p.batch * ((p.rows + sw - 1) / sw);
    return groups * p.L * P * sw;
}
inline int64_t rows_coop_chunk(int xsz) { return xsz == 8 ? 4 * 8 * 256 : 4 * 16 * 256; }
inline int64_t rows_coop_members(int64_t K, int xsz) {
    const int64_t ch = rows_coop_chunk(xsz);
    return K <= 0 ? 1 : (K + ch - 1) / ch;
}
inline int64_t rows_coop_slots(const SplitParams &p, int xsz) {
    const int64_t P = rows_coop_members(p.K, xsz);
    return P > 1 ? p.batch * p.rows * p.L * P : 0;
}
// split_pair_kernel's row configurations: classes 4 and 5 (4 waves per row,
// K <= 4096 / 8192)
inline int pair_nc(const SplitPlan &a) {
    return a.path == kSplitRows ? (a.variant == 4 ? 4 : a.variant == 5 ? 8 : 0) : 0;
}

// The tag a wait looks for and its time limit: the test hook makes every wait
// look for a tag that is never written and give up at its first check, so
// the timeout path runs with no wait longer than one poll.
struct WaitRule {
    uint32_t tag;
    uint64_t ticks;
};
WaitRule wait_rule();
// Clears n exchange words and the status word after them.
hipError_t clear_slots(uint64_t *slot, int64_t n, hipStream_t st);
// Follows a cooperative launch whose status word is `status` (see
// poison_scales_kernel).
hipError_t launch_poison(const SplitParams &p, const uint64_t *status, hipStream_t st);

template <typename ST> struct SplitLaunch {
    // p0 and (unless null) p1 by split_fused_kernel, K of class cls, columns
    // by the groups of this width (0: no columns, 1: narrow, 2: wide)
    static hipError_t fused(const SplitParams *p0, const SplitParams *p1, int cls, int width,
                            int x_dtype, hipStream_t st);
    // one fp64 / fp32 operand by any other kernel
    static hipError_t one(const SplitParams &p, const SplitPlan &plan, int x_dtype, hipStream_t st);
    // A's rows and B's columns by split_pair_kernel (fp64)
    static hipError_t pair(const SplitParams &pa, const SplitPlan &plan_a, const SplitParams &pb,
                           hipStream_t st);
    // the fewest workgroups per CU over the kernels that wait
    static void coop_occupancy(int &occ, bool &ok);
};

}  // namespace ozk
