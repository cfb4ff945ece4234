// vct_split.h -- how launches are split over workgroups and passes: host rules
// in plain integers, without HIP.
#pragma once

#include <algorithm>

namespace vct {

// ------------------------------------------------- tile adjoint (vct_trace.hip)

constexpr int kAdjMaxViews = 256;  // views per workgroup (its tables in LDS)
// Rays per workgroup: what 2^19 rays add to a voxel at the full fixed-point
// scale stays within the sums' 51 bits (a ray adds at most sqrt(2) 2^30: its
// first segment and its others there).  8192 channels take at most 64 views.
constexpr int kAdjMaxRays = 1 << 19;

struct AdjointSplit {
    int views, chunks;  // per chunk (the last may hold fewer); chunks
};

// Chunks of the views of one tile: at most 2048 workgroups, four full rounds
// of two per CU (380^2 x 722 views 1.15 ms with the 2160 of 15 chunks, 1.13 with
// the 2016 of 14; 4096 take 1.08, but a voxel's float adds and their rounding
// double), or more where a chunk would exceed its views or rays; the chunks as
// even as they go.  asked: VCT_OPT_ADJOINT_VIEWS.
inline AdjointSplit adjoint_split(int ntiles, int views, int channels, int asked)
{
    const int most = std::max(1, std::min(kAdjMaxViews, kAdjMaxRays / channels));
    auto chunks_of = [&](int per) { return (views + per - 1) / per; };
    int per = std::min(asked, most);
    if (asked <= 0) {
        const int n = std::max(std::min(views, 2048 / ntiles), chunks_of(most));
        per = chunks_of(n);
    }
    return {per, chunks_of(per)};
}

// ------------------------------ several sinograms per call (vct_backproject_ws)

constexpr int kIlWidth = 12;  // widest slice
constexpr int kIlPass = 48;   // most sinograms that one pass interleaves (bounds the workspace)

// Width of the interleaved slices that S sinograms of N^2 pixels take, 0 for
// none (a single sinogram, the exact option).  The fewest slices of at most
// kIlWidth (max_k: VCT_OPT_BP_SINOS_PER_LANE), but enough that the launch has
// kIlLanes lanes, and then the narrowest width that holds an even share.
// Measured (us, one launch, 800 views): 16 sinograms at 512^2 as 3 x 6, 2 x 8,
// 12 + 4 and 1 x 16 867, 889, 1103 and 1235; 12 at 300^2 as 2 x 6, 12 and 3 x 4
// 291, 319 and 363; 12 at 200^2 x 360 views as 3 x 4, 2 x 6, 12 and 6 x 2 104,
// 114, 117 and 148.
inline int bp_interleave_width(int N, bool exact, int max_k, int S)
{
    constexpr long long kIlLanes = 1 << 17;
    if (S < 2 || exact) return 0;
    const long long px = (long long)N * N;
    const int cap = max_k >= 2 && max_k < kIlWidth ? max_k / 2 * 2 : kIlWidth;
    const int slices = std::max((S + cap - 1) / cap, (int)std::min<long long>((S + 1) / 2, (kIlLanes + px - 1) / px));
    return ((S + slices - 1) / slices + 1) / 2 * 2;
}

// Sinograms per pass of slices of K, and the slots that S of them take.
inline int bp_interleave_pass(int K) { return kIlPass / K * K; }
inline int bp_interleave_slots(int S, int K) { return std::min((S + K - 1) / K * K, bp_interleave_pass(K)); }

// Slots that serve up to S sinograms at any width that such a call can take,
// whatever the options: it grows with S, so a workspace sized for the largest
// call serves the others.
inline int bp_interleave_bound(int S)
{
    int slots = 0;
    for (int K = 2; K <= std::min(kIlWidth, (S + 1) / 2 * 2); K += 2)
        if (S >= 2) slots = std::max(slots, bp_interleave_slots(S, K));
    return slots;
}

}  // namespace vct
