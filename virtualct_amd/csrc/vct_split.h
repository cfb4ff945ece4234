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

}  // namespace vct
