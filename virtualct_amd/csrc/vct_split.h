// vct_split.h -- how launches are split over workgroups and passes: host rules
// in plain integers, without HIP.
#pragma once

#include <algorithm>

namespace vct {

// ------------------------------------------------ segment tracer (vct_trace.hip)

// log2 of the orbits of a workgroup: 6, or 5 or 4 where n, the workgroups of 64
// orbits (16 channels of 4 base views), are too few to share the chip's L1s; the
// more voxels a march passes, the more they are worth against the closer lanes
// of 64.  The densities' type and count do not enter (calls of a plan share the
// redo bits, whose layout this is).  us with 64, 32 and 16 orbits, u16, M = 6, 609
// channels (n): 1024^2 x 40 views (117) 271, 168, 148; x 160 (390) 567, 469, 462; x
// 240 (585) 763, 583, 686; x 480 (1170) 881, 913, 1344; 512^2 x 40 102, 63, 54; x 160
// 154, 116, 112; x 200 (507) 191, 127, 133; x 480 218, 215, 276; 256^2 x 80 (195) 43, 39,
// 41; x 200 58, 59, 69; 128^2 x 40 28, 23, 24; x 160 36, 38, 49; 64^2 x 40 21, 19, 21; x 80
// 21, 23, 29.
inline int seg_shift(int N, int base_views, int channel_tiles)
{
    const double n = (base_views + 3) / 4 * (double)channel_tiles;
    if (n <= std::min(0.6 * N, 350.0)) return 4;
    return n <= std::min(std::max(1.8 * N, 128.0), 1000.0) ? 5 : 6;
}

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

// Lanes of a workgroup of sp.views views: 512, or 256 where its rays would leave
// most of them without one, three such workgroups of M materials fit into a
// CU's LDS and there are enough of them to fill the chip.  tile_channels:
// channels of a tile's width at the isocentre, of which it covers 1.27 times as
// many on average (|cos| + |sin|); with more materials the LDS adds count for
// more and idle lanes for less.  M = 1 and 6, 512 and 256 lanes: 128^2 x 80
// views on 51.2 cm (178 rays) 172 and 190 us, 133 and 165; 512^2 x 40 views of 300
// channels 192 and 206, 140 and 170; 256^2 x 100 views (340 rays) 154 and 172, 144
// and 184; 101^2 x 80 (220 rays) 108 and 130, 91 and 138; M = 8 at 128^2 203 and 214; 8^2
// x 4 views of 22 channels, M = 6, 17 and 19.
inline int adjoint_lanes(int M, int ntiles, AdjointSplit sp, int channels, double tile_channels)
{
    const bool few = sp.views * std::min((double)channels, 1.27 * tile_channels) <= 256.0 - 8.0 * M;
    return M <= 6 && few && (long long)ntiles * sp.chunks > 512 ? 256 : 512;
}

// ---------------------------------------- batched spectral sums (vct_batch.hip)

// Workgroups that share the S spectra of one phantom's rays: one where the
// blocks of rays fill two workgroups per CU, else as many as do (a phantom of 8
// views x 609 channels and 64 spectra of 1024 bins 3557 us with one, 118 with
// 64).
inline int spectral_parts(int ray_blocks, int phantoms, int S)
{
    const long long blocks = std::max(1LL, (long long)ray_blocks * phantoms);
    return (int)std::min<long long>(S, (512 + blocks - 1) / blocks);
}

// ------------------------------ several sinograms per call (vct_backproject_ws)

constexpr int kIlWidth = 12;  // widest slice
constexpr int kIlPass = 48;   // most sinograms that one pass interleaves (bounds the workspace)
constexpr long long kIlLanes = 1 << 17;  // lanes of a pass that fill the chip

struct Interleave {
    int width, per;  // sinograms per slice and per pass; width 0: not interleaved
};

// A call of so little work that the interleaving launch costs as much as it
// saves: few views, whose chain of adds is short, on few pixels (us of the call,
// plain and interleaved: 16^2 x 2 views 7 and 14, 32^2 x 40 11 and 14, 128^2 x 40
// with 4 and 13 sinograms 11 and 14, 18 and 15; 64^2 x 80 19 and 20, x 800 170 to 248
// and 144 to 170).
inline bool bp_interleave_small(int N, int views, int S)
{
    return views < 64 && (long long)N * N * views * S < 1 << 25;
}

// How S sinograms of N^2 pixels are interleaved: the fewest slices of at most
// kIlWidth (max_k: VCT_OPT_BP_SINOS_PER_LANE), but enough that the launch has
// kIlLanes lanes, and then the narrowest width that holds an even share, in
// passes of as many whole slices as kIlPass holds.  Images so small that a whole
// pass has fewer lanes run better in one plain launch than in several (50
// sinograms, plain and interleaved: 128^2 x 160 views 79 and 132 us; 200^2 x 360
// 404 and 369).  Measured (us, one launch, 800 views): 16 sinograms at 512^2 as
// 3 x 6, 2 x 8, 12 + 4 and 1 x 16 867, 889, 1103 and 1235; 12 at 300^2 as 2 x 6,
// 12 and 3 x 4 291, 319 and 363; 12 at 200^2 x 360 views as 3 x 4, 2 x 6, 12 and
// 6 x 2 104, 114, 117 and 148.
inline Interleave bp_interleave(int N, int views, bool exact, int max_k, int S)
{
    if (S < 2 || exact || bp_interleave_small(N, views, S)) return {0, S};
    const long long px = (long long)N * N;
    const int cap = max_k >= 2 && max_k < kIlWidth ? max_k / 2 * 2 : kIlWidth;
    const int slices = std::max((S + cap - 1) / cap, (int)std::min<long long>((S + 1) / 2, (kIlLanes + px - 1) / px));
    const int K = ((S + slices - 1) / slices + 1) / 2 * 2, per = kIlPass / K * K;
    if (S > per && kIlPass / K * px < kIlLanes) return {0, S};
    return {K, per};
}

// Slots that n sinograms of one pass take in slices of K.
inline int bp_interleave_slots(int n, int K) { return (n + K - 1) / K * K; }

// Slots that serve up to S sinograms at any width that such a call can take,
// whatever the options: it grows with S, so a workspace sized for the largest
// call serves the others.
inline int bp_interleave_bound(int N, int views, int S)
{
    if (S < 2 || bp_interleave_small(N, views, S)) return 0;
    int slots = 0;
    for (int K = 2; K <= std::min(kIlWidth, (S + 1) / 2 * 2); K += 2)
        slots = std::max(slots, bp_interleave_slots(std::min(S, kIlPass / K * K), K));
    return slots;
}

}  // namespace vct
