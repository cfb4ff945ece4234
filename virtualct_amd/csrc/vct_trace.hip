// vct_trace.hip -- MBFPA ray tracer, polyenergetic detector sum, detector
// noise and phantom packing for CDNA4 (gfx950).
//
// Design (64 adjacent channels of one view per wave):
//   k_trace_fwd  marches each fan ray once through the image in FP64 and
//                accumulates the per-element path integrals
//                L_m = sum_seg rho_m(voxel) * length in FP64 registers; the
//                segment decomposition (entry/exit clip, integer-cm start
//                plane, midpoint voxel, minor-axis crossing split) follows
//                M/reprojection_TOMO.cpp:53-283 operation for operation, so
//                it is bit-identical to the reference when compiled with
//                -ffp-contract=off.  The reference re-traces every ray once
//                per energy bin (M/main.cpp:492); here the trace is done once
//                and the spectrum is applied afterwards.
//   k_spectral   I_s = sum_E pdf_s(E) exp(-sum_m mu_s,m(E) L_m) with the
//                spectrum tables of spectrum s in LDS (k_spectral_grad: with
//                its derivatives in the L_m), plus the per-spectrum
//                max/min used by the normalisation and the noise clamp.
//   k_detector   max-normalisation + Gaussian noise (Philox4x32-10 +
//                Box-Muller) + the reference's clamps.
//   k_trace_seg  the same path integrals with one segment per loop iteration,
//                one march for the rays of views v, v + V/4, v + V/2,
//                v + 3V/4 (or v, v + V/2, or one ray); k_trace_redo marches
//                what it leaves undecided.
//   k_trace_fwd_rot  the quarter- (or half-) turn orbit form of k_trace_fwd,
//                split over eight lanes by step windows, for the grids that
//                k_trace_seg does not take (seg_grid).
//   k_trace_adj_tile  the adjoint by image tiles: windowed marches of the
//                rays that cross a tile, w_m * length summed in LDS in
//                fixed point, one float atomic per voxel at the end.
#include "vct_internal.h"
#include "vct_march.h"
#include "vct_spectral.h"
#include "vct_split.h"

#include <algorithm>
#include <climits>
#include <cstring>
#include <cmath>

namespace vct {

// ------------------------------------------------------------------ sinks

// Forward sinks accumulate L_m += rho_m(voxel) * length in FP64 (the u16
// sink per 32-bit word of two materials: the word as one integer and its high
// half, which resolves the low half to ~1e-11 relative).  add2
// takes the two candidate segments of one march step and issues both gathers
// before using either, each only on the lanes where it is a segment in the
// image: the gathers' texture path, not the FP64 arithmetic, is what the
// march keeps busiest (78% / 84% TA / TD busy with unmasked gathers).
template <int M>
struct SinkU16 {
    static constexpr bool kAdd2 = true;
    const char* __restrict__ vox;
    // word k of a voxel holds materials 2k (low half) and 2k+1 (high half);
    // accw[k] sums the whole word as one integer lo + 65536 hi and acch[k]
    // the high half, so material 2k is accw[k] - 65536 acch[k] at the end
    double accw[(M + 1) / 2], acch[M / 2];
    double acc[M];
    __device__ __forceinline__ void init(const void* p)
    {
        vox = reinterpret_cast<const char*>(p);
#pragma unroll
        for (int k = 0; k < (M + 1) / 2; k++) accw[k] = 0.0;
#pragma unroll
        for (int k = 0; k < M / 2; k++) acch[k] = 0.0;
    }
    __device__ __forceinline__ uint4 load(int v) const
    {
        // 32-bit byte offset (N*N*16 bytes < 4 GB)
        return *reinterpret_cast<const uint4*>(vox + (uint32_t)v * 16u);
    }
    __device__ __forceinline__ void accumulate(const uint4& q, double rr)
    {
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int k = 0; k < (M + 1) / 2; k++) {
            // odd M: the last word's high half is not a material of this call
            const uint32_t wk = (2 * k + 1 < M) ? w[k] : (w[k] & 0xffffu);
            accw[k] = __builtin_fma((double)wk, rr, accw[k]);
        }
#pragma unroll
        for (int k = 0; k < M / 2; k++) acch[k] = __builtin_fma((double)(w[k] >> 16), rr, acch[k]);
    }
    __device__ __forceinline__ void add(int v, double rr) { accumulate(load(v), rr); }
    // the two candidate segments of a committed step, each only on lanes
    // where it is a segment (ok1, ok2): the others issue no gather
    __device__ __forceinline__ void add2(bool ok1, int v1, double r1, bool ok2, int v2, double r2)
    {
        uint4 q1, q2;
        if (ok1) q1 = load(v1);
        if (ok2) q2 = load(v2);
        if (ok1) accumulate(q1, r1);
        if (ok2) accumulate(q2, r2);
    }
    __device__ __forceinline__ void finish()
    {
#pragma unroll
        for (int m = 0; m < M; m++)
            acc[m] = (m & 1) ? acch[m >> 1] : accw[m >> 1] - (m / 2 < M / 2 ? 65536.0 * acch[m >> 1] : 0.0);
    }
};

template <int M>
struct SinkF32 {
    static constexpr bool kAdd2 = true;
    const float4* __restrict__ vox;
    double acc[M];
    struct Vox {
        float4 lo, hi;
    };
    __device__ __forceinline__ void init(const void* p)
    {
        vox = reinterpret_cast<const float4*>(p);
#pragma unroll
        for (int m = 0; m < M; m++) acc[m] = 0.0;
    }
    __device__ __forceinline__ Vox load(int v) const
    {
        Vox q;
        q.lo = vox[2 * v];
        q.hi = M > 4 ? vox[2 * v + 1] : make_float4(0.f, 0.f, 0.f, 0.f);
        return q;
    }
    __device__ __forceinline__ void accumulate(const Vox& q, double rr)
    {
        const float r[8] = {q.lo.x, q.lo.y, q.lo.z, q.lo.w, q.hi.x, q.hi.y, q.hi.z, q.hi.w};
#pragma unroll
        for (int m = 0; m < M; m++) {
            // a negative density contributes nothing (reference ph = 0, :155):
            // fmaxf gives 0 for negatives and NaN, and -0 adds the same zero
            const double rho = (double)fmaxf(r[m], 0.f);
            acc[m] = __builtin_fma(rho, rr, acc[m]);
        }
    }
    __device__ __forceinline__ void add(int v, double rr) { accumulate(load(v), rr); }
    __device__ __forceinline__ void add2(bool ok1, int v1, double r1, bool ok2, int v2, double r2)
    {
        Vox q1, q2;
        if (ok1) q1 = load(v1);
        if (ok2) q2 = load(v2);
        if (ok1) accumulate(q1, r1);
        if (ok2) accumulate(q2, r2);
    }
};

// Orbit sink: the segments of the ray of view v, taken also as the segments
// of the rays of views v + kV/R (k = 1..R-1, turned by k/R of a turn), each
// at the turned voxel.  Ray k accumulates rho(voxel) * length as the
// single-ray sinks do.  The march hands over, for every candidate segment,
// the floors (fa, fb) of its major and minor index values; the x and y floors
// (fx, fy) of ray k are those of ray 0 turned: a quarter turn maps (fx, fy)
// to (N-1-fy, fx).  Each ray then takes the reference's own rule: index
// trunc(q) = f + (f < 0), in the image when both lie in 0..N-1, i.e.
// f in -1..N-1 (a midpoint less than a pixel beyond the low edge counts into
// the edge voxel, one beyond the high edge does not).
// unsafe: a decision of the march that a turned ray might take otherwise did
// not clear the margin (the caller then traces rays 1..R-1 by themselves;
// ray 0 is right in any case).
__host__ __device__ __forceinline__ void swap_d(double& x, double& y)
{
    const double t = x;
    x = y;
    y = t;
}

template <int M, int DT, int R>
struct SinkRot {
    static_assert(R == 1 || R == 2 || R == 4, "orbits of 1, 2 or 4 rays");
    static constexpr bool kAdd2 = true;
    static constexpr bool kRot = true;
    static constexpr int NW = (M + 1) / 2;  // u16: 32-bit words of two materials
    // Bytes per voxel of the work copies: u16 with M <= 6 keeps the three
    // words that hold the materials, other u16 all four, f32 eight floats.
    static constexpr int VB = DT == VCT_DENS_U16 ? (M <= 6 ? 12 : 16) : 32;
    // Gathers read the copy of the densities whose rows run along the
    // minor axis of the slot's ray ([y][x] voxels when y is its major axis,
    // the transposed [x][y] copy when x is), so the lanes of a wave, which
    // hold neighbouring rays at the same major step, meet neighbouring voxels
    // of one row.  Slot k holds ray k (the base ray turned k quarter turns),
    // except that rays 1 and 3 trade slots when y is the base ray's major
    // axis; finish() puts them back.  Both copies are padded by two voxels
    // on every side (NP = N + 4 per row): row and column -1 repeat row and
    // column 0 (the reference truncates index -1 to voxel 0), rows and
    // columns -2, N and N + 1 are zero, so the committed steps' gathers need
    // no in-image test (a voxel outside the image reads zeros).
    const char* __restrict__ voxE;  // slots 0 and 2 (and 1 when R == 2)
    const char* __restrict__ voxO;  // slots 1 and 3 when R == 4
    bool xmajor;
    int N;
    int NP;   // row pitch of the copies in voxels, N + 4
    int ORG;  // index of voxel (0, 0), 2 NP + 2
    bool unsafe;
    double accw[R][NW], acch[R][M / 2];  // u16: word sums and high halves
    double acc[R][M];                    // f32: sums; u16: after finish()
    // pt: the two padded copies, [y][x] then [x][y]
    __host__ __device__ void init(const void* pt, bool xm, int n)
    {
        NP = n + 4;
        ORG = 2 * NP + 2;
        const char* P = reinterpret_cast<const char*>(pt);
        const char* T = P + (size_t)NP * NP * VB;
        voxE = xm ? T : P;
        voxO = xm ? P : T;
        xmajor = xm;
        N = n;
        unsafe = false;
        #pragma unroll
        for (int k = 0; k < R; k++) {
            #pragma unroll
            for (int w = 0; w < NW; w++) accw[k][w] = 0.0;
            #pragma unroll
            for (int w = 0; w < M / 2; w++) acch[k][w] = 0.0;
            #pragma unroll
            for (int m = 0; m < M; m++) acc[k][m] = 0.0;
        }
    }
    // slot k of a segment whose floors are (fa, fb) on the base ray's (major,
    // minor) axes: the (major, minor) coordinates of the turned ray, indexed
    // minor + NP * major in its copy, with the reference's truncation of
    // index -1 to voxel 0 (0 with rr = 0 when outside the image)
    __host__ __device__ __forceinline__ void voxels(int fa, int fb, double rr, int (&v)[R], double (&r)[R]) const
    {
        const int n1 = N - 1;
        const int ta = n1 - fa, tb = n1 - fb;
        #pragma unroll
        for (int k = 0; k < R; k++) {
            int ma, mi;
            if (R == 1 || k == 0) { ma = fa; mi = fb; }
            else if (R == 2 || k == 2) { ma = ta; mi = tb; }
            else if (k == 1) { ma = fa; mi = tb; }
            else { ma = ta; mi = fb; }
            const bool in = (unsigned)(ma + 1) <= (unsigned)N && (unsigned)(mi + 1) <= (unsigned)N;
            v[k] = in ? ORG + max(mi, 0) + mul24(max(ma, 0), NP) : 0;
            r[k] = in ? rr : 0.0;
        }
    }
    struct Vox {
        uint4 lo, hi;  // u16: lo = the 8 materials; f32: lo = materials 0-3, hi = 4-7
    };
    // the voxel at byte offset o of the copy of slot k
    __host__ __device__ __forceinline__ Vox load_at(int k, uint32_t o) const
    {
        const char* vox = (R == 4 && (k & 1)) ? voxO : voxE;
        Vox q;
        if constexpr (VB == 12) {
            const uint3 t = *reinterpret_cast<const uint3*>(vox + o);
            q.lo = make_uint4(t.x, t.y, t.z, 0u);
            q.hi = make_uint4(0u, 0u, 0u, 0u);
        } else if constexpr (VB == 16) {
            q.lo = *reinterpret_cast<const uint4*>(vox + o);
            q.hi = make_uint4(0u, 0u, 0u, 0u);
        } else {
            const uint4* f = reinterpret_cast<const uint4*>(vox + o);
            q.lo = f[0];
            q.hi = M > 4 ? f[1] : make_uint4(0u, 0u, 0u, 0u);
        }
        return q;
    }
    __host__ __device__ __forceinline__ Vox load(int k, int v) const { return load_at(k, (uint32_t)v * (uint32_t)VB); }
    __host__ __device__ __forceinline__ void accumulate(int k, const Vox& q, double rr)
    {
        if constexpr (DT == VCT_DENS_U16) {
            const uint32_t w[4] = {q.lo.x, q.lo.y, q.lo.z, q.lo.w};
            #pragma unroll
            for (int j = 0; j < NW; j++) {
                const uint32_t wj = (2 * j + 1 < M) ? w[j] : (w[j] & 0xffffu);
                accw[k][j] = __builtin_fma((double)wj, rr, accw[k][j]);
            }
            #pragma unroll
            for (int j = 0; j < M / 2; j++) acch[k][j] = __builtin_fma((double)(w[j] >> 16), rr, acch[k][j]);
        } else {
            const uint32_t b[8] = {q.lo.x, q.lo.y, q.lo.z, q.lo.w, q.hi.x, q.hi.y, q.hi.z, q.hi.w};
            #pragma unroll
            for (int m = 0; m < M; m++) {
                float rho;
                memcpy(&rho, &b[m], sizeof(float));
                acc[k][m] = __builtin_fma((double)fmaxf(rho, 0.f), rr, acc[k][m]);  // as SinkF32
            }
        }
    }
    // one candidate segment whose index values clear the margin (floors)
    __host__ __device__ __forceinline__ void add_fl(int fa, int fb, double rr)
    {
        int v[R];
        double r[R];
        voxels(fa, fb, rr, v, r);
        Vox q[R];
        #pragma unroll
        for (int k = 0; k < R; k++) q[k] = load(k, v[k]);
        #pragma unroll
        for (int k = 0; k < R; k++) accumulate(k, q[k], r[k]);
    }
    // one candidate segment of a general march step from the signed quotients
    // (ta, tb) of its index values t + N/2: ray k takes fl(+-t + N/2) on each
    // of its axes (minus where the turn flips the axis) and the reference's
    // trunc and in-image test
    __host__ __device__ __forceinline__ void add_t(double ta, double tb, double rr)
    {
        int v[R];
        double r[R];
        voxels_t(ta, tb, rr, v, r);
        Vox q[R];
        #pragma unroll
        for (int k = 0; k < R; k++) q[k] = load(k, v[k]);
        #pragma unroll
        for (int k = 0; k < R; k++) accumulate(k, q[k], r[k]);
    }
    __host__ __device__ __forceinline__ void voxels_t(double ta, double tb, double rr, int (&v)[R], double (&r)[R]) const
    {
        const double tx = xmajor ? ta : tb, ty = xmajor ? tb : ta;
        const double c = (double)(N / 2);
        #pragma unroll
        for (int k = 0; k < R; k++) {
            double gx, gy;
            if (R == 1 || k == 0) { gx = tx + c; gy = ty + c; }
            else if (R == 2 || k == 2) { gx = -tx + c; gy = -ty + c; }
            else if (k == 1) { gx = -ty + c; gy = tx + c; }
            else { gx = ty + c; gy = -tx + c; }
            const int ix = trunc_i32(gx), iy = trunc_i32(gy);
            const bool in = ix >= 0 && ix <= N - 1 && iy >= 0 && iy <= N - 1;
            // ray k goes to slot k, but rays 1 and 3 trade slots when y is the
            // base ray's major axis; its major axis is x when xmajor differs
            // from its own quarter-turn parity
            const bool odd = R == 4 && (k & 1);
            const int slot = (odd && !xmajor) ? 4 - k : k;
            const bool majx = xmajor != odd;
            v[slot] = in ? ORG + (majx ? iy + NP * ix : ix + NP * iy) : 0;
            r[slot] = in ? rr : 0.0;
        }
    }
    // byte offsets of the four slots of one candidate, its coordinates
    // clamped to [-2, N + 1] (values outside read zeros there too)
    __host__ __device__ __forceinline__ void offsets(int fa, int fb, uint32_t (&o)[R]) const
    {
        const int a = min(max(fa + 2, 0), N + 3), b = min(max(fb + 2, 0), N + 3);
        const int ta = N + 3 - a, tb = N + 3 - b;  // (N - 1 - f) + 2
        const uint32_t ra = (uint32_t)mul24(a, VB * NP), rt = (uint32_t)mul24(ta, VB * NP);
        const uint32_t cb = (uint32_t)mul24(b, VB), ct = (uint32_t)mul24(tb, VB);
        #pragma unroll
        for (int k = 0; k < R; k++) {
            if (R == 1 || k == 0) o[k] = ra + cb;
            else if (R == 2 || k == 2) o[k] = rt + ct;
            else if (k == 1) o[k] = ra + ct;
            else o[k] = rt + cb;
        }
    }
    // the two candidate segments of a committed step; the first only on lanes
    // whose step crosses a minor grid line (cross), so lanes without a
    // crossing issue no gathers for it (the gathers' texture path is what the
    // kernel keeps busiest); a segment of length 0 would add exactly nothing
    __host__ __device__ __forceinline__ void add2_fl(bool cross, int fa1, int fb1, double r1, int fa2, int fb2,
                                                     double r2)
    {
        uint32_t o1[R], o2[R];
        offsets(fa1, fb1, o1);
        offsets(fa2, fb2, o2);
        Vox q1[R], q2[R];
        if (cross) {
            #pragma unroll
            for (int k = 0; k < R; k++) q1[k] = load_at(k, o1[k]);
        }
        #pragma unroll
        for (int k = 0; k < R; k++) q2[k] = load_at(k, o2[k]);
        if (cross) {
            #pragma unroll
            for (int k = 0; k < R; k++) accumulate(k, q1[k], r1);
        }
        #pragma unroll
        for (int k = 0; k < R; k++) accumulate(k, q2[k], r2);
    }
    __host__ __device__ __forceinline__ void finish()
    {
        if (R == 4 && !xmajor) {
            // slots 1 and 3 hold rays 3 and 1
            #pragma unroll
            for (int w = 0; w < NW; w++) swap_d(accw[1 % R][w], accw[3 % R][w]);
            #pragma unroll
            for (int w = 0; w < M / 2; w++) swap_d(acch[1 % R][w], acch[3 % R][w]);
            #pragma unroll
            for (int m = 0; m < M; m++) swap_d(acc[1 % R][m], acc[3 % R][m]);
        }
        if constexpr (DT == VCT_DENS_U16) {
            #pragma unroll
            for (int k = 0; k < R; k++)
                #pragma unroll
                for (int m = 0; m < M; m++)
                    acc[k][m] = (m & 1) ? acch[k][m >> 1]
                                        : accw[k][m >> 1] - (m / 2 < M / 2 ? 65536.0 * acch[k][m >> 1] : 0.0);
        }
    }
};

// Adjoint sink of one image tile: a segment whose voxel lies in the tile adds
// w[m] * length to the tile's accumulator in LDS, [m][row][col] with a row
// pitch of TS + 1 (a wave's lanes are adjacent channels of one view, which
// meet a column of the tile at one step when x is the major axis).  FIXED:
// the accumulator is 51-bit fixed point, each contribution rounded to an
// integer after scaling by a power of two that keeps it below 2^30 in
// magnitude; the sums of up to kAdjMaxRays rays are then exact (and
// independent of the order of the adds), and ds_add_u64 runs about ten times
// faster than ds_add_f32 on gfx950 (0.3 vs 3.4 lane-operations per clock per
// CU, measured).  The float
// form serves workgroups whose weights are not all finite, so NaN and
// infinity reach the gradient as with float sums.
constexpr int kAdjTile = 32;
constexpr int kAdjBlock = 512;  // most lanes of a workgroup (adjoint_lanes)

template <int M, bool FIXED>
struct SinkTile {
    static constexpr bool kAdd2 = false;
    static constexpr bool kAB = true;
    // (a plane's padding moves the next one by eight banks)
    static constexpr int TS = kAdjTile, PITCH = TS + 1, PLANE = (TS * PITCH + 31) / 32 * 32 + 4;
    unsigned long long* acc;  // [M][TS][PITCH], int64 or (FIXED false) float in the same memory
    int x0, y0;
    bool xmajor;
    double w[M];  // (FIXED: times 2^S)
    // FIXED: w r + 1.5 2^52 holds the product rounded to an integer in its low
    // bits, so one fused multiply-add makes the addend; the magic's own bits
    // are multiples of 2^51 and leave the sum's low 51 bits (fixed_sum) alone.
    static constexpr double kMagic = 6755399441055744.0;
    static __device__ __forceinline__ long long fixed_sum(unsigned long long acc) { return (long long)(acc << 13) >> 13; }
    __device__ __forceinline__ void add_at(int off, double r)
    {
#pragma unroll
        for (int m = 0; m < M; m++) {
            if constexpr (FIXED)
                atomicAdd(acc + off + m * PLANE,
                          (unsigned long long)__double_as_longlong(__builtin_fma(w[m], r, kMagic)));
            else
                atomicAdd(reinterpret_cast<float*>(acc) + off + m * PLANE, (float)w[m] * (float)r);
        }
    }
    __device__ __forceinline__ void add_ab(int ia, int ib, double rr)
    {
        const int x = xmajor ? ia : ib, y = xmajor ? ib : ia;
        const uint32_t lx = (uint32_t)(x - x0), ly = (uint32_t)(y - y0);
        if (lx < (uint32_t)TS && ly < (uint32_t)TS) add_at((int)(ly * PITCH + lx), rr);
    }
};

// Steps k0..k1 (k0 >= 1) of ray r into a tile, one segment per loop iteration
// as k_trace_seg forms them, for grids that seg_planes accepts.  The margin
// tests are looked at after the loop; false: one failed, and the window has
// been taken out of the tile again by the same loop with the weights negated
// (the fixed-point sums are exact, so nothing of it remains), for the caller to
// march it step by step.  w is left as it was or negated.
template <int M>
__device__ __forceinline__ bool seg_window(const TraceArgs& a, const RayConst& r, SinkTile<M, true>& sink, bool& ovf,
                                           int k0, int k1)
{
    using Sink = SinkTile<M, true>;
    const double ai = r.ai, af = r.af, Lb = r.Lb, D = a.D;
    const double kAB = r.dB / r.dA, kBA = r.dA / r.dB;
    const double sA = r.xmajor ? 1.0 : -1.0, nxm = (double)a.nxm;
    const double pha = af > ai ? 1.0 : -1.0;
    // integer-cm start plane, M/reprojection_TOMO.cpp:115-119
    const int ain = ((ai < 0 && af < ai) || (ai > 0 && af > ai)) ? trunc_i32(trunc_i32(ai) + pha) : trunc_i32(ai);
    const double uain = pha * (double)ain;
    // last plane inside the square (exactly u_0 + fl(k D) <= Lb)
    int ka = (int)fmin(fmax((Lb - uain) / D, -1.0), 1.0e8);
    if (uain + (double)(ka + 1) * D <= Lb) ka++;
    if (ka >= 0 && uain + (double)ka * D > Lb) ka--;
    const int kend = min(k1, ka + 1), kstop = min(kend, a.max_steps - 1);
    // plane k0 - 1: the minor cell and the first line ahead
    const double u_start = uain + (double)(k0 - 1) * D;
    const double b0 = __builtin_fma(pha * u_start - r.sa, kAB, r.sb);
    const double qb = __builtin_fma(b0, -sA * a.invD, nxm), fb = floor(qb);
    const double margin = kMarchMargin * fmax(1.0, a.invD);
    const bool up = (r.bf > r.bi) == (sA < 0.0);  // the minor index grows
    const int dm = up ? 1 : -1;
    const int mi0 = (int)fmin(fmax(fb, -2.0), (double)a.N + 1.0);
    const double c1 = pha * kBA * (-sA * D), c0 = pha * (r.sa - r.sb * kBA);
    // (the last test bounds the loop: each further line lies ahead)
    if (!(fabs(qb - fb - 0.5) < 0.5 - margin && fabs(af - ai) >= kMarchMargin && fabs(r.bf - r.bi) >= kMarchMargin &&
          fabs(kBA) <= 1.0e6 && c1 * (double)dm > 0.5 * D))
        return false;
    const int inside = 2 * a.nxm;
    // the window's first plane must be in the square, as march_loop tests
    if (k0 - 1 > ka || (unsigned)mi0 >= (unsigned)inside || k0 > kend) return true;
    if (k0 >= a.max_steps) {
        ovf = true;
        return true;
    }
    const int T = kstop - k0;
    const double uk0 = uain + (double)k0 * D, dux = c1 * (double)dm;
    const double ux0 = __builtin_fma((double)(up ? mi0 + 1 : mi0) - nxm, c1, c0);
    const double near = margin * D * fabs(kBA), sec = sqrt(1.0 + kAB * kAB);
    const double hA = 0.5 * sA * pha * a.invD, q2 = nxm + 2.0;
    // tile coordinates; index -1 is 0 by truncation, so the tiles at 0 take it
    const int oA = r.xmajor ? sink.x0 : sink.y0, oB = r.xmajor ? sink.y0 : sink.x0;
    const int loA = oA == 0 ? -1 : 0, loB = oB == 0 ? -1 : 0;
    const int stA = r.xmajor ? 1 : Sink::PITCH, stB = r.xmajor ? Sink::PITCH : 1;
    for (int pass = 0;; pass++) {
        bool unsure = false;
        double uold = u_start;
        int t = 0, nc = 0, mi = mi0;
        for (;;) {
            const double uk = __builtin_fma((double)t, D, uk0), ux = __builtin_fma((double)nc, dux, ux0);
            const double unew = fmin(ux, uk);
            const bool cross = ux < uk;
            unsure |= fabs(uk - ux) < near;
            // the middle's major index (+ 2, so truncation is floor)
            const double qa = __builtin_fma(uold + unew, hA, q2);
            unsure |= fabs(__builtin_amdgcn_fract(qa) - 0.5) > 0.5 - kMarchMargin;
            // (what lies beyond N - 1 is not stored)
            const int la = (int)qa - (oA + 2), lb = mi - oB;
            if ((unsigned)(la - loA) < (unsigned)(Sink::TS - loA) && (unsigned)(lb - loB) < (unsigned)(Sink::TS - loB))
                sink.add_at((int)(__umul24(max(la, 0), stA) + __umul24(max(lb, 0), stB)), (unew - uold) * sec);
            uold = unew;
            // after a plane the march goes on while it lies in the square
            const bool out = (unsigned)mi >= (unsigned)inside;
            if (!cross && (t >= T || out)) {
                if (!out && kstop < kend) ovf = true;
                break;
            }
            t += cross ? 0 : 1;
            nc += cross ? 1 : 0;
            mi += cross ? dm : 0;
        }
        if (pass == 1) return false;
        if (!unsure) return true;
#pragma unroll
        for (int m = 0; m < M; m++) sink.w[m] = -sink.w[m];
    }
}

// ---------------------------------------------------------------- kernels

// Sum over the P lanes of a group (P a power of two dividing 64, groups
// aligned): every lane of the group gets the same sum.
template <int P>
__device__ __forceinline__ double group_sum(double x)
{
#pragma unroll
    for (int d = 1; d < P; d <<= 1) x += __shfl_xor(x, d);
    return x;
}
template <int P>
__device__ __forceinline__ int group_sum(int x)
{
#pragma unroll
    for (int d = 1; d < P; d <<= 1) x += __shfl_xor(x, d);
    return x;
}

// One ray per P lanes, each marching one window of its steps (P = 1: the whole
// march, in the reference's order).  Small calls have too few rays to hide a
// march's latency, and the march of the r >= rmax test divides at every step:
// 64^2 x 80 views 75 us with P = 1, 44, 46 and 48 with 4, 8 and 16; 64^2 x 800
// 298, 270, 292 and 351; 128^2 (51.2 cm) x 81 153, 67, 64 and 59.
template <int M, int DT, int P>
__global__ __launch_bounds__(256) void k_trace_fwd(TraceArgs a)
{
    using Sink = std::conditional_t<DT == VCT_DENS_U16, SinkU16<M>, SinkF32<M>>;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int local = t / P, piece = t % P;
    if (local >= a.n_rays) return;  // (all lanes of a ray)
    const int ray = a.ray_offset + local;
    const int view = ray / a.W;
    const int ch = ray - view * a.W;
    float out[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    int iks = 0;
    if (view < a.VT) {
        bool ovf = false;
        Sink sink;
        sink.init(a.dens);
        if constexpr (P == 1) {
            iks = march_ray<true>(a, view, ch, sink, ovf);
        } else {
            RayConst r;
            if (setup_ray(a, view, ch, r)) {
                const int len = (march_step_estimate(a, r) + P - 1) / P;
                const int k0 = piece * len, k1 = piece == P - 1 ? INT_MAX : k0 + len - 1;
                iks = r.dB != 0.0 && !a.rcheck && !a.exact ? march_loop<true>(a, r, sink, ovf, k0, k1)
                                                           : march_loop<false>(a, r, sink, ovf, k0, k1);
            }
        }
        if constexpr (DT == VCT_DENS_U16) sink.finish();
#pragma unroll
        for (int m = 0; m < M; m++) out[m] = (float)(group_sum<P>(sink.acc[m]) * a.out_scale);
        iks = group_sum<P>(iks);
        if (ovf) atomicOr(a.err, 1);
    }
    if (piece != 0) return;
    float4* dst = reinterpret_cast<float4*>(a.L) + (size_t)ray * 2;
    dst[0] = make_float4(out[0], out[1], out[2], out[3]);
    dst[1] = make_float4(out[4], out[5], out[6], out[7]);
    if (a.counts) a.counts[ray] = iks;
}

// One ray of k_trace_fwd, written to L (and counts).
template <int M, int DT>
__device__ __forceinline__ void trace_one(const TraceArgs& a, int view, int ch)
{
    const int ray = view * a.W + ch;
    float out[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    int iks = 0;
    bool ovf = false;
    if (DT == VCT_DENS_U16) {
        SinkU16<M> sink;
        sink.init(a.dens);
        iks = march_ray<true>(a, view, ch, sink, ovf);
        sink.finish();
#pragma unroll
        for (int m = 0; m < M; m++) out[m] = (float)(sink.acc[m] * a.out_scale);
    } else {
        SinkF32<M> sink;
        sink.init(a.dens);
        iks = march_ray<true>(a, view, ch, sink, ovf);
#pragma unroll
        for (int m = 0; m < M; m++) out[m] = (float)(sink.acc[m] * a.out_scale);
    }
    if (ovf) atomicOr(a.err, 1);
    float4* dst = reinterpret_cast<float4*>(a.L) + (size_t)ray * 2;
    dst[0] = make_float4(out[0], out[1], out[2], out[3]);
    dst[1] = make_float4(out[4], out[5], out[6], out[7]);
    if (a.counts) a.counts[ray] = iks;
}

// Orbits of R rays: the base ray (view v < V/R, channel) is marched once and
// gives the rays of views v + kV/R their path integrals from the turned
// voxels (SinkRot).  The march of one orbit is split over a group of P
// adjacent lanes: lane p runs steps [p len, (p + 1) len) of the windowed
// march (the last lane to the end), len = ceil(steps / P), and the group adds
// its partial sums and segment counts with cross-lane shuffles.  When a march
// piece reports a decision within the margin, or the ray needs the exact
// march, the group traces rays 1..R-1 (and the base ray, unless marched) one
// by one, one ray per lane.  Every ray's segments are the reference's; the
// orbit shares the base ray's lengths, which differ from a ray's own
// |da| * sec by rounding.  Every branch before a shuffle depends only on the
// orbit, so the P lanes of a group stay together through the shuffles.
template <int M, int DT, int R, int P>
__global__ __launch_bounds__(256) void k_trace_fwd_rot(TraceArgs a)
{
    static_assert(P >= 1 && P <= 64 && (P & (P - 1)) == 0, "P: a power of two");
    const int gl = blockIdx.x * blockDim.x + threadIdx.x;
    const int orbit = gl / P, piece = gl % P;
    const int Vq = a.V / R;
    if (orbit >= Vq * a.W) return;  // whole groups
    const int view = orbit / a.W;
    const int ch = orbit - view * a.W;
    RayConst r;
    bool safe = false;
    const bool hit = setup_ray(a, view, ch, r, &safe);
    bool done = false;
    if (safe && !hit) {
        // the whole orbit misses the image: no segment, path integrals 0
        for (int k = piece; k < R; k += P) {
            const int ray = (view + k * Vq) * a.W + ch;
            float4* dst = reinterpret_cast<float4*>(a.L) + (size_t)ray * 2;
            dst[0] = make_float4(0.f, 0.f, 0.f, 0.f);
            dst[1] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (a.counts) a.counts[ray] = 0;
        }
        done = true;
    } else if (safe && r.dB != 0.0 && !a.rcheck && !a.exact) {
        SinkRot<M, DT, R> sink;
        sink.init(a.dens_t, r.xmajor, a.N);
        bool ovf = false;
        int k0 = 0, k1 = INT_MAX;
        if (P > 1) {
            const int len = (march_step_estimate(a, r) + P - 1) / P;
            k0 = piece * len;
            k1 = piece == P - 1 ? INT_MAX : k0 + len - 1;
        }
        int iks = march_loop<true>(a, r, sink, ovf, k0, k1);
        if (ovf) atomicOr(a.err, 1);
        if (P > 1) {
            iks = group_sum<P>(iks);
            sink.unsafe = group_sum<P>(sink.unsafe ? 1 : 0) != 0;
            if constexpr (DT == VCT_DENS_U16) {
#pragma unroll
                for (int k = 0; k < R; k++) {
#pragma unroll
                    for (int w = 0; w < SinkRot<M, DT, R>::NW; w++) sink.accw[k][w] = group_sum<P>(sink.accw[k][w]);
#pragma unroll
                    for (int w = 0; w < M / 2; w++) sink.acch[k][w] = group_sum<P>(sink.acch[k][w]);
                }
            } else {
#pragma unroll
                for (int k = 0; k < R; k++)
#pragma unroll
                    for (int m = 0; m < M; m++) sink.acc[k][m] = group_sum<P>(sink.acc[k][m]);
            }
        }
        sink.finish();
        // ray 0 is right in any case (its own march); the turned rays only
        // when no decision was within the margin
#pragma unroll
        for (int k = 0; k < R; k++) {
            if (k % P != piece || (k > 0 && sink.unsafe)) continue;
            const int ray = (view + k * Vq) * a.W + ch;
            float out[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int m = 0; m < M; m++) out[m] = (float)(sink.acc[k][m] * a.out_scale);
            float4* dst = reinterpret_cast<float4*>(a.L) + (size_t)ray * 2;
            dst[0] = make_float4(out[0], out[1], out[2], out[3]);
            dst[1] = make_float4(out[4], out[5], out[6], out[7]);
            if (a.counts) a.counts[ray] = iks;
        }
        if (sink.unsafe) {
            for (int k = 1 + piece; k < R; k += P) trace_one<M, DT>(a, view + k * Vq, ch);
        }
        done = true;
    }
    if (!done) {
        for (int k = piece; k < R; k += P) trace_one<M, DT>(a, view + k * Vq, ch);
    }
}

// ------------------------------------------------ tracer, segment by segment
//
// k_trace_seg: orbits of R rays as k_trace_fwd_rot, but each loop iteration is
// one segment of the lane's ray instead of one major step with its two
// candidate segments.  Along u = the major coordinate in the direction of
// travel, the segments after plane 0 end at the major planes u_k = u_0 + k D
// and at the minor grid lines, whose crossings x_n = c0 + c1 n are linear in
// the line index too, so the next end is the smaller of two products; the
// minor cell moves by one per crossing and the major index comes from the
// segment's middle.  A step's crossing is then no masked half of the wave's
// work, and per ray-segment about half the instructions remain.
//
// Decisions are those of march_loop: a plane and a line closer than the
// margin, a middle within it of a major grid line or a set-up decision within
// it leave the orbit to k_trace_redo, which marches its rays one by one; the
// tests are kept
// as running extremes and looked at once, after the loop.  The host rules out
// grids whose plane-to-plane middles lie on grid lines (seg_grid).
//
// A workgroup holds 64 neighbouring orbits, 16 channels of 4 views; each of its
// kSegWaves waves runs one window of the march, so all lanes of a wave are at
// about the same place and its gathers fall into few cache lines: requests to
// L2 bound the tracer before the instructions do (64 channels of one view per
// wave drift apart by rows: 0.44 ms where 16 x 4 take 0.30; 8 x 8 and 32 x 2
// 0.31 and 0.32; eight windows of eight orbits, the split before, 0.53).  Few
// views make too few such workgroups for the chip's L1s: they hold 32 or 16
// orbits then, in 16 or 32 windows (seg_shift).  The windows' sums meet in LDS,
// one ray of the orbits after the other.
// 800 x 609, against k_trace_fwd_rot: u16 M = 6 512^2 0.53 -> 0.29 ms, M = 8
// 0.62 -> 0.33; float M = 6 512^2 1.08 -> 0.48, 768^2 2.53 -> 0.95; one ray
// per march (401 views) against k_trace_fwd 0.60 -> 0.28.  Orbits read the
// plan's work copies; one ray per march reads the packed densities, so that
// calls of such a plan (odd views or grid) on several streams stay apart: the
// redo bits, which all calls share, and the orbits per workgroup, which lay them
// out, depend on the geometry alone.
constexpr int kSegWaves = 8;

// Bytes per voxel of the tracer's work copies: the materials in use.
template <int M, int DT>
constexpr int seg_voxel()
{
    return DT == VCT_DENS_U16 ? 4 * ((M + 1) / 2) : 8 * ((M + 1) / 2);
}

// A workgroup's 16 V orbits (V = 4, 2 or 1): kSegCh neighbouring channels of V
// neighbouring base views.
constexpr int kSegCh = 16;
__host__ __device__ __forceinline__ void seg_orbit(int block, int orbit, int V, int W, int& view, int& ch)
{
    const int ct = (W + kSegCh - 1) / kSegCh, vt = block / ct;
    view = vt * V + orbit / kSegCh;
    ch = (block - vt * ct) * kSegCh + orbit % kSegCh;
}

template <int M, int DT, int R>
struct SegSums {
    static constexpr int NW = (M + 1) / 2;
    // bytes of a voxel in the work copies (R == 1: a unit of the minor index)
    static constexpr int ND = seg_voxel<M, DT>() / 4, VB = R == 1 ? 1 : 4 * ND;
    // u16: sums of the 32-bit words and of their high halves (SinkU16)
    double accw[R][NW], acch[R][NW];
    struct Vox {
        uint32_t w[ND];
    };
    __device__ __forceinline__ void init()
    {
#pragma unroll
        for (int k = 0; k < R; k++)
#pragma unroll
            for (int j = 0; j < NW; j++) accw[k][j] = acch[k][j] = 0.0;
    }
    static __device__ __forceinline__ Vox load(const char* base, uint32_t o)
    {
        Vox q;
        const char* p = base + o;
        if constexpr (ND % 4 == 0) {
#pragma unroll
            for (int j = 0; j < ND / 4; j++) {
                const uint4 t = reinterpret_cast<const uint4*>(p)[j];
                q.w[4 * j] = t.x; q.w[4 * j + 1] = t.y; q.w[4 * j + 2] = t.z; q.w[4 * j + 3] = t.w;
            }
        } else if constexpr (ND == 6) {  // 8-byte aligned voxels
            struct alignas(8) Six { uint32_t w[6]; };
            const Six t = *reinterpret_cast<const Six*>(p);
#pragma unroll
            for (int j = 0; j < 6; j++) q.w[j] = t.w[j];
        } else if constexpr (ND == 3) {
            const uint3 t = *reinterpret_cast<const uint3*>(p);
            q.w[0] = t.x; q.w[1] = t.y; q.w[2] = t.z;
        } else if constexpr (ND == 2) {
            const uint2 t = *reinterpret_cast<const uint2*>(p);
            q.w[0] = t.x; q.w[1] = t.y;
        } else {
            q.w[0] = *reinterpret_cast<const uint32_t*>(p);
        }
        return q;
    }
    __device__ __forceinline__ void add(int k, const Vox& q, double rr)
    {
        if constexpr (DT == VCT_DENS_U16) {
#pragma unroll
            for (int j = 0; j < NW; j++) {
                // odd M: the last word's high half is not a material of this call
                const uint32_t w = 2 * j + 1 < M ? q.w[j] : q.w[j] & 0xffffu;
                accw[k][j] = __builtin_fma((double)w, rr, accw[k][j]);
                if (2 * j + 1 < M) acch[k][j] = __builtin_fma((double)(q.w[j] >> 16), rr, acch[k][j]);
            }
        } else {
            // (a negative density contributes nothing, as SinkF32; the work
            // copies hold max(rho, 0))
            auto rho = [](uint32_t w) { return (double)(R == 1 ? fmaxf(__uint_as_float(w), 0.f) : __uint_as_float(w)); };
#pragma unroll
            for (int j = 0; j < NW; j++) {
                accw[k][j] = __builtin_fma(rho(q.w[2 * j]), rr, accw[k][j]);
                if (2 * j + 1 < M) acch[k][j] = __builtin_fma(rho(q.w[2 * j + 1]), rr, acch[k][j]);
            }
        }
    }
    __device__ __forceinline__ void scale(double f)
    {
#pragma unroll
        for (int k = 0; k < R; k++)
#pragma unroll
            for (int j = 0; j < NW; j++) {
                accw[k][j] *= f;
                acch[k][j] *= f;
            }
    }
    // material m of ray k
    __device__ __forceinline__ double sum(int k, int m) const
    {
        const int j = m >> 1;
        if (m & 1) return acch[k][j];
        if (DT == VCT_DENS_U16 && m + 1 < M) return accw[k][j] - 65536.0 * acch[k][j];
        return accw[k][j];
    }
};

template <int M, int DT, int R>
__global__ __launch_bounds__(64 * kSegWaves) void k_trace_seg(TraceArgs a, int sh)
{
    using Sums = SegSums<M, DT, R>;
    constexpr int VB = Sums::VB;
    __shared__ double part[64 * kSegWaves * M];  // [window][material][orbit]
    __shared__ int cnt[64], redo[64];
    // 2^sh orbits (seg_shift), of which a lane marches one in one of the windows
    const int pieces = 64 * kSegWaves >> sh, lane = threadIdx.x & ((1 << sh) - 1), piece = (int)threadIdx.x >> sh;
    const int Vq = (R == 1 ? a.VT : a.V / R);
    int view, ch;
    seg_orbit(blockIdx.x, lane, (1 << sh) / kSegCh, a.W, view, ch);
    const bool valid = view < Vq && ch < a.W;
    if (piece == 0) {
        cnt[lane] = 0;
        redo[lane] = 0;
    }
    __syncthreads();
    Sums sums;
    sums.init();
    RayConst r;
    bool safe = false;
    const bool hit = valid && setup_ray(a, view, ch, r, &safe);
    bool bad = valid && !safe;
    if (hit && safe) {
        const double ai = r.ai, af = r.af, Lb = r.Lb, D = a.D;
        const double kAB = r.dB / r.dA, kBA = r.dA / r.dB;
        const double sec = sqrt(1.0 + kAB * kAB);
        const double pha = af > ai ? 1.0 : -1.0;
        // integer-cm start plane, M/reprojection_TOMO.cpp:115-119
        const int ain = ((ai < 0 && af < ai) || (ai > 0 && af > ai)) ? trunc_i32(trunc_i32(ai) + pha) : trunc_i32(ai);
        const double uain = pha * (double)ain;
        const double sA = r.xmajor ? 1.0 : -1.0, nxm = (double)a.nxm;
        // set-up decisions that a turned ray might take otherwise, and slopes
        // too small for the lines' crossings
        bad = !((fabs(ai) == Lb || trunc_safe(ai)) && fabs(af - ai) >= kMarchMargin &&
                fabs(r.bf - r.bi) >= kMarchMargin && fabs(kBA) <= 1.0e6);
        // window of planes: this piece ends segments at planes k0 .. kstop
        const int len = (march_step_estimate(a, r) + pieces - 1) / pieces;
        const int k0 = max(piece * len, 1), k1 = piece == pieces - 1 ? a.max_steps : (piece + 1) * len - 1;
        // last plane inside the square (exactly u_0 + fl(k D) <= Lb)
        int ka = (int)fmin(fmax((Lb - uain) / D, -1.0), 1.0e8);
        if (uain + (double)(ka + 1) * D <= Lb) ka++;
        if (ka >= 0 && uain + (double)ka * D > Lb) ka--;
        const int kend = min(k1, ka + 1), kstop = min(kend, a.max_steps - 1);
        // minor index value of plane k0 - 1: the cell and the first line ahead
        const double u_start = uain + (double)(k0 - 1) * D;
        const double b0 = __builtin_fma(pha * u_start - r.sa, kAB, r.sb);
        const double hB = -sA * a.invD;
        const double qb = __builtin_fma(b0, hB, nxm), fb = floor(qb);
        // the general march's margins: 1e-9 voxel, and 1e-9 cm where it is the
        // larger (a line is also where it compares signs and the square's edge)
        const double margin = kMarchMargin * fmax(1.0, a.invD);
        bad = bad || !(fabs(qb - fb - 0.5) < 0.5 - margin);
        const bool up = (r.bf > r.bi) == (sA < 0.0);  // the minor index grows
        const int dm = up ? 1 : -1;
        int mi = (int)fmin(fmax(fb, -2.0), (double)a.N + 1.0);
        double nd = (double)(up ? mi + 1 : mi) - nxm;  // next line, counted from the centre
        const double c1 = pha * kBA * (-sA * D), c0 = pha * (r.sa - r.sb * kBA);
        // each further line lies ahead, at least about a pitch on (|slope| <= 1),
        // so the loop below ends
        bad = bad || !(c1 * (double)dm > 0.5 * D);
        const double hA = 0.5 * sA * pha * a.invD, q2 = nxm + 2.0;
        // byte offsets in the two copies: row (major) and column (minor) parts
        // of a voxel and of its turned images; slots 1 and 3 read the other copy
        const int NP = a.N + 4, row = VB * NP;
        const uint32_t size = (uint32_t)(NP * NP) * (uint32_t)VB;
        const uint32_t baseE = r.xmajor ? size : 0u, dO = r.xmajor ? 0u - size : size;
        const uint32_t rT = (uint32_t)((a.N + 3) * row) + 2u * baseE, cT = (uint32_t)((a.N + 3) * VB);
        const char* copies = reinterpret_cast<const char*>(R == 1 ? a.dens : a.dens_t);
        // R == 1: the packed densities themselves, by the ray's own axes
        constexpr int IB = DT == VCT_DENS_U16 ? 16 : 32;
        const int stA = (r.xmajor ? 1 : a.N) * IB, stB = (r.xmajor ? a.N : 1) * IB;
        // voxel (ma, mb) of a lone ray, index -1 being 0 by truncation; outside
        // the image the length is 0
        auto lone = [&](int ma, int mb, double& rr) {
            const bool in = (unsigned)(ma + 1) <= (unsigned)a.N && (unsigned)(mb + 1) <= (unsigned)a.N;
            rr = in ? rr : 0.0;
            return in ? (uint32_t)__umul24(max(ma, 0), stA) + (uint32_t)__umul24(max(mb, 0), stB) : 0u;
        };
        int n = 0;
        const int inside = 2 * a.nxm;  // minor cells 0 .. inside - 1 lie in the square
        bool ovf = false;
        if (piece == 0 && !bad) {
            // step 0: one segment from the entry to plane 0 (up to 1 cm, not cut
            // at grid lines); its indices from the reference's exact expressions,
            // whose ties on the major axis turn with the ray when the entry lies
            // on a major side of the square (march_loop's a_sym)
            const double be = ((double)ain - r.sa) / r.dA * r.dB + r.sb;
            if (ka >= 0 && (unsigned)mi < (unsigned)inside) {
                if (a.max_steps < 1) ovf = true;
                else {
                    n = 1;
                    const double rr = fabs((double)ain - ai);
                    const double ta = sA * ((ai + (double)ain) * 0.5) / D, tb = -sA * ((r.bi + be) * 0.5) / D;
                    const double qa = ta + nxm, qm = tb + nxm;
                    const bool sure_a = fabs(fabs(qa - trunc(qa)) - 0.5) < 0.5 - kMarchMargin;
                    const bool sure_b = fabs(fabs(qm - trunc(qm)) - 0.5) < 0.5 - kMarchMargin;
                    if (rr != 0.0) {
                        if (!sure_b || !(sure_a || fabs(ai) == Lb)) bad = true;
                        // each ray takes fl(+-t + N/2) of its own axis and its trunc:
                        // index t + N/2 and N/2 - t, here as voxel numbers
                        const int pa = trunc_i32(ta + nxm), na = trunc_i32(-ta + nxm);
                        const int pb = trunc_i32(tb + nxm), nb = trunc_i32(-tb + nxm);
                        auto in = [&](int v) { return v >= 0 && v <= a.N - 1; };
                        auto one = [&](int k, uint32_t base, int ma, int mb) {
                            if (!in(ma) || !in(mb)) return;
                            sums.add(k, Sums::load(copies, base + (uint32_t)((ma + 2) * row) + (uint32_t)((mb + 2) * VB)),
                                     rr);
                        };
                        if constexpr (R == 1) {
                            if (in(pa) && in(pb)) {
                                double l = rr;
                                const uint32_t o = lone(pa, pb, l);
                                sums.add(0, Sums::load(copies, o), l);
                            }
                        } else {
                            one(0, baseE, pa, pb);
                        }
                        if constexpr (R == 2) one(1, baseE, na, nb);
                        if constexpr (R == 4) {
                            one(2, baseE, na, nb);
                            one(1, baseE + dO, pa, nb);
                            one(3, baseE + dO, na, pb);
                        }
                    }
                }
            }
        }
        // the window's first plane k0 - 1 must be in the square, as march_loop
        // tests before each step
        if (!bad && k0 - 1 <= ka && (unsigned)mi < (unsigned)inside) {
            if (k0 >= a.max_steps) ovf = k0 <= k1;
            else if (k0 <= kend) {
                // after i segments nc of them ended at a line and i - nc at a plane;
                // i is the same on every lane
                const int T = kstop - k0;
                const double uk0 = uain + (double)k0 * D, ux0 = __builtin_fma(nd, c1, c0), dux = c1 * (double)dm;
                const double near = margin * D * fabs(kBA);
                const int dc = dm * VB;
                const uint32_t cin = (uint32_t)(inside * VB);
                uint32_t cu = (uint32_t)((mi + 2) * VB);
                double uold = u_start;
                int nc = 0;
                int i = 0;
                bool unsure = false;
                struct Pending {
                    typename Sums::Vox q[R];
                    double rr;
                };
                // segment i: its gathers are issued into p; true if it is the last
                auto step = [&](Pending& p) {
                    const int t = i - nc;
                    const double uk = __builtin_fma((double)t, D, uk0), ux = __builtin_fma((double)nc, dux, ux0);
                    const double unew = fmin(ux, uk);
                    p.rr = unew - uold;
                    const bool cross = ux < uk;
                    unsure |= fabs(uk - ux) < near;
                    // the middle's major index (+ 2, so truncation is floor), and its
                    // distance from the grid lines
                    const double qa = __builtin_fma(uold + unew, hA, q2);
                    unsure |= fabs(__builtin_amdgcn_fract(qa) - 0.5) > 0.5 - kMarchMargin;
                    uold = unew;
                    // (clamped: what lies outside reads the zero border)
                    if constexpr (R == 1) {
                        p.q[0] = Sums::load(copies, lone((int)qa - 2, (int)(cu / VB) - 2, p.rr));
                    } else {
                        const uint32_t ia = min((uint32_t)(int)qa, (uint32_t)(a.N + 3)), c = min(cu, cT);
                        const uint32_t ra = __umul24(ia, (uint32_t)row) + baseE;
                        const uint32_t rt = rT - ra, ct = cT - c;
                        p.q[0] = Sums::load(copies, ra + c);
                        p.q[R == 4 ? 2 : 1] = Sums::load(copies, rt + ct);
                        if constexpr (R == 4) {
                            p.q[1] = Sums::load(copies, ra + dO + ct);
                            p.q[3] = Sums::load(copies, rt + dO + c);
                        }
                    }
                    // after a plane the march goes on while it lies in the square
                    const bool out = cu - 2u * VB >= cin;
                    const bool end = !cross && (t >= T || out);
                    if (end && !out && kstop < kend) ovf = true;
                    nc += cross ? 1 : 0;
                    cu += (uint32_t)(cross ? dc : 0);
                    i++;
                    return end;
                };
                // (outside the image a lone ray holds voxel 0 with length 0, which an
                // infinite density would turn into NaN; an orbit reads the zero border)
                auto add = [&](const Pending& p) {
                    if (R == 1 && DT == VCT_DENS_F32 && p.rr == 0.0) return;
#pragma unroll
                    for (int k = 0; k < R; k++) sums.add(k, p.q[k], p.rr);
                };
                // a segment's voxels are added while the next one's are fetched, in
                // two register sets in turn; four rays of more than 6 materials add
                // each at once (the second set would take the kernel past 128
                // registers: 0.33 against 0.39 ms at 512^2, u16, M = 8)
                Pending p0, p1;
                if constexpr (R == 4 && M > 6) {
                    bool end = false;
                    while (!end) {
                        end = step(p0);
                        add(p0);
                    }
                } else if (step(p0)) {
                    add(p0);
                } else {
                    for (;;) {
                        bool end = step(p1);
                        add(p0);
                        if (end) {
                            add(p1);
                            break;
                        }
                        end = step(p0);
                        add(p1);
                        if (end) {
                            add(p0);
                            break;
                        }
                    }
                }
                n += i;
                bad = unsure;
            }
        }
        // (the lengths above lack the factor sec)
        sums.scale(sec);
        if (ovf) atomicOr(a.err, 1);
        if (!bad && n) atomicAdd(&cnt[lane], n);
    }
    if (bad) redo[lane] = 1;
    // the windows' sums, ray k of the orbits at a time: lane t adds and writes
    // slot t >> sh of its orbit
    const bool xmaj = hit && r.xmajor;
#pragma unroll
    for (int k = 0; k < R; k++) {
        __syncthreads();
#pragma unroll
        for (int m = 0; m < M; m++) part[((piece * M + m) << sh) + lane] = sums.sum(k, m);
        __syncthreads();
        // slots 1 and 3 hold rays 3 and 1 when y is the base ray's major axis
        const int ray_k = (R == 4 && (k & 1) && !xmaj) ? 4 - k : k;
        if (valid && !redo[lane] && piece < 8) {
            const int ray = (view + ray_k * Vq) * a.W + ch, m = piece;
            double t = 0.0;
            if (m < M) {
                auto eight = [&](int w0) {
#pragma unroll
                    for (int w = 0; w < kSegWaves; w++) t += part[(((w0 + w) * M + m) << sh) + lane];
                };
                // (not a loop: with one the compiler forms all rays' sums before it,
                // in half as many registers again)
                eight(0);
                if (sh < 6) eight(8);
                if (sh < 5) {
                    eight(16);
                    eight(24);
                }
            }
            a.L[(size_t)ray * 8 + m] = (float)(t * a.out_scale);
            if (piece == 0 && a.counts) a.counts[ray] = cnt[lane];
        }
    }
    if (threadIdx.x < 64) {
        const unsigned long long m = __ballot(piece == 0 && valid && redo[lane]);
        if (threadIdx.x == 0) a.redo[blockIdx.x] = m;
    }
}

// The rays of the orbits that k_trace_seg left (bit l of redo[w]: orbit l of
// workgroup w), each by its own march in the 64 windows of a wave (a kernel of
// its own, so that the general march's registers do not count against the
// segment loop's).  One workgroup, a wave per ray of an orbit, per 64 words;
// they are nearly always all zero.
template <int M, int DT, int R>
__global__ __launch_bounds__(64 * R) void k_trace_redo(TraceArgs a, int words, int sh)
{
    constexpr int P = 64;
    using Sink = std::conditional_t<DT == VCT_DENS_U16, SinkU16<M>, SinkF32<M>>;
    const int w0 = blockIdx.x * 64, lane = threadIdx.x & 63, Vq = (R == 1 ? a.VT : a.V / R);
    const unsigned long long mine = w0 + lane < words ? a.redo[w0 + lane] : 0ull;
    unsigned long long any = __ballot(mine != 0ull);
    while (any) {
        const int w = __ffsll((long long)any) - 1;
        any &= any - 1;
        unsigned long long m = __shfl(mine, w);
        while (m) {
            int v0, ch;
            seg_orbit(w0 + w, __ffsll((long long)m) - 1, (1 << sh) / kSegCh, a.W, v0, ch);
            m &= m - 1;
            const int view = v0 + (int)(threadIdx.x >> 6) * Vq, piece = lane;
            RayConst r;
            Sink sink;
            sink.init(a.dens);
            int iks = 0;
            bool ovf = false;
            if (setup_ray(a, view, ch, r)) {
                const int len = (march_step_estimate(a, r) + P - 1) / P;
                const int k0 = piece * len, k1 = piece == P - 1 ? INT_MAX : k0 + len - 1;
                iks = r.dB != 0.0 ? march_loop<true>(a, r, sink, ovf, k0, k1) : march_loop<false>(a, r, sink, ovf, k0, k1);
            }
            if (ovf) atomicOr(a.err, 1);
            if constexpr (DT == VCT_DENS_U16) sink.finish();
            float out[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < M; q++) out[q] = (float)(group_sum<P>(sink.acc[q]) * a.out_scale);
            iks = group_sum<P>(iks);
            if (piece == 0) {
                const int ray = view * a.W + ch;
                float4* dst = reinterpret_cast<float4*>(a.L) + (size_t)ray * 2;
                dst[0] = make_float4(out[0], out[1], out[2], out[3]);
                dst[1] = make_float4(out[4], out[5], out[6], out[7]);
                if (a.counts) a.counts[ray] = iks;
            }
        }
    }
}

// Whether k_trace_seg serves this geometry: the guarded march without the
// r >= rmax test, 32-bit offsets into the two copies, and no start plane whose
// plane-to-plane middles fall on a major grid line (u_0 integer, middles at
// u_0/D + k + 1/2: a grid of 128 voxels on 51.2 cm has such planes at every
// odd centimetre, and each of their steps would be undecided).
static bool seg_planes(const TraceArgs& a);
static bool seg_grid(const TraceArgs& a, int vb)
{
    if (!a.redo || (a.rot > 1 && !a.dens_t)) return false;
    const double np = a.N + 4.0;
    if (2.0 * np * np * vb >= 4294967296.0 || (double)vb * np >= 8388608.0) return false;
    return seg_planes(a);
}
static bool seg_planes(const TraceArgs& a)
{
    if (a.exact || a.rcheck) return false;
    const int last = (int)((double)a.nxm * a.D) + 2;
    for (int c = 0; c <= last; c++) {
        const double f = (double)c * a.invD + 0.5;
        if (fabs(f - nearbyint(f)) < 1.0e-6) return false;
    }
    return true;
}

// Adjoint by image tiles.  Workgroup (chunk, tile) takes the views of one
// chunk and one TS^2 tile of the image; for each view it finds the channels
// whose rays can cross the tile (box_channels), and each such ray runs only
// the march steps that can land in the tile (box_steps, the windowed
// march_loop), adding w[m] * length into the tile in LDS.  Each segment of
// each ray lands in exactly one tile, so the tiles of one chunk together add
// every segment once.  A first pass over the workgroup's rays takes the
// largest |w|, which sets the fixed-point scale (SinkTile); at the end the
// tile is added to grad with one float atomic per voxel and material (zero
// where the voxel's density of that material is negative, the tracer's sign
// test).  Work items are dealt to XCDs (workgroup g runs on XCD g % 8) in
// contiguous runs, tile fastest, so the workgroups of one XCD share view
// chunks and read their rays' weights through one L2.
// Instruction issue and the LDS atomics (3.4 lane-operations per clock and CU)
// bound it.  Two workgroups of 512 lanes per CU within 128 registers instead
// of three of 256 lanes with 135: 380^2 x 722 views, M = 6, 1.38 -> 1.16 ms,
// M = 8 1.87 -> 1.28; the addend by one fused multiply-add 1.53 -> 1.38; the
// segment loop 1.91 -> 1.53; workgroups with few rays take 256 lanes
// (adjoint_lanes); larger tiles (40) 1.11, but 0.14 instead of 0.12
// at 64^2.
template <int M>
__device__ __forceinline__ void adj_weights(const TraceArgs& a, int ray, float (&w)[M])
{
    const float gscale = (a.g ? a.g[ray] : 1.f) * (float)a.out_scale;
    const float4* wv = reinterpret_cast<const float4*>(a.wts) + (size_t)ray * 2;
    const float4 w0 = wv[0];
    const float4 w1 = M > 4 ? wv[1] : make_float4(0.f, 0.f, 0.f, 0.f);
    const float wa[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
#pragma unroll
    for (int m = 0; m < M; m++) w[m] = wa[m] * gscale;
}

template <int M>
__global__ __launch_bounds__(kAdjBlock, 4) void k_trace_adj_tile(TraceArgs a, int ntx, int ntiles, int cv, int per_xcd, int seg)
{
    using Fixed = SinkTile<M, true>;
    using Float = SinkTile<M, false>;
    constexpr int TS = Fixed::TS, PITCH = Fixed::PITCH, PLANE = Fixed::PLANE;
    __shared__ unsigned long long acc[M * PLANE];
    __shared__ int pref[kAdjMaxViews + 1];
    __shared__ int clo[kAdjMaxViews];
    __shared__ uint32_t wmax_bits, nonfinite;
    const int item = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    const int nchunk = (a.VT + cv - 1) / cv;
    if (item >= ntiles * nchunk) return;  // whole workgroup, before any barrier
    const int chunk = item / ntiles, tile = item - chunk * ntiles;
    const int x0 = (tile % ntx) * TS, y0 = (tile / ntx) * TS;
    const int v0 = chunk * cv;
    const int nv = min(cv, a.VT - v0);
    for (int i = threadIdx.x; i < M * PLANE; i += blockDim.x) acc[i] = 0ull;
    if (threadIdx.x == 0) {
        wmax_bits = 0u;
        nonfinite = 0u;
    }
    // the tile plus two voxels, in cm (x index i covers [(i - nxm) D, (i + 1 - nxm) D),
    // y index j covers (-(j + 1 - nxm) D, -(j - nxm) D])
    const double D = a.D;
    const double x_lo = (double)(x0 - 2 - a.nxm) * D, x_hi = (double)(x0 + TS + 2 - a.nxm) * D;
    const double y_lo = -(double)(y0 + TS + 2 - a.nxm) * D, y_hi = -(double)(y0 - 2 - a.nxm) * D;
    for (int i = threadIdx.x; i < nv; i += blockDim.x) {
        int lo, hi;
        box_channels(a, v0 + i, x_lo, x_hi, y_lo, y_hi, lo, hi);
        clo[i] = lo;
        pref[i + 1] = hi >= lo ? hi - lo + 1 : 0;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        pref[0] = 0;
        for (int i = 0; i < nv; i++) pref[i + 1] += pref[i];
    }
    __syncthreads();
    const int total = pref[nv];
    // view slot j with pref[j] <= i < pref[j + 1], and the ray of item i
    auto item_ray = [&](int i, int& view, int& ch) {
        int lo = 0, hi = nv - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (pref[mid] <= i) lo = mid;
            else hi = mid - 1;
        }
        view = v0 + lo;
        ch = clo[lo] + (i - pref[lo]);
    };
    // pass 1: the largest |w| of the workgroup's rays (non-negative float bits
    // order as unsigned integers) and whether any weight is not finite
    {
        float wmax = 0.f;
        bool bad = false;
        for (int i = threadIdx.x; i < total; i += blockDim.x) {
            int view, ch;
            item_ray(i, view, ch);
            float w[M];
            adj_weights<M>(a, view * a.W + ch, w);
#pragma unroll
            for (int m = 0; m < M; m++) {
                const float u = fabsf(w[m]);
                bad = bad || !(u <= 3.0e38f);
                wmax = fmaxf(wmax, u);
            }
        }
        if (wmax > 0.f) atomicMax(&wmax_bits, __float_as_uint(wmax));
        if (bad) atomicOr(&nonfinite, 1u);
    }
    __syncthreads();
    const float wmax = __uint_as_float(wmax_bits);
    // segment lengths are at most sqrt(2) max(1 cm, D): the first step runs from
    // the entry to the integer-cm start plane, the others one pitch
    // (weights so small that the scale would leave float's range, wl below
    // 2^-80, sum in float too, as non-finite ones do)
    const float wl = wmax * (float)(2.0 * fmax(1.0, D));
    if (nonfinite == 0u && !(wmax > 0.f)) return;  // nothing to add (uniform over the workgroup)
    const bool fixed = nonfinite == 0u && wl <= 3.0e38f && wl >= 0x1p-80f;
    int S = 0;
    if (fixed) {
        int e;
        frexpf(wl, &e);  // wl < 2^e, e >= -79
        S = 30 - e;      // <= 109
    }
    const double scale = ldexp(1.0, S);
    bool ovf = false;
    for (int i = threadIdx.x; i < total; i += blockDim.x) {
        int view, ch;
        item_ray(i, view, ch);
        float w[M];
        adj_weights<M>(a, view * a.W + ch, w);
        bool any = false;
#pragma unroll
        for (int m = 0; m < M; m++) any = any || (w[m] != 0.f);
        if (!any) continue;
        RayConst r;
        if (!setup_ray(a, view, ch, r)) continue;
        int k0, k1;
        if (!box_steps(a, r, x_lo, x_hi, y_lo, y_hi, k0, k1)) continue;
        const bool fast = r.dB != 0.0 && !a.rcheck && !a.exact;
        if (fixed) {
            Fixed sink{acc, x0, y0, r.xmajor, {}};
#pragma unroll
            for (int m = 0; m < M; m++) sink.w[m] = w[m] * scale;
            // (the segment loop starts after the entry's step 0)
            if (fast && seg) {
                if (k0 == 0) {
                    march_loop<true>(a, r, sink, ovf, 0, 0);
                    k0 = 1;
                }
                if (k0 <= k1 && !seg_window<M>(a, r, sink, ovf, k0, k1)) {
#pragma unroll
                    for (int m = 0; m < M; m++) sink.w[m] = w[m] * scale;
                    march_loop<true>(a, r, sink, ovf, k0, k1);
                }
            } else if (fast) march_loop<true>(a, r, sink, ovf, k0, k1);
            else march_loop<false>(a, r, sink, ovf, k0, k1);
        } else {
            Float sink{acc, x0, y0, r.xmajor, {}};
#pragma unroll
            for (int m = 0; m < M; m++) sink.w[m] = w[m];
            if (fast) march_loop<true>(a, r, sink, ovf, k0, k1);
            else march_loop<false>(a, r, sink, ovf, k0, k1);
        }
    }
    if (ovf) atomicOr(a.err, 1);
    __syncthreads();
    const float* dens = reinterpret_cast<const float*>(a.dens);
    const double unscale = ldexp(1.0, -S);
    // (a lane per material of a voxel, so that a wave's adds cover whole lines of grad)
    constexpr int MP = M > 4 ? 8 : M > 2 ? 4 : M;
    for (int i = threadIdx.x; i < TS * TS * MP; i += blockDim.x) {
        const int m = i % MP, lx = i / MP % TS, ly = i / MP / TS;
        const int x = x0 + lx, y = y0 + ly;
        if (m >= M || x >= a.N || y >= a.N) continue;
        const size_t v = (size_t)y * a.N + x;
        const int off = ly * PITCH + lx + m * PLANE;
        float val = fixed ? (float)((double)Fixed::fixed_sum(acc[off]) * unscale) : reinterpret_cast<const float*>(acc)[off];
        if (dens && !(dens[v * 8 + m] >= 0.f)) val = 0.f;
        if (val != 0.f) unsafeAtomicAdd(a.grad + v * 8 + m, val);
    }
}

// Polyenergetic sums.  Rays per workgroup: each workgroup adds its max and min
// of I to the spectrum's two statistics words with one atomic each, and those
// atomics serialise on the one address (1904 workgroups of 256 rays took as
// long as the sums at 800 x 609), so workgroups are large, but for calls whose
// large ones would leave CUs without any.
constexpr int kSpecBlock = 1024;

// Adds the workgroup's max and min of I (non-negative floats order like their
// bits) to stats[0..1].  Every lane takes part.
__device__ __forceinline__ void spec_stats(uint32_t* stats, bool valid, float I, uint32_t (&red)[2][kSpecBlock / 64])
{
    uint32_t mx = valid ? __float_as_uint(I) : 0u;
    uint32_t mn = valid ? __float_as_uint(I) : 0x7f800000u;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        mx = max(mx, (uint32_t)__shfl_xor((int)mx, off, 64));
        mn = min(mn, (uint32_t)__shfl_xor((int)mn, off, 64));
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) { red[0][wave] = mx; red[1][wave] = mn; }
    __syncthreads();
    if (threadIdx.x == 0) {
        const int nw = (blockDim.x + 63) >> 6;
        for (int w = 1; w < nw; w++) { mx = max(mx, red[0][w]); mn = min(mn, red[1][w]); }
        atomicMax(stats, mx);
        atomicMin(stats + 1, mn);
    }
}

// The sums alone (spec_sum), one spectrum per blockIdx.y.
template <int M>
__global__ __launch_bounds__(kSpecBlock) void k_spectral(SpectralArgs a)
{
    extern __shared__ float lds[];
    __shared__ uint32_t red[2][kSpecBlock / 64];
    __shared__ int last[kSpecBlock / 64];
    const int s = blockIdx.y, nr = a.V * a.W, traced = a.VT * a.W;
    const SpecTable<M> tab =
        SpecTable<M>::fill(lds, last, a.att + (size_t)s * M * a.NE, a.pdf + (size_t)s * a.NE, a.NE);
    const int ray = blockIdx.x * blockDim.x + threadIdx.x, ray0 = ray & ~63;
    SpecRays<M> L;
    L.load([&](int t, int m) { return ray0 + t < traced ? a.L[(size_t)(ray0 + t) * 8 + m] : 0.f; });
    float I = spec_sum<M>(tab, L);
    if (ray >= traced) I = 0.f;
    if (ray < nr) a.raw[(size_t)s * nr + ray] = I;
    spec_stats(a.stats + 2 * s, ray < nr, I, red);
}

// The sums and their derivatives in the path integrals, one ray per lane; tables
// in LDS as mu2[e][8] = -mu_m(E_e) * log2(e) and pdf[e].
template <int M>
__global__ __launch_bounds__(kSpecBlock) void k_spectral_grad(SpectralArgs a)
{
    extern __shared__ float lds[];
    float* mu2 = lds;
    float* pdf = lds + a.NE * 8;
    __shared__ uint32_t red[2][kSpecBlock / 64];
    const int s = blockIdx.y;
    const int NE = a.NE;
    const float kLog2e = 1.4426950408889634f;
    for (int i = threadIdx.x; i < NE * 8; i += blockDim.x) {
        const int e = i >> 3, m = i & 7;
        mu2[i] = (m < M) ? -a.att[((size_t)s * M + m) * NE + e] * kLog2e : 0.f;
    }
    for (int e = threadIdx.x; e < NE; e += blockDim.x) pdf[e] = a.pdf[(size_t)s * NE + e];
    __syncthreads();

    const int nr = a.V * a.W;
    const int ray = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = ray < nr;
    float I = 0.f;
    float d[M];
#pragma unroll
    for (int m = 0; m < M; m++) d[m] = 0.f;
    if (valid && ray / a.W < a.VT) {
        const float4* Lv = reinterpret_cast<const float4*>(a.L) + (size_t)ray * 2;
        const float4 l0 = Lv[0], l1 = Lv[1];
        const float Lm[8] = {l0.x, l0.y, l0.z, l0.w, l1.x, l1.y, l1.z, l1.w};
        for (int e = 0; e < NE; e++) {
            // the 8 table entries of bin e in two 16-byte LDS reads
            const float4 m0 = reinterpret_cast<const float4*>(mu2)[2 * e];
            const float4 m1 = reinterpret_cast<const float4*>(mu2)[2 * e + 1];
            const float mu[8] = {m0.x, m0.y, m0.z, m0.w, m1.x, m1.y, m1.z, m1.w};
            float x = 0.f;
#pragma unroll
            for (int m = 0; m < M; m++) x = fmaf(mu[m], Lm[m], x);
            // hardware exp2: only terms below 2^-126 (flushed) differ from exp2f
            const float t = pdf[e] * __builtin_amdgcn_exp2f(x);
            I += t;
#pragma unroll
            for (int m = 0; m < M; m++) d[m] = fmaf(t, mu[m], d[m]);
        }
    }
    if (valid) {
        a.raw[(size_t)s * nr + ray] = I;
        const float kLn2 = 0.69314718055994531f;
        float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < M; m++) o[m] = d[m] * kLn2;
        float4* dst = reinterpret_cast<float4*>(a.dIdL) + ((size_t)s * nr + ray) * 2;
        dst[0] = make_float4(o[0], o[1], o[2], o[3]);
        dst[1] = make_float4(o[4], o[5], o[6], o[7]);
    }
    spec_stats(a.stats + 2 * s, valid, I, red);
}

__global__ void k_stats_init(uint32_t* stats, int S)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < S) {
        stats[2 * i] = 0u;
        stats[2 * i + 1] = 0x7f800000u;
    }
}

// Order-preserving uint image of a float (for atomic min/max of any sign).
__device__ __forceinline__ uint32_t ord_of(float f)
{
    const uint32_t b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

__device__ __forceinline__ float float_of_ord(uint32_t o)
{
    return __uint_as_float((o & 0x80000000u) ? (o & 0x7fffffffu) : ~o);
}

__global__ void k_minmax_init(uint32_t* st)
{
    st[0] = 0u;           // max, ordered
    st[1] = 0xffffffffu;  // min, ordered
}

__global__ __launch_bounds__(256) void k_minmax(const float* __restrict__ x, int n, uint32_t* st)
{
    __shared__ uint32_t red[2][4];
    uint32_t mx = 0u, mn = 0xffffffffu;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const uint32_t o = ord_of(x[i]);
        mx = max(mx, o);
        mn = min(mn, o);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        mx = max(mx, (uint32_t)__shfl_xor((int)mx, off, 64));
        mn = min(mn, (uint32_t)__shfl_xor((int)mn, off, 64));
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) { red[0][wave] = mx; red[1][wave] = mn; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x >> 6); w++) { mx = max(mx, red[0][w]); mn = min(mn, red[1][w]); }
        atomicMax(st, mx);
        atomicMin(st + 1, mn);
    }
}

// Converts the ordered images back to float bit patterns {max, min}.
__global__ void k_minmax_final(uint32_t* st)
{
    st[0] = __float_as_uint(float_of_ord(st[0]));
    st[1] = __float_as_uint(float_of_ord(st[1]));
}

// Philox4x32-10 (Salmon et al., SC'11).
__device__ __forceinline__ uint4 philox4x32_10(uint4 c, uint32_t k0, uint32_t k1)
{
#pragma unroll
    for (int r = 0; r < 10; r++) {
        if (r) { k0 += 0x9E3779B9u; k1 += 0xBB67AE85u; }
        const uint32_t lo0 = 0xD2511F53u * c.x, hi0 = __umulhi(0xD2511F53u, c.x);
        const uint32_t lo1 = 0xCD9E8D57u * c.z, hi1 = __umulhi(0xCD9E8D57u, c.z);
        c = make_uint4(hi1 ^ c.y ^ k0, lo1, hi0 ^ c.w ^ k1, lo0);
    }
    return c;
}

__global__ __launch_bounds__(256) void k_detector(DetectorArgs a)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n * a.S) return;
    const int s = i / a.n;
    const int r = i - s * a.n;
    const float mx = __uint_as_float(a.stats[2 * s]);
    const float p = a.raw[i] / mx;  // M/main.cpp:521
    float o = p;
    if (a.sigma != 0.0) {
        // M/main.cpp:63-74 with Philox uniforms in (0,1) in place of rand()
        const uint4 u = philox4x32_10(make_uint4((uint32_t)r, a.stream_id + (uint32_t)s, 0u, 0u), a.key0, a.key1);
        const double u1 = ((double)u.x + 1.0) / 4294967297.0;
        const double u2 = ((double)u.y + 1.0) / 4294967297.0;
        const double z = sqrt(-2.0 * log(u1)) * sin(2.0 * 3.141592653589793238462643383279 * u2);
        const double nstar = (double)p + (0 + a.sigma * z);
        o = (float)nstar;
        if (nstar < 0) {
            const float pmin = __uint_as_float(a.stats[2 * s + 1]) / mx;
            o = (float)((double)pmin / 10);
        }
        if (nstar > 1.0) o = 1.0f;
    }
    a.out[i] = o;
}

__global__ __launch_bounds__(256) void k_pack_i16(const int16_t* __restrict__ src, int M, int NN,
                                                  uint16_t* __restrict__ dst)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= NN) return;
    uint32_t w[4] = {0u, 0u, 0u, 0u};
    for (int m = 0; m < M; m++) {
        const int x = src[(size_t)m * NN + v];
        const uint32_t u = x > 0 ? (uint32_t)x : 0u;
        w[m >> 1] |= (m & 1) ? (u << 16) : u;
    }
    reinterpret_cast<uint4*>(dst)[v] = make_uint4(w[0], w[1], w[2], w[3]);
}

__global__ __launch_bounds__(256) void k_pack_f32(const float* __restrict__ src, int M, int NN,
                                                  float* __restrict__ dst)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= NN) return;
    float r[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int m = 0; m < M; m++) r[m] = src[(size_t)m * NN + v];
    float4* d = reinterpret_cast<float4*>(dst) + (size_t)v * 2;
    d[0] = make_float4(r[0], r[1], r[2], r[3]);
    d[1] = make_float4(r[4], r[5], r[6], r[7]);
}

// Zero path integrals (and counts) of n rays.
__global__ __launch_bounds__(256) void k_trace_zero(float* __restrict__ L, int32_t* __restrict__ counts, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4* d = reinterpret_cast<float4*>(L) + (size_t)i * 2;
    d[0] = d[1] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (counts) counts[i] = 0;
}

// One voxel of the tracer's work copies: the first VB bytes of a packed
// voxel (two bytes per u16 material, four per float one, in whole pairs).
template <int VB>
struct alignas(VB % 16 == 0 ? 16 : VB % 8 == 0 ? 8 : 4) WorkVox {
    uint32_t w[VB / 4];
};

// The tracer's two work copies of the packed densities (IB bytes per voxel),
// padded by two voxels on every side (NP = N + 4 per row): yx[y + 2][x + 2]
// and xy[x + 2][y + 2] hold voxel (x, y) for x, y in [-1, N - 1], index -1
// reading voxel 0 as the reference's truncation does, and zeros elsewhere;
// by 32 x 32 tiles of the padded grid through LDS.  CLAMP: float densities
// below zero (and NaN) as 0, which is what they contribute
// (M/reprojection_TOMO.cpp:155), so the sums need no test.
template <int IB, int VB, bool CLAMP>
__global__ __launch_bounds__(256) void k_pack_copies(const char* __restrict__ in, WorkVox<VB>* __restrict__ yx,
                                                     WorkVox<VB>* __restrict__ xy, int N)
{
    static_assert(VB % 4 == 0 && VB <= IB, "a work voxel is a prefix of the packed voxel");
    __shared__ WorkVox<VB> tile[32][33];
    const int NP = N + 4;
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;  // padded coordinates
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int j = ty; j < 32; j += 8) {
        const int pr = r0 + j, pc = c0 + tx;
        const int y = pr - 2, x = pc - 2;
        WorkVox<VB> t;
#pragma unroll
        for (int q = 0; q < VB / 4; q++) t.w[q] = 0u;
        if (y >= -1 && y < N && x >= -1 && x < N)
            t = *reinterpret_cast<const WorkVox<VB>*>(in + ((size_t)max(y, 0) * N + max(x, 0)) * IB);
        if constexpr (CLAMP) {
#pragma unroll
            for (int q = 0; q < VB / 4; q++) t.w[q] = __float_as_uint(fmaxf(__uint_as_float(t.w[q]), 0.f));
        }
        tile[j][tx] = t;
        if (pr < NP && pc < NP) yx[(size_t)pr * NP + pc] = t;
    }
    __syncthreads();
    for (int i = ty; i < 32; i += 8) {
        const int pr = c0 + i, pc = r0 + tx;  // row x + 2, column y + 2
        if (pr < NP && pc < NP) xy[(size_t)pr * NP + pc] = tile[tx][i];
    }
}

template <int IB, int VB, bool CLAMP = false>
static void launch_pack_copies(const TraceArgs& a, hipStream_t s)
{
    const int NP = a.N + 4;
    const dim3 grid((unsigned)((NP + 31) / 32), (unsigned)((NP + 31) / 32));
    WorkVox<VB>* yx = reinterpret_cast<WorkVox<VB>*>(a.dens_t);
    hipLaunchKernelGGL((k_pack_copies<IB, VB, CLAMP>), grid, dim3(256), 0, s, reinterpret_cast<const char*>(a.dens), yx,
                       yx + (size_t)NP * NP, a.N);
}

// --------------------------------------------------------------- launchers

// Lanes per orbit: eight, so that the launch holds eight times as many waves
// as orbits/64 (121,800 orbits at 800 x 609 give ~15,200 waves); measured at
// 512^2 (u16, 64-lane workgroups): 2 lanes 0.621 ms, 4 0.538, 8 0.531, 16 0.600.
constexpr int kOrbitLanes = 8;

template <int M, int DT, int R>
static void launch_trace_rot(const TraceArgs& a, hipStream_t s)
{
    const long long lanes = (long long)(a.V / R) * a.W * kOrbitLanes;
    hipLaunchKernelGGL((k_trace_fwd_rot<M, DT, R, kOrbitLanes>), dim3((unsigned)((lanes + a.block - 1) / a.block)),
                       dim3(a.block), 0, s, a);
}

template <int M, int DT>
static vct_status launch_trace_seg(const TraceArgs& a, hipStream_t s)
{
    if (a.rot > 1) launch_pack_copies<DT == VCT_DENS_U16 ? 16 : 32, seg_voxel<M, DT>(), DT == VCT_DENS_F32>(a, s);
    const int base_views = a.rot > 1 ? a.V / a.rot : a.VT;
    const int ct = (a.W + kSegCh - 1) / kSegCh, sh = seg_shift(a.N, base_views, ct), vt = (1 << sh) / kSegCh;
    const dim3 grid((unsigned)((base_views + vt - 1) / vt * ct));
    const dim3 block(64 * kSegWaves);
    if (a.VT < a.V) {
        // an odd count's last view is not traced
        const size_t done = (size_t)a.VT * a.W, rest = (size_t)(a.V - a.VT) * a.W;
        hipLaunchKernelGGL(k_trace_zero, dim3((unsigned)((rest + 255) / 256)), dim3(256), 0, s, a.L + done * 8,
                           a.counts ? a.counts + done : nullptr, (int)rest);
    }
    if (base_views > 0) {
        const int words = (int)grid.x;
        const dim3 rgrid((unsigned)((words + 63) / 64));
#define VCT_SEG(RR)                                                                  \
    hipLaunchKernelGGL((k_trace_seg<M, DT, RR>), grid, block, 0, s, a, sh);          \
    hipLaunchKernelGGL((k_trace_redo<M, DT, RR>), rgrid, dim3(64 * RR), 0, s, a, words, sh);
        if (a.rot == 4) { VCT_SEG(4) }
        else if (a.rot == 2) { VCT_SEG(2) }
        else { VCT_SEG(1) }
#undef VCT_SEG
    }
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

template <int M>
static vct_status launch_trace_m(const TraceArgs& a, int dens_type, bool adjoint, hipStream_t s)
{
    const dim3 block(a.block);
    const dim3 grid((a.n_rays + a.block - 1) / a.block);
    const bool whole = a.ray_offset == 0 && a.n_rays == a.V * a.W;
    if (!adjoint && whole && seg_grid(a, dens_type == VCT_DENS_U16 ? seg_voxel<M, VCT_DENS_U16>() : seg_voxel<M, VCT_DENS_F32>()))
        return dens_type == VCT_DENS_U16 ? launch_trace_seg<M, VCT_DENS_U16>(a, s) : launch_trace_seg<M, VCT_DENS_F32>(a, s);
    if (!adjoint && whole && (a.rot == 4 || a.rot == 2)) {
        if (a.V % a.rot != 0 || a.N % 2 != 0 || a.VT != a.V || a.exact || a.rcheck || !a.dens_t)
            return set_error(VCT_ERR_INTERNAL, "orbit trace with V %d, N %d", a.V, a.N);
        // the orbit gathers read two padded work copies, [y][x] and [x][y]
        if (dens_type == VCT_DENS_U16) {
            if constexpr (M <= 6) launch_pack_copies<16, 12>(a, s);
            else launch_pack_copies<16, 16>(a, s);
        } else {
            launch_pack_copies<32, 32>(a, s);
        }
        if (dens_type == VCT_DENS_U16) {
            if (a.rot == 4) launch_trace_rot<M, VCT_DENS_U16, 4>(a, s);
            else launch_trace_rot<M, VCT_DENS_U16, 2>(a, s);
        } else {
            if (a.rot == 4) launch_trace_rot<M, VCT_DENS_F32, 4>(a, s);
            else launch_trace_rot<M, VCT_DENS_F32, 2>(a, s);
        }
    } else if (adjoint) {
        if (a.VT > 0) {
            const int ntx = (a.N + kAdjTile - 1) / kAdjTile, ntiles = ntx * ntx;
            const AdjointSplit sp = adjoint_split(ntiles, a.VT, a.W, a.adj_views);
            const int per_xcd = (ntiles * sp.chunks + 7) / 8;
            const int lanes = adjoint_lanes(M, ntiles, sp, a.W, std::min(a.N, kAdjTile) * a.D / a.ch_cm);
            hipLaunchKernelGGL((k_trace_adj_tile<M>), dim3(per_xcd * 8), dim3(lanes), 0, s, a, ntx, ntiles, sp.views,
                               per_xcd, seg_planes(a) ? 1 : 0);
        }
    } else if (!a.exact && a.n_rays <= INT_MAX / 8) {
        // (the exact option keeps the reference's order of the sums)
        const dim3 split((4 * a.n_rays + a.block - 1) / a.block);
        if (dens_type == VCT_DENS_U16) hipLaunchKernelGGL((k_trace_fwd<M, VCT_DENS_U16, 4>), split, block, 0, s, a);
        else hipLaunchKernelGGL((k_trace_fwd<M, VCT_DENS_F32, 4>), split, block, 0, s, a);
    } else if (dens_type == VCT_DENS_U16) {
        hipLaunchKernelGGL((k_trace_fwd<M, VCT_DENS_U16, 1>), grid, block, 0, s, a);
    } else {
        hipLaunchKernelGGL((k_trace_fwd<M, VCT_DENS_F32, 1>), grid, block, 0, s, a);
    }
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

bool trace_uses_block(const TraceArgs& a, int dens_type, int M)
{
    return !seg_grid(a, (dens_type == VCT_DENS_U16 ? 4 : 8) * ((M + 1) / 2));
}

size_t trace_redo_words(int V, int W)
{
    return (size_t)V * (size_t)((W + kSegCh - 1) / kSegCh);
}

vct_status launch_trace(const TraceArgs& a, int dens_type, int M, bool adjoint, hipStream_t s)
{
    if (a.n_rays <= 0) return VCT_OK;
    switch (M) {
    case 1: return launch_trace_m<1>(a, dens_type, adjoint, s);
    case 2: return launch_trace_m<2>(a, dens_type, adjoint, s);
    case 3: return launch_trace_m<3>(a, dens_type, adjoint, s);
    case 4: return launch_trace_m<4>(a, dens_type, adjoint, s);
    case 5: return launch_trace_m<5>(a, dens_type, adjoint, s);
    case 6: return launch_trace_m<6>(a, dens_type, adjoint, s);
    case 7: return launch_trace_m<7>(a, dens_type, adjoint, s);
    case 8: return launch_trace_m<8>(a, dens_type, adjoint, s);
    default: return set_error(VCT_ERR_ARG, "number of materials %d outside 1..8", M);
    }
}

template <int M>
static void launch_spectral_m(const SpectralArgs& a, hipStream_t s)
{
    const int nr = a.V * a.W;
    const int block = (long long)nr * a.S >= 128 * kSpecBlock ? kSpecBlock : 256;
    const dim3 grid((nr + block - 1) / block, a.S);
    if (a.dIdL)
        hipLaunchKernelGGL((k_spectral_grad<M>), grid, dim3(block), sizeof(float) * (size_t)a.NE * 9, s, a);
    else
        hipLaunchKernelGGL((k_spectral<M>), grid, dim3(block), sizeof(float) * SpecTable<M>::floats(a.NE), s, a);
}

vct_status launch_spectral(const SpectralArgs& a, hipStream_t s)
{
    if (a.NE <= 0 || a.NE > kMaxBins) return set_error(VCT_ERR_ARG, "NE=%d outside 1..%d", a.NE, kMaxBins);
    if (a.S <= 0 || a.S > 65535) return set_error(VCT_ERR_ARG, "n_spectra=%d invalid", a.S);
    switch (a.M) {
    case 1: launch_spectral_m<1>(a, s); break;
    case 2: launch_spectral_m<2>(a, s); break;
    case 3: launch_spectral_m<3>(a, s); break;
    case 4: launch_spectral_m<4>(a, s); break;
    case 5: launch_spectral_m<5>(a, s); break;
    case 6: launch_spectral_m<6>(a, s); break;
    case 7: launch_spectral_m<7>(a, s); break;
    case 8: launch_spectral_m<8>(a, s); break;
    default: return set_error(VCT_ERR_ARG, "number of materials %d outside 1..8", a.M);
    }
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

vct_status launch_stats_init(uint32_t* stats, int S, hipStream_t s)
{
    hipLaunchKernelGGL(k_stats_init, dim3((S + 63) / 64), dim3(64), 0, s, stats, S);
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

vct_status launch_minmax(const float* x, int n, uint32_t* stats, hipStream_t s)
{
    if (n <= 0) return set_error(VCT_ERR_ARG, "empty array");
    hipLaunchKernelGGL(k_minmax_init, dim3(1), dim3(1), 0, s, stats);
    const int blocks = min((n + 255) / 256, 2048);
    hipLaunchKernelGGL(k_minmax, dim3(blocks), dim3(256), 0, s, x, n, stats);
    hipLaunchKernelGGL(k_minmax_final, dim3(1), dim3(1), 0, s, stats);
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

vct_status launch_detector(const DetectorArgs& a, hipStream_t s)
{
    const long long total = (long long)a.n * a.S;
    if (total <= 0 || total > INT_MAX) return set_error(VCT_ERR_ARG, "detector size %lld invalid", total);
    hipLaunchKernelGGL(k_detector, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, a);
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

vct_status launch_pack_i16(const int16_t* src, int M, int N, uint16_t* dst, hipStream_t s)
{
    const int NN = N * N;
    hipLaunchKernelGGL(k_pack_i16, dim3((NN + 255) / 256), dim3(256), 0, s, src, M, NN, dst);
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

vct_status launch_pack_f32(const float* src, int M, int N, float* dst, hipStream_t s)
{
    const int NN = N * N;
    hipLaunchKernelGGL(k_pack_f32, dim3((NN + 255) / 256), dim3(256), 0, s, src, M, NN, dst);
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

}  // namespace vct
