// vct_npf.hip -- the npf side output of the MBFPA program for CDNA4 (gfx950):
// a pixel-driven, chord-weighted backprojection of a normalised sinogram
// (M/lengthproj_TOMO.cpp:14-185, called from M/main.cpp:407-419).
//
// k_lengthproj: one thread per pixel of a 16x16 tile.  Per view the thread forms the
// reference's chord length of the ray from the source through the pixel
// (:72-106), intersects that ray with the detector arc about the source
// (:109-131), converts the hit to a fractional channel with acos (:133-150),
// interpolates the view's row of the sinogram and adds sample * chord in
// float, views ascending (:152-170).  All geometry is FP64 in the
// reference's operation order (contraction off); the sinogram window
// (<= 2 MB) stays in L2/MALL.  The channel pitch and isocentre channel are
// the detector's (the plan's geometry); a window row may hold fewer channels
// (measured data keep 582 or fewer), and hits past its last channel take that
// channel's value (the reference, whose pitch is fixed by its 609-channel
// End_Channel, interpolates there with the narrower row as stride, i.e. reads
// the next row's first channels).  The reference also fills two per-pixel,
// per-view caches for its disabled iterative loop; they are not produced.
// k_lengthproj_fan: the same sums for the machine's own geometry, where the
// channel follows from the fan angle.
#include "vct_internal.h"

#include <cmath>

namespace vct {

constexpr int kNpfTile = 16;

// prepareMaskData, M/misc_TOMO.cpp:21-36
__device__ __forceinline__ bool npf_inside(const LengthprojArgs& a, int jx, int jy)
{
    const double mr = (double)(a.N - 1) / 2.0;
    return ((double)jy - mr) * ((double)jy - mr) + ((double)jx - mr) * ((double)jx - mr) <= mr * mr;
}
__device__ __forceinline__ double npf_y(const LengthprojArgs& a, int jy)
{
    return a.N * a.pix * 0.5 - (jy + 0.5) * a.pix;  // :56
}
__device__ __forceinline__ double npf_x(const LengthprojArgs& a, int jx)
{
    return -a.N * a.pix * 0.5 + (jx + 0.5) * a.pix;  // :61
}

// The term of window row j, view jr, for the pixel at (rx, ry), in the
// reference's operation order.
__device__ __forceinline__ float npf_term(const LengthprojArgs& a, double rx, double ry, int j, int jr)
{
    const double pix = a.pix, rz = a.rz, R = a.det_radius;
    const int last = a.pw - 1;  // the window's last channel
    const double c = a.cosT[jr], s = a.sinT[jr];
    const double sx = a.sid * s, sy = a.sid * c, sz = rz;
    const double yslope = fabs(ry - sy), xslope = fabs(rx - sx);
    double rr;
    if (xslope > yslope) {  // :84-92
        const double q0 = (rx - 0.5 * pix - sx) / (rx - sx);
        const double q1 = (rx + 0.5 * pix - sx) / (rx - sx);
        const double xx0 = rx - 0.5 * pix, xx1 = rx + 0.5 * pix;
        const double yy0 = q0 * (ry - sy) + sy, yy1 = q1 * (ry - sy) + sy;
        const double zz0 = q0 * (rz - sz) + sz, zz1 = q1 * (rz - sz) + sz;
        rr = sqrt((xx0 - xx1) * (xx0 - xx1) + (yy0 - yy1) * (yy0 - yy1) + (zz0 - zz1) * (zz0 - zz1));
    } else {  // :94-101, whose far end reuses yy0: xx1 == xx0
        const double yy0 = ry - 0.5 * pix, yy1 = ry + 0.5 * pix;
        const double q0 = (yy0 - sy) / (ry - sy);
        const double xx0 = q0 * (rx - sx) + sx, xx1 = xx0;
        const double zz0 = q0 * (rz - sz) + sz, zz1 = zz0;
        rr = sqrt((xx0 - xx1) * (xx0 - xx1) + (yy0 - yy1) * (yy0 - yy1) + (zz0 - zz1) * (zz0 - zz1));
    }
    // detector hit, :109-131
    const double dx = a.det_src_iso * s, dy = a.det_src_iso * c;
    const double aa = (sy - ry) / (sx - rx);
    const double bb = -sx * (sy - ry) / (sx - rx) + sy;
    const double A = 1.0 + aa * aa;
    const double B = 2.0 * aa * bb - 2.0 * aa * dy - 2.0 * dx;
    const double C = dx * dx + bb * bb + dy * dy - 2.0 * bb * dy - R * R;
    const double root = sqrt(B * B - 4.0 * A * C);
    const double px1 = (-B + root) / (2.0 * A), py1 = aa * px1 + bb;
    const double px2 = (-B - root) / (2.0 * A), py2 = aa * px2 + bb;
    const bool second = px1 * px1 + py1 * py1 > px2 * px2 + py2 * py2;
    const double px = second ? px2 : px1, py = second ? py2 : py1;
    // fractional channel, :133-150
    const double ox = -a.iso_det * s, oy = -a.iso_det * c;
    const double dis = (px - ox) * (px - ox) + (py - oy) * (py - oy);
    const double angle = acos(1.0 - dis / (2.0 * R * R));
    const double rot_px = px * c - py * s;
    const double dj = rot_px > 0.0 ? a.iso_channel - angle / a.delta : a.iso_channel + angle / a.delta;
    const float* row = a.proj + (size_t)j * a.pw;
    double np;
    if (0 <= dj && dj < last) {  // :152-158
        const int i0 = (int)dj;
        const double w = dj - (double)i0;
        np = (1.0 - w) * row[i0] + w * row[i0 + 1];
    } else if (0 > dj) {
        np = row[0];
    } else if (dj >= last) {
        np = row[last];
    } else {
        return 0.f;  // NaN channel: the reference adds nothing (the sum is never -0, so +0 leaves it)
    }
    return (float)(np * rr);
}

__global__ __launch_bounds__(256) void k_lengthproj(LengthprojArgs a)
{
    const int jx = blockIdx.x * kNpfTile + (threadIdx.x & (kNpfTile - 1));
    const int jy = blockIdx.y * kNpfTile + threadIdx.x / kNpfTile;
    if (jx >= a.N || jy >= a.N) return;
    float acc = 0.f;
    if (npf_inside(a, jx, jy)) {
        const double ry = npf_y(a, jy), rx = npf_x(a, jx);
        for (int j = 0; j < a.count; j++) {
            int jr = a.base + j;
            if (jr >= a.V) jr -= a.V;  // :70-71
            acc += npf_term(a, rx, ry, j, jr);
        }
    }
    a.npf[(size_t)jy * a.N + jx] = acc;
}

// Coefficients of atan(t)/t in t^2, |t| <= 0.5, highest power first: the
// interpolant at 13 Chebyshev nodes that the backprojection's exact form uses
// (<= 1.2 ulp).  The launcher passes them over the channel pitch.
static const double kAtan[kNpfPoly] = {0.010030841489968486, -0.027302779603074177, 0.041775850326747944,
                                       -0.05118531938647954, 0.05857435765165694,   -0.06663667844183857,
                                       0.07692057989976618,  -0.09090895058092312,  0.11111110602305971,
                                       -0.14285714274692063, 0.19999999999875542,   -0.3333333333333278, 1.0};
__device__ __forceinline__ double rcp_refined(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    r = __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
    return __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
}
// 1/sqrt(x) to a few ulp: the hardware estimate and two Newton steps
__device__ __forceinline__ double rsq_refined(double x)
{
    double r = __builtin_amdgcn_rsq(x);
    r = __builtin_fma(0.5 * r, __builtin_fma(-x * r, r, 1.0), r);
    return __builtin_fma(0.5 * r, __builtin_fma(-x * r, r, 1.0), r);
}

// The machine's geometry: the detector arc is centred on the source (radius R)
// and the isocentre's hit lies on it (sid + iso_det = R).  In the frame turned
// by the view the pixel is at (X, Y), the source at (0, sid); the hit is
// R (sin g, ..) with tan g = X / (sid - Y), its chord from the isocentre's
// hit subtends |g|, so the channel is isocentre - g / pitch: one reciprocal and
// one polynomial in place of the circle's quadratic (four divisions, a square
// root) and acos.  The pixel's chord is pix on the steep side (the reference's
// far end reuses the near point) and pix |P - S| / |rx - sx| on the other.
// Terms agree with the reference's to ~1e-12 relative, below their rounding to
// float; a ray within 1e-4 of the image's y direction, where the reference's
// line slope (and with it its own rounding) grows without bound, takes its
// expression.
//
// FP64 issue bounds both forms (about 55 vector instructions per pixel-view
// here): 2.00 -> 0.44 ms at 512^2, 800 views.  Four waves share 64 pixels: each
// computes kNpfChunk views of a round into LDS and the first adds them, views
// ascending.  One pixel per lane with all its views took 0.50 ms (every
// workgroup is resident from the start, and those on the mask's edge leave
// their CU idle); with 4 times the workgroups the chip fills as they end, and
// small images have waves enough.
constexpr int kNpfWaves = 4, kNpfChunk = 4;

__global__ __launch_bounds__(64 * kNpfWaves) void k_lengthproj_fan(LengthprojArgs a)
{
    constexpr int K = kNpfChunk;
    __shared__ float part[kNpfWaves * K][64];
    const int p = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int jx = blockIdx.x * 8 + (p & 7), jy = blockIdx.y * 8 + (p >> 3);
    const bool in_img = jx < a.N && jy < a.N;
    const bool inside = in_img && npf_inside(a, jx, jy);
    const double ry = npf_y(a, jy), rx = npf_x(a, jx);
    const int last = a.pw - 1;
    float acc = 0.f;
    // terms of window rows j0 .. j0 + K - 1 (zero past the window)
    auto terms = [&](int j0, float (&out)[K]) {
        float t0[K], t1[K];
        double w[K], rr[K];
        bool in[K];
        int odd = 0;
#pragma unroll
        for (int u = 0; u < K; u++) {
            const int j = min(j0 + u, a.count - 1);
            int jr = a.base + j;
            if (jr >= a.V) jr -= a.V;
            const double c = a.cosT[jr], s = a.sinT[jr];
            const double X = __builtin_fma(rx, c, -(ry * s));
            const double den = __builtin_fma(-rx, s, __builtin_fma(-ry, c, a.sid));
            const double tg = X * rcp_refined(den), q = tg * tg;
            double p = a.poly[0];
#pragma unroll
            for (int i = 1; i < kNpfPoly; i++) p = __builtin_fma(p, q, a.poly[i]);
            const double dj = __builtin_fma(-tg, p, a.iso_channel);
            // (rounded as the reference does: a pixel on the diagonal of the
            // source takes the side that its rounding gives)
            const double ex = rx - a.sid * s, ey = ry - a.sid * c;
            const double h = ex * ex, g = __builtin_fma(ey, ey, h);
            odd |= (fabs(ex) < 1.0e-4 * fabs(ey) && j0 + u < a.count) ? 1 << u : 0;
            rr[u] = fabs(ex) > fabs(ey) ? a.pix * (g * rsq_refined(g * h)) : a.pix;
            in[u] = dj >= 0.0 && dj < (double)last;
            const int i0 = min(max((int)dj, 0), last);
            w[u] = dj - (double)i0;
            // (scalar base of the row, the lane's channel as a 32-bit offset)
            const float* row = a.proj + (size_t)j * a.pw;
            t0[u] = row[(uint32_t)i0];
            t1[u] = row[(uint32_t)(in[u] ? i0 + 1 : i0)];
        }
#pragma unroll
        for (int u = 0; u < K; u++) {
            const double np = (1.0 - w[u]) * t0[u] + w[u] * t1[u];
            out[u] = j0 + u < a.count ? (float)((in[u] ? np : (double)t0[u]) * rr[u]) : 0.f;
        }
        if (__any(odd)) {  // rare: one copy of the reference's expression
#pragma unroll 1
            for (int u = 0; u < K; u++) {
                if (!(odd >> u & 1)) continue;
                int jr = a.base + j0 + u;
                if (jr >= a.V) jr -= a.V;
                const float t = npf_term(a, rx, ry, j0 + u, jr);
#pragma unroll
                for (int x = 0; x < K; x++) out[x] = x == u ? t : out[x];
            }
        }
    };
    for (int j0 = 0; j0 < a.count; j0 += kNpfWaves * K) {
        float o[K];
#pragma unroll
        for (int u = 0; u < K; u++) o[u] = 0.f;
        if (inside) terms(j0 + wave * K, o);
#pragma unroll
        for (int u = 0; u < K; u++) part[wave * K + u][p] = o[u];
        __syncthreads();
        if (wave == 0) {
#pragma unroll
            for (int u = 0; u < kNpfWaves * K; u++) acc += part[u][p];
        }
        __syncthreads();
    }
    if (wave == 0 && in_img) a.npf[(size_t)jy * a.N + jx] = acc;
}

// The fan form needs the machine's geometry (above; sid + iso_det equals R to
// rounding) and pixels seen from the source within |tan| <= 0.5 (the
// polynomial's range).
static bool npf_fan(const LengthprojArgs& a)
{
    const double r = (a.N - 1) * 0.5 * a.pix;
    return a.det_src_iso == a.sid && std::fabs(a.sid + a.iso_det - a.det_radius) <= 1.0e-13 * a.det_radius &&
           r < a.sid && r / std::sqrt(a.sid * a.sid - r * r) <= 0.49;
}

vct_status launch_lengthproj(const LengthprojArgs& args, hipStream_t s)
{
    LengthprojArgs a = args;
    for (int i = 0; i < kNpfPoly; i++) a.poly[i] = kAtan[i] / a.delta;
    const dim3 grid((a.N + kNpfTile - 1) / kNpfTile, (a.N + kNpfTile - 1) / kNpfTile);
    const dim3 small((a.N + 7) / 8, (a.N + 7) / 8);
    if (npf_fan(a)) hipLaunchKernelGGL(k_lengthproj_fan, small, dim3(64 * kNpfWaves), 0, s, a);
    else hipLaunchKernelGGL(k_lengthproj, grid, dim3(kNpfTile * kNpfTile), 0, s, a);
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

}  // namespace vct
