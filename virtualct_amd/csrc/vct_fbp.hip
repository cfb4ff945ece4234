// vct_fbp.hip -- fan-beam FBP for CDNA4 (gfx950).
//
//   k_filter_prep  q[r][k] = -ln p[r][k] * sid * cos((k - W/2) * dbeta), the
//                  reference's per-channel pre-weight (F/filterSinogramTOMO.cpp:236-242),
//                  written straight into the register layout of the MFMA A
//                  operand (zero padded to Kp).
//   k_filter_gemm  fltd = q . C'^T with v_mfma_f32_32x32x2f32, where
//                  C'[m][k] = C[m][k] * dbeta is the reference's filter
//                  matrix (prepareConstMap, F/filterSinogramTOMO.cpp:9-138;
//                  Shepp-Logan or Ram-Lak).  Its rows are Toeplitz except the
//                  41 edge rows that prepareConstMap renormalises, so most
//                  column tiles read C' from an LDS copy of its Toeplitz
//                  generator and only edge tiles read the packed matrix.  A
//                  workgroup owns a 32x32 output tile, one wave per quarter
//                  of K; the quarters meet in LDS.
//   k_backproject  pixel-driven fan backprojection
//                  (F/reconstructImageTOMO.cpp:46-100): a 16x16 pixel tile per
//                  workgroup, one lane per pixel, the view loop uniform over
//                  the wave, FP64 geometry and the reference's float
//                  accumulation order.
//   k_backproject_multi  the same for 2..16 sinograms of one geometry per
//                  lane, sharing each pixel-view's geometry.
//   k_backproject_sym  one sinogram by orbits of the quarter turn: each
//                  pixel-view geometry serves four pixels (views a multiple
//                  of 4, N even; sums in another order).
//   k_backproject_lone  one sinogram on other grids and view counts: orbits of
//                  four, two or one pixels, FP64 sums.
#include "vct_internal.h"

#include <algorithm>
#include <climits>
#include <cmath>

namespace vct {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kBpTile = 16;   // pixel tile edge
constexpr int kBpSinos = 16;  // most sinograms per lane in k_backproject_multi
constexpr long long kBpMinLanes = 1 << 18;  // lanes a backprojection launch keeps (4 waves per SIMD)

__device__ __forceinline__ int trunc_i32_bp(double v)
{
    return (v > -2147483649.0 && v < 2147483648.0) ? (int)v : INT_MIN;
}

// Packed operand index: tile (32 rows or columns), K position k, row/col in
// tile rr.  Lane l = rr + 32*(k&1) holds step t = k>>1; four consecutive
// steps share one float4.
__host__ __device__ __forceinline__ size_t pack_index(int tile, int k, int rr, int Kp)
{
    const int t = k >> 1, hi = k & 1;
    const int q = t >> 2, j = t & 3;
    const int l = rr + 32 * hi;
    return ((((size_t)tile * (Kp / 8) + q) * 64 + l) * 4) + j;
}

// Single-precision log rounded from the double log: the correctly rounded
// logf up to double rounding, which is what the C library's logf returns on
// all but ~0.06% of sinogram values (the device logf differs on about a third).
__device__ __forceinline__ float logf_rounded(float x) { return (float)log((double)x); }

// One workgroup per 32 rows x 32 channels: the rows are read along the
// channels (coalesced), pre-weighted into LDS, and written out as the 4 x 64
// float4 of their packed operand block (contiguous), so the writes are whole
// lines instead of 4-byte scatters.
__global__ __launch_bounds__(256) void k_filter_prep(FilterPrepArgs a)
{
    __shared__ float t[32][33];
    const int kc = blockIdx.x, tr = blockIdx.y;
    for (int e = threadIdx.x; e < 32 * 32; e += blockDim.x) {
        const int rr = e >> 5, kk = e & 31;
        const int r = tr * 32 + rr, k = kc * 32 + kk;
        float v = 0.f;
        if (r < a.R && k < a.W) {
            const double p = a.proj[(size_t)r * a.W + k];
            double y;
            if (a.bhc) {
                // beam-hardening correction, M/beam_hardening_correction.cpp:51-55 (whose
                // log of a float is the single-precision overload)
                y = -(double)logf_rounded((float)p);
                y = fabs(y) + (a.bhc_alpha * pow(fabs(y), a.bhc_beta));
            } else {
                y = -log(p);
            }
            v = (float)(y * a.coeff[k]);
        }
        t[rr][kk] = v;
    }
    __syncthreads();
    // float4 (q, l) of the tile holds k = 8q + 2j + (l >> 5), j = 0..3, of
    // row l & 31 (pack_index)
    const int i = threadIdx.x, qq = i >> 6, l = i & 63, rr = l & 31, hi = l >> 5;
    const float* row = t[rr] + 8 * qq + hi;
    float4* out = reinterpret_cast<float4*>(a.apk) + ((size_t)tr * (a.Kp / 8) + kc * 4 + qq) * 64 + l;
    *out = make_float4(row[0], row[2], row[4], row[6]);
}

constexpr int kFiltWaves = 4;  // K quarters of an output tile, one wave each
constexpr int kFiltU = 10;     // quads (4 MFMA steps each) of A that a lane loads one chunk ahead
constexpr int kFiltStrip = 4;  // column tiles per workgroup of a tall product

// NT 32x32 output tiles side by side per workgroup; wave w sums the w-th quarter
// of K of each, and the quarters meet in LDS in a fixed order.  Operands are the
// pre-packed register order: lane l = i + 32*h holds row/column i at
// k = 8q + 2j + h in element j of float4 q.  Every lane loads a whole chunk of
// A (and, NT = 1, of B) before the last chunk's MFMAs run, so that 10 loads or
// more are in flight per lane.
//
// B is the filter matrix.  For a column tile whose rows are not renormalised
// (edge_lo < m < edge_hi) it is Toeplitz, B[k][m] = toep[m - k + Kp - 1]: the
// workgroup copies its tiles' window of the generator into LDS and reads B
// from there, so only the few edge tiles read the packed matrix from memory.
//
// NT = 1 for a single sinogram, whose 500 tiles of 80 MFMAs a wave need every
// wave they can get; a tall product (stacked sinograms) re-read A once per column tile and
// was bound by that, so there an A quad serves NT tiles.  Every output is the
// same sum in the same order for any NT.  Prep and product of 96 and 12
// sinograms of 800 x 609: NT = 1 1160 and 155 us, 2 1050 and 137, 4 926 and 123,
// 5 963 and 141 (the product then at 80 TFLOP/s); below 2000 tiles one per workgroup
// is as fast or faster (2 sinograms 32 and 31 us, 4 of 300 channels 23 and 27).
//
// Workgroups are dealt to XCDs in contiguous row-major ranges (workgroup g runs
// on XCD g % 8), so an XCD reads about an eighth of A, once, into its L2.
template <int NT>
__global__ __launch_bounds__(64 * kFiltWaves) void k_filter_gemm(FilterGemmArgs a, int ct, int cs, int nitems, int per_xcd)
{
    constexpr int U = NT == 1 ? kFiltU : kFiltU / 2;
    extern __shared__ float tw[];  // Toeplitz window, Kp + 32 NT - 1 floats
    __shared__ float part[kFiltWaves][16][64];
    const int xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
    const int item = xcd * per_xcd + slot;
    if (slot >= per_xcd || item >= nitems) return;  // the whole workgroup
    const int tr = item / cs, tc0 = (item - tr * cs) * NT;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int Q = a.Kp / 8, Qw = Q / kFiltWaves;
    const int qb = wave * Qw, qe = qb + Qw;
    const int nt = min(NT, ct - tc0);
    bool toep[NT], any = false;  // uniform over the workgroup
#pragma unroll
    for (int n = 0; n < NT; n++) {
        const int m0 = (tc0 + n) * 32;
        toep[n] = n < nt && m0 > a.edge_lo && m0 + 31 < a.edge_hi;
        any = any || toep[n];
    }
    if (any) {
        for (int j = threadIdx.x; j < a.Kp - 1 + 32 * nt; j += blockDim.x) tw[j] = a.toep[32 * tc0 + j];
        __syncthreads();
    }
    const float4* A = reinterpret_cast<const float4*>(a.apk) + ((size_t)tr * Q) * 64 + lane;
    const float4* B = reinterpret_cast<const float4*>(a.bpk) + ((size_t)tc0 * Q) * 64 + lane;
    // window index of B[k = 0] for this lane: column m = 32 tc + (lane & 31), k = lane >> 5
    const int t0 = (lane & 31) - (lane >> 5) + a.Kp - 1;
    auto b_quad = [&](int n, int q) {
        if (toep[n]) {
            const int t = t0 + 32 * n - 8 * q;
            return make_float4(tw[t], tw[t - 2], tw[t - 4], tw[t - 6]);
        }
        return B[((size_t)n * Q + q) * 64];
    };
    floatx16 acc[NT];
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[n][i] = 0.f;
    auto quad = [&](floatx16& c, const float4& x, const float4& y) {
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(x.x, y.x, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(x.y, y.y, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(x.z, y.z, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(x.w, y.w, c, 0, 0, 0);
    };
    float4 ca[U], cb[U];
#pragma unroll
    for (int u = 0; u < U; u++)
        if (qb + u < qe) {
            ca[u] = A[(size_t)(qb + u) * 64];
            if (NT == 1) cb[u] = b_quad(0, qb + u);
        }
    for (int qs = qb; qs < qe; qs += U) {
        float4 na[U], nb[U];
#pragma unroll
        for (int u = 0; u < U; u++)
            if (qs + U + u < qe) {
                na[u] = A[(size_t)(qs + U + u) * 64];
                if (NT == 1) nb[u] = b_quad(0, qs + U + u);
            }
        if constexpr (NT == 1) {
#pragma unroll
            for (int u = 0; u < U; u++)
                if (qs + u < qe) quad(acc[0], ca[u], cb[u]);
        } else {
#pragma unroll
            for (int n = 0; n < NT; n++) {
                if (n >= nt) break;
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (qs + u < qe) cb[u] = b_quad(n, qs + u);
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (qs + u < qe) quad(acc[n], ca[u], cb[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            ca[u] = na[u];
            if (NT == 1) cb[u] = nb[u];
        }
    }
    // each wave adds and writes a quarter of the rows of a tile
#pragma unroll
    for (int n = 0; n < NT; n++) {
        if (n >= nt) break;
        if (n > 0) __syncthreads();
#pragma unroll
        for (int i = 0; i < 16; i++) part[wave][i][lane] = acc[n][i];
        __syncthreads();
        const int col = (tc0 + n) * 32 + (lane & 31);
#pragma unroll
        for (int ii = 0; ii < 16 / kFiltWaves; ii++) {
            const int i = wave * (16 / kFiltWaves) + ii;
            const int row = tr * 32 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
            float v = part[0][i][lane];
#pragma unroll
            for (int w = 1; w < kFiltWaves; w++) v += part[w][i][lane];
            if (a.in_mode && (v < 1000.0f || v > 300000.0f)) v = 0.f;  // :250-255
            if (row < a.R && col < a.W) a.out[(size_t)row * a.W + col] = v;
        }
    }
}

// atan(t) for |t| <= 0.5 as t * P(t^2), P of degree 12: the interpolant of
// atan(sqrt(u))/sqrt(u) at 13 Chebyshev nodes of [0, 0.25], computed in 50-digit
// arithmetic (relative error 4e-18 before rounding; <= 1.2 ulp evaluated in
// FP64 over |t| <= 0.5).  Masked pixels see |t| <= tan(asin(r_mask / sid))
// (0.32 for the reference geometry); larger |t| take the library atan.
constexpr double kAtanSmall[13] = {
    0.010030841489968486, -0.027302779603074177, 0.041775850326747944, -0.05118531938647954,
    0.05857435765165694, -0.06663667844183857, 0.07692057989976618, -0.09090895058092312,
    0.11111110602305971, -0.14285714274692063, 0.19999999999875542, -0.3333333333333278, 1.0};
__device__ __forceinline__ double atan_small(double t)
{
    const double u = t * t;
    double p = kAtanSmall[0];
#pragma unroll
    for (int i = 1; i < 13; i++) p = __builtin_fma(p, u, kAtanSmall[i]);
    return t * p;
}

// 1/x to ~1 ulp: hardware estimate + two Newton steps.
__device__ __forceinline__ double rcp_f64(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    double e = __builtin_fma(-x, r, 1.0);
    r = __builtin_fma(r, e, r);
    e = __builtin_fma(-x, r, 1.0);
    return __builtin_fma(r, e, r);
}

// Coefficients of atan(t)/t for |t| <= 0.5, highest power of t^2 first
// (Chebyshev interpolant of degree 8 on [0, 0.25]): error below 2.5e-13 rad, a
// 2e-10 channel shift of the detector coordinate at 0.326 rad over 304
// channels.  The launchers pass them times the channels per radian (poly), so
// a channel takes no further product and the kernels read them as scalars.
static const double kAtanSym[kBpPoly] = {0.023298796324010433,  -0.05296597132474749, 0.07378028372611917,
                                         -0.09047114852983332,  0.1110744933786942,   -0.1428554012478447,
                                         0.19999995815529828,   -0.3333333329437766,  0.9999999999993997};
// Largest |tan(gamma)| of a masked pixel, the tangent from the source to the
// mask circle of radius r (pixel centres lie within mask_r pitches), beyond
// the polynomials' range; also for a degenerate geometry, whose NaN channels
// only the wide form tests for.
static bool bp_wide(const BackprojArgs& a)
{
    const double r = a.mask_r * a.pix;
    return a.degenerate || !(r < a.sid) || r / std::sqrt(a.sid * a.sid - r * r) > 0.49;
}

static void set_poly(BackprojArgs& a)
{
    for (int i = 0; i < kBpPoly; i++) a.poly[i] = kAtanSym[i] * a.inv_dbeta_ch;
}

// The exact order (VCT_OPT_EXACT_BACKPROJECT).  One lane per pixel, a 16x16
// pixel tile per workgroup.  The view loop is the same on every lane of a wave, so each view's cos/sin and the base of its
// filtered-sinogram row are scalar loads, and four views are unrolled so that
// their geometry and gathers overlap.  The float accumulation adds the views
// in the reference's order (F/reconstructImageTOMO.cpp:57-95); the filtered
// sinogram (1.95 MB at 800 x 609) is read through L2 without staging.
//
// WIDE: some masked pixel may see |tan(gamma)| > 0.5, beyond the polynomial;
// those take the library atan.  The host picks the variant from the bound
// |tan(gamma)| <= r / sqrt(sid^2 - r^2) over the mask radius r; without the
// fallback the view loop has no branch.
template <bool WIDE>
__global__ __launch_bounds__(kBpTile * kBpTile) void k_backproject(BackprojArgs a)
{
    const int tx = threadIdx.x & (kBpTile - 1), ty = threadIdx.x / kBpTile;
    const int x = blockIdx.x * kBpTile + tx;
    const int y = blockIdx.y * kBpTile + ty;
    const int s = blockIdx.z;
    const float* fl = a.fltd + (size_t)s * a.V * a.W;
    const bool in_img = x < a.N && y < a.N;
    // prepareMaskData, F/misc.cpp:20-36
    const double dyc = (double)y - a.mask_r, dxc = (double)x - a.mask_r;
    const bool masked = in_img && (dyc * dyc + dxc * dxc <= a.mask_r2);
    const double xx = -(x - a.center) * a.pix;  // :52-53
    const double yy = -(y - a.center) * a.pix;
    float acc = 0.f;
    if (masked) {
#pragma unroll 4
        for (int v = 0; v < a.use_views; v++) {
            const double c = a.cosT[v], sn = a.sinT[v];
            const double X = xx * c + yy * sn;
            const double Y = -xx * sn + yy * c;
            const double den = a.sid - Y;
            const double L2 = den * den + X * X;
            const double tg = X * rcp_f64(den);
            double gam = atan_small(tg);
            if (WIDE && fabs(tg) > 0.5) gam = atan(X / den);
            const double fGAM = gam * a.inv_dbeta_ch + a.cent;
            const int GAM = trunc_i32_bp(fGAM);
            const double w = fGAM - GAM;
            const bool ok = GAM >= 0 && GAM < a.W - 1;
            const float* row = fl + (size_t)v * a.W + (ok ? GAM : 0);
            // the reference's sum is 1.0 * sum1 + 0.0 * 0 (:92), which only turns
            // -0 into +0; acc is never -0 (it starts at +0, and x + (-x) is +0),
            // and acc + (-0) = acc + (+0) = acc, so the add is left out
            const double sum = (1 - w) * row[0] + w * row[1];
            const float term = (float)(rcp_f64(L2) * sum * a.dbeta_view * a.xfactor);
            acc = ok ? acc + term : acc;
        }
    }
    if (in_img) a.img[((size_t)s * a.N + y) * a.N + x] = acc;
}

// The sinogram-independent part of one pixel-view: detector weights, 1/L^2,
// whether the bin pair is on the detector, and its first bin (0 if it is not).
struct BpView {
    double w, w0, rL2;
    float w1s, w0s;  // FW: the two interpolation weights times 1/L^2 and the view step, in float
    int col;
    bool ok;
};

// FW: the float-weight form (the degree-8 atan, 1/L^2 in float), whose
// terms differ from the exact ones by ~1e-7 relative.  Its geometry stays FP64
// but takes fused multiply-adds where the exact form repeats the reference's
// separate roundings, the source distance sid - Y in one pair of them, and the
// bin without the range test of the cast (|gamma| < pi / 2 keeps it in range;
// WIDE fields hold pixels level with the source, where den = 0 makes tg NaN or
// infinite: the library atan of X / den and the tested cast put them off the
// detector as the exact form does, X = den = 0 included).
// About 30 instead of 45 vector instructions per geometry, and per sinogram
// three instead of four (a branch in place of a select): 512^2 x 800, one
// sinogram in orbits 0.124 -> 0.106 ms, 12 per lane 1.12 -> 0.93 ms.
template <bool WIDE, bool FW = false>
__device__ __forceinline__ BpView bp_view(const BackprojArgs& a, double xx, double yy, int v)
{
    const double c = a.cosT[v], sn = a.sinT[v];
    BpView g;
    if constexpr (FW) {
        const double X = __builtin_fma(xx, c, yy * sn);
        const double den = __builtin_fma(xx, sn, __builtin_fma(-yy, c, a.sid));
        const double L2 = __builtin_fma(den, den, X * X);
        // one Newton step on the reciprocal estimate: within ~11 ulp of the
        // quotient, a 1e-12 channel shift
        const double r = __builtin_amdgcn_rcp(den);
        const double tg = X * __builtin_fma(r, __builtin_fma(-den, r, 1.0), r);
        const double u = tg * tg;
        double p = a.poly[0];
#pragma unroll
        for (int i = 1; i < kBpPoly; i++) p = __builtin_fma(p, u, a.poly[i]);
        double fGAM = __builtin_fma(tg, p, a.cent);
        if (WIDE && !(fabs(tg) <= 0.5)) fGAM = __builtin_fma(atan(X / den), a.inv_dbeta_ch, a.cent);
        const int GAM = WIDE ? trunc_i32_bp(fGAM) : (int)fGAM;
        // (1 - w in FP64: both weights keep 24 bits where they are small)
        const double w = fGAM - GAM;
        const float sf = __builtin_amdgcn_rcpf((float)L2) * (float)(a.dbeta_view * a.xfactor);
        g.w1s = (float)w * sf;
        g.w0s = (float)(1.0 - w) * sf;
        g.ok = (unsigned)GAM < (unsigned)(a.W - 1);
        g.col = g.ok ? GAM : 0;
    } else {
        const double X = xx * c + yy * sn;
        const double Y = -xx * sn + yy * c;
        const double den = a.sid - Y;
        const double L2 = den * den + X * X;
        const double tg = X * rcp_f64(den);
        double gam = atan_small(tg);
        if (WIDE && fabs(tg) > 0.5) gam = atan(X / den);
        const double fGAM = gam * a.inv_dbeta_ch + a.cent;
        const int GAM = trunc_i32_bp(fGAM);
        g.w = fGAM - GAM;
        g.w0 = 1 - g.w;
        g.rL2 = rcp_f64(L2);
        g.ok = GAM >= 0 && GAM < a.W - 1;
        g.col = g.ok ? GAM : 0;
    }
    return g;
}

// k_backproject for K >= 2 sinograms of the same geometry per lane.  The pixel-view geometry (X,
// Y, L^2, gamma, the detector bin and its weights) does not depend on the
// sinogram, so a lane computes it once and applies it to K sinograms, each
// with the single-sinogram expression; the images are bit-identical for
// every K.  Workgroup z covers sinograms K*z ... K*z + K - 1; past S the
// lane re-reads sinogram S - 1 and stores nothing.  bp_multi_tile is one
// tile (bx, by) of workgroup z = bz.  FW (float weights, the default unless
// the plan asks for the exact backprojection): the interpolation and
// distance weights of a term are computed in the float-weight form of
// bp_view and applied in float, as in k_backproject_sym (within ~1e-6 of
// the exact terms); otherwise every term is the single-sinogram FP64
// expression and the images equal k_backproject's bit for bit.
// IL (K even): a.fltd holds the sinograms interleaved in slices of K,
// [S/K][V][W][K] (k_interleave_sinos), so the K tap pairs of a pixel-view are
// 2K contiguous floats, read as K/2 16-byte loads (8-byte aligned where K is
// no multiple of 4) instead of 2K 4-byte ones; the same values, so the same
// images.  Narrow slices leave registers for U views at once, whose geometry
// chains and gathers overlap: each pixel adds its views one after the other,
// so at 4 waves per SIMD and below the chain's latency bounds the kernel.  One
// view per set -> U: K = 2 at 128^2 x 800 views 251 -> 143 us, K = 4 at 300^2
// 215 -> 194, K = 12 at 768^2 1214 -> 1105; four per set lose what they gain
// from K = 4 on (registers).  Wide slices are bound by the L1's 64 bytes per
// clock: K = 12 at 512^2, 48 us per image.
template <bool WIDE, int K, bool FW, bool IL = false>
__device__ __forceinline__ void bp_multi_tile(const BackprojArgs& a, int S, int bx, int by, int bz)
{
    constexpr int U = !IL || K > 12 ? 1 : K == 2 ? 4 : 2;
    static_assert(!IL || K % 2 == 0, "interleaved slices hold an even number of sinograms");
    const double dbx = a.dbeta_view * a.xfactor;
    const int tx = threadIdx.x & (kBpTile - 1), ty = threadIdx.x / kBpTile;
    const int x = bx * kBpTile + tx;
    const int y = by * kBpTile + ty;
    const int s0 = bz * K;
    const float* fl[K];
#pragma unroll
    for (int k = 0; k < K; k++) fl[k] = a.fltd + (size_t)min(s0 + k, S - 1) * a.V * a.W;
    // IL: the tap pairs of view v's bin pair col are floats [o K, o K + 2K),
    // o = v W + col <= V W - 2, of slice bz, so they stay inside the slice
    const float* slice = a.fltd + (size_t)bz * a.V * a.W * K;
    auto taps = [&](int v, const BpView& g, float (&t0)[K], float (&t1)[K]) {
        // scalar base of the view's rows, the lane's bin as a 32-bit offset
        const uint32_t row = (uint32_t)(v * a.W);
        const uint32_t col = (uint32_t)g.col;
        if constexpr (IL) {
            struct alignas(K % 4 == 0 ? 16 : 8) Four { float v[4]; };
            const Four* q = reinterpret_cast<const Four*>(slice + (size_t)row * K + col * (uint32_t)K);
#pragma unroll
            for (int h = 0; h < K / 2; h++) {
                const Four u = q[h];
#pragma unroll
                for (int j = 0; j < 4; j++) (4 * h + j < K ? t0[4 * h + j] : t1[4 * h + j - K]) = u.v[j];
            }
        } else {
#pragma unroll
            for (int k = 0; k < K; k++) {
                // (one pointer: col + 1 as a 32-bit index may wrap, and the pair
                // would be two loads, each of which spreads over as many lines
                // where pixels are wider than channels: 256^2 x 800 views, 13
                // sinograms, 379 us with one load, 599 with two)
                const float* p = fl[k] + row + col;
                t0[k] = p[0];
                t1[k] = p[1];
            }
        }
    };
    const bool in_img = x < a.N && y < a.N;
    // prepareMaskData, F/misc.cpp:20-36
    const double dyc = (double)y - a.mask_r, dxc = (double)x - a.mask_r;
    const bool masked = in_img && (dyc * dyc + dxc * dxc <= a.mask_r2);
    const double xx = -(x - a.center) * a.pix;  // :52-53
    const double yy = -(y - a.center) * a.pix;
    float acc[K];
#pragma unroll
    for (int k = 0; k < K; k++) acc[k] = 0.f;
    if (masked && a.use_views > 0) {
        // software pipeline: the geometry and gathers of view v + 1 are
        // issued before the terms of view v are summed (the last view loads
        // itself again), so the gathers' latency overlaps the arithmetic
        auto add = [&](const BpView& g, const float (&t0)[K], const float (&t1)[K]) {
            if constexpr (FW) {
                // (a branch, not a select per sinogram: nearly always every
                // lane of the wave sees the detector)
                if (g.ok) {
#pragma unroll
                    for (int k = 0; k < K; k++) acc[k] += fmaf(g.w1s, t1[k], g.w0s * t0[k]);
                }
            } else {
#pragma unroll
                for (int k = 0; k < K; k++) {
                    const double sum = g.w0 * t0[k] + g.w * t1[k];  // + 0.0 left out as above
                    const float term = (float)(g.rL2 * sum * a.dbeta_view * a.xfactor);
                    acc[k] = g.ok ? acc[k] + term : acc[k];
                }
            }
        };
        // two sets of U views in registers: the next set is fetched while one
        // is summed (no copies between them); what lies past the last view
        // re-reads it and is not summed
        struct Set {
            BpView g[U];
            float t0[U][K], t1[U][K];
        };
        const int nv = a.use_views;
        auto fetch = [&](Set& q, int v) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int w = min(v + u, nv - 1);
                q.g[u] = bp_view<WIDE, FW>(a, xx, yy, w);
                taps(w, q.g[u], q.t0[u], q.t1[u]);
            }
        };
        auto sum = [&](const Set& q, int v) {
#pragma unroll
            for (int u = 0; u < U; u++)
                if (u == 0 || v + u < nv) add(q.g[u], q.t0[u], q.t1[u]);
        };
        Set p, q;
        fetch(p, 0);
#pragma unroll 1
        for (int v = 0; v < nv; v += 2 * U) {
            fetch(q, v + U);
            sum(p, v);
            if (v + U >= nv) break;
            fetch(p, v + 2 * U);
            sum(q, v + U);
        }
    }
    if (in_img) {
#pragma unroll
        for (int k = 0; k < K; k++)
            if (s0 + k < S) a.img[((size_t)(s0 + k) * a.N + y) * a.N + x] = acc[k];
    }
}

template <bool WIDE, int K, bool FW, bool IL = false>
__global__ __launch_bounds__(kBpTile * kBpTile) void k_backproject_multi(BackprojArgs a, int S)
{
    bp_multi_tile<WIDE, K, FW, IL>(a, S, blockIdx.x, blockIdx.y, blockIdx.z);
}

// Several geometries in one launch: workgroup l belongs to the group g with
// pref[g] <= l < pref[g + 1] (a scalar search, uniform over the workgroup)
// and runs tile l - pref[g] of that group's tiles x slices, exactly as
// k_backproject_multi would.
template <bool WIDE, int K, bool FW, bool IL = false>
__global__ __launch_bounds__(kBpTile * kBpTile) void k_backproject_groups(BpGroups ga)
{
    const int l = blockIdx.x;
    int g = 0;
    while (g + 1 < ga.n && l >= ga.pref[g + 1]) g++;
    const int local = l - ga.pref[g];
    const int tx = ga.tiles_x[g];
    const int per_slice = tx * tx;
    const int bz = local / per_slice, r = local - bz * per_slice;
    bp_multi_tile<WIDE, K, FW, IL>(ga.a[g], ga.S[g], r % tx, r / tx, bz);
}

// Sinograms [S][VW] -> slices of K, dst[S/K][VW][K] (zeros past S): lane p
// of slice sl gathers the K values of pixel-row entry p (each read coalesced
// over the lanes) and stores them as 16-byte (K a multiple of 4) or 8-byte
// stores.
template <int K>
__global__ __launch_bounds__(256) void k_interleave_sinos(const float* __restrict__ src, int S, int VW,
                                                          float* __restrict__ dst)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x, sl = blockIdx.y;
    if (p >= VW) return;
    float v[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int s = sl * K + k;
        v[k] = s < S ? src[(size_t)s * VW + p] : 0.f;
    }
    float* d = dst + ((size_t)sl * VW + p) * K;
    if constexpr (K % 4 == 0) {
#pragma unroll
        for (int h = 0; h < K / 4; h++)
            reinterpret_cast<float4*>(d)[h] = make_float4(v[4 * h], v[4 * h + 1], v[4 * h + 2], v[4 * h + 3]);
    } else {
#pragma unroll
        for (int h = 0; h < K / 2; h++) reinterpret_cast<float2*>(d)[h] = make_float2(v[2 * h], v[2 * h + 1]);
    }
}

// One sinogram by orbits of the quarter turn.  With V views over 360 degrees
// (V a multiple of 4, Q = V/4) and a centred N x N grid (N even), pixel p at
// view v + Q has the geometry of pixel T(p) = (y, N-1-x) at view v, so the
// geometry G(p, v) of a base pixel p (x, y < N/2) serves the four pixels
// T^-k(p), k = 0..3, at views v + kQ (mod V):
//   T^0 = (x, y), T^-1 = (N-1-y, x), T^-2 = (N-1-x, N-1-y), T^-3 = (y, N-1-x).
// A workgroup holds 64 base pixels (an 8 x 8 tile of the quadrant); wave w
// runs the w-th eighth of the base views with the software pipeline of
// k_backproject_multi, and each pixel's partial sums are added in the waves'
// order through LDS.  (Eight waves because a small grid's are few: against
// four 128^2 x 800 views 50 -> 31 us, 200^2 x 360 24 -> 16; 512^2 107 -> 105.)  The geometry follows the single-sinogram
// expression in FP64; the interpolation and distance weights of a term are
// applied in float, and the order of the float sum differs from the
// reference's ascending views (images within 1e-5 of the reference's).
constexpr int kBpSymWaves = 8;
template <bool WIDE>
__global__ __launch_bounds__(64 * kBpSymWaves) void k_backproject_sym(BackprojArgs a)
{
    __shared__ float part[kBpSymWaves - 1][4][64];
    // the view range is per wave: made scalar, so the four rows of a view
    // are scalar bases and their wrap a scalar test
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int h = a.N / 2, Q = a.V / 4;
    const int x = blockIdx.x * 8 + (lane & 7), y = blockIdx.y * 8 + (lane >> 3);
    const bool in_q = x < h && y < h;
    // prepareMaskData, F/misc.cpp:20-36 (the circle is invariant under T)
    const double dyc = (double)y - a.mask_r, dxc = (double)x - a.mask_r;
    const bool masked = in_q && (dyc * dyc + dxc * dxc <= a.mask_r2);
    const double xx = -(x - a.center) * a.pix;  // :52-53
    const double yy = -(y - a.center) * a.pix;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    const int len = (a.V + kBpSymWaves - 1) / kBpSymWaves;
    const int vb = wave * len, ve = min(vb + len, a.V);
    if (masked && vb < ve) {
        // rows of view v + kQ (mod V); vb + kQ < V + 3Q, one wrap at most (a
        // scalar base; V * W <= 2^28)
        auto row_of = [&](int v, int k) {
            const int r = v + k * Q;
            return a.fltd + (uint32_t)((r >= a.V ? r - a.V : r) * a.W);
        };
        // the pixel-view geometry in the float-weight form: the sums already
        // run in another order than the reference's, and its roundings (~1e-7
        // relative per term) stay far below that difference
        auto fetch = [&](int v, const BpView& g, float (&t0)[4], float (&t1)[4]) {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float* row = row_of(v, k) + (uint32_t)g.col;
                t0[k] = row[0];
                t1[k] = row[1];
            }
        };
        auto add = [&](const BpView& g, const float (&t0)[4], const float (&t1)[4]) {
            if (g.ok) {
#pragma unroll
                for (int k = 0; k < 4; k++) acc[k] = fmaf(g.w1s, t1[k], fmaf(g.w0s, t0[k], acc[k]));
            }
        };
        // two views per iteration in two register sets (as in bp_multi_tile)
        BpView g = bp_view<WIDE, true>(a, xx, yy, vb), gn;
        float r0[4], r1[4], n0[4], n1[4];
        fetch(vb, g, r0, r1);
#pragma unroll 1
        for (int v = vb; v < ve; v += 2) {
            const int v1 = min(v + 1, ve - 1);
            gn = bp_view<WIDE, true>(a, xx, yy, v1);
            fetch(v1, gn, n0, n1);
            add(g, r0, r1);
            if (v + 1 == ve) break;
            const int v2 = min(v + 2, ve - 1);
            g = bp_view<WIDE, true>(a, xx, yy, v2);
            fetch(v2, g, r0, r1);
            add(gn, n0, n1);
        }
    }
    if (wave > 0) {
#pragma unroll
        for (int k = 0; k < 4; k++) part[wave - 1][k][lane] = acc[k];
    }
    __syncthreads();
    if (wave == 0 && in_q) {
        const int n1 = a.N - 1;
        const int px[4] = {x, n1 - y, n1 - x, y};
        const int py[4] = {y, x, n1 - y, n1 - x};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            float v = acc[k];
#pragma unroll
            for (int w = 0; w < kBpSymWaves - 1; w++) v += part[w][k][lane];
            a.img[(size_t)py[k] * a.N + px[k]] = v;
        }
    }
}

// atan(t) = t P(t^2) with P's coefficients in arguments (atan_small's, times
// the channels per radian), so the kernel reads them as scalars.
constexpr int kBpLonePoly = (int)(sizeof(kAtanSmall) / sizeof(double));
struct BackprojLoneArgs {
    BackprojArgs a;
    double poly[kBpLonePoly];
};

// One sinogram where k_backproject_sym does not serve (a view count that is no
// multiple of 4, or N odd): orbits of R = 4, 2 or 1 turns, each term and each
// sum in FP64 as k_backproject's terms are.  One lane per pixel left an odd
// grid of 301^2 at 1.4 waves per SIMD, each a serial chain of 630 views, and
// every pixel-view computed its geometry.  Here kBpLoneWaves waves share the
// views of 64 base pixels, two views per iteration in two register sets, and a
// geometry serves the R pixels of its orbit:
//   R = 4 (V % 4 == 0): T^0 .. T^-3 of k_backproject_sym; for N odd the base
//         pixels are x <= c, y < c (c the middle) and the centre,
//   R = 2 (V even): (x, y) at view v and (N-1-x, N-1-y) at view v + V/2; base
//         pixels are the upper rows and, N odd, the middle row's x <= c,
//   R = 1: every pixel by itself (V odd: its last view measures nothing).
// The centre is its own image; its orbit's slots hold the same sum and slot 0
// stores it.  Results are within the FP64 sum's rounding to float, closer to
// the exact image than one float add per view.  FP64 issue bounds it.
// FBP of one sinogram against k_backproject: 301^2 x 630 views 197 -> 75 us.
constexpr int kBpLoneWaves = 8;
template <bool WIDE, int R>
__global__ __launch_bounds__(64 * kBpLoneWaves) void k_backproject_lone(BackprojLoneArgs la)
{
    const BackprojArgs& a = la.a;
    __shared__ double part[kBpLoneWaves - 1][R][64];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int x = blockIdx.x * 8 + (lane & 7), y = blockIdx.y * 8 + (lane >> 3);
    const int h = a.N / 2;
    const bool mid = a.N % 2 != 0 && y == h;  // the middle row of an odd grid
    const bool base = R == 1   ? x < a.N && y < a.N
                      : R == 2 ? x < a.N && (y < h || (mid && x <= h))
                               : x < a.N - h && (y < h || (mid && x == h));
    // prepareMaskData, F/misc.cpp:20-36 (the circle is invariant under turns)
    const double dyc = (double)y - a.mask_r, dxc = (double)x - a.mask_r;
    const bool masked = base && (dyc * dyc + dxc * dxc <= a.mask_r2);
    const double xx = -(x - a.center) * a.pix;  // :52-53
    const double yy = -(y - a.center) * a.pix;
    const double dbx = a.dbeta_view * a.xfactor;
    // this wave's run of the views; a turn adds Q (R > 1: use_views == V)
    const int Q = a.V / R, nv = a.use_views, len = (nv + kBpLoneWaves - 1) / kBpLoneWaves;
    const int vb = wave * len, ve = min(vb + len, nv);
    double acc[R];
#pragma unroll
    for (int k = 0; k < R; k++) acc[k] = 0.0;
    if (masked && vb < ve) {
        struct View {
            double w0, w1;
            uint32_t col;
            bool ok;
        };
        auto geometry = [&](int v) {
            const double c = a.cosT[v], sn = a.sinT[v];
            View g;
            const double X = __builtin_fma(xx, c, yy * sn);
            const double den = __builtin_fma(xx, sn, __builtin_fma(-yy, c, a.sid));
            const double L2 = __builtin_fma(den, den, X * X);
            const double tg = X * rcp_f64(den);
            const double u = tg * tg;
            double p = la.poly[0];
#pragma unroll
            for (int i = 1; i < kBpLonePoly; i++) p = __builtin_fma(p, u, la.poly[i]);
            double fGAM = __builtin_fma(tg, p, (double)a.cent);
            if (WIDE && !(fabs(tg) <= 0.5)) fGAM = __builtin_fma(atan(X / den), a.inv_dbeta_ch, (double)a.cent);
            const int GAM = WIDE ? trunc_i32_bp(fGAM) : (int)fGAM;  // (as bp_view)
            const double s = rcp_f64(L2) * dbx;
            g.w1 = (fGAM - GAM) * s;
            g.w0 = s - g.w1;
            g.ok = (unsigned)GAM < (unsigned)(a.W - 1);
            g.col = g.ok ? GAM : 0;
            return g;
        };
        auto fetch = [&](int v, const View& g, float (&t0)[R], float (&t1)[R]) {
#pragma unroll
            for (int k = 0; k < R; k++) {
                const int r = v + k * Q;
                // (a scalar base; V * W <= 2^28)
                const float* row = a.fltd + (uint32_t)((R > 1 && r >= a.V ? r - a.V : r) * a.W) + g.col;
                t0[k] = row[0];
                t1[k] = row[1];
            }
        };
        auto add = [&](const View& g, const float (&t0)[R], const float (&t1)[R]) {
            if (g.ok) {
#pragma unroll
                for (int k = 0; k < R; k++)
                    acc[k] = __builtin_fma(g.w1, (double)t1[k], __builtin_fma(g.w0, (double)t0[k], acc[k]));
            }
        };
        View g = geometry(vb), gn;
        float r0[R], r1[R], n0[R], n1[R];
        fetch(vb, g, r0, r1);
#pragma unroll 1
        for (int v = vb; v < ve; v += 2) {
            const int v1 = min(v + 1, ve - 1);
            gn = geometry(v1);
            fetch(v1, gn, n0, n1);
            add(g, r0, r1);
            if (v + 1 == ve) break;
            const int v2 = min(v + 2, ve - 1);
            g = geometry(v2);
            fetch(v2, g, r0, r1);
            add(gn, n0, n1);
        }
    }
    if (wave > 0) {
#pragma unroll
        for (int k = 0; k < R; k++) part[wave - 1][k][lane] = acc[k];
    }
    __syncthreads();
    if (wave == 0 && base) {
        const int n1 = a.N - 1;
        const bool centre = mid && x == h;
        const int px[4] = {x, R == 2 ? n1 - x : n1 - y, n1 - x, y};
        const int py[4] = {y, R == 2 ? n1 - y : x, n1 - y, n1 - x};
#pragma unroll
        for (int k = 0; k < R; k++) {
            double v = acc[k];
#pragma unroll
            for (int w = 0; w < kBpLoneWaves - 1; w++) v += part[w][k][lane];
            if (k == 0 || !centre) a.img[(size_t)py[k] * a.N + px[k]] = (float)v;
        }
    }
}

// The beam-hardening tool M/beam_hardening_correction.cpp:47-60 elementwise:
// y = -ln p (single-precision log, as the tool's C++ overload resolution
// gives), y' = |y| + alpha |y|^beta, out = exp(-y') in FP64, stored as float.
__global__ __launch_bounds__(256) void k_beam_hardening(const float* __restrict__ in, float* __restrict__ out, int n,
                                                        double alpha, double beta)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double yi = -(double)logf_rounded(in[i]);  // the tool's log of a float is logf
    yi = fabs(yi) + (alpha * pow(fabs(yi), beta));
    out[i] = (float)exp(-yi);
}

vct_status launch_beam_hardening(const float* in, float* out, int n, double alpha, double beta, hipStream_t s)
{
    if (n <= 0) return set_error(VCT_ERR_ARG, "empty sinogram");
    hipLaunchKernelGGL(k_beam_hardening, dim3((n + 255) / 256), dim3(256), 0, s, in, out, n, alpha, beta);
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

vct_status launch_filter(const FilterPrepArgs& p, const FilterGemmArgs& g, hipStream_t s)
{
    if (p.Kp % (8 * kFiltWaves) != 0)
        return set_error(VCT_ERR_INTERNAL, "filter K padding %d not a multiple of %d", p.Kp, 8 * kFiltWaves);
    if ((size_t)(p.Kp + 31) * sizeof(float) > 48 * 1024) return set_error(VCT_ERR_ARG, "too many channels for the filter");
    const int Rp = (p.R + 31) / 32 * 32;
    hipLaunchKernelGGL(k_filter_prep, dim3(p.Kp / 32, Rp / 32), dim3(256), 0, s, p);
    VCT_HIP(hipGetLastError());
    const int Wp = (g.W + 31) / 32 * 32;
    const int ct = Wp / 32;
    const long long ntiles = (long long)(Rp / 32) * ct;
    if (ntiles > INT_MAX / 2) return set_error(VCT_ERR_ARG, "filter GEMM too large");
    const int nt = ntiles >= 2000 ? kFiltStrip : 1;
    const int cs = (ct + nt - 1) / nt, nitems = Rp / 32 * cs, per_xcd = (nitems + 7) / 8;
    const size_t lds = (size_t)(g.Kp + 32 * nt - 1) * sizeof(float);
    const dim3 grid(8 * per_xcd), blk(64 * kFiltWaves);
    if (nt == 1) hipLaunchKernelGGL(k_filter_gemm<1>, grid, blk, lds, s, g, ct, cs, nitems, per_xcd);
    else hipLaunchKernelGGL(k_filter_gemm<kFiltStrip>, grid, blk, lds, s, g, ct, cs, nitems, per_xcd);
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

// k_backproject_multi with K sinograms per lane, for K = K0 ... kBpSinos.
template <bool WIDE, int K0>
static void launch_bp_multi(const BackprojArgs& a, int S, int K, hipStream_t s)
{
    if constexpr (K0 < kBpSinos) {
        if (K > K0) {
            launch_bp_multi<WIDE, K0 + 1>(a, S, K, s);
            return;
        }
    }
    const dim3 grid((a.N + kBpTile - 1) / kBpTile, (a.N + kBpTile - 1) / kBpTile, (S + K0 - 1) / K0);
    if (a.exact)
        hipLaunchKernelGGL((k_backproject_multi<WIDE, K0, false>), grid, dim3(kBpTile * kBpTile), 0, s, a, S);
    else
        hipLaunchKernelGGL((k_backproject_multi<WIDE, K0, true>), grid, dim3(kBpTile * kBpTile), 0, s, a, S);
}

template <bool WIDE, bool FW, int K0>
static void launch_bp_groups_k(const BpGroups& ga, int K, hipStream_t s)
{
    if constexpr (K0 < kBpSinos) {
        if (K > K0) {
            launch_bp_groups_k<WIDE, FW, K0 + 1>(ga, K, s);
            return;
        }
    }
    hipLaunchKernelGGL((k_backproject_groups<WIDE, K0, FW>), dim3(ga.pref[ga.n]), dim3(kBpTile * kBpTile), 0, s, ga);
}

vct_status launch_backproject_groups(BpGroups& ga, int K, hipStream_t s, bool il)
{
    for (int g = 0; g < std::min(ga.n, kMaxBpGroups); g++) set_poly(ga.a[g]);
    if (ga.n < 1 || ga.n > kMaxBpGroups) return set_error(VCT_ERR_ARG, "%d groups (1..%d)", ga.n, kMaxBpGroups);
    if (K < 2) K = 2;
    if (K > kBpSinos) K = kBpSinos;
    bool wide = false, exact = false;
    long long total = 0;
    ga.pref[0] = 0;
    for (int g = 0; g < ga.n; g++) {
        const BackprojArgs& a = ga.a[g];
        exact = exact || a.exact;
        if (ga.S[g] < 1) return set_error(VCT_ERR_ARG, "group %d has no sinograms", g);
        wide = wide || bp_wide(a);
        ga.tiles_x[g] = (a.N + kBpTile - 1) / kBpTile;
        total += (long long)ga.tiles_x[g] * ga.tiles_x[g] * ((ga.S[g] + K - 1) / K);
        if (total > INT_MAX) return set_error(VCT_ERR_ARG, "grouped backprojection too large");
        ga.pref[g + 1] = (int)total;
    }
    if (il) {
        const dim3 grid(ga.pref[ga.n]), blk(kBpTile * kBpTile);
#define VCT_BP_IL(KK)                                                                                   \
    case KK:                                                                                            \
        if (wide && exact) hipLaunchKernelGGL((k_backproject_groups<true, KK, false, true>), grid, blk, 0, s, ga);  \
        else if (wide) hipLaunchKernelGGL((k_backproject_groups<true, KK, true, true>), grid, blk, 0, s, ga);  \
        else if (exact) hipLaunchKernelGGL((k_backproject_groups<false, KK, false, true>), grid, blk, 0, s, ga); \
        else hipLaunchKernelGGL((k_backproject_groups<false, KK, true, true>), grid, blk, 0, s, ga);   \
        break;
        switch (K) {
            VCT_BP_IL(4) VCT_BP_IL(8) VCT_BP_IL(12) VCT_BP_IL(16)
        default: return set_error(VCT_ERR_ARG, "interleaved slices of %d sinograms (4, 8, 12 or 16)", K);
        }
#undef VCT_BP_IL
    } else if (wide && exact) launch_bp_groups_k<true, false, 2>(ga, K, s);
    else if (wide) launch_bp_groups_k<true, true, 2>(ga, K, s);
    else if (exact) launch_bp_groups_k<false, false, 2>(ga, K, s);
    else launch_bp_groups_k<false, true, 2>(ga, K, s);
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

vct_status launch_interleave_sinos(const float* src, int S, int VW, int K, float* dst, hipStream_t s)
{
    if (S < 1 || VW < 1) return set_error(VCT_ERR_ARG, "empty sinograms");
    const dim3 grid((VW + 255) / 256, (S + K - 1) / K), blk(256);
    switch (K) {
    case 2: hipLaunchKernelGGL(k_interleave_sinos<2>, grid, blk, 0, s, src, S, VW, dst); break;
    case 4: hipLaunchKernelGGL(k_interleave_sinos<4>, grid, blk, 0, s, src, S, VW, dst); break;
    case 6: hipLaunchKernelGGL(k_interleave_sinos<6>, grid, blk, 0, s, src, S, VW, dst); break;
    case 8: hipLaunchKernelGGL(k_interleave_sinos<8>, grid, blk, 0, s, src, S, VW, dst); break;
    case 10: hipLaunchKernelGGL(k_interleave_sinos<10>, grid, blk, 0, s, src, S, VW, dst); break;
    case 12: hipLaunchKernelGGL(k_interleave_sinos<12>, grid, blk, 0, s, src, S, VW, dst); break;
    case 16: hipLaunchKernelGGL(k_interleave_sinos<16>, grid, blk, 0, s, src, S, VW, dst); break;
    default: return set_error(VCT_ERR_ARG, "interleaved slices of %d sinograms (2, 4 .. 12 or 16)", K);
    }
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

vct_status launch_backproject_il(const BackprojArgs& args, int S, int K, hipStream_t s)
{
    BackprojArgs a = args;
    set_poly(a);
    const dim3 grid((a.N + kBpTile - 1) / kBpTile, (a.N + kBpTile - 1) / kBpTile, (S + K - 1) / K),
        blk(kBpTile * kBpTile);
#define VCT_BP_IL(KK)                                                                                      \
    case KK:                                                                                               \
        if (bp_wide(a)) hipLaunchKernelGGL((k_backproject_multi<true, KK, true, true>), grid, blk, 0, s, a, S); \
        else hipLaunchKernelGGL((k_backproject_multi<false, KK, true, true>), grid, blk, 0, s, a, S);      \
        break;
    switch (K) {
        VCT_BP_IL(2) VCT_BP_IL(4) VCT_BP_IL(6) VCT_BP_IL(8) VCT_BP_IL(10) VCT_BP_IL(12)
    default: return set_error(VCT_ERR_INTERNAL, "interleaved slices of %d sinograms", K);
    }
#undef VCT_BP_IL
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

template <bool WIDE, int R>
static void launch_bp_lone(const BackprojArgs& a, hipStream_t s)
{
    BackprojLoneArgs la{a, {}};
    for (int i = 0; i < kBpLonePoly; i++) la.poly[i] = kAtanSmall[i] * a.inv_dbeta_ch;
    const int bx = R == 4 ? (a.N + 1) / 2 : a.N, by = R == 1 ? a.N : (a.N + 1) / 2;
    hipLaunchKernelGGL((k_backproject_lone<WIDE, R>), dim3((bx + 7) / 8, (by + 7) / 8), dim3(64 * kBpLoneWaves), 0, s,
                       la);
}

template <bool WIDE>
static void launch_bp_w(const BackprojArgs& a, int S, hipStream_t s)
{
    // the fewest workgroup slices of at most kBpSinos sinograms, split evenly
    // (S = 20: two slices of 10, not 16 + 4), but enough slices that the launch
    // has kBpMinLanes lanes: 256^2 pixels x 3 sinograms in one slice would
    // leave one wave per SIMD, and 3 slices of one sinogram run 2-3x faster
    const long long px = (long long)a.N * a.N;
    const long long floor_slices = (kBpMinLanes + px - 1) / px;
    const int cap = a.max_k >= 2 && a.max_k < kBpSinos ? a.max_k : kBpSinos;
    int slices = (S + cap - 1) / cap;
    if (slices < floor_slices) slices = (int)std::min<long long>(S, floor_slices);
    const int K = (S + slices - 1) / slices;
    if (S == 1 && !a.exact && a.V % 4 == 0 && a.N % 2 == 0 && a.use_views == a.V && a.N >= 2) {
        const int h = a.N / 2;
        const dim3 grid((h + 7) / 8, (h + 7) / 8);
        hipLaunchKernelGGL(k_backproject_sym<WIDE>, grid, dim3(64 * kBpSymWaves), 0, s, a);
        return;
    }
    if (S == 1 && !a.exact) {
        const int R = a.use_views != a.V ? 1 : a.V % 4 == 0 ? 4 : 2;
        if (R == 4) launch_bp_lone<WIDE, 4>(a, s);
        else if (R == 2) launch_bp_lone<WIDE, 2>(a, s);
        else launch_bp_lone<WIDE, 1>(a, s);
        return;
    }
    if (K == 1 && a.exact) {
        const dim3 grid((a.N + kBpTile - 1) / kBpTile, (a.N + kBpTile - 1) / kBpTile, S);
        hipLaunchKernelGGL(k_backproject<WIDE>, grid, dim3(kBpTile * kBpTile), 0, s, a);
        return;
    }
    // (several sinograms one per lane take the float-weight template too, so
    // an image does not depend on how the call was split)
    launch_bp_multi<WIDE, 1>(a, S, K, s);
}

vct_status launch_backproject(const BackprojArgs& args, int S, hipStream_t s)
{
    BackprojArgs a = args;
    set_poly(a);
    if (S <= 0) return set_error(VCT_ERR_ARG, "no sinograms to backproject");
    if (bp_wide(a))
        launch_bp_w<true>(a, S, s);
    else
        launch_bp_w<false>(a, S, s);
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

}  // namespace vct
