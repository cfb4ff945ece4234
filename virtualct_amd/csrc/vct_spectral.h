// vct_spectral.h -- the polyenergetic sum over a spectrum's bins on the matrix
// cores (device code, included by .hip files only).
//
// A wave holds 64 rays in four tiles of 16.  For 16 bins at a time the
// exponents x[bin][ray] = sum_m mu2[bin][m] L[ray][m] are one or two
// v_mfma_f32_16x16x4f32 per tile (M <= 4, M <= 8; FP32 throughout), which
// leave lane l four bins, 4 (l >> 4) + i, of ray l & 15; the lane adds pdf *
// exp2(x) of its bins, and the four lane groups meet at the end.  The tables
// are then read from LDS once per 64 rays and 16 bins instead of once per ray
// and bin, and a sum is four chains of a quarter of the bins (error against 64
// bits 6e-8 instead of 1.6e-7 at 120 bins, 1.0e-7 instead of 4.0e-7 at 650).
// What bounds it: an exponential is 9 cycles of a SIMD, the 16x16x4 product 35
// per 256 exponents, and their times add (four products and 16 exponentials
// take 289 cycles): 35 cycles per 64 bin-rays of 5 to 8 materials, where one ray per
// lane took 50 (the tables' reads), and 28 is what its multiply-adds alone
// would.  800 x 609 rays: 650 bins 115 -> 85 us, two spectra of 120 bins and 8
// materials 55 -> 45.  (For the derivatives a second product costs as much as
// it saves: their kernels sum one ray per lane.)
#pragma once

#include "vct_internal.h"

namespace vct {

typedef float floatx4 __attribute__((ext_vector_type(4)));

// One past the highest bin with a nonzero probability among the bins this
// wave's lanes hold (bin e on this lane, consecutive bins on consecutive
// lanes), or 0; called by every active lane, it needs no atomics.
__device__ __forceinline__ int last_nonzero_bin(int e, float p)
{
    const unsigned long long m = __ballot(p != 0.f);
    const int base = e - (int)(threadIdx.x & 63);  // the bin of lane 0
    return m ? base + 64 - __clzll((long long)m) : 0;
}

// LDS of one spectrum: [nblk][ST][64] mu2 (= -mu log2 e) in operand order,
// lane l of step st holding bin l & 15 of the block and material 4 st + (l >> 4),
// and [nblk * 16] pdf.
template <int M>
struct SpecTable {
    static constexpr int ST = (M + 3) / 4;
    const float *frag, *pdf;
    int ne;  // bins up to the last nonzero probability; those past it add exactly +0
    static __host__ __device__ int floats(int NE) { return (NE + 15) / 16 * (64 * ST + 16); }
    // by the whole workgroup (at most 16 waves), all of whose waves see it on
    // return; att [M][NE] and pdf [NE] of the spectrum, last[16] in LDS
    static __device__ __forceinline__ SpecTable fill(float* lds, int* last, const float* __restrict__ att,
                                                     const float* __restrict__ pdf, int NE)
    {
        const float kLog2e = 1.4426950408889634f;
        const int nblk = (NE + 15) / 16;
        float *frag = lds, *p = frag + nblk * 64 * ST;
        for (int i = threadIdx.x; i < nblk * 64 * ST; i += blockDim.x) {
            const int l = i & 63, bin = (i / (64 * ST)) * 16 + (l & 15), m = 4 * ((i >> 6) % ST) + (l >> 4);
            frag[i] = m < M && bin < NE ? -att[(size_t)m * NE + bin] * kLog2e : 0.f;
        }
        int mine = 0;
        for (int i = threadIdx.x; i < nblk * 16; i += blockDim.x) {
            p[i] = i < NE ? pdf[i] : 0.f;
            mine = max(mine, last_nonzero_bin(i, p[i]));
        }
        // (lane 0 holds bins wherever its wave does)
        if ((threadIdx.x & 63) == 0) last[threadIdx.x >> 6] = mine;
        __syncthreads();
        int ne = 0;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) ne = max(ne, last[w]);
        return {frag, p, ne};
    }
};

// L of the wave's 64 rays in operand order; elem(t, m) is material m of the
// ray of lane t.
template <int M>
struct SpecRays {
    static constexpr int ST = (M + 3) / 4;
    float b[4][ST];
    template <class F>
    __device__ __forceinline__ void load(F&& elem)
    {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int st = 0; st < ST; st++) {
                const int m = 4 * st + (lane >> 4);
                b[r][st] = m < M ? elem(16 * r + (lane & 15), m) : 0.f;
            }
    }
};

// The lane's own ray's sum.  Every lane of the wave takes part.
template <int M>
__device__ __forceinline__ float spec_sum(const SpecTable<M>& tab, const SpecRays<M>& L)
{
    constexpr int ST = SpecTable<M>::ST;
    const int lane = threadIdx.x & 63, grp = lane >> 4, ne = tab.ne;
    float I[4] = {0.f, 0.f, 0.f, 0.f};
    auto block = [&](int j, bool tail) {
        float a[ST];
#pragma unroll
        for (int st = 0; st < ST; st++) a[st] = tab.frag[(j * ST + st) * 64 + lane];
        const float4 pv = *reinterpret_cast<const float4*>(tab.pdf + 16 * j + 4 * grp);
        const float p[4] = {pv.x, pv.y, pv.z, pv.w};
        floatx4 x[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            x[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[0], L.b[r][0], floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            if constexpr (ST > 1) x[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[1], L.b[r][1], x[r], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // (a bin past the spectrum's end adds nothing, whatever its x)
            const bool on = !tail || 16 * j + 4 * grp + i < ne;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                // hardware exp2: only terms below 2^-126 (flushed) differ from exp2f
                const float e = __builtin_amdgcn_exp2f(x[r][i]);
                I[r] = on ? fmaf(p[i], e, I[r]) : I[r];
            }
        }
    };
    const int full = ne / 16;
    for (int j = 0; j < full; j++) block(j, false);
    if (ne & 15) block(full, true);
    // the four lane groups' sums of tiles 0..3: lane l gets the total of tile l >> 4
    const bool hi = grp >= 2, odd = grp & 1;
    const float s0 = hi ? I[0] : I[2], s1 = hi ? I[1] : I[3];
    const float k0 = (hi ? I[2] : I[0]) + __shfl_xor(s0, 32), k1 = (hi ? I[3] : I[1]) + __shfl_xor(s1, 32);
    const float s = odd ? k0 : k1;
    return (odd ? k1 : k0) + __shfl_xor(s, 16);
}

}  // namespace vct
