// fold.h — running DFT of one chunk of contour samples (calculate_JandM's
// accumulation, FDTD_GPU.cu:231-280).
//
// Phase e^{-j w (step + t0) dt}: evaluated in FP64 for every step of the chunk
// (<= 64 steps) into an LDS table and rounded once to FP32 (a rotation
// recurrence would drift by an ulp per step); the chunk is summed in FP32 and
// added to the long-running accumulator with Kahan compensation.  A thread
// folds one contour point for nf frequencies from fb on, kFoldGroup at a time:
// few items (one simulation) take one frequency per thread, so the
// frequencies spread over more blocks; many items take groups of 8, so each
// sample is read once per 8 frequencies.  Every frequency's sum runs in the
// same order either way.
#pragma once
#include "device.h"

namespace tomo {
namespace {

// Samples of contour point p at the chunk's step k: H, and Ez at the face and
// at its outer neighbour.  Global-address-space views (flat loads would also
// count against the LDS counter, so every phase-table wait would drain the
// sample loads); the rows go round after S->srows.
struct FoldSamples {
    gcfloat *h, *e0, *e1;
    int P, rows, r0;
    __device__ __forceinline__ FoldSamples(const DevSim* S, const LaunchItem& it, int p)
        : h((gcfloat*)S->samp + p), e0(h + (size_t)S->srows * S->P), e1(e0 + (size_t)S->srows * S->P), P(S->P),
          rows(S->srows), r0(it.samp0) {}
    __device__ __forceinline__ size_t at(int k) const {
        const int r = r0 + k;
        return (size_t)(r >= rows ? r - rows : r) * P;
    }
};

// Fold nk steps of item `it`; every thread of the workgroup calls it (the
// phases are shared out over the workgroup), p beyond the contour included.
// wJ, wM: [>= nf][64] in LDS.
template <int kFoldGroup>
__device__ __forceinline__ void fold_fp32(const DevSim* S, const LaunchItem& it, int nk, int fb, int nf, int p, float2* wJ,
                                          float2* wM) {
    for (int i = threadIdx.x; i < 2 * nf * nk; i += blockDim.x) {
        const int which = i / (nf * nk), f = (i / nk) % nf, k = i % nk;
        double s0, c0;
        sincos(-S->wdt[fb + f] * ((double)it.step0 + k + (which ? S->tM : S->tJ)), &s0, &c0);
        (which ? wM : wJ)[f * 64 + k] = make_float2((float)c0, (float)s0);
    }
    __syncthreads();
    const int P = S->P;
    if (p >= P) return;
    const int leg = p < S->L1 ? 0 : (p < S->L2 ? 1 : (p < S->L3 ? 2 : 3));
    const float sdt = S->sgn_dt[leg];
    const FoldSamples Z(S, it, p);
    for (int f0 = 0; f0 < nf; f0 += kFoldGroup) {
        float jr[kFoldGroup], ji[kFoldGroup], mr[kFoldGroup], mi[kFoldGroup];
#pragma unroll
        for (int q = 0; q < kFoldGroup; ++q) jr[q] = ji[q] = mr[q] = mi[q] = 0.f;
        // unrolled so that several steps' samples are in flight at once
        // (the accumulation order is unchanged); one frequency per thread
        // leaves the registers for 20 steps' loads
#pragma unroll kFoldGroup == 1 ? 20 : 8
        for (int k = 0; k < nk; ++k) {
            const size_t o = Z.at(k);
            const float h = Z.h[o];
            const float e = (Z.e0[o] + Z.e1[o]) / 2;
#pragma unroll
            for (int q = 0; q < kFoldGroup; ++q) {
                const float2 a = wJ[(f0 + q) * 64 + k], b = wM[(f0 + q) * 64 + k];
                jr[q] += h * a.x;
                ji[q] += h * a.y;
                mr[q] += e * b.x;
                mi[q] += e * b.y;
            }
        }
#pragma unroll
        for (int q = 0; q < kFoldGroup; ++q) {
            if (f0 + q >= nf) break;
            float4* aJ = (float4*)S->accJ + (size_t)(fb + f0 + q) * P + p;
            float4* aM = (float4*)S->accM + (size_t)(fb + f0 + q) * P + p;
            float4 vJ = *aJ, vM = *aM;
            // Kahan: value (x, y), compensation (z, w)
            float yv, tv;
            yv = sdt * jr[q] - vJ.z; tv = vJ.x + yv; vJ.z = (tv - vJ.x) - yv; vJ.x = tv;
            yv = sdt * ji[q] - vJ.w; tv = vJ.y + yv; vJ.w = (tv - vJ.y) - yv; vJ.y = tv;
            yv = sdt * mr[q] - vM.z; tv = vM.x + yv; vM.z = (tv - vM.x) - yv; vM.x = tv;
            yv = sdt * mi[q] - vM.w; tv = vM.y + yv; vM.w = (tv - vM.y) - yv; vM.y = tv;
            *aJ = vJ;
            *aM = vM;
        }
    }
}

// FP64 study mode: exact phases; the M phase is the J phase rotated by
// -w (tM - tJ).  dJ: [>= nf][64], dRot: [>= nf] in LDS.
template <int kFoldGroup>
__device__ __forceinline__ void fold_fp64(const DevSim* S, const LaunchItem& it, int nk, int fb, int nf, int p, double2* dJ,
                                          double2* dRot) {
    for (int i = threadIdx.x; i < nf * nk; i += blockDim.x) {
        const int f = i / nk, k = i % nk;
        double s, c;
        sincos(-S->wdt[fb + f] * ((double)it.step0 + k + S->tJ), &s, &c);
        dJ[f * 64 + k] = make_double2(c, s);
    }
    if (threadIdx.x < nf) {
        double s, c;
        sincos(-S->wdt[fb + threadIdx.x] * (S->tM - S->tJ), &s, &c);
        dRot[threadIdx.x] = make_double2(c, s);
    }
    __syncthreads();
    const int P = S->P;
    if (p >= P) return;
    const int leg = p < S->L1 ? 0 : (p < S->L2 ? 1 : (p < S->L3 ? 2 : 3));
    const float sdt = S->sgn_dt[leg];
    const FoldSamples Z(S, it, p);
    for (int f0 = 0; f0 < nf; f0 += kFoldGroup) {
        double jr[kFoldGroup], ji[kFoldGroup], mr[kFoldGroup], mi[kFoldGroup];
#pragma unroll
        for (int q = 0; q < kFoldGroup; ++q) jr[q] = ji[q] = mr[q] = mi[q] = 0.0;
#pragma unroll 8
        for (int k = 0; k < nk; ++k) {
            const size_t o = Z.at(k);
            const double h = Z.h[o];
            const double e = 0.5 * ((double)Z.e0[o] + (double)Z.e1[o]);
#pragma unroll
            for (int q = 0; q < kFoldGroup; ++q) {
                const double2 a = dJ[(f0 + q) * 64 + k], r = dRot[f0 + q];
                const double2 b = make_double2(a.x * r.x - a.y * r.y, a.x * r.y + a.y * r.x);
                jr[q] += h * a.x;
                ji[q] += h * a.y;
                mr[q] += e * b.x;
                mi[q] += e * b.y;
            }
        }
#pragma unroll
        for (int q = 0; q < kFoldGroup; ++q) {
            if (f0 + q >= nf) break;
            double2* aJ = (double2*)S->accJ + (size_t)(fb + f0 + q) * P + p;
            double2* aM = (double2*)S->accM + (size_t)(fb + f0 + q) * P + p;
            double2 vJ = *aJ, vM = *aM;
            vJ.x += sdt * jr[q]; vJ.y += sdt * ji[q]; vM.x += sdt * mr[q]; vM.y += sdt * mi[q];
            *aJ = vJ;
            *aM = vM;
        }
    }
}

}  // namespace
}  // namespace tomo
