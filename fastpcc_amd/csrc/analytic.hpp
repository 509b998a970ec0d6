// Analytic signals of real windows of even length through half-length transforms.
//
// The analytic signal of AnalyticSignal_plan_float (src/FFTapps.c:104-124) has the
// window itself as real part and its Hilbert transform u as imaginary part.  With
// z[m] = x[2m] + i x[2m+1], Z = FFT_h(z), h = N/2, and theta = 2 pi k / N,
//   U[k] = cos(theta) conj Z[h-k] + i sin(theta) Z[k]  (0 < k < h),  U[0] = 0,
//   u[2m] + i u[2m+1] = IFFT_h(U)[m] / h:
// two h-point transforms and real factors between them instead of two N-point ones.
#pragma once
#include "fft_core.hpp"

namespace fpcc {

// Z -> U / h (its conjugate if CONJ) in place (by the whole workgroup, between barriers); cs[k] =
// exp(2 pi i k / N), at(k) the LDS index of element k.
template <bool CONJ, typename At>
__device__ __forceinline__ void hilbert_half(cf32 *lds, int h, const cf32 *__restrict__ cs, At at)
{
    const float inv = 1.0f / (float)h;
    for (int k = threadIdx.x; 2 * k <= h; k += blockDim.x) {
        if (k == 0) {
            lds[at(0)] = cf32{0.0f, 0.0f};
            continue;
        }
        const cf32 a = lds[at(k)], c = lds[at(h - k)], w = cs[k];
        const float cc = w.x * inv, ss = w.y * inv;
        const cf32 u = cf32{cc * c.x - ss * a.y, ss * a.x - cc * c.y};
        const cf32 v = cf32{-cc * a.x - ss * c.y, cc * a.y + ss * c.x};
        lds[at(k)] = CONJ ? conj(u) : u;
        if (2 * k < h) lds[at(h - k)] = CONJ ? conj(v) : v;
    }
}

}  // namespace fpcc
