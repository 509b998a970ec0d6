// Epilogue of the two-pass inverse transforms: one lag of the window, normalised.
#pragma once
#include "bigfft.hpp"
#include "edge.hpp"

namespace fpcc {

// Lag l of pair p (stations i, j) and window w from vx, the unnormalised n-point
// inverse's value there.
__device__ __forceinline__ void lagwin_store(const ColArgs &a, int p, int w, int i, int j, int n, int l, float vx)
{
    const int lag = a.lag0 + l;
    double o = (double)(a.scale * vx);
    const int m = a.Nsig - abs(lag);
    if (a.edge && m > 0 && m < a.K) {
        // short overlap: the FP32 transform's absolute error, divided by
        // the overlap's small energy, would dominate; sum it exactly
        int ei = i, ej = j;
        if (a.norm != 1) pair_index(p, a.S, ei, ej);
        const int w0 = a.esum ? 0 : w, w1 = a.esum ? a.Wall : w + 1;
        const double c = edge_corr(a.edge, a.K, a.Wall, ei, ej, w0, w1, lag, m, a.norm == 2);
        o = c * (double)a.scale * (double)n;  // the transform's scale: vx is n c
    }
    if (a.norm == 1) {
        const double *P1 = a.E + (long long)(i * a.Wfull + w) * a.lde;
        const double *P2 = a.E + (long long)(j * a.Wfull + w) * a.lde;
        const int N = a.Nsig;
        const int a1 = max(0, -lag), b1 = min(N, N - lag);
        const int a2 = max(0, lag), b2 = min(N, N + lag);
        o = o / sqrt((P1[b1] - P1[a1]) * (P2[b2] - P2[a2]));
    } else if (a.norm == 2) {
        o = o / (double)(a.Nsig - abs(lag));
    }
    if (a.accumulate) a.y[(long long)p * a.L + l] += (float)o;
    else a.y[((long long)p * a.Wfull + w) * a.L + l] = (float)o;
}

}  // namespace fpcc
