// Transforms of several rows or columns by one workgroup of 256 threads, in place in
// one LDS buffer (the two-pass FFTs of bigfft.hip, the pair stage of longpair.hip).
#pragma once
#include "engine.hpp"

namespace fpcc {

// W_n^m from the two-factor table of get_split_twiddles (m < n): two small
// cached lookups instead of a gather over an n-entry table
template <typename R> __device__ __forceinline__ C2<R> tw_m(const C2<R> *__restrict__ twN, unsigned m)
{
    return cmul(twN[kTwLo + m / kTwLo], twN[m % kTwLo]);
}

// Compile-time batched transforms for the common splits (2^17 .. 2^19 as 256 x
// 512 .. 256 x 2048): NTR transforms of NPT points transform in place in one LDS
// buffer, transform t at t * LDT, point i at ct_pad(i) (one pad slot per 16
// values), 256 threads, each pass reading all of a thread's butterflies before
// writing.  Columns: 16 x 256 points, radix 16 x 16, stride 274; rows: 4 x 512
// (8 x 8 x 8, stride 544) or 4 x 1024 (16 x 8 x 8, stride 1088).  The strides keep
// the loads, passes and stores within 1.5x of conflict-free LDS access.

template <int NPT, int NTR, int LDT, int DIR, int R, int NS, int NT = 256>
__device__ __forceinline__ void ctb_pass(cf32 *lds, const cf32 *__restrict__ tw)
{
    constexpr int NBF = NPT / R, TOT = NTR * NBF, BPT = (TOT + NT - 1) / NT;
    cf32 v[BPT][R];
#pragma unroll
    for (int i = 0; i < BPT; ++i) {
        const int bb = threadIdx.x + NT * i;
        if (TOT % NT == 0 || bb < TOT) {
            const int t = bb / NBF, b = bb % NBF;
#pragma unroll
            for (int r = 0; r < R; ++r) v[i][r] = lds[t * LDT + ct_pad(b + r * NBF)];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < BPT; ++i) {
        const int bb = threadIdx.x + NT * i;
        if (TOT % NT == 0 || bb < TOT) {
            const int t = bb / NBF, b = bb % NBF;
            const int k = b % NS;
            if (NS > 1) {
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    cf32 w = tw[(r - 1) * NS + k];
                    if (DIR > 0) w.y = -w.y;
                    v[i][r] = cmul(v[i][r], w);
                }
            }
            Dft<R, DIR>::run(v[i]);
            const int base = (b - k) * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) lds[t * LDT + ct_pad(base + r * NS)] = v[i][r];
        }
    }
    __syncthreads();
}

// Register-ended passes of a tile's in-place transforms (transform t's point p at
// lds[t * LDT + ct_pad(p)]), one butterfly b of transform t a call.  First pass
// (stride 1): the butterfly's inputs, points b + r NPT/R, are in v; its outputs go
// to LDS (the caller puts a barrier after every thread's call).
template <int NPT, int LDT, int DIR, int R>
__device__ __forceinline__ void ctb_first_regs(cf32 *v, int t, int b, cf32 *lds)
{
    Dft<R, DIR>::run(v);
#pragma unroll
    for (int r = 0; r < R; ++r) lds[t * LDT + ct_pad(b * R + r)] = v[r];
}
// Last pass (stride NPT/R): the butterfly's outputs, points b + r NPT/R, stay in v.
template <int NPT, int LDT, int DIR, int R>
__device__ __forceinline__ void ctb_last_regs(const cf32 *lds, int t, int b, cf32 *v, const cf32 *__restrict__ tw)
{
    constexpr int NS = NPT / R;
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = lds[t * LDT + ct_pad(b + r * NS)];
#pragma unroll
    for (int r = 1; r < R; ++r) {
        cf32 w = tw[(r - 1) * NS + b];
        if (DIR > 0) w.y = -w.y;
        v[r] = cmul(v[r], w);
    }
    Dft<R, DIR>::run(v);
}

template <int NT, int NPT, int NTR, int LDT, int DIR, int NS, int OFF, int R, int... Rest>
__device__ __forceinline__ void ctb_passes(cf32 *lds, const cf32 *__restrict__ tw)
{
    ctb_pass<NPT, NTR, LDT, DIR, R, NS, NT>(lds, tw + OFF);
    if constexpr (sizeof...(Rest) > 0) ctb_passes<NT, NPT, NTR, LDT, DIR, NS * R, OFF + (R - 1) * NS, Rest...>(lds, tw);
}

// tw: the per-pass twiddles of the plan with radices Rs (in that order)
template <int NPT, int NTR, int LDT, int DIR, int... Rs>
__device__ __forceinline__ cf32 *ctb_fft(cf32 *lds, const cf32 *__restrict__ tw)
{
    static_assert((Rs * ... * 1) == NPT, "radices must multiply to NPT");
    ctb_passes<256, NPT, NTR, LDT, DIR, 1, 0, Rs...>(lds, tw);
    return lds;
}

}  // namespace fpcc
