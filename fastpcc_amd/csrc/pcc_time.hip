// Time-domain PCC1 and PCC-v (src/FFTapps.c:251-278, 309-336, 475-783) on gfx950.
//
// For each lag, with a = phi2[n+lag] and b = phi1[n] over the overlap
// n in [max(0,-lag), min(N,N-lag)) (the lowlevels are called with the phasors of
// x2 first, src/FFTapps.c:598, :735):
//   PCC1:  y = sum(|a+b| - |a-b|) / (2 count)               (sqrtf terms)
//   PCC-v: y = sum(|a+b|^v - |a-b|^v) / (2^(v/2) count)     (powf(|.|^2, v/2) terms)
//
// The station stage keeps the half-angle phasors alpha, alpha^2 = a (half_phasor,
// cplx.hpp).  With alpha conj(beta) = p + i q and d = |alpha|^2 - |beta|^2,
//   |a + b|^2 = 4 p^2 + d^2,   |a - b|^2 = 4 q^2 + d^2
// are sums of squares: no cancellation where a is close to -b or to b (the identity
// through 2 Re(a conj b) loses the terms there).  P = 2p and Q = 2q are products of
// rank 2 of the samples of a row and a column, so a 32 x 32 tile (i, j) of terms is two
// MFMAs.  FP32 MFMAs take the vector unit's own multipliers (measured: 2 ns each a wave
// of terms on top of the terms), bf16 ones run beside it (0.3 ns): every component is
// split into three bf16 parts (24 bits, exact) and the products of two components
// except lowest x lowest (2^-32) fill K = 16.
//
// PCC1 needs |a+b| - |a-b| = |P| - |Q| + (corr(P) - corr(Q)), 0 <= corr(x) =
// sqrt(x^2 + d^2) - |x| <= d^2 / (2|x|).  Square roots run at a quarter of the vector
// rate, so groups of four terms a lane first test that corr <= 2^-24, FP32's rounding
// of a term (|a+b| <= 2), throughout the wave, with a bound of |d| over the group's
// rows; only groups that fail take the roots.  d is the difference of two
// regularisers 1e-6 max|z| / |z|: 1e-5 in noise, where 1 in 10 groups fails; windows
// with an event 30 times the noise fail mostly and take the roots as well.
// 16 stations x 24 windows of 3600, 2001 lags: 9.40 ms with 12 vector operations a term
// (sums, differences and squares formed term by term), 5.21 ms here, bound by the
// vector unit (83% busy, 6.8 operations a term).
#include <algorithm>
#include "engine.hpp"
#include "kernels.hpp"
#include "profile.hpp"
#include "pairs.hpp"

namespace fpcc {

// Hardware square root and power (v_sqrt_f32; v_log_f32 and v_exp_f32, i.e.
// 2^(V log2 x)), about 1 ulp and a few ulp per term, as the reference's CUDA
// engine compiles its terms (fast math); the correctly rounded library versions
// cost several times more instructions.  Sums over N terms of either sign keep
// the output within 1e-8 of the correctly rounded terms.  x^V for V <= 0 keeps powf
// (k_pcc_direct).
__device__ __forceinline__ float hw_sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ float hw_pow(float x, float V)
{
    return __builtin_amdgcn_exp2f(V * __builtin_amdgcn_logf(x));
}

typedef float f16v __attribute__((ext_vector_type(16)));
typedef __bf16 b8v __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));

enum { PT_SQRT = 0, PT_SQUARE = 1, PT_HWPOW = 2, PT_POW = 3 };  // PT_POW: k_pcc_direct

constexpr float kPtD = 2896.3093757400986f;  // (2^11.5 d)^2 <= |x|: corr(x) <= 2^-24

// A component's 8 K slots from its bf16 parts h + m + l, each the rounded rest: left
// (h h m m h l m l) against right (h m h m l h l m)
__device__ __forceinline__ unsigned round_bf16(float v)  // in the upper half
{
    const unsigned u = __float_as_uint(v);
    return (u + 0x7fffu + ((u >> 16) & 1u)) & 0xffff0000u;
}
__device__ __forceinline__ void split3(float v, unsigned &h, unsigned &m, unsigned &l)
{
    h = round_bf16(v);
    const float r = v - __uint_as_float(h);
    m = round_bf16(r);
    l = __float_as_uint(r - __uint_as_float(m));  // at most 8 bits are left
}
// the upper halves of a (low) and b (high)
__device__ __forceinline__ unsigned pack_hi(unsigned a, unsigned b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }
__device__ __forceinline__ u4v slots_left(float v)
{
    unsigned h, m, l;
    split3(v, h, m, l);
    return u4v{pack_hi(h, h), pack_hi(m, m), pack_hi(h, l), pack_hi(m, l)};
}
__device__ __forceinline__ u4v slots_right(float v)
{
    unsigned h, m, l;
    split3(v, h, m, l);
    const unsigned hm = pack_hi(h, m);
    return u4v{hm, hm, pack_hi(l, h), pack_hi(l, m)};
}
// 1 - |alpha|^2, and a bound of |1 - |alpha|^2| such that the difference of two is at
// most the larger bound, times 2^11.5; one that lets no group pass where the bound is
// past 0.8 or the magnitude past 1 by more than rounding (records near FP32's smallest
// squares)
__device__ __forceinline__ float pt_delta(cf32 v) { return (float)(1.0 - ((double)v.x * v.x + (double)v.y * v.y)); }
__device__ __forceinline__ float pt_bound(float delta)
{
    const float b = kPtD * (delta + 1.2e-7f);
    return delta < -1.2e-7f || b > 0.8f ? 1e6f : b;
}

// The 16 terms of a lane, added to acc.  db: delta of the lane's column, bb its bound;
// rd: deltas of the tile's rows, rb the bounds' maxima over runs of 8 rows, in LDS
// (lane rows 8 g + 4 h + r, g, r < 4).
template <int FN>
__device__ __forceinline__ void pt_tile(float (&acc)[16], f16v P, f16v Q, float db, float bb, const float *rd,
                                        const float *rb, int h, float V)
{
    if constexpr (FN == PT_SQUARE) {  // |a+b|^2 - |a-b|^2: d cancels
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = fmaf(-Q[r], Q[r], fmaf(P[r], P[r], acc[r]));
        return;
    }
    const auto roots = [&](int g) {  // P, Q of group g as |a+b|^v, |a-b|^v
        const f4v da = *reinterpret_cast<const f4v *>(rd + 8 * g + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int r = 4 * g + e;
            const float d = da[e] - db, dd = d * d, s = fmaf(P[r], P[r], dd), u = fmaf(Q[r], Q[r], dd);
            if constexpr (FN == PT_SQRT) {
                P[r] = hw_sqrt(s);
                Q[r] = hw_sqrt(u);
            } else {
                P[r] = hw_pow(s, V);
                Q[r] = hw_pow(u, V);
            }
        }
    };
    if constexpr (FN == PT_SQRT) {
        // min(|P|, |Q|) >= tau, tau = b^2 for the larger bound b = 2^11.5 B, follows from
        // ||P| - |Q|| <= 2 - 2B - 1.3 tau: P^2 + Q^2 = 4 |alpha beta|^2 >= 4 (1 - B)^2, and
        // sqrt(4 rho^2 - m^2) - m falls with m; 1e-6 for the rounding of the difference
        const f4v ra = *reinterpret_cast<const f4v *>(rb);
        float f[4], z[16];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            float m = 0.0f;
#pragma unroll
            for (int r = 4 * g; r < 4 * g + 4; ++r) {
                z[r] = fabsf(P[r]) - fabsf(Q[r]);
                m = fmaxf(m, fabsf(z[r]));
            }
            const float b = fmaxf(ra[g], bb);
            f[g] = fmaf(b, fmaf(1.3f, b, 2.0f / kPtD), m);
        }
        const float fm = fmaxf(fmaxf(f[0], f[1]), fmaxf(f[2], f[3]));
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(fm > 2.0f - 1e-6f) != 0, 0)) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                if (__builtin_amdgcn_ballot_w64(f[g] > 2.0f - 1e-6f) == 0) continue;
                roots(g);
#pragma unroll
                for (int r = 4 * g; r < 4 * g + 4; ++r) z[r] = P[r] - Q[r];
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] += z[r];
        return;
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) roots(g);
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] += P[r] - Q[r];  // the small difference first
}

constexpr int kPtWaves = 4;
constexpr int kPtChunk = 512;  // samples staged at a time
constexpr int kPtFlush = 4;    // chunks (16 terms a lane and tile each) summed in FP32 before FP64

__host__ __device__ constexpr int pt_bands(int tpw) { return kPtWaves * tpw - 1; }  // 32-lag bands a workgroup

// How the terms of one output row (a pair-window, or a pair whose rw windows are
// averaged) are spread: G units, each a run of windows, or (ns > 1) one of ns equal
// parts of one window's samples.
struct PtSplit {
    int G, ns, nblk;  // units a row, parts a window, lag blocks a row
};

// Workgroup of 4 waves: one lag block of 32 (4 TPW - 1) lags of one unit.  Tile c
// (wave c mod 4) is the square of terms (m, n) = (n0 + lagA + 32 c + i, n0 + j),
// i, j < 32, walked down the diagonal n0 = nstart, nstart + 32, ...: its sums over
// i - j = r belong to lag lagA + 32 c + r, so 4 TPW tiles cover 4 TPW - 1 bands of 32
// lags.  Each chunk of samples is staged in LDS by components (out-of-range samples
// as alpha = 0, whose terms are zero for V > 0).  The 16 FP32 sums a lane are added along the
// tile's diagonals in FP64 every 4 chunks (64 terms).
// Two or three waves a SIMD asked for: within 256 registers the MFMA results land in
// ordinary registers (else the compiler puts them in accumulation registers, three
// more moves a term).
// MFMA 32x32x16 layout: lane l holds A[l%32][8 (l/32) ..], B[8 (l/32) ..][l%32] and
// D[8 (r/4) + 4 (l/32) + r%4][l%32], r < 16; its half-wave holds the slots of one
// component: P (ax | ay)(2bx | 2by), Q (ax | ay)(-2by | 2bx).
template <int FN, int TPW>
__global__ void __launch_bounds__(64 * kPtWaves) __attribute__((amdgpu_waves_per_eu(TPW == 4 ? 2 : 3)))
k_pcc_time(const cf32 *__restrict__ phi, int S, int W, int N, int lag_first, int L, float V, double div, int mode,
           PtSplit sp, int row0, float *__restrict__ y, int out_ld, int out_off, double *__restrict__ part)
{
    constexpr int kT = 64 * kPtWaves, kTiles = kPtWaves * TPW, kA = kPtChunk + 32 * (kTiles - 1);
    __shared__ u4v bc[3][kPtChunk], ac[2][kA];                  // 2bx, 2by, -2by; ax, ay
    __shared__ __align__(16) float bd[kPtChunk], ad[kA], ab[kA / 8];  // deltas; the rows' bounds by 8
    // between chunks the operands' space serves the sums along diagonals
    float (*tile)[32 * 33] = reinterpret_cast<float (*)[32 * 33]>(ac);
    double (*diag)[64] = reinterpret_cast<double (*)[64]>(bc);
    static_assert(sizeof(float) * kPtWaves * 32 * 33 <= sizeof(ac) && sizeof(double) * kTiles * 64 <= sizeof(bc), "fit");
    const int t = threadIdx.x, lane = t & 63, h = lane >> 5, lj = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int ru = blockIdx.x / sp.nblk, u = ru % sp.G, row = row0 + ru / sp.G;
    // Workgroups go to the 8 XCDs in turn and the last lag block of a unit is short.  An even
    // number of blocks would put it on the same XCDs in every unit (780 pairs x 24 windows of
    // 1800, 481 lags: 8.7 ms, half the chip idle), so the blocks of a unit move on by one
    // each time the pattern of units over XCDs repeats (7.3 ms).
    const int g = sp.nblk & -sp.nblk, lb = (blockIdx.x % sp.nblk + (g > 1 ? ru / max(8 / g, 1) : 0)) % sp.nblk;
    const int p = mode == 0 ? row / W : row;
    // windows and sample range of this unit
    int w0, w1, part_i = 0;
    if (mode == 0) {
        w0 = row - p * W;
        w1 = w0 + 1;
        part_i = u;
    } else if (sp.ns > 1) {
        w0 = u / sp.ns;
        w1 = w0 + 1;
        part_i = u - w0 * sp.ns;
    } else {
        w0 = (int)((long long)u * W / sp.G);
        w1 = (int)((long long)(u + 1) * W / sp.G);
    }
    int i, j;
    pair_index(p, S, i, j);
    const int lagA = lag_first + lb * 32 * pt_bands(TPW);
    const int lagB = min(lagA + 32 * pt_bands(TPW) - 1, lag_first + L - 1);
    const int Lb = lagB - lagA + 1;
    int nstart = max(0, -lagB), nend = min(N, N - lagA);
    if (sp.ns > 1) {
        const int per = ((nend - nstart + sp.ns - 1) / sp.ns + 31) / 32 * 32;
        nstart += part_i * per;
        nend = min(nend, nstart + per);
    }
    const u4v *bp = bc[h] + lj, *bq = bc[h ? 0 : 2] + lj, *ap = ac[h] + lj;  // by half-wave

    float acc[TPW][16];
    double dsum[TPW];  // lane l < 63: the tile's diagonal r = l - 31
#pragma unroll
    for (int k = 0; k < TPW; ++k) {
        dsum[k] = 0.0;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[k][r] = 0.f;
    }
    auto flush = [&]() {
        float *sc = tile[wave];
#pragma unroll
        for (int k = 0; k < TPW; ++k) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                sc[(8 * (r >> 2) + 4 * h + (r & 3)) * 33 + lj] = acc[k][r];
                acc[k][r] = 0.f;
            }
            // the scratch is the wave's own: its writes land before its reads
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_wave_barrier();
            const int r = lane - 31;
#pragma unroll 8
            for (int jj = 0; jj < 32; ++jj) {
                const int ii = jj + r;
                if (ii >= 0 && ii < 32) dsum[k] += (double)sc[ii * 33 + jj];
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_wave_barrier();
        }
    };
    int chunks = 0;
    for (int w = w0; w < w1; ++w) {
        const cf32 *p1 = phi + (long long)(i * W + w) * N;
        const cf32 *p2 = phi + (long long)(j * W + w) * N;
        cf32 fb[kPtChunk / kT], fa[(kA + kT - 1) / kT];  // the next chunk's samples, loaded ahead
        auto fetch = [&](int n0) {
#pragma unroll
            for (int i = 0; i < kPtChunk / kT; ++i) {
                const int n = n0 + t + kT * i;
                fb[i] = n < nend ? p1[n] : cf32{0.f, 0.f};
            }
#pragma unroll
            for (int i = 0; i < (kA + kT - 1) / kT; ++i) {
                const int m = n0 + lagA + t + kT * i;
                fa[i] = m >= 0 && m < N ? p2[m] : cf32{0.f, 0.f};
            }
        };
        fetch(nstart);
        for (int n0 = nstart; n0 < nend; n0 += kPtChunk) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kPtChunk / kT; ++i) {
                const int e = t + kT * i;
                const u4v sy = slots_right(2 * fb[i].y);
                bc[0][e] = slots_right(2 * fb[i].x);
                bc[1][e] = sy;
                bc[2][e] = sy ^ 0x80008000u;
                bd[e] = pt_delta(fb[i]);
            }
#pragma unroll
            for (int i = 0; i < (kA + kT - 1) / kT; ++i) {
                const int e = t + kT * i;
                const float d = pt_delta(fa[i]);
                // the maximum over 8 samples: 8 lanes
                float b = pt_bound(d);
                b = fmaxf(b, __shfl_xor(b, 1, 64));
                b = fmaxf(b, __shfl_xor(b, 2, 64));
                b = fmaxf(b, __shfl_xor(b, 4, 64));
                if (e < kA) {
                    ac[0][e] = slots_left(fa[i].x);
                    ac[1][e] = slots_left(fa[i].y);
                    ad[e] = d;
                    if ((e & 7) == 0) ab[e >> 3] = b;
                }
            }
            __syncthreads();
            if (n0 + kPtChunk < nend) fetch(n0 + kPtChunk);
            // tiles of all steps in one sequence, software-pipelined: the operands of the
            // tile after next load and the next tile's MFMAs run while a tile's terms are
            // summed (its results in the other half of P, Q)
            const int nst = min(kPtChunk, nend - n0);
            f16v P[2], Q[2];
            u4v b_p = bp[0], b_q = bq[0], a_p = ap[32 * wave];
            auto mfma = [&](int x) {
                const f16v z = {};
                P[x] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(b8v, a_p), __builtin_bit_cast(b8v, b_p), z, 0, 0, 0);
                Q[x] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(b8v, a_p), __builtin_bit_cast(b8v, b_q), z, 0, 0, 0);
            };
            // operands of tile k of the step at n (a wave's tiles are c = wave, wave + 4, ...);
            // past the last step they are loaded, not used
            auto load = [&](int n, int k) {
                const int nb = min(n, kPtChunk - 32);
                if (k == 0) {
                    b_p = bp[nb];
                    b_q = bq[nb];
                }
                a_p = ap[nb + 32 * (wave + kPtWaves * k)];
            };
            mfma(0);
            load(0, 1);
            for (int n = 0; n < nst; n += 32) {
                const float db = bd[n + lj], bb = pt_bound(db);
#pragma unroll
                for (int k = 0; k < TPW; ++k) {
                    mfma((k + 1) & 1);
                    load(k + 2 < TPW ? n : n + 32, (k + 2) % TPW);
                    const int e0 = n + 32 * (wave + kPtWaves * k), m0 = n0 + lagA + e0;
                    // tiles of no lag of this block, or outside the other window, hold no terms
                    if (32 * (wave + kPtWaves * k) - 31 < Lb && m0 + 31 >= 0 && m0 < N)
                        pt_tile<FN>(acc[k], P[k & 1], Q[k & 1], db, bb, ad + e0, ab + e0 / 8, h, V);
                }
            }
            if (++chunks == kPtFlush) {
                chunks = 0;
                __syncthreads();
                flush();
            }
        }
    }
    __syncthreads();
    if (chunks) flush();
#pragma unroll
    for (int k = 0; k < TPW; ++k) diag[wave + kPtWaves * k][lane] = dsum[k];
    __syncthreads();
    // lag lagA + 32 c + r: diagonal r of tile c and diagonal r - 32 of tile c + 1
    for (int l = t; l < Lb; l += kT) {
        const int c = l >> 5, r = l & 31;
        const double sum = diag[c][31 + r] + (r ? diag[c + 1][r - 1] : 0.0);
        const int gl = lb * 32 * pt_bands(TPW) + l;
        if (sp.G > 1) {
            part[(long long)ru * L + gl] = sum;
        } else {
            const int lag = lagA + l, count = max(0, min(N, N - lag) - max(0, -lag));
            y[(long long)row * out_ld + out_off + gl] = (float)(sum / (div * count));
        }
    }
}

// x y - z w, within 1.5 ulp: 0 where x = z and y = w (or x = w and y = z)
__device__ __forceinline__ float prod_diff(float x, float y, float z, float w)
{
    const float p = z * w, e = fmaf(-z, w, p);
    return fmaf(x, y, -p) + e;
}

// 256 lags of one output row a workgroup, one a thread, over the overlap alone: for launches
// that the tiles' blocks of lags and chunks of samples do not fill (pt_direct_faster), and
// for V <= 0, where the terms of samples outside the windows are not zero (0^V) and a term
// grows without bound as a nears b or -b (P and Q without cancellation: exactly 0 for
// a = -b and a = b).  Bound by the vector unit, 12 operations a term: 2.4 T PCC1 terms/s
// (18720 pair-windows of 2000, 2001 lags) where the tiles reach 3.3, and 2.8 against 2.3
// at 241 lags.  LDS rows of 8 and 4 bytes: as rows of 16 their reads were the bound (1.3x
// the time at 241 lags); two lags a thread halved the reads but left most launches too
// few waves (0.6 .. 0.9x).
constexpr int kPdLags = 256, kPdChunk = 256, kPdRun = 64;  // terms summed in FP32 before FP64

template <int FN>
__device__ __forceinline__ float pd_term(cf32 a, float ad, cf32 b, float bd, float V)
{
    // b holds 2 beta: P, Q as in the tiles
    float P, Q;
    if constexpr (FN == PT_POW) {
        P = prod_diff(a.x, b.x, -a.y, b.y);
        Q = prod_diff(a.y, b.x, a.x, b.y);
    } else {
        P = fmaf(a.x, b.x, a.y * b.y);
        Q = fmaf(a.y, b.x, -(a.x * b.y));
    }
    if constexpr (FN == PT_SQUARE) return fmaf(P, P, -(Q * Q));
    const float d = ad - bd, dd = d * d, s = fmaf(P, P, dd), u = fmaf(Q, Q, dd);
    if constexpr (FN == PT_SQRT) return hw_sqrt(s) - hw_sqrt(u);
    if constexpr (FN == PT_HWPOW) return hw_pow(s, V) - hw_pow(u, V);
    return powf(s, V) - powf(u, V);
}

template <int FN>
__global__ void __launch_bounds__(kPdLags)
k_pcc_direct(const cf32 *__restrict__ phi, int S, int W, int N, int lag_first, int L, float V, double div, int mode,
             int nblk, int row0, float *__restrict__ y, int out_ld, int out_off)
{
    constexpr int kA = kPdChunk + kPdLags;
    __shared__ cf32 sb[kPdChunk], sa[kA];    // 2 beta, alpha (0 outside the window)
    __shared__ float db[kPdChunk], da[kA];   // 1 - |.|^2
    const int t = threadIdx.x, lb = blockIdx.x % nblk, row = row0 + blockIdx.x / nblk;
    const int p = mode == 0 ? row / W : row;
    const int w0 = mode == 0 ? row - p * W : 0, w1 = mode == 0 ? w0 + 1 : W;
    int i, j;
    pair_index(p, S, i, j);
    const int lagA = lag_first + lb * kPdLags, lagB = min(lagA + kPdLags - 1, lag_first + L - 1), lag = lagA + t;
    const int nstart = max(0, -lagB), nend = min(N, N - lagA);
    // samples this lag takes (V <= 0), or any lag of the wave: the others' terms are zero
    int lo0 = max(0, -lag), hi0 = lag <= lagB ? min(N, N - lag) : lo0;
    if constexpr (FN != PT_POW) {
        const int wl = lagA + 64 * __builtin_amdgcn_readfirstlane(t >> 6);
        lo0 = max(0, -min(wl + 63, lagB));
        hi0 = wl <= lagB ? min(N, N - wl) : lo0;
    }
    double acc = 0.0;
    for (int w = w0; w < w1; ++w) {
        const cf32 *p1 = phi + (long long)(i * W + w) * N;
        const cf32 *p2 = phi + (long long)(j * W + w) * N;
        for (int n0 = nstart; n0 < nend; n0 += kPdChunk) {
            __syncthreads();
            const int nc = min(kPdChunk, nend - n0);
            if (t < nc) {
                const cf32 v = p1[n0 + t];
                sb[t] = cf32{2.f * v.x, 2.f * v.y};
                db[t] = pt_delta(v);
            }
            // lanes past lagB in a wave that holds it read on: up to the next 64 lags
            const int na = nc + ((lagB - lagA) | 63);
            for (int e = t; e < na; e += kPdLags) {
                const int m = n0 + lagA + e;
                const cf32 v = m >= 0 && m < N ? p2[m] : cf32{0.f, 0.f};
                sa[e] = v;
                da[e] = pt_delta(v);
            }
            __syncthreads();
            const int lo = max(lo0 - n0, 0), hi = min(hi0 - n0, nc);
            for (int e0 = lo; e0 < hi; e0 += kPdRun) {
                const int e1 = min(e0 + kPdRun, hi);
                float sum = 0.f;
#pragma unroll 8
                for (int e = e0; e < e1; ++e) sum += pd_term<FN>(sa[e + t], da[e + t], sb[e], db[e], V);
                acc += (double)sum;
            }
        }
    }
    if (lag > lagB) return;
    const int count = max(0, min(N, N - lag) - max(0, -lag));
    y[(long long)row * out_ld + out_off + lb * kPdLags + t] = (float)(acc / (div * count));
}

// The G partial sums of every lag of a row, in order, normalised.
__global__ void __launch_bounds__(256)
k_pcc_time_sum(const double *__restrict__ part, int N, int lag_first, int L, int G, double div, float *__restrict__ y,
               int out_ld, int out_off)
{
    const int l = blockIdx.x * 256 + threadIdx.x;
    const long long row = blockIdx.y;  // G > 1 only where rows are few
    if (l >= L) return;
    double sum = 0.0;
    for (int u = 0; u < G; ++u) sum += part[(row * G + u) * L + l];
    const int lag = lag_first + l, count = max(0, min(N, N - lag) - max(0, -lag));
    y[row * out_ld + out_off + l] = (float)(sum / (div * count));
}

namespace {

// Lag blocks and units of a launch (rows: output rows; rw: windows a row sums).  The
// widest lag block that still gives kPtFill workgroups with one window a unit (the
// tile beyond the block's bands costs 1 in 4 TPW), then as many units a row as fill
// the chip that often: a row's windows in G runs, or each window's samples in ns
// parts of at least 512.  One workgroup a lag block ran 2.7 ms for 3 stations x 14
// windows of 2879 samples (42 workgroups), the split 0.25 ms.
constexpr long long kPtFill = 3072;

int pt_tpw(long long rows, int rw, int L)
{
    return rows * rw * ((L + 32 * pt_bands(4) - 1) / (32 * pt_bands(4))) >= kPtFill / 2 ? 4 : 2;
}

PtSplit pt_split(long long rows, int rw, int N, int L, int tpw)
{
    PtSplit s{1, 1, (L + 32 * pt_bands(tpw) - 1) / (32 * pt_bands(tpw))};
    const long long want = (kPtFill + rows * s.nblk - 1) / (rows * s.nblk);
    if (want <= rw) {
        s.G = (int)want;
    } else {
        s.ns = (int)std::min<long long>((want + rw - 1) / rw, std::max(1, N / 512));
        s.G = rw * s.ns;
    }
    return s;
}

// Whether one lag a thread is faster than the tiles: both times in us from the launch's
// shape.  Tiles: workgroups (two of TPW 4 or three of TPW 2 a CU run at once) of a fixed
// cost and, per 32 samples, the staging and products of all tiles and the terms of those
// that hold lags; a chip they do not fill runs them faster.  One lag a thread: the
// vector work of its waves, or a lone wave's latency.  The constants are those that pick
// the faster one in 240 measured launches (S 2 .. 100, W 1 .. 30, N 16 .. 4096, up to 2001
// lags; at worst 1.15x of the faster one's time, where the two are near each other and the
// records decide how many roots the tiles take).  The tiles alone ran at 0.1x of this
// kernel's speed for 18720 windows of 16, 0.65 .. 0.85x for as many of 600 .. 2000 and up
// to 501 lags; this kernel at 0.1x of theirs for few long windows.
bool pt_direct_faster(int fn, long long rows, int rw, int N, int lag_first, int L, int tpw, const PtSplit &sp)
{
    struct Cost {
        double unit, step4, tile4, step2, tile2, wave, serial, group;
    };
    static constexpr Cost kSqrt{11, 0.82, 0.14, 0.13, 1.0, 5.4e-4, 0.053, 3.5e-4};
    static constexpr Cost kPow{6.5, 0.3, 0.58, 0.25, 0.30, 7.6e-4, 0.056, 4.5e-4};
    static constexpr Cost kSquare{9, 0.5, 0.06, 0.26, 0.09, 5.5e-4, 0.040, 2.7e-4};
    const Cost &c = fn == PT_SQRT ? kSqrt : fn == PT_SQUARE ? kSquare : kPow;
    // samples a lag takes of a window, on average
    const double a = lag_first, b = lag_first + L - 1;
    const double n = N - (a < 0 && b > 0 ? (a * a + b * b) / (2 * (b - a)) : std::abs(a + b) / 2);
    // tiles
    const double windows = sp.ns > 1 ? 1.0 : (double)rw / sp.G, steps = n / 32 / sp.ns;
    // tiles a wave of a lag block, on average: all of them but in the last one
    const int last = L - (sp.nblk - 1) * 32 * pt_bands(tpw), tiles = std::min((last + 62) / 32, kPtWaves * tpw);
    const double deep = (double)((sp.nblk - 1) * tpw + (tiles + kPtWaves - 1) / kPtWaves) / sp.nblk;
    const double rounds = (double)rows * sp.G * sp.nblk / (tpw == 4 ? 512 : 768);
    const double turns = rounds <= 1 ? 0.6 : rounds < 3 ? std::ceil(rounds) : rounds + 0.5;
    const double step = tpw == 4 ? c.step4 + c.tile4 * deep : c.step2 + c.tile2 * deep;
    const double tiled = turns * (c.unit + windows * steps * step);
    // one lag a thread: between the larger of the two bounds (the longest lag's, for one wave)
    // and their sum
    const double work = rw * n / 32 * rows * (c.wave * ((L + 63) / 64) + c.group * ((L + kPdLags - 1) / kPdLags));
    const double alone = rw * (N - (a < 0 && b > 0 ? 0.0 : std::min(std::abs(a), std::abs(b)))) * c.serial;
    return std::pow(std::pow(work, 2.5) + std::pow(alone, 2.5), 0.4) < tiled;
}

template <int TPW>
int launch_pt(int fn, const cf32 *d_phi, int S, int W, int N, int lag_first, int L, float V, double div, int mode,
              const PtSplit &sp, int row0, unsigned blocks, float *d_y, int out_ld, int out_off, double *part, hipStream_t st)
{
    const dim3 g(blocks), b(64 * kPtWaves);
#define FPCC_PT(FN)                                                                                               \
    hipLaunchKernelGGL((k_pcc_time<FN, TPW>), g, b, 0, st, d_phi, S, W, N, lag_first, L, V, div, mode, sp, row0, d_y,    \
                       out_ld, out_off, part)
    switch (fn) {
    case PT_SQRT: FPCC_PT(PT_SQRT); break;
    case PT_SQUARE: FPCC_PT(PT_SQUARE); break;
    default: FPCC_PT(PT_HWPOW); break;
    }
#undef FPCC_PT
    FPCC_CHECK(hipGetLastError());
    return 0;
}

}  // namespace

size_t pcc_time_scratch(int S, int W, int N, int L, int mode)
{
    if (L <= 0) return 0;
    const long long P = (long long)S * (S - 1) / 2, rows = mode == 0 ? P * W : P;
    const int rw = mode == 0 ? 1 : W;
    const PtSplit sp = pt_split(rows, rw, N, L, pt_tpw(rows, rw, L));
    return sp.G > 1 ? sizeof(double) * (size_t)rows * sp.G * (size_t)L : 0;
}

int launch_pcc_time(const cf32 *d_phi, int S, int W, int N, int lag_first, int L, double v, int pcc1, int mode,
                    float *d_y, int out_ld, int out_off, double *part, hipStream_t st)
{
    if (L <= 0) return 0;
    const long long P = (long long)S * (S - 1) / 2, rows = mode == 0 ? P * W : P;
    if (!rows) return 0;
    const int rw = mode == 0 ? 1 : W;
    const int tpw = pt_tpw(rows, rw, L);
    PtSplit sp = pt_split(rows, rw, N, L, tpw);
    if (!part) sp.G = sp.ns = 1;
    if (rows > 0x7fffffff) {
        fprintf(stderr, "fastpcc: %lld output rows exceed one job\n", rows);
        return -1;
    }
    const float V = (float)(v / 2);
    // PCC1, and PCC-v at v = 1 (|.|^2 to the power 1/2), take square roots; PCC-v at
    // v = 2 takes the squared magnitudes themselves (powf(x, 1) = x)
    const int fn = pcc1 || V == 0.5f ? PT_SQRT : V == 1.0f ? PT_SQUARE : V > 0.f ? PT_HWPOW : PT_POW;
    // per lag: sum / (2 count) (:276) or sum / (2^(v/2) count) (:334), over the windows of a row
    const double div = (pcc1 ? 2.0 : pow(2.0, (double)V)) * rw;
    const bool direct = fn == PT_POW || pt_direct_faster(fn, rows, rw, N, lag_first, L, tpw, sp);
    ProfScope prof(direct ? (pcc1 ? "pcc1_direct" : "pccv_direct") : pcc1 ? "pcc1_time" : "pccv_time", st);
    // the rows of one launch at a time; rows that are split (G > 1) are few
    const int nblk = direct ? (L + kPdLags - 1) / kPdLags : sp.nblk, G = direct ? 1 : sp.G;
    const long long step = std::max(1LL, kMostBlocks / ((long long)nblk * G));
    for (long long r0 = 0; r0 < rows; r0 += step) {
        const int row0 = (int)r0;
        const unsigned blocks = (unsigned)(std::min(step, rows - r0) * G * nblk);
        if (direct) {
            const dim3 g(blocks), b(kPdLags);
#define FPCC_PD(FN)                                                                                               \
    hipLaunchKernelGGL(k_pcc_direct<FN>, g, b, 0, st, d_phi, S, W, N, lag_first, L, V, div, mode, nblk, row0, d_y,    \
                       out_ld, out_off)
            switch (fn) {
            case PT_SQRT: FPCC_PD(PT_SQRT); break;
            case PT_SQUARE: FPCC_PD(PT_SQUARE); break;
            case PT_HWPOW: FPCC_PD(PT_HWPOW); break;
            default: FPCC_PD(PT_POW); break;
            }
#undef FPCC_PD
            FPCC_CHECK(hipGetLastError());
            continue;
        }
        const auto launch = tpw == 4 ? launch_pt<4> : launch_pt<2>;
        const int r = launch(fn, d_phi, S, W, N, lag_first, L, V, div, mode, sp, row0, blocks, d_y, out_ld, out_off, part, st);
        if (r) return r;
    }
    if (G == 1) return 0;
    hipLaunchKernelGGL(k_pcc_time_sum, dim3((L + 255) / 256, (unsigned)rows), dim3(256), 0, st, part, N, lag_first, L,
                       sp.G, div, d_y, out_ld, out_off);
    FPCC_CHECK(hipGetLastError());
    return 0;
}

}  // namespace fpcc
