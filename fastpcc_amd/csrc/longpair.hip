// Pair stage of transforms longer than one workgroup's LDS, without a pass through HBM.
//
// The correlation is real and only the lags of a window are wanted, so from the
// spectra in the two-pass order (bin k1 + N1 k2 at k1 N2 + k2) one kernel
//  - folds the cross spectrum Y = conj(F_i) F_j (or a Gram row) to the half-length
//    spectrum Z of M = Nz/2 bins, y[2m] + i y[2m+1] = IFFT_M(Z)[m] (pcc2.hip); Z of rows
//    k1 and N1 - k1 needs only those two rows of Y,
//  - inverts each row over k2 (H = N2/2 points) in LDS: x[k1][n2], times W_M^{-k1 n2},
//  - and, instead of the N1-point transforms over k1, adds the row pair's terms
//    x[k1] W^{k1 n1} + x[N1-k1] conj(W^{k1 n1}), W = exp(2 pi i / N1), to the outputs
//    m = n1 H + n2 whose n1 the lag window reads (a few of N1), in registers.
// With s = x[k1] + x[N1-k1] and d = x[k1] - x[N1-k1] outputs n1 and -n1 share the sums
// E = sum s cos and O = sum d sin: out[+-n1] = E +- i O, four multiply-adds a row pair.
//
// A workgroup takes a share of the row pairs of one pair (or pair-window) and leaves
// its sums in the scratch row's own place; k_long_lags adds the shares and writes the
// normalised lags.  Shares go to consecutive workgroups, so each XCD keeps reading
// the same eighth (or quarter ..) of every station's spectrum, which its L2 holds.
// Twiddles are products of FP64 table entries rounded once, and the shares are added in
// FP64: with FP32 ones the fold and the sums cost more accuracy than the passes saved
// (16 stations x 86400, 1-bit: error against 64 bits 1.90e-7 in two passes, 2.03e-7 with
// FP32 twiddles, 1.78e-7 so; at most 3% of the time).
// Against the inverse row and column passes (rows of Nz written and read again, both
// of full length): 32 stations x 86400, +-2000 lags 477 -> 214 us, one pair x 649
// windows x 21600, +-3000 lags 282 -> 167 us; bound by the latency of its loads and folds
// (vector unit 21-30% busy, 1.7 TB/s of HBM).
#include <algorithm>
#include <cstdlib>
#include "bigfft.hpp"
#include "kernels.hpp"
#include "lagwin.hpp"
#include "pairs.hpp"
#include "profile.hpp"
#include "tile_fft.hpp"

namespace fpcc {

enum { LP_CROSS = 0, LP_REAL = 1, LP_GRAM = 2 };  // LP_REAL: spectra of real signals, Y[Nz-k] = conj Y[k]

struct LongArgs {
    const cf32 *F, *F2;         // spectra (stations i, j), or Gram rows (F)
    cf32 *dst;                  // scratch rows (may be the Gram rows)
    long long bstride;
    int N1, S, W, Wb, wsel, wsum, pair0;  // as RowArgs
    int G, upg, A;              // shares an item, units a share, largest |n1|
    const cf32 *twH, *twR;      // passes of H, full table of N1
    const cf64 *twN, *twC;      // split table of Nz, full table of N2
};

__host__ __device__ constexpr int lp_ld(int H) { return H == 256 ? 274 : H == 512 ? 544 : 1088; }

template <int H>
__device__ __forceinline__ void lp_rows_ifft(cf32 *lds, const cf32 *__restrict__ tw)
{
    if constexpr (H == 256) ctb_fft<256, 16, lp_ld(256), +1, 16, 16>(lds, tw);
    else if constexpr (H == 512) ctb_fft<512, 8, lp_ld(512), +1, 8, 8, 8>(lds, tw);
    else ctb_fft<1024, 4, lp_ld(1024), +1, 16, 8, 8>(lds, tw);
}

__device__ __forceinline__ cf32 lp_round(cf64 w) { return cf32{(float)w.x, (float)w.y}; }

// Z[k] of the fold from a = Y[k] + conj Y[Nz-k] and c = Y[M-k] + conj Y[M+k], w = W_Nz^{-k}
__device__ __forceinline__ cf32 lp_fold(cf32 a, cf32 c, cf32 w)
{
    const cf32 P = cf32{a.x + c.x, a.y - c.y}, Q = cf32{a.x - c.x, a.y + c.y}, wq = cmul(w, Q);
    return cf32{P.x - wq.y, P.y + wq.x};
}

// H = N2/2; AB: bound of the outputs' |n1| (registers); 16 rows of 256 points (8 of 512,
// 4 of 1024), i.e. 4096 points, a unit.
template <int H, int AB, int SRC>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(H == 256 ? 3 : 2)))
k_long_pair(LongArgs a)
{
    constexpr int N2 = 2 * H, PU = 2048 / H, TP = 256 / PU, LD = lp_ld(H), EP = H / 256;
    static_assert(H / TP == 8, "eight folds a thread and unit");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cf32 *lds = reinterpret_cast<cf32 *>(smem_raw);
    const int t = threadIdx.x, N1 = a.N1;
    const int b = blockIdx.x / a.G, g = blockIdx.x - b * a.G;
    const long long n = (long long)N1 * N2;
    const cf32 *Fi = nullptr, *Fj = nullptr;
    int W = 1;
    if (SRC == LP_GRAM) {
        Fi = a.F + (long long)b * a.bstride;
    } else {
        int ci, cj;
        const int q = b / a.Wb;
        pair_index(a.pair0 + q, a.S, ci, cj);
        const int w0 = a.wsum ? 0 : a.wsel + (b - q * a.Wb);
        W = a.wsum ? a.W : 1;
        Fi = a.F + (long long)(ci * a.W + w0) * n;
        Fj = a.F2 + (long long)(cj * a.W + w0) * n;
    }
    const int pq = t / TP, c = t % TP;  // fold: row pair of the unit, first k2
    const cf64 wc = conj(a.twC[c]);  // exp(2 pi i c / N2)
    // sums: outputs n2 = t + 256 e
    cf32 E[EP][AB + 1], O[EP][AB + 1];
#pragma unroll
    for (int e = 0; e < EP; ++e) {
#pragma unroll
        for (int i = 0; i <= AB; ++i) E[e][i] = O[e][i] = cf32{0.f, 0.f};
    }
    for (int u = g * a.upg; u < (g + 1) * a.upg; ++u) {
        {
            const int pi = u * PU + pq;  // row pair (pi, N1 - pi); (0, N1/2) for pi = 0
            const int ra = pi, rb = pi ? N1 - pi : N1 / 2;
            // row factor of the fold twiddles, exp(2 pi i pi / Nz) wc
            const cf64 wr = cmul(conj(a.twN[pi]), wc);  // pi < kTwLo
            // four of a thread's eight bins at a time: their loads in flight together fill
            // the registers three workgroups a CU leave
#pragma unroll 1
            for (int hs = 0; hs < 2; ++hs) {
                const cf64 wrh = hs ? rot<+1>(wr) : wr;  // W_16^4 = i
                const int k0 = c + 4 * TP * hs;
                cf32 av[4], cv[4];
#pragma unroll
                for (int s = 0; s < 4; ++s) av[s] = cv[s] = cf32{0.f, 0.f};
                for (int w = 0; w < W; ++w) {
                    const cf32 *fi = Fi + w * n, *fj = Fj + w * n;
                    auto Y = [&](int r, int k) {
                        const int o = r * N2 + k;
                        return SRC == LP_GRAM ? fi[o] : cmulc(fi[o], fj[o]);
                    };
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        const int k = k0 + TP * s;
                        // bins k, M - k (and Nz - k, M + k); row 0 is its own mirror, k2 -> -k2
                        const cf32 y0 = Y(ra, k), y2 = pi ? Y(rb, H - 1 - k) : Y(0, H - k);
                        if (SRC == LP_REAL) {
                            av[s] = av[s] + y0;
                            cv[s] = cv[s] + y2;
                        } else {
                            const cf32 y1 = pi ? Y(rb, N2 - 1 - k) : Y(0, (N2 - k) & (N2 - 1)), y3 = Y(ra, k + H);
                            av[s] = av[s] + cf32{y0.x + y1.x, y0.y - y1.y};
                            cv[s] = cv[s] + cf32{y2.x + y3.x, y2.y - y3.y};
                        }
                    }
                }
                sfor<4>([&](auto sc) {
                    constexpr int s = sc();
                    const int k = k0 + TP * s;
                    const cf32 w = lp_round(twc<+1, 16, s>(wrh));  // exp(2 pi i TP s / N2) = W_16^s
                    cf32 x = av[s], z = cv[s];
                    if (SRC == LP_REAL && pi == 0 && k == 0) x.y = z.y = 0.f;  // DC and Nyquist of a real signal
                    lds[pq * LD + ct_pad(k)] = lp_fold(x, z, w);
                    if (pi) lds[(PU + pq) * LD + ct_pad(H - 1 - k)] = lp_fold(z, x, cf32{-w.x, w.y});
                });
            }
            if (pi == 0) {  // row N1/2: its own mirror, k2 -> N2 - 1 - k2
                const cf64 wh = cmul(wr, conj(a.twN[N1 / 2]));
#pragma unroll 1
                for (int s = 0; s < 8; ++s) {
                    const int k = c + TP * s;
                    cf32 x = cf32{0.f, 0.f}, z = cf32{0.f, 0.f};
                    for (int w = 0; w < W; ++w) {
                        const cf32 *fi = Fi + w * n + (long long)rb * N2, *fj = Fj + w * n + (long long)rb * N2;
                        auto Y = [&](int q) { return SRC == LP_GRAM ? fi[q] : cmulc(fi[q], fj[q]); };
                        const cf32 y0 = Y(k), y2 = Y(H - 1 - k);
                        if (SRC == LP_REAL) {
                            x = x + y0;
                            z = z + y2;
                        } else {
                            const cf32 y1 = Y(N2 - 1 - k), y3 = Y(k + H);
                            x = x + cf32{y0.x + y1.x, y0.y - y1.y};
                            z = z + cf32{y2.x + y3.x, y2.y - y3.y};
                        }
                    }
                    lds[(PU + pq) * LD + ct_pad(k)] = lp_fold(x, z, lp_round(cmul(wh, conj(a.twC[TP * s]))));
                }
            }
        }
        __syncthreads();
        lp_rows_ifft<H>(lds, a.twH);
#pragma unroll 2
        for (int q = 0; q < PU; ++q) {
            const int pi = __builtin_amdgcn_readfirstlane(u * PU + q);
#pragma unroll
            for (int e = 0; e < EP; ++e) {
                const int n2 = t + 256 * e;
                const cf32 xa = lds[q * LD + ct_pad(n2)], xb = lds[(PU + q) * LD + ct_pad(n2)];
                if (pi == 0) {  // rows 0 and N1/2: W^{(N1/2) n1} = (-1)^n1, W_M^{(N1/2) n2} = W_Nz^{N1 n2}
                    const cf32 x1 = cmul(xb, lp_round(conj(tw_m(a.twN, (unsigned)N1 * (unsigned)n2))));
                    const cf32 s = xa + x1, d = xa - x1;
#pragma unroll
                    for (int i = 0; i <= AB; ++i) E[e][i] = E[e][i] + (i & 1 ? d : s);
                } else {
                    const cf64 wt = conj(tw_m(a.twN, 2u * (unsigned)pi * (unsigned)n2));
                    const cf32 x0 = cmul(xa, lp_round(wt)), x1 = cmul(xb, lp_round(conj(cmul(wt, a.twC[2 * n2]))));
                    const cf32 s = x0 + x1, d = x0 - x1;
#pragma unroll
                    for (int i = 0; i <= AB; ++i) {
                        const cf32 w = a.twR[(unsigned)(pi * i) & (unsigned)(N1 - 1)];  // (cos, -sin)
                        E[e][i].x = fmaf(s.x, w.x, E[e][i].x);
                        E[e][i].y = fmaf(s.y, w.x, E[e][i].y);
                        O[e][i].x = fmaf(-d.x, w.y, O[e][i].x);
                        O[e][i].y = fmaf(-d.y, w.y, O[e][i].y);
                    }
                }
            }
        }
        __syncthreads();
    }
    // out[n1] at (n1 + A) H + n2 of this share's place: the first rows it read
    cf32 *out = a.dst + (long long)b * a.bstride + (long long)g * a.upg * 4096;
#pragma unroll
    for (int e = 0; e < EP; ++e)
#pragma unroll
        for (int i = 0; i <= AB; ++i) {
            if (i > a.A) break;
            const cf32 x = E[e][i], o = O[e][i];
            const int n2 = t + 256 * e;
            out[(a.A + i) * H + n2] = cf32{x.x - o.y, x.y + o.x};
            if (i) out[(a.A - i) * H + n2] = cf32{x.x + o.y, x.y - o.x};
        }
}

// Lags of item b from its shares' outputs, with the two-pass inverse's epilogue.  f: what
// one share's outputs are to the n-point inverse's value (1/2 where the fold holds twice
// the half spectrum); not part of ca.scale, which the exact short overlaps take as well.
__global__ void __launch_bounds__(256)
k_long_lags(ColArgs ca, const cf32 *__restrict__ C, long long bstride, int H, int n, int G, int gstride, int A, float f)
{
    const int l = blockIdx.x * 256 + threadIdx.x, b = blockIdx.y;
    if (l >= ca.L) return;
    const int q = b / ca.Wb, w = ca.wsel + (b - q * ca.Wb), p = ca.pair0 + q;
    int i = 0, j = 0;
    if (ca.norm == 1) pair_index(p, ca.S, i, j);
    const int lag = ca.lag0 + l, m = lag >> 1;  // floor
    const float *row = reinterpret_cast<const float *>(C + (long long)b * bstride + (A * H + m)) + (lag & 1);
    double v = 0.0;
    for (int s = 0; s < G; ++s) v += (double)row[2LL * s * gstride];
    lagwin_store(ca, p, w, i, j, n, l, f * (float)v);
}

namespace {

// largest |n1| of the lags' half-length index m = n1 H + n2
int lp_reach(int lag0, int L, int H)
{
    auto fdiv = [](int v, int d) { return v >= 0 ? v / d : -((-v + d - 1) / d); };
    return std::max(std::abs(fdiv(lag0, 2 * H)), std::abs(fdiv(lag0 + L - 1, 2 * H)));
}

template <int H, int AB>
int launch_lp(const LongArgs &a, int src, int blocks, hipStream_t st)
{
    const size_t lds = sizeof(cf32) * (4096 / H) * (size_t)lp_ld(H);
    const dim3 g(blocks), t(256);
    if (src == LP_CROSS) hipLaunchKernelGGL((k_long_pair<H, AB, LP_CROSS>), g, t, lds, st, a);
    else if (src == LP_REAL) hipLaunchKernelGGL((k_long_pair<H, AB, LP_REAL>), g, t, lds, st, a);
    else hipLaunchKernelGGL((k_long_pair<H, AB, LP_GRAM>), g, t, lds, st, a);
    FPCC_CHECK(hipGetLastError());
    return 0;
}

}  // namespace

// Rows of 512, 1024 or 2048 bins (the splits of 2^14 .. 2^20), at least one whole unit,
// lags whose sums stay in registers (|n1| H <= 3072: within +-6144; the sums cost 2 |n1|
// multiply-adds a bin) and fit the rows a share read.
// And work for half the chip: the units of all items are its workgroups, against one
// for every four rows of the two passes.  1-bit, one window: 72 units 0.98x of the two
// passes' speed, 144 1.09x, 182 1.22x (N 10000, 24000, 10000); with windows summed
// unit by unit 6 units ran at half their speed (3 pairs x 40 windows of 12001).
bool long_pair_ok(const BigPlan &bp, int lag0, int L, long long nbatch, int wsum)
{
    if (!bp.ok || (bp.n2 != 512 && bp.n2 != 1024 && bp.n2 != 2048)) return false;
    const int H = bp.n2 / 2, PU = 2048 / H, U = bp.n1 / (2 * PU);
    if (U < 1 || (bp.n1 & (bp.n1 - 1))) return false;
    if (nbatch * U < (wsum > 1 ? 512 : 128)) return false;
    const int A = lp_reach(lag0, L, H);
    return A * H <= 3072 && (long long)(2 * A + 1) * H <= (long long)U * 4096;
}

int run_long_pair(const BigPlan &bp, const RowArgs &ra, const ColArgs &ca, bool real, int nbatch, hipStream_t st,
                  const char *name)
{
    if (nbatch <= 0) return 0;
    if (!long_pair_ok(bp, ca.lag0, ca.L, nbatch, ra.wsum ? ra.Wfull : 1) || nbatch > 65535) return -1;
    const int H = bp.n2 / 2, PU = 2048 / H, U = bp.n1 / (2 * PU);
    LongArgs a{};
    const bool gram = ra.op == ROW_INV_PLAIN;
    a.F = gram ? ra.src : ra.F;
    a.F2 = ra.F2 ? ra.F2 : ra.F;
    a.dst = ra.dst;
    a.bstride = ra.bstride;
    a.N1 = bp.n1;
    a.S = ra.Sst;
    a.W = ra.Wfull;
    a.Wb = ra.Wb;
    a.wsel = ra.wsel;
    a.wsum = ra.wsum;
    a.pair0 = ra.pair0;
    a.A = lp_reach(ca.lag0, ca.L, H);
    // as many shares as keep the sums within the rows each read, fewer (less to add up)
    // where the items alone give the chip eight workgroups a CU
    a.upg = 1;
    while ((2 * a.A + 1) * H > a.upg * 4096) a.upg *= 2;
    while (2 * a.upg <= U && (long long)nbatch * (U / (2 * a.upg)) >= 2048) a.upg *= 2;
    a.G = U / a.upg;
    a.twN = (const cf64 *)get_split_twiddles(bp.n, true);
    a.twH = (const cf32 *)(H == 256 ? get_order_twiddles(256, {16, 16}) : H == 512 ? get_order_twiddles(512, {8, 8, 8})
                                                                          : get_order_twiddles(1024, {16, 8, 8}));
    a.twR = (const cf32 *)get_full_twiddles(bp.n1, false);
    a.twC = (const cf64 *)get_full_twiddles(bp.n2, true);
    if (!a.twN || !a.twH || !a.twR || !a.twC) return -1;
    if ((long long)nbatch * a.G > 0x7fffffff) return -1;
    const int src = gram ? LP_GRAM : real ? LP_REAL : LP_CROSS, blocks = nbatch * a.G, e = a.A * H / 256;
    int r;
    {
        ProfScope prof(name, st);
        if (H == 256) r = e <= 4 ? launch_lp<256, 4>(a, src, blocks, st) : e <= 8 ? launch_lp<256, 8>(a, src, blocks, st)
                                                                                   : launch_lp<256, 12>(a, src, blocks, st);
        else if (H == 512) r = e <= 4 ? launch_lp<512, 2>(a, src, blocks, st) : e <= 8 ? launch_lp<512, 4>(a, src, blocks, st)
                                                                                        : launch_lp<512, 6>(a, src, blocks, st);
        else r = e <= 4 ? launch_lp<1024, 1>(a, src, blocks, st) : e <= 8 ? launch_lp<1024, 2>(a, src, blocks, st)
                                                                          : launch_lp<1024, 3>(a, src, blocks, st);
    }
    if (r) return r;
    const float f = src == LP_REAL ? 1.0f : 0.5f;
    ProfScope prof("long_lags", st);
    hipLaunchKernelGGL(k_long_lags, dim3((ca.L + 255) / 256, nbatch), dim3(256), 0, st, ca, (const cf32 *)a.dst, a.bstride, H,
                       bp.n, a.G, a.upg * 4096, a.A, f);
    FPCC_CHECK(hipGetLastError());
    return 0;
}

}  // namespace fpcc
