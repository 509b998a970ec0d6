// Pair stage of windows with zero-pad lengths Nz = 512 .. 8192 (M = Nz/2 = 256 .. 4096) on
// compile-time FP32 inverses: PCC2 spectra (Nz up to 4096; pair stage of 8192 in gram.hip),
// 1-bit half spectra, Gram rows (Nz up to 4096).
//
// A transform takes M/8 threads (one radix-8 butterfly a thread and pass) and two LDS
// buffers of M values, and a workgroup of 256 threads (512 at M 4096) runs 2048/M of
// them: 32 KB, so that a CU holds several workgroups at every length.  Thread t folds
// bins k = t + i M/8 (i < 4) and M - k from one load of each.  Where every window counts
// alike (PCC2 and 1-bit: the overlap normalisation does not depend on the window) the mean
// over windows is one inverse of the spectra's sum (in FP64); per-window outputs are a transform
// each, spread over the chip however few the pairs.
// Whole jobs, against the runtime plan with 512 threads a transform and an inverse per
// window: 45 stations x 30 windows of 1800, 1-bit, every window 526 us, here 240 us
// (output 142 MB), their mean 459 us, 135 us; 50 stations x 20 x 600 PCC2, every window
// 248 us, 84 us; 97 stations x 17 x 2880 Gram 312 us, 291 us.  Bound by reading the
// spectra through the caches.
#include <algorithm>
#include <type_traits>
#include "edge.hpp"
#include "engine.hpp"
#include "kernels.hpp"
#include "pairs.hpp"
#include "profile.hpp"

namespace fpcc {

enum { PS_PCC2 = 0, PS_REAL = 1, PS_GRAM = 2 };

struct PsArgs {
    const cf32 *A, *B;  // spectra of stations i and j (rows of ld), or Gram rows (A, layout gl)
    long long ld;
    GLayout gl;
    int S, W, N, lag0, L, units;
    float scale;
    int count;          // PS_GRAM: divide by the overlap
    const float *edge;  // window edges (exact short overlaps), or null
    int K;
    float *y;
    const cf32 *tw, *twc;
};

// One pass of fft_core.hpp's ct_pass_oop by the NT threads of a transform.
template <int M, int NT, int R, int NS, int LIN, int LOUT>
__device__ __forceinline__ void ps_pass(const cf32 *in, cf32 *out, const cf32 *__restrict__ tw, int t)
{
    constexpr int NB = M / R, BPT = (NB + NT - 1) / NT;
#pragma unroll
    for (int i = 0; i < BPT; ++i) {
        const int b = t + i * NT;
        if (NB % NT == 0 || b < NB) {
            cf32 v[R];
#pragma unroll
            for (int r = 0; r < R; ++r) v[r] = in[ct_lay<LIN>(b + r * NB)];
            const int k = b % NS;
            if (NS > 1) {
#pragma unroll
                for (int r = 1; r < R; ++r) v[r] = cmulc(tw[(r - 1) * NS + k], v[r]);
            }
            Dft<R, +1>::run(v);
            const int base = (b - k) * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) out[ct_lay<LOUT>(base + r * NS)] = v[r];
        }
    }
    __syncthreads();
}

// Last radix: 8 x 8 x .. with the rest
__host__ __device__ constexpr int ps_last(int M) { return M == 256 || M == 2048 ? 4 : M == 1024 ? 2 : 8; }

template <int M>
__device__ __forceinline__ cf32 *ps_ifft(cf32 *a, cf32 *b, const cf32 *__restrict__ tw, int t)
{
    constexpr int NT = M / 8, RL = ps_last(M);
    ps_pass<M, NT, 8, 1, 0, 2>(a, b, tw, t);
    if constexpr (M <= 512) {
        ps_pass<M, NT, 8, 8, 2, 0>(b, a, tw + 7, t);
        ps_pass<M, NT, RL, 64, 0, 0>(a, b, tw + 7 + 56, t);
        return b;
    } else {
        ps_pass<M, NT, 8, 8, 2, 2>(b, a, tw + 7, t);
        ps_pass<M, NT, 8, 64, 2, 0>(a, b, tw + 7 + 56, t);
        ps_pass<M, NT, RL, 512, 0, 0>(b, a, tw + 7 + 56 + 448, t);
        return a;
    }
}

// MODE 0: every window, y[p][w][L]; 1: the windows' mean (Gram rows: already summed)
template <int M, int SRC, int MODE, bool BATCH>
__global__ void __launch_bounds__(M == 4096 ? 512 : 256)
k_pair_short(PsArgs a, GnBatch jb, int block0)
{
    constexpr int NT = M / 8, TB = M == 4096 ? 512 : 256, TPB = TB / NT, Nz = 2 * M;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int g = threadIdx.x / NT, t = threadIdx.x % NT;
    cf32 *buf0 = reinterpret_cast<cf32 *>(smem_raw) + g * 2 * M, *buf1 = buf0 + M;
    const int unit = (blockIdx.x + block0) * TPB + g;
    const bool live = unit < a.units;
    int u = live ? unit : a.units - 1;
    if (BATCH) {
        int j = 0;
        while (j + 1 < jb.n && u >= jb.b0[j + 1]) ++j;
        u -= jb.b0[j];
        a.A = (const cf32 *)jb.Xa[j];
        a.B = (const cf32 *)jb.Xb[j];
        a.S = jb.S[j];
        a.W = jb.W[j];
        a.N = jb.N[j];
        a.lag0 = jb.lag0[j];
        a.L = jb.L[j];
        a.y = jb.y[j];
        a.edge = jb.edge[j];
        a.K = jb.K[j];
    }
    const int W = a.W;
    const int p = MODE == 0 ? u / W : u;
    const int w0 = MODE == 0 ? u - p * W : 0, w1 = MODE == 0 ? w0 + 1 : W;
    int i = 0, j = 0;
    if (SRC != PS_GRAM || a.edge) pair_index(p, a.S, i, j);
    // folded sums (see pcc2.hip): av at bin k, cv at M - k, ph at M/2
    typedef std::conditional_t<SRC != PS_GRAM && MODE == 1, cf64, cf32> Acc;  // the windows' sums
    Acc av[4], cv[4], ph{};
#pragma unroll
    for (int q = 0; q < 4; ++q) av[q] = cv[q] = Acc{};
    auto add = [](Acc &s, cf32 v) {
        s.x += v.x;
        s.y += v.y;
    };
    if constexpr (SRC == PS_GRAM) {
        auto G = [&](int k) {
            return a.A[(long long)(k >> a.gl.sh) * a.gl.gs + p * a.gl.pl + (k & ((1 << a.gl.sh) - 1))];
        };
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int k = t + NT * q;
            av[q] = G(k);
            cv[q] = G(M - k);
        }
        if (t == 0) ph = G(M / 2);
    } else {
        for (int w = w0; w < w1; ++w) {
            const cf32 *f = a.A + (long long)(i * W + w) * a.ld, *h = a.B + (long long)(j * W + w) * a.ld;
            auto Y = [&](int k) { return cmulc(f[k], h[k]); };
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int k = t + NT * q;
                const cf32 y0 = Y(k), y2 = Y(M - k);
                if (SRC == PS_REAL) {
                    add(av[q], y0);
                    add(cv[q], y2);
                } else {
                    const cf32 y1 = Y((Nz - k) & (Nz - 1)), y3 = Y(M + k);
                    add(av[q], cf32{y0.x + y1.x, y0.y - y1.y});
                    add(cv[q], cf32{y2.x + y3.x, y2.y - y3.y});
                }
            }
            if (t == 0) {
                const cf32 u0 = Y(M / 2);
                if (SRC == PS_REAL) {
                    add(ph, u0);
                } else {
                    const cf32 u1 = Y(Nz - M / 2);
                    add(ph, cf32{u0.x + u1.x, u0.y - u1.y});
                }
            }
        }
    }
    auto fold = [&](cf32 x, cf32 z, cf32 w) {
        const cf32 P = cf32{x.x + z.x, x.y - z.y}, Q = cf32{x.x - z.x, x.y + z.y}, wq = cmul(w, Q);
        return cf32{P.x - wq.y, P.y + wq.x};
    };
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int k = t + NT * q;
        cf32 x = cf32{(float)av[q].x, (float)av[q].y}, z = cf32{(float)cv[q].x, (float)cv[q].y};
        if (k == 0) x.y = z.y = 0.f;  // DC and Nyquist of a real signal's spectrum are real
        const cf32 w = a.twc[k];
        buf0[k] = fold(x, z, w);
        if (k) buf0[M - k] = fold(z, x, cf32{-w.x, w.y});
    }
    if (t == 0) buf0[M / 2] = cf32{2.f * (float)ph.x, -2.f * (float)ph.y};
    __syncthreads();
    const cf32 *z = ps_ifft<M>(buf0, buf1, a.tw, t);
    if (!live) return;
    float *dst = a.y + (long long)u * a.L;
    for (int l = t; l < a.L; l += NT) {
        const int lag = a.lag0 + l, n = lag & (Nz - 1);
        const cf32 v = z[n >> 1];
        const float r = a.scale * ((n & 1) ? v.y : v.x);
        if (SRC == PS_PCC2 || (SRC == PS_GRAM && !a.count)) {
            dst[l] = MODE == 1 && SRC == PS_PCC2 ? r / (float)W : r;
        } else {
            // counts: exact sums over short overlaps, the mean over the windows, the overlap
            const int m = a.N - abs(lag);
            double c = (double)r;
            if (a.edge && m > 0 && m < a.K)
                c = edge_corr(a.edge, a.K, W, i, j, w0, w1, lag, m, true) * (SRC == PS_GRAM ? (double)a.scale * (double)Nz : 1.0);
            if (SRC == PS_REAL && MODE == 1) c /= (double)W;
            dst[l] = (float)(c / (double)m);
        }
    }
}

namespace {

template <int M, int SRC, int MODE, bool BATCH>
int launch_ps_t(const PsArgs &a, const GnBatch &jb, hipStream_t st)
{
    constexpr int NT = M / 8, TB = M == 4096 ? 512 : 256, TPB = TB / NT;
    const size_t lds = sizeof(cf32) * 2 * M * TPB;
    const long long blocks = ((long long)a.units + TPB - 1) / TPB;
    for (long long b = 0; b < blocks; b += kMostBlocks)
        hipLaunchKernelGGL((k_pair_short<M, SRC, MODE, BATCH>), dim3((unsigned)std::min(kMostBlocks, blocks - b)), dim3(TB), lds,
                           st, a, jb, (int)b);
    FPCC_CHECK(hipGetLastError());
    return 0;
}

template <int M>
int launch_ps_m(int src, int mode, bool batch, const PsArgs &a, const GnBatch &jb, hipStream_t st)
{
    if constexpr (M < 4096) {
        if (src == PS_PCC2) return mode == 0 ? launch_ps_t<M, PS_PCC2, 0, false>(a, jb, st) : launch_ps_t<M, PS_PCC2, 1, false>(a, jb, st);
        if (src == PS_GRAM) return launch_ps_t<M, PS_GRAM, 1, false>(a, jb, st);
    }
    if (src != PS_REAL) return -1;
    if (batch) return mode == 0 ? launch_ps_t<M, PS_REAL, 0, true>(a, jb, st) : launch_ps_t<M, PS_REAL, 1, true>(a, jb, st);
    return mode == 0 ? launch_ps_t<M, PS_REAL, 0, false>(a, jb, st) : launch_ps_t<M, PS_REAL, 1, false>(a, jb, st);
}

int launch_ps(int src, int mode, bool batch, int Nz, PsArgs a, const GnBatch &jb, hipStream_t st, const char *name)
{
    const int M = Nz / 2;
    if (a.units <= 0) return 0;
    a.tw = (const cf32 *)(M == 4096   ? get_order_twiddles(4096, {8, 8, 8, 8})
                          : M == 2048 ? get_order_twiddles(2048, {8, 8, 8, 4})
                          : M == 1024 ? get_order_twiddles(1024, {8, 8, 8, 2})
                          : M == 512  ? get_order_twiddles(512, {8, 8, 8})
                                      : get_order_twiddles(256, {8, 8, 4}));
    a.twc = (const cf32 *)get_c2r_twiddles(Nz, false);
    if (!a.tw || !a.twc) return -1;
    ProfScope prof(name, st);
    switch (M) {
    case 4096: return launch_ps_m<4096>(src, mode, batch, a, jb, st);
    case 2048: return launch_ps_m<2048>(src, mode, batch, a, jb, st);
    case 1024: return launch_ps_m<1024>(src, mode, batch, a, jb, st);
    case 512: return launch_ps_m<512>(src, mode, batch, a, jb, st);
    case 256: return launch_ps_m<256>(src, mode, batch, a, jb, st);
    }
    return -1;
}

}  // namespace

bool pair_short_ok(int Nz) { return Nz == 512 || Nz == 1024 || Nz == 2048 || Nz == 4096 || Nz == 8192; }

int launch_short_pcc2(const cf32 *d_F, int S, int W, int N, int Nz, int lag0, int L, int mode, float *d_y, hipStream_t st)
{
    const long long P = (long long)S * (S - 1) / 2, units = mode == 0 ? P * W : P;
    if (!pair_short_ok(Nz) || units > 0x7fffffff) return -1;
    PsArgs a{};
    a.A = a.B = d_F;
    a.ld = Nz;
    a.S = S;
    a.W = W;
    a.N = N;
    a.lag0 = lag0;
    a.L = L;
    a.units = (int)units;
    a.scale = 0.5f * (1 / ((float)Nz * (float)N));  // the fold holds twice the half spectrum
    a.y = d_y;
    return launch_ps(PS_PCC2, mode ? 1 : 0, false, Nz, a, GnBatch{}, st, mode ? "pair_pcc2_mean" : "pair_pcc2_none");
}

int launch_short_1bit(const cf32 *d_Xa, const cf32 *d_Xb, long long ld, int S, int W, int N, int Nz, int lag0, int L,
                      int mode, float *d_y, const float *d_edge, hipStream_t st)
{
    const long long P = (long long)S * (S - 1) / 2, units = mode == 0 ? P * W : P;
    if (!pair_short_ok(Nz) || units > 0x7fffffff) return -1;
    PsArgs a{};
    a.A = d_Xa;
    a.B = d_Xb;
    a.ld = ld;
    a.S = S;
    a.W = W;
    a.N = N;
    a.lag0 = lag0;
    a.L = L;
    a.units = (int)units;
    a.scale = 1.0f / (float)Nz;
    a.edge = d_edge;
    a.K = d_edge ? edge_len(N) : 0;
    a.y = d_y;
    return launch_ps(PS_REAL, mode, false, Nz, a, GnBatch{}, st, mode ? "pair_1bit_mean" : "pair_1bit_none");
}

int launch_short_1bit_batch(const GnBatch &jb, int units, long long ld, int Nz, int mode, hipStream_t st)
{
    if (!pair_short_ok(Nz)) return -1;
    PsArgs a{};
    a.ld = ld;
    a.units = units;
    a.scale = 1.0f / (float)Nz;
    return launch_ps(PS_REAL, mode, true, Nz, a, jb, st, mode ? "pair_1bit_mean_batch" : "pair_1bit_none_batch");
}

int launch_short_gram(const cf32 *d_G, const GLayout &gl, int P, int Nz, int N, int W, int lag0, int L, float scale,
                      int count, float *d_y, const float *d_edge, int K, int S, hipStream_t st)
{
    if (!pair_short_ok(Nz)) return -1;
    PsArgs a{};
    a.A = d_G;
    a.gl = gl;
    a.S = S;
    a.W = W;
    a.N = N;
    a.lag0 = lag0;
    a.L = L;
    a.units = P;
    a.scale = scale;
    a.count = count;
    a.edge = d_edge;
    a.K = K;
    a.y = d_y;
    return launch_ps(PS_GRAM, 1, false, Nz, a, GnBatch{}, st, "pair_c2r");
}

}  // namespace fpcc
