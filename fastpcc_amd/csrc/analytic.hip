// Analytic signals of long windows in one workgroup's LDS (analytic.hpp): N even, N/2
// 7-smooth, up to about 38 500 samples (half a window as complex values with one pad slot
// per 16, in place in 160 KB).  Reads the window, writes the analytic row and its
// maximum: 12 bytes a sample instead of the 56 of three passes over full-length
// rows (two-pass transform, mask and inverse).  1298 windows of 21600: 785 -> 265 us;
// bound by the passes' vector work at one workgroup (16 waves) a CU.
#include "analytic.hpp"
#include "engine.hpp"
#include "kernels.hpp"
#include "profile.hpp"

namespace fpcc {

namespace {

constexpr int kAlT = 1024;       // threads
constexpr int kAlMax = 19264;    // largest h: (h + h/16 + 1) values and 16 floats in 160 KB

// One Stockham pass of fft_core.hpp in place: every butterfly of a thread is read
// before any is written.
template <int R>
__device__ __forceinline__ void al_pass(cf32 *lds, int n, int Ns, const cf32 *__restrict__ tw)
{
    constexpr int BPT = (kAlMax / R + kAlT - 1) / kAlT;
    const int nb = n / R;
    const float rns = 1.0f / (float)Ns;
    int t0 = threadIdx.x;
    // opaque: the compiler would keep every radix's indices across the loop over passes
    asm volatile("" : "+v"(t0));
    cf32 v[BPT][R];
#pragma unroll
    for (int i = 0; i < BPT; ++i) {
        const int b = t0 + kAlT * i;
        if (b < nb) {
#pragma unroll
            for (int r = 0; r < R; ++r) v[i][r] = lds[ct_pad(b + r * nb)];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < BPT; ++i) {
        const int b = t0 + kAlT * i;
        if (b < nb) {
            const int k = b - (int)(((float)b + 0.5f) * rns) * Ns;  // b mod Ns, exact below 2^20
            if (Ns > 1) {
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    v[i][r] = cmul(v[i][r], tw[(r - 1) * Ns + k]);
                }
            }
            Dft<R, -1>::run(v[i]);
            const int base = (b - k) * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) lds[ct_pad(base + r * Ns)] = v[i][r];
        }
        __builtin_amdgcn_sched_barrier(0);  // one butterfly's twiddles and temporaries at a time
    }
    __syncthreads();
}

__device__ __forceinline__ void al_fft(cf32 *lds, const FftPlan &plan, const cf32 *__restrict__ tw)
{
    int Ns = 1;
    for (int p = 0; p < plan.npass; ++p) {
        const int R = plan.radix[p];
        const cf32 *twp = tw + plan.tw_off[p];
        switch (R) {
        case 2: al_pass<2>(lds, plan.n, Ns, twp); break;
        case 3: al_pass<3>(lds, plan.n, Ns, twp); break;
        case 4: al_pass<4>(lds, plan.n, Ns, twp); break;
        case 5: al_pass<5>(lds, plan.n, Ns, twp); break;
        case 7: al_pass<7>(lds, plan.n, Ns, twp); break;
        case 8: al_pass<8>(lds, plan.n, Ns, twp); break;
        case 9: al_pass<9>(lds, plan.n, Ns, twp); break;
        case 16: al_pass<16>(lds, plan.n, Ns, twp); break;
        case 25: al_pass<25>(lds, plan.n, Ns, twp); break;
        default: break;
        }
        Ns *= R;
    }
}

__global__ void __launch_bounds__(kAlT)
k_analytic_lds(const float *__restrict__ x, long long stride, int W, int N, FftPlan plan, const cf32 *__restrict__ tw,
               const cf32 *__restrict__ cs, cf32 *__restrict__ Z, float *__restrict__ mx)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cf32 *lds = reinterpret_cast<cf32 *>(smem_raw);
    const int sw = blockIdx.x, s = sw / W, w = sw - s * W, h = N >> 1, t = threadIdx.x;
    float *red = reinterpret_cast<float *>(lds + h + h / 16 + 1);
    const float *in = x + (long long)s * stride + (long long)w * N;
    const bool even = ((size_t)in & 7) == 0;  // rows of odd stride start between pairs
    auto pair = [&](int m) {
        if (even) return reinterpret_cast<const cf32 *>(in)[m];
        return cf32{in[2 * m], in[2 * m + 1]};
    };
    for (int m = t; m < h; m += kAlT) lds[ct_pad(m)] = pair(m);
    __syncthreads();
    // the inverse as the conjugate of the conjugate's forward transform: one copy of the
    // passes (two spilled their registers)
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass) {
        al_fft(lds, plan, tw);
        if (pass) break;
        hilbert_half<true>(lds, h, cs, [](int k) { return ct_pad(k); });
        __syncthreads();
    }
    float4 *row = reinterpret_cast<float4 *>(Z + (long long)sw * N);  // N even: 16-byte rows
    float mv = 0.0f;
    for (int m = t; m < h; m += kAlT) {
        const cf32 v = pair(m), u = conj(lds[ct_pad(m)]);
        row[m] = float4{v.x, u.x, v.y, u.y};
        mv = fmaxf(mv, fmaxf(v.x * v.x + u.x * u.x, v.y * v.y + u.y * u.y));
    }
    mv = block_max(mv, red);
    if (t == 0) mx[sw] = mv;
}

}  // namespace

bool analytic_lds_ok(int N)
{
    FftPlan p;
    return N >= 4096 && !(N & 1) && N / 2 <= kAlMax && factor_plan(N / 2, p);
}

int launch_analytic_lds(const float *x, long long stride, int S, int W, int N, cf32 *Z, float *mx, hipStream_t st)
{
    if (!analytic_lds_ok(N)) return -1;
    const int h = N / 2;
    const DevPlan &p = get_plan(h, false);
    const cf32 *cs = (const cf32 *)get_c2r_twiddles(N, false);
    if (!p.ok || !cs) return -1;
    const size_t lds = sizeof(cf32) * (size_t)(h + h / 16 + 1) + sizeof(float) * 16;
    if (lds > 65536)
        (void)hipFuncSetAttribute((const void *)k_analytic_lds, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    ProfScope prof("analytic_lds", st);
    hipLaunchKernelGGL(k_analytic_lds, dim3(S * W), dim3(kAlT), lds, st, x, stride, W, N, p.plan, (const cf32 *)p.tw, cs,
                       Z, mx);
    FPCC_CHECK(hipGetLastError());
    return 0;
}

}  // namespace fpcc
