// Compress: divide by weight (emc_cuda.cu:758-786), normalisation to mean 1 (emc_cuda.cu:639-661,
// 788-798; FP64 grid-wide sums instead of the reference's single-block FP32 reduction) and the
// masked Gaussian blur (the intended math of emc_cuda.cu:1404-1492), in that order.
//
// The reference averages the model over its positive voxels.  Which voxels are positive after the
// divide depends on where the responsibilities underflow (a voxel whose every contribution is a
// P below the float range is 0 in FP32 and positive in FP64: 6 % of the voxels at 32^3), and after
// the blur on the sign of rounding-level ringing.  Here the mean is taken over the voxels that
// received weight (Wt > 0, zeros included) of the divided model: the same set in every precision
// and at every summation order, and the same mean wherever the support holds no zero.  The
// initial model (no weights yet) is averaged over its positive voxels as in the reference.
//
// Blur: the Fourier multiplier exp(-2 pi^2 sigma^2 |d|^2 / L^2), d = min(k, L-k) per axis, is
// separable and real-symmetric, so it equals three periodic 1-D convolutions with taps
// g[d] = (1/L) sum_k h(k) cos(2 pi k d / L) (FP64, rounded to float).  At L = 64 this is
// 3 * L^4 = 5e7 FMAs on an L2-resident volume, cheaper than a 3-D FFT round trip.
//
// Launches: divide + statistics, then one pass per axis; the first axis pass finishes the statistics itself
// (every workgroup adds the 256 block partials in the same order, so all get the same normaliser) and
// scales what it reads, the last scales what it keeps.  At small sides the launches are
// the time (about 4.6 us each in a stream).  emc_compress_device at 41^3 27 us, and 128^3 62 us (its passes 10,
// 22, 16 and 20 us against 25 MB of traffic and 1.6 GFLOP); with a voxel per thread and axis, separate
// divide, scale and average launches and a thread per tap 41 and 222 us.
#include <algorithm>

#include "../emc_internal.h"

namespace emc {
namespace {

template <typename T>
__device__ __forceinline__ T wave_sum(T v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

constexpr int kPartBlocks = 256;

// Blur taps g[d], one wavefront per d: lane l adds the terms k = l, l + 64, ..., then a fixed butterfly.
__device__ __forceinline__ void blur_tap(int L, double sigma, int d, float *taps)
{
    const int lane = threadIdx.x & 63;
    double acc = 0.0;
    for (int k = lane; k < L; k += 64) {
        const int kk = min(k, L - k);
        acc += exp(-2.0 * M_PI * M_PI * sigma * sigma * (double)kk * kk / ((double)L * L)) *
               cos(2.0 * M_PI * (double)k * d / L);
    }
    acc = wave_sum(acc);
    if (lane == 0) taps[d] = (float)(acc / L);
}

__global__ __launch_bounds__(256) void k_blur_taps(int L, double sigma, float *__restrict__ taps)
{
    const int d = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (d < L) blur_tap(L, sigma, d, taps);
}

// Per-block FP64 sum and count over the averaged voxels (those with Wt > 0 when Wt is given, else
// the positive ones, emc_cuda.cu:639-661), the max (emc_cuda.cu:629-637) and the sum of Wt.
// DIVIDE: the model is first formed as Mnum / Wt (-1 where Wt <= 0, emc_cuda.cu:758-786).  The workgroups
// past kPartBlocks form the blur taps, when taps is given.
template <bool DIVIDE, bool QUADS>
__global__ __launch_bounds__(256) void k_model_partial(float *__restrict__ M, const float *__restrict__ Mnum,
                                                       const float *__restrict__ Wt, int64_t n,
                                                       double *__restrict__ part, int L, double sigma,
                                                       float *__restrict__ taps)
{
    if (blockIdx.x >= kPartBlocks) {
        const int d = (blockIdx.x - kPartBlocks) * 4 + (threadIdx.x >> 6);
        if (d < L) blur_tap(L, sigma, d, taps);
        return;
    }
    __shared__ double rs[4], rc[4], rm[4], rw[4];
    double s = 0.0, cnt = 0.0, mx = -1e300, ws = 0.0;
    auto one = [&](float x, float w) {
        if (Wt ? w > 0.0f : x > 0.0f) { s += x; cnt += 1.0; }
        mx = fmax(mx, (double)x);
        ws += w;
    };
    auto div = [](float m, float w) { return w > 0.0f ? m / w : -1.0f; };
    if (DIVIDE && QUADS) {  // four voxels per thread and step
        const int64_t n4 = n / 4;
        for (int64_t v = blockIdx.x * (int64_t)256 + threadIdx.x; v < n4; v += (int64_t)kPartBlocks * 256) {
            const float4 a = reinterpret_cast<const float4 *>(Mnum)[v], w = reinterpret_cast<const float4 *>(Wt)[v];
            const float4 x = make_float4(div(a.x, w.x), div(a.y, w.y), div(a.z, w.z), div(a.w, w.w));
            reinterpret_cast<float4 *>(M)[v] = x;
            one(x.x, w.x);
            one(x.y, w.y);
            one(x.z, w.z);
            one(x.w, w.w);
        }
        const int64_t v = 4 * n4 + threadIdx.x;
        if (blockIdx.x == 0 && v < n) {
            const float w = Wt[v], x = div(Mnum[v], w);
            M[v] = x;
            one(x, w);
        }
    } else {
        for (int64_t v = blockIdx.x * (int64_t)256 + threadIdx.x; v < n; v += (int64_t)kPartBlocks * 256) {
            const float w = Wt ? Wt[v] : 0.0f;
            one(DIVIDE ? (M[v] = div(Mnum[v], w)) : M[v], w);
        }
    }
    s = wave_sum(s);
    cnt = wave_sum(cnt);
    ws = wave_sum(ws);
    for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
    if ((threadIdx.x & 63) == 0) {
        rs[threadIdx.x >> 6] = s; rc[threadIdx.x >> 6] = cnt; rm[threadIdx.x >> 6] = mx; rw[threadIdx.x >> 6] = ws;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        part[4 * blockIdx.x + 0] = rs[0] + rs[1] + rs[2] + rs[3];
        part[4 * blockIdx.x + 1] = rc[0] + rc[1] + rc[2] + rc[3];
        part[4 * blockIdx.x + 2] = fmax(fmax(rm[0], rm[1]), fmax(rm[2], rm[3]));
        part[4 * blockIdx.x + 3] = rw[0] + rw[1] + rw[2] + rw[3];
    }
}

// The statistics from the kPartBlocks block partials, by a whole workgroup of NT threads: load_stats reads
// the thread's share (before other loads, so that they fly together); finish_stats returns 1 / average
// in every thread, and workgroup 0 writes the scalars (and the average to avg_out, when given).
template <int NT>
struct StatLoads {
    double2 p[kPartBlocks / NT], q[kPartBlocks / NT];
};
template <int NT>
__device__ __forceinline__ StatLoads<NT> load_stats(const double *__restrict__ part)
{
    StatLoads<NT> x;
#pragma unroll
    for (int k = 0; k < kPartBlocks / NT; ++k) {
        x.p[k] = reinterpret_cast<const double2 *>(part)[2 * (threadIdx.x + k * NT)];
        x.q[k] = reinterpret_cast<const double2 *>(part)[2 * (threadIdx.x + k * NT) + 1];
    }
    return x;
}
template <int NT>
__device__ __forceinline__ double finish_stats(const StatLoads<NT> &x, double *__restrict__ scal, bool with_wt,
                                               double *__restrict__ avg_out)
{
    constexpr int NW = NT / 64;
    __shared__ double rs[NW], rc[NW], rm[NW], rw[NW];
    double s = 0.0, cnt = 0.0, mx = -1e300, ws = 0.0;
#pragma unroll
    for (int k = 0; k < kPartBlocks / NT; ++k) {
        s += x.p[k].x;
        cnt += x.p[k].y;
        mx = fmax(mx, x.q[k].x);
        ws += x.q[k].y;
    }
    s = wave_sum(s);
    cnt = wave_sum(cnt);
    ws = wave_sum(ws);
    for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
    if ((threadIdx.x & 63) == 0) {
        rs[threadIdx.x >> 6] = s; rc[threadIdx.x >> 6] = cnt; rm[threadIdx.x >> 6] = mx; rw[threadIdx.x >> 6] = ws;
    }
    __syncthreads();
    double S = 0.0, C = 0.0, MX = -1e300, W = 0.0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        S += rs[w];
        C += rc[w];
        MX = fmax(MX, rm[w]);
        W += rw[w];
    }
    const double avg = C > 0.0 ? S / C : 0.0, inv = avg > 0.0 ? 1.0 / avg : 1.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        scal[SC_AVG] = avg;
        scal[SC_COUNT] = C;
        scal[SC_INV] = inv;
        scal[SC_MAX] = MX;
        if (with_wt) scal[SC_WSUM] = W;
        if (!(avg > 0.0) || !isfinite(avg)) scal[SC_NONFINITE] = 2.0;
        if (avg_out) *avg_out = avg;
    }
    return inv;
}

__global__ __launch_bounds__(256) void k_model_final(const double *__restrict__ part, double *__restrict__ scal,
                                                     bool with_wt)
{
    finish_stats<256>(load_stats<256>(part), scal, with_wt, nullptr);
}

// M *= 1/avg on every voxel, the negative (missing) ones included (emc_cuda.cu:795).
__device__ __forceinline__ float scaled(float m, double inv) { return (float)((double)m * inv); }

__global__ __launch_bounds__(256) void k_scale(float *__restrict__ M, int64_t n, const double *__restrict__ part,
                                               double *__restrict__ scal, bool with_wt, double *__restrict__ avg_out)
{
    const double inv = finish_stats<256>(load_stats<256>(part), scal, with_wt, avg_out);
    for (int64_t v = blockIdx.x * (int64_t)256 + threadIdx.x; v < n; v += (int64_t)gridDim.x * 256) M[v] = scaled(M[v], inv);
}

// One axis of the periodic convolution: out[c] = sum_t g[(c - t) mod L] in[t], t ascending, on NL lines of the
// axis per workgroup, held in LDS.  A thread computes 4 outputs of 4 lines: per 4 inputs it reads 4 line
// quads and the 7 taps they meet (two quads of the doubled tap table), 6 LDS reads for 64 FMAs, so the
// vector ALU bounds it (a thread per voxel with its inputs from L2 took 56 us per axis at 128^3).
// AXIS 0: lines are rows (x); it reads the divided model, finishes the statistics, scales and takes negatives
// as 0.  AXIS 1 (y) and 2 (z): lines are columns, neighbouring lines contiguous in x.  AXIS 2 writes into the
// model, where a voxel that is negative once scaled (a missing one) keeps that value.
constexpr int kBlurThreads = 128;
template <int AXIS, int NL>
__global__ __launch_bounds__(kBlurThreads) void k_blur(const float *__restrict__ in, float *__restrict__ out,
                                                       const float *__restrict__ taps, int L,
                                                       const double *__restrict__ part, double *__restrict__ scal,
                                                       double *__restrict__ avg_out, bool quads)
{
    extern __shared__ float4 blur_lds[];
    const int Lr = (L + 3) & ~3, ld = Lr + 4;
    float *line = reinterpret_cast<float *>(blur_lds);  // [NL][ld], zero past L
    float *gg = line + NL * ld;                         // [2 Lr + 4]: gg[k] = g[(k - Lr) mod L]
    const int tid = threadIdx.x;
    const int l0 = blockIdx.x * NL, nl = min(NL, L * L - l0);
    // first element of line l, and the step along it
    const int64_t step = AXIS == 0 ? 1 : AXIS == 1 ? L : (int64_t)L * L;
    auto first = [&](int l) -> int64_t {
        return AXIS == 0 ? (int64_t)l * L : AXIS == 1 ? (int64_t)(l / L) * L * L + l % L : (int64_t)l;
    };
    auto fill_taps = [&] {
        for (int k = tid; k < 2 * Lr + 4; k += kBlurThreads) {
            int d = k - Lr;
            while (d < 0) d += L;
            while (d >= L) d -= L;
            gg[k] = taps[d];
        }
    };
    double inv = 1.0;
    const auto kept = [&inv](float m, float x) {  // AXIS 2: the scaled value where it is negative, else the blurred one
        if (!(m < 0.0f)) return x;
        const float s = scaled(m, inv);
        return s < 0.0f ? s : x;
    };
    if constexpr (AXIS == 0) {
        const StatLoads<kBlurThreads> sl = load_stats<kBlurThreads>(part);
        for (int r = tid >> 6; r < NL; r += kBlurThreads / 64)
            for (int t = tid & 63; t < ld; t += 64) line[r * ld + t] = r < nl && t < L ? in[first(l0 + r) + t] : 0.0f;
        fill_taps();
        inv = finish_stats<kBlurThreads>(sl, scal, true, avg_out);
        for (int r = tid >> 6; r < NL; r += kBlurThreads / 64)  // each thread its own elements again
            for (int t = tid & 63; t < ld; t += 64) {
                const float a = scaled(line[r * ld + t], inv);
                line[r * ld + t] = a < 0.0f ? 0.0f : a;
            }
    } else {
        const int r = tid % NL;
        const int64_t f = first(l0 + r);
        for (int t = tid / NL; t < ld; t += kBlurThreads / NL) line[r * ld + t] = r < nl && t < L ? in[f + t * step] : 0.0f;
        fill_taps();
        if (AXIS == 2) inv = scal[SC_INV];
    }
    __syncthreads();
    constexpr int G = NL / 4;  // line groups
    const int nq = Lr / 4;
    for (int it = tid; it < nq * G; it += kBlurThreads) {
        const int cg = AXIS == 0 ? it % nq : it / G, lg = AXIS == 0 ? it / nq : it % G;
        const int c0 = 4 * cg;
        const float *a0 = line + 4 * lg * ld;
        float acc[4][4];  // [line][output]
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[r][i] = 0.0f;
        for (int t = 0; t < Lr; t += 4) {
            const float4 glo = *reinterpret_cast<const float4 *>(gg + c0 - t + Lr - 4);
            const float4 ghi = *reinterpret_cast<const float4 *>(gg + c0 - t + Lr);
            const float gv[8] = {glo.x, glo.y, glo.z, glo.w, ghi.x, ghi.y, ghi.z, ghi.w};  // gv[4 + i - u]
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float4 a = *reinterpret_cast<const float4 *>(a0 + r * ld + t);
                const float av[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[r][i] = __builtin_fmaf(gv[4 + i - u], av[u], acc[r][i]);
            }
        }
        int64_t f[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) f[r] = first(l0 + 4 * lg + r) + c0 * step;
        // sides of a multiple of 4: the four lines (or outputs) are whole and contiguous, one 16-byte store each
        if (quads) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (AXIS == 0) {
                    *reinterpret_cast<float4 *>(out + f[i]) = make_float4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]);
                } else {
                    float4 *o = reinterpret_cast<float4 *>(out + f[0] + i * step);
                    float4 v = make_float4(acc[0][i], acc[1][i], acc[2][i], acc[3][i]);
                    if (AXIS == 2) {
                        const float4 m = *o;
                        v = make_float4(kept(m.x, v.x), kept(m.y, v.y), kept(m.z, v.z), kept(m.w, v.w));
                    }
                    *o = v;
                }
            }
            continue;
        }
        float m[4][4];
        if (AXIS == 2)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) m[r][i] = c0 + i < L && 4 * lg + r < nl ? out[f[r] + i * step] : 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (c0 + i < L && 4 * lg + r < nl)
                    out[f[r] + i * step] = AXIS == 2 ? kept(m[r][i], acc[r][i]) : acc[r][i];
    }
}

template <int AXIS>
void launch_axis(const float *in, float *out, const float *taps, int L, const double *part, double *scal,
                 double *avg_out, hipStream_t st)
{
    const size_t Lr = (L + 3) & ~3;
    auto lds = [&](size_t nl) { return sizeof(float) * (nl * (Lr + 4) + 2 * Lr + 4); };
    const int lines = L * L;
    const bool quads = L % 4 == 0 && (uintptr_t)out % 16 == 0;
    if (L <= 512)
        hipLaunchKernelGGL((k_blur<AXIS, 16>), dim3((lines + 15) / 16), dim3(kBlurThreads), lds(16), st, in, out, taps, L,
                           part, scal, avg_out, quads);
    else  // 8 lines: 41 KB of LDS at the largest side
        hipLaunchKernelGGL((k_blur<AXIS, 8>), dim3((lines + 7) / 8), dim3(kBlurThreads), lds(8), st, in, out, taps, L, part,
                           scal, avg_out, quads);
}

}  // namespace

hipError_t launch_blur_taps(int L, double sigma, float *taps, hipStream_t st)
{
    hipLaunchKernelGGL(k_blur_taps, dim3((L + 3) / 4), dim3(256), 0, st, L, sigma, taps);
    return hipGetLastError();
}

// The steps of one compress on explicit buffers: divide, normalise over the voxels with weight,
// blur (t1 and t2: two L^3 volumes of scratch).  With new_taps the taps are formed too.
hipError_t launch_compress_buffers(int L, double blur_sigma, bool new_taps, const float *Mnum, const float *Wt,
                                   float *model, float *taps, float *t1, float *t2, double *red, double *scal,
                                   double *avg_out, hipStream_t st)
{
    const int64_t N3 = (int64_t)L * L * L;
    const bool blur = blur_sigma > 0.0, aligned = (((uintptr_t)Mnum | (uintptr_t)Wt | (uintptr_t)model) & 15) == 0;
    const dim3 grid(kPartBlocks + (blur && new_taps ? (L + 3) / 4 : 0));
    // the quads need 16-byte aligned volumes (a caller's may not be)
    if (aligned)
        hipLaunchKernelGGL((k_model_partial<true, true>), grid, dim3(256), 0, st, model, Mnum, Wt, N3, red, L, blur_sigma, taps);
    else
        hipLaunchKernelGGL((k_model_partial<true, false>), grid, dim3(256), 0, st, model, Mnum, Wt, N3, red, L, blur_sigma, taps);
    if (blur) {
        launch_axis<0>(model, t1, taps, L, red, scal, avg_out, st);
        launch_axis<1>(t1, t2, taps, L, nullptr, scal, nullptr, st);
        launch_axis<2>(t2, model, taps, L, nullptr, scal, nullptr, st);
    } else {
        hipLaunchKernelGGL(k_scale, dim3((unsigned)std::min<int64_t>((N3 + 255) / 256, 2048)), dim3(256), 0, st, model, N3,
                           red, scal, true, avg_out);
    }
    return hipGetLastError();
}

hipError_t launch_normalize(const emc_ctx *c, bool apply, bool support, hipStream_t st)
{
    static_assert(4 * kPartBlocks <= kRedLen, "model statistics partials");
    hipLaunchKernelGGL((k_model_partial<false, false>), dim3(kPartBlocks), dim3(256), 0, st, c->model, nullptr,
                       support ? c->Wt : nullptr, c->N3, c->red, 0, 0.0, nullptr);
    if (apply)
        hipLaunchKernelGGL(k_scale, dim3((unsigned)std::min<int64_t>((c->N3 + 255) / 256, 2048)), dim3(256), 0, st, c->model,
                           c->N3, c->red, c->scal, support, nullptr);
    else
        hipLaunchKernelGGL(k_model_final, dim3(1), dim3(256), 0, st, c->red, c->scal, support);
    return hipGetLastError();
}

}  // namespace emc
