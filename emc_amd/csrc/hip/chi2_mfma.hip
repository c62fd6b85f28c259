// chi^2 likelihood kinds on the matrix cores (emc_cuda.cu:160-216, 242-276), with the optional
// per (rotation, pattern) intensity scaling (emc_cuda.cu:438-455, 516-531).
//
// The reference's D = sum_{valid p} a (W - K/phi)^2 (a = 1/(W + 0.02), 1 or 1/W^2 by kind) expands to
//   D = sum a W^2  -  2 ip sum (a W) K  +  ip^2 sum a K^2,      ip = 1/phi,
// two contractions over pixels of split-BF16 slice operands with the counts and the counts
// squared (both exact in BF16: K, and K^2 as hi + lo), plus a per-rotation constant.  The scaling's
// sums are two more contractions: sum K^2 over {W > 1e-10} (indicator operand, exact) and sum W K
// over the same pixels.  The FP32 products go through the contraction kernels' store epilogue; one
// elementwise pass combines them into the logits (in double) and 1/phi.
#include "../emc_internal.h"
#include "geom.h"

namespace emc {
namespace {

template <typename T>
__device__ __forceinline__ T wave_sum(T v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// x -> NT BF16 terms whose sum carries ~8 NT significant bits of x; two values, packed, per store.
template <int NT>
__device__ __forceinline__ void split(const float *x, uint32_t *const *t, size_t o)
{
    uint32_t h[2], m[2], l[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const bf16_t hb = f2bf(x[q]);
        const float r1 = x[q] - bf2f(hb);
        const bf16_t mb = f2bf(r1);
        h[q] = hb;
        m[q] = mb;
        l[q] = f2bf(r1 - bf2f(mb));
    }
    t[0][o] = h[0] | (h[1] << 16);
    if (NT > 1) t[1][o] = m[0] | (m[1] << 16);
    if (NT > 2) t[2][o] = l[0] | (l[1] << 16);
}

// One workgroup per chunk row r: the four operands from the slices kept by the statistics pass (W, 0 on
// invalid samples; masked pixels and padding rows count as 0) and Aw[r] = sum a W^2.  Two pixels per thread.
template <int NT>
__global__ __launch_bounds__(256) void k_chi2_operands(const float *__restrict__ Wk, int cs, int Pa, int Pp, int kind,
                                                       int64_t plane, bool scaling, bf16_t *__restrict__ Cx,
                                                       double *__restrict__ Aw)
{
    __shared__ double red[4];
    const int r = blockIdx.x;
    double acc = 0.0;
    uint32_t *t[4][3];
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int q = 0; q < 3; ++q)
            t[p][q] = reinterpret_cast<uint32_t *>(Cx + (int64_t)(p * NT + (q < NT ? q : 0)) * plane);
    for (int j = 2 * threadIdx.x; j < Pp; j += 512) {  // Pp is even
        const size_t o = ((size_t)r * Pp + j) / 2;
        float W[2] = {0.0f, 0.0f}, a[2], aW[2], in[2], Wi[2];
        if (r < cs) {
            const float2 v = *reinterpret_cast<const float2 *>(Wk + (size_t)r * Pp + j);
            if (j < Pa) W[0] = v.x;
            if (j + 1 < Pa) W[1] = v.y;
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            a[q] = W[q] > 0.0f ? chi2_weight(W[q], kind) : 0.0f;
            aW[q] = a[q] * W[q];
            acc += (double)a[q] * W[q] * W[q];
            const bool ok = W[q] > 1.0e-10f;  // emc_cuda.cu:444 (a zero count adds nothing to either sum)
            in[q] = ok ? 1.0f : 0.0f;
            Wi[q] = ok ? W[q] : 0.0f;
        }
        split<NT>(aW, t[0], o);
        split<NT>(a, t[1], o);
        if (scaling) {
            split<1>(in, t[2], o);  // the indicator is exact in one term
            split<NT>(Wi, t[3], o);
        }
    }
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) Aw[r] = red[0] + red[1] + red[2] + red[3];
}

// R rows hold sum a W K on entry (rows [s0, s0 + cs), patterns [0, I)); G2 = sum a K^2,
// G3 = sum_{W>1e-10} K^2, G4 = sum_{W>1e-10} W K.  ip = G4 / G3 when both are > 0 (else 1).
__global__ void k_chi2_combine(float *__restrict__ R, const float *__restrict__ G2, const float *__restrict__ G3,
                               const float *__restrict__ G4, const double *__restrict__ Aw,
                               const float *__restrict__ bias, const float *__restrict__ rscale, int cs, int I,
                               int64_t ld, bool scaling, float *__restrict__ iphi)
{
    const int64_t n = (int64_t)cs * ld;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x) {
        const int r = (int)(t / ld), i = (int)(t % ld);
        if (i >= I) continue;
        double ip = 1.0;
        if (scaling) {
            const float a = G3[t], b = G4[t];
            const float f = (a > 0.0f && b > 0.0f) ? b / a : 1.0f;
            iphi[t] = f;
            ip = f;
        }
        const double D = Aw[r] - 2.0 * ip * (double)R[t] + ip * ip * (double)G2[t];
        R[t] = (float)((double)bias[r] - D * (double)rscale[r]);
    }
}

unsigned grid_for(int64_t n) { return (unsigned)std::min<int64_t>((n + 255) / 256, 16384); }

}  // namespace

hipError_t launch_logl_chi2_mfma(const emc_ctx *c, int s0, int cs, hipStream_t st)
{
    const int NT = c->la_terms;
    const int64_t plane = (int64_t)c->chunkp * c->Pp;
    const bool scaling = c->opt.scaling != 0;
    const float *Wk = c->lw32 + (size_t)s0 * c->Pp;
    const auto operands = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(c->chunkp), dim3(256), 0, st, Wk, cs, c->Pa, c->Pp, (int)c->opt.diff, plane, scaling,
                           c->Cx, c->Aw);
    };
    if (NT == 3) operands(k_chi2_operands<3>);
    else operands(k_chi2_operands<2>);
    hipError_t e = hipGetLastError();
    auto op = [&](int p, int q) { return c->Cx + (int64_t)(p * NT + q) * plane; };
    auto with_counts = [&](int p, float *C) {  // C = X_p . K^T (hi + lo counts above 256)
        hipError_t err = launch_gemm_store_mfma(c, NT, op(p, 0), op(p, 1), NT == 3 ? op(p, 2) : nullptr, 1, c->K16,
                                                nullptr, c->K8, C, false, st);
        if (err == hipSuccess && c->k_split)
            err = launch_gemm_store_mfma(c, NT, op(p, 0), op(p, 1), NT == 3 ? op(p, 2) : nullptr, 1, c->K16lo, nullptr,
                                         nullptr, C, true, st);
        return err;
    };
    // C = X_p . (K^2)^T with na terms of X_p; the low half of K^2 meets na - 1 of them (at least
    // one): the dropped product of the two lowest terms is below 2^-16 of the sum's terms.
    auto with_squares = [&](int p, int na, float *C) {
        return launch_gemm_store_mfma(c, na, op(p, 0), op(p, 1), na == 3 ? op(p, 2) : nullptr, c->k2_split ? 2 : 1,
                                      c->K2h, c->K2l, nullptr, C, false, c->side);
    };
    // The contractions do not depend on each other: those with the squares run on a second stream, so that the last,
    // partly filled round of one is filled with tiles of the next (6,300 x 4,000 at 64^3: 400 tiles each, 1.56
    // rounds of the chip).
    float *R = c->R + (size_t)s0 * c->Ip;
    if (e == hipSuccess) e = fork_side(c, st);
    if (e != hipSuccess) return e;
    e = with_squares(1, NT, c->G2);
    if (e == hipSuccess && scaling) e = with_squares(2, 1, c->G3);
    hipError_t e2 = with_counts(0, R);
    if (e2 == hipSuccess && scaling) e2 = with_counts(3, c->G4);
    const hipError_t e3 = join_side(c, st);
    for (hipError_t x : {e, e2, e3})
        if (x != hipSuccess) return x;
    const int64_t n = (int64_t)cs * c->Ip;
    hipLaunchKernelGGL(k_chi2_combine, dim3(grid_for(n)), dim3(256), 0, st, R, c->G2, c->G3, c->G4, c->Aw,
                       c->bias + s0, c->rscale + s0, cs, c->I, (int64_t)c->Ip, scaling,
                       scaling ? c->iphi + (size_t)s0 * c->Ip : nullptr);
    return hipGetLastError();
}

}  // namespace emc
