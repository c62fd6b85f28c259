// Expand: quaternion slicing of the 3D model (emc_cuda.cu:102-157) and the per-rotation
// quantities the likelihood needs.
//
// Layout: active (mask != 0) pixels are compacted to j in [0, Pa) with coordinates axyz[3][Pp];
// slices are written row-per-rotation [chunkp][Pp] so that both contractions read them with
// the reduction index contiguous.  One workgroup owns one rotation row: the rotation matrix is
// wave-uniform, coordinate reads are coalesced, and model reads are gathers that hit L2
// (the 64^3 model is 1 MiB).
#include <algorithm>

#include "../emc_internal.h"
#include "geom.h"

namespace emc {
namespace {

// rotations per workgroup in the statistics pass: 8 keeps 4 waves per SIMD (16 needed 210 VGPRs,
// 2 waves per SIMD: 0.77 instead of 0.61 ms at 64^3 / 25,680 rotations)
constexpr int kStatsG = 8, kStatsH = 4;  // kStatsH: whose samples' loads are in flight together

template <typename T>
__device__ __forceinline__ T wave_sum(T v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__global__ void k_rotmat(const float *__restrict__ q, const float *__restrict__ w, int S, int Sp,
                         float *__restrict__ rotm, float *__restrict__ logw)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= Sp) return;
    float m[12] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    float lw = 0.0f;
    if (s < S) {
        rotmat(q[4 * s], q[4 * s + 1], q[4 * s + 2], q[4 * s + 3], m);
        lw = logf(w[s]);
    }
    for (int k = 0; k < 12; ++k) rotm[12 * (size_t)s + k] = m[k];
    logw[s] = lw;
}

template <typename T>
__global__ void k_fill(T *__restrict__ p, T v, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// Bound by the host link; few workgroups reach its rate (32 as fast as 512).
__global__ __launch_bounds__(256) void k_export(const float *__restrict__ a, const float *__restrict__ b, int64_t N3,
                                                int64_t o, int n, float *__restrict__ out)
{
    for (int t = blockIdx.x * 256 + threadIdx.x; t < n; t += gridDim.x * 256) {
        const int64_t k = o + t;
        out[t] = k < N3 ? a[k] : b[k - N3];
    }
}

__global__ void k_quad_model(const float *__restrict__ model, int L, float4 *__restrict__ modelq)
{
    const int nb = (int)quad_blocks(L);
    const int64_t n = (int64_t)nb * nb * nb * 8;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x) {
        const int k = (int)(t & 7);
        const int64_t b = t >> 3;
        const int x = (int)(b % nb) * 2 + (k & 1), y = (int)(b / nb % nb) * 2 + ((k >> 1) & 1);
        const int z = (int)(b / ((int64_t)nb * nb)) * 2 + (k >> 2);
        float4 q = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (x < L && y < L && z < L) {
            const int64_t v = ((int64_t)z * L + y) * L + x;
            const bool xe = x + 1 < L, ye = y + 1 < L;
            q = make_float4(model[v], xe ? model[v + 1] : 0.0f, ye ? model[v + L] : 0.0f, xe && ye ? model[v + L + 1] : 0.0f);
        }
        modelq[t] = q;
    }
}

// What the statistics pass keeps of its samples, so that no later pass gathers from the model again.
enum { KEEP_NONE, KEEP_LOG, KEEP_W, KEEP_WA };

// Per-rotation slice sum over V_s = {active j : W > 0}, |V_s|, and per pixel the workgroup's sum of
// log W and number of rotations with a valid sample (colp[block][j] = (sum, count); summed over
// the blocks in a fixed order by k_colsum_*, so the column sums are deterministic).
// kStatsG rotations per workgroup; each thread walks pixels j = tid, tid+256, ... and keeps the
// kStatsG partial sums in registers.  KEEP_LOG keeps log W ([S][Pp], -inf where W <= 0) for the
// operand split, KEEP_W keeps W (0 where invalid) for the chi^2 operands, KEEP_WA the FP32 chi^2
// contraction's operands W and a themselves: a second gather from the model costs as much as this one
// (64^3 / 6,300 rotations 125 us), reading back what was kept 20 to 50 us.
// What bounds it: the lines that the gathers touch and their latency.  Samples load whether the point is inside or
// not, four rotations' at once, from a quad-packed model in 2 x 2 x 2 blocks (geom.h), us at 64^3 / 25,680
// rotations, 128^3 / 6,300 and 64^3 / 6,300: 382, 838, 107 with the loads behind each sample's test and lines along x;
// 325, 847 with the loads ahead alone; 285, 578, 91 with the blocks too, eight rotations at once (143 registers);
// 240, 552, 78 four at once (89).
template <int INTERP, int KEEP>
__global__ __launch_bounds__(256) void k_slice_stats(const float *__restrict__ model,
                                                     const float4 *__restrict__ modelq, int L,
                                                     const float *__restrict__ rotm, int S,
                                                     const float *__restrict__ axyz, int Pa, int Pp, int kind,
                                                     double *__restrict__ sumW, int32_t *__restrict__ ns,
                                                     float2 *__restrict__ colp, float *__restrict__ out0,
                                                     float *__restrict__ out1, double *__restrict__ scal)
{
    __shared__ double red_w[kStatsG][256];
    __shared__ __attribute__((aligned(16))) float rm[kStatsG][12];
    __shared__ int red_n[kStatsG][256];
    static_assert(kStatsG * 32 == 256, "32 lanes per rotation in the final sums");
    const int s0 = blockIdx.x * kStatsG;
    const int tid = threadIdx.x;
    const int ng = min(kStatsG, S - s0);
    if (tid < kStatsG * 12) rm[tid / 12][tid % 12] = rotm[12 * (size_t)min(s0 + tid / 12, S - 1) + tid % 12];
    __syncthreads();
    if (blockIdx.x == 0 && tid == 0) scal[SC_NONFINITE] = 0.0;  // the first kernel of an E-step
    float sw[kStatsG];
    int cnt[kStatsG];
#pragma unroll
    for (int g = 0; g < kStatsG; ++g) { sw[g] = 0.0f; cnt[g] = 0; }
    if (KEEP == KEEP_WA)  // the contraction reads whole tiles: padding pixels and rotations are zeros
        for (int g = 0; g < kStatsG; ++g)
            for (int j = (g < ng ? Pa : 0) + tid; j < Pp; j += 256) {
                out0[(size_t)(s0 + g) * Pp + j] = 0.0f;
                out1[(size_t)(s0 + g) * Pp + j] = 0.0f;
            }
    for (int j = tid; j < Pa; j += 256) {
        const float X = axyz[j], Y = axyz[Pp + j], Z = axyz[2 * Pp + j];
        float col = 0.0f;
        int colv = 0;
#pragma unroll
        for (int h = 0; h < kStatsG; h += kStatsH) {
            float Wh[kStatsH];
#pragma unroll
            for (int g = 0; g < kStatsH; ++g) {
                float m[12];
#pragma unroll
                for (int q = 0; q < 12; q += 4)
                    *reinterpret_cast<float4 *>(m + q) = *reinterpret_cast<const float4 *>(&rm[h + g][q]);
                Wh[g] = INTERP == EMC_INTERP_TRILINEAR ? sample_quad(modelq, L, m, X, Y, Z) : sample<INTERP>(model, L, m, X, Y, Z);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = h; g < h + kStatsH; ++g) {
                if (g >= ng) continue;
                const float W = Wh[g - h];
                const size_t o = (size_t)(s0 + g) * Pp + j;
                float v0 = KEEP == KEEP_LOG ? -INFINITY : 0.0f, v1 = 0.0f;
                if (W > 0.0f) {
                    sw[g] += W;
                    cnt[g] += 1;
                    if (KEEP == KEEP_LOG) {
                        v0 = logf(W);
                        col += v0;
                        colv += 1;
                    } else {
                        v0 = W;
                        if (KEEP == KEEP_WA) v1 = chi2_weight(W, kind);
                    }
                }
                if (KEEP != KEEP_NONE) out0[o] = v0;
                if (KEEP == KEEP_WA) out1[o] = v1;
            }
        }
        if (KEEP == KEEP_LOG && colp) colp[(size_t)blockIdx.x * Pp + j] = make_float2(col, (float)colv);
    }
    // per-rotation sums over the workgroup's 256 threads through LDS, in a fixed order: 32 lanes per
    // rotation add 8 values each, then five shuffle steps
    const int lane = tid & 63;
#pragma unroll
    for (int g = 0; g < kStatsG; ++g) {
        red_w[g][tid] = (double)sw[g];
        red_n[g][tid] = cnt[g];
    }
    __syncthreads();
    {
        const int g = tid >> 5, part = lane & 31;
        double a = 0.0;
        int b = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            a += red_w[g][part + 32 * q];
            b += red_n[g][part + 32 * q];
        }
#pragma unroll
        for (int o = 16; o > 0; o >>= 1) {
            a += __shfl_xor(a, o, 64);
            b += __shfl_xor(b, o, 64);
        }
        if (part == 0 && g < ng) {
            sumW[s0 + g] = a;
            ns[s0 + g] = b;
        }
    }
}

// Column sums of the statistics pass, in two fixed-order steps: part r of the blocks
// [r * per, (r + 1) * per) per pixel here, then the kColParts parts in order (k_bias).
constexpr int kColParts = 32;

__global__ __launch_bounds__(256) void k_colsum_part(const float2 *__restrict__ colp, int nblk, int Pa, int Pp,
                                                     double2 *__restrict__ cpart)
{
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= Pa) return;
    const int r = blockIdx.y, per = (nblk + kColParts - 1) / kColParts;
    const int b0 = r * per, b1 = min(nblk, b0 + per);
    double a = 0.0, n = 0.0;
    int b = b0;
    for (; b + 4 <= b1; b += 4) {  // four independent loads, added in order
        const float2 v0 = colp[(size_t)b * Pp + j], v1 = colp[(size_t)(b + 1) * Pp + j];
        const float2 v2 = colp[(size_t)(b + 2) * Pp + j], v3 = colp[(size_t)(b + 3) * Pp + j];
        a += v0.x; n += v0.y;
        a += v1.x; n += v1.y;
        a += v2.x; n += v2.y;
        a += v3.x; n += v3.y;
    }
    for (; b < b1; ++b) {
        const float2 v = colp[(size_t)b * Pp + j];
        a += v.x;
        n += v.y;
    }
    cpart[(size_t)r * Pp + j] = make_double2(a, n);
}

// FP32 slice rows for the plain contraction.  KIND: TRUE_POISSON -> A0 = log(phi0 W) (0 if
// invalid; log phi0 is read from the device scalars written by k_bias);
// chi^2 kinds -> A0 = W, A1 = pixel weight a (0 if invalid):
//   poisson (reference chi^2) a = 1/(W+0.02), absolute a = 1, relative a = 1/W^2.
template <int INTERP, int KIND>
__global__ __launch_bounds__(256) void k_slice_f32(const float *__restrict__ model, int L,
                                                   const float *__restrict__ rotm, int s0, int cs,
                                                   const float *__restrict__ axyz, int Pa, int Pp,
                                                   const double *__restrict__ scal,
                                                   float *__restrict__ A0, float *__restrict__ A1)
{
    const int r = blockIdx.x;
    const bool row_ok = r < cs;
    const float logphi0 = KIND == EMC_DIFF_TRUE_POISSON ? (float)scal[SC_LOGPHI0] : 0.0f;
    float m[9];
    if (row_ok) load_rot(rotm, s0 + r, m);
    for (int j = threadIdx.x; j < Pp; j += 256) {
        float a0 = 0.0f, a1 = 0.0f;
        if (row_ok && j < Pa) {
            const float W = sample<INTERP>(model, L, m, axyz[j], axyz[Pp + j], axyz[2 * Pp + j]);
            if (W > 0.0f) {
                if (KIND == EMC_DIFF_TRUE_POISSON) {
                    a0 = logf(W) + logphi0;
                } else {
                    a0 = W;
                    a1 = chi2_weight(W, KIND);
                }
            }
        }
        A0[(size_t)r * Pp + j] = a0;
        if (KIND != EMC_DIFF_TRUE_POISSON) A1[(size_t)r * Pp + j] = a1;
    }
}

// log W kept by the statistics pass -> A0 = log(phi0 W) (0 where invalid and in the padding), in place.
__global__ __launch_bounds__(256) void k_log_phi0(float *__restrict__ A0, int cs, int rows, int Pa, int Pp,
                                                  const double *__restrict__ scal)
{
    const float logphi0 = (float)scal[SC_LOGPHI0];
    const int quads = Pp / 4;  // Pp is a multiple of 128
    const int64_t n = (int64_t)rows * quads;
    for (int64_t t = blockIdx.x * 256 + threadIdx.x; t < n; t += (int64_t)gridDim.x * 256) {
        const int r = (int)(t / quads), j = (int)(t % quads) * 4;
        float4 *p = reinterpret_cast<float4 *>(A0) + t;
        const float4 v = *p;
        const float l[4] = {v.x, v.y, v.z, v.w};
        float x[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = r < cs && j + q < Pa && l[q] > -INFINITY ? l[q] + logphi0 : 0.0f;
        *p = make_float4(x[0], x[1], x[2], x[3]);
    }
}

// cst_i = sum_j K_ij colmean_j - B0 (FP64), one wavefront per pattern.
__device__ __forceinline__ void pattern_const(const bf16_t *__restrict__ K16, const bf16_t *__restrict__ K16lo,
                                              const uint8_t *__restrict__ K8, int i, int Pp,
                                              const float *__restrict__ colmean, double B0,
                                              double *__restrict__ cst)
{
    const int lane = threadIdx.x & 63;
    double acc = 0.0;
    if (K8) {  // byte counts (exact): 16 per lane and 16-byte load (Pp % 16 == 0)
        for (int j = lane * 16; j < Pp; j += 64 * 16) {
            const uint4 v = *reinterpret_cast<const uint4 *>(K8 + (size_t)i * Pp + j);
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 m = *reinterpret_cast<const float4 *>(colmean + j + 4 * q);
                acc = fma((double)(w[q] & 0xffu), (double)m.x, acc);
                acc = fma((double)((w[q] >> 8) & 0xffu), (double)m.y, acc);
                acc = fma((double)((w[q] >> 16) & 0xffu), (double)m.z, acc);
                acc = fma((double)(w[q] >> 24), (double)m.w, acc);
            }
        }
    } else {  // eight per lane and 16-byte load
        for (int j = lane * 8; j < Pp; j += 64 * 8) {
            const uint4 v = *reinterpret_cast<const uint4 *>(K16 + (size_t)i * Pp + j);
            const uint4 u = K16lo ? *reinterpret_cast<const uint4 *>(K16lo + (size_t)i * Pp + j) : make_uint4(0, 0, 0, 0);
            const uint32_t w[4] = {v.x, v.y, v.z, v.w}, l[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float2 m = *reinterpret_cast<const float2 *>(colmean + j + 2 * q);
                const float k0 = __uint_as_float(w[q] << 16) + __uint_as_float(l[q] << 16);
                const float k1 = __uint_as_float(w[q] & 0xffff0000u) + __uint_as_float(l[q] & 0xffff0000u);
                acc = fma((double)k0, (double)m.x, acc);
                acc = fma((double)k1, (double)m.y, acc);
            }
        }
    }
    acc = wave_sum(acc);
    if (lane == 0) cst[i] = acc - B0;
}

// Centred log-slice x = (log W + log phi0, or 0 where W <= 0) - colmean[j], from the log W kept by the
// statistics pass, split into NT BF16 terms (hi, [mid,] lo) whose sum carries ~8*NT significant bits
// of x.  The workgroups past the first gx * nsplit (gx for a row of groups) form the patterns' constants, which
// depend on the same column means (a launch of their own took 13 us at 32^3 / 1,000 patterns and 60 us with
// split counts read element by element).  One flat grid: a second dimension is documented to 65,536 groups, which
// 262,144 patterns of up to 1,024 pixels would pass.  Four pixels per thread and kSplitRows rows per workgroup, whose loads are issued
// together (the column means are read once for all of them).  Pp is a multiple of 128.
constexpr int kSplitRows = 8;

template <int NT>
__global__ __launch_bounds__(256) void k_split_bf16(const float *__restrict__ lw, int s0, int cs, int Pa, int Pp,
                                                    const float *__restrict__ colmean,
                                                    const double *__restrict__ scal, bf16_t *__restrict__ Lh,
                                                    bf16_t *__restrict__ Lm, bf16_t *__restrict__ Ll, int gx, int nsplit,
                                                    const bf16_t *__restrict__ K16, const bf16_t *__restrict__ K16lo,
                                                    const uint8_t *__restrict__ K8, int I, double *__restrict__ cst)
{
    if ((int)blockIdx.x >= gx * nsplit) {
        const int i = ((int)blockIdx.x - gx * nsplit) * 4 + (int)(threadIdx.x >> 6);
        if (i < I) pattern_const(K16, K16lo, K8, i, Pp, colmean, scal[SC_B0], cst);  // a whole wavefront
        return;
    }
    const int r0 = blockIdx.x / gx * kSplitRows;
    const int j0 = (blockIdx.x % gx * 256 + threadIdx.x) * 4;
    if (j0 >= Pp) return;
    const float logphi0 = (float)scal[SC_LOGPHI0];
    float cm[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) cm[q] = j0 + q < Pa ? colmean[j0 + q] : 0.0f;
    float4 v[kSplitRows];
#pragma unroll
    for (int rr = 0; rr < kSplitRows; ++rr) {
        v[rr] = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
        if (r0 + rr < cs) v[rr] = *reinterpret_cast<const float4 *>(lw + (size_t)(s0 + r0 + rr) * Pp + j0);
    }
    auto pack = [](const uint16_t *w) {
        return make_uint2((uint32_t)w[0] | ((uint32_t)w[1] << 16), (uint32_t)w[2] | ((uint32_t)w[3] << 16));
    };
#pragma unroll
    for (int rr = 0; rr < kSplitRows; ++rr) {
        const int r = r0 + rr;  // rows of the padded chunk past cs are written as zeros
        const float l[4] = {v[rr].x, v[rr].y, v[rr].z, v[rr].w};
        uint16_t h[4], mi[4], lo[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int j = j0 + q;
            float x = 0.0f;
            if (r < cs && j < Pa) x = (l[q] > -INFINITY ? l[q] + logphi0 : 0.0f) - cm[q];
            h[q] = f2bf(x);
            const float r1 = x - bf2f(h[q]);
            mi[q] = f2bf(r1);
            lo[q] = f2bf(r1 - bf2f(mi[q]));
        }
        const size_t o = (size_t)r * Pp + j0;
        *reinterpret_cast<uint2 *>(Lh + o) = pack(h);
        if (NT == 2) {
            *reinterpret_cast<uint2 *>(Ll + o) = pack(mi);
        } else {
            *reinterpret_cast<uint2 *>(Lm + o) = pack(mi);
            *reinterpret_cast<uint2 *>(Ll + o) = pack(lo);
        }
    }
}

template <int INTERP>
__global__ __launch_bounds__(256) void k_expand(const float *__restrict__ model, int L,
                                                const float *__restrict__ rotm, int s0,
                                                const float *__restrict__ coords, int P,
                                                float *__restrict__ out)
{
    const int r = blockIdx.x;
    float m[9];
    load_rot(rotm, s0 + r, m);
    for (int p = threadIdx.x; p < P; p += 256)
        out[(size_t)r * P + p] = sample<INTERP>(model, L, m, coords[p], coords[P + p], coords[2 * P + p]);
}

// Fluence, per-rotation logit terms and pixel column means.  Every workgroup forms the total
// sum_s sumW_s itself (the same fixed order in each, so the same value) and writes its share of the
// rotations and pixels; workgroup 0 writes the scalars.  No more workgroups than the chip holds at once, since each reads
// every sumW_s (an iteration of 1,000,000 rotations x 64 patterns at 12^3: 6,360 us with one per 256 rotations, 4,790 so).
//   TRUE_POISSON: phi0 = fluence or (sumK/I)/(sum_s sumW_s / S);
//                 bias_s = log w_s - phi0 sumW_s + B0, B0 = phi0 * mean_s sumW_s (a global
//                 shift that keeps the stored logits small; it is returned through cst).
//   chi^2 kinds:  bias_s = log w_s, rscale_s = 1/(2 n_s sigma^2) (0 when n_s = 0).
constexpr int kBiasGroups = 512;
__global__ __launch_bounds__(1024) void k_bias(const double *__restrict__ sumW, const int32_t *__restrict__ ns,
                                               const float *__restrict__ logw, int S, int Sp, int I,
                                               double sumK_total, double fluence, int diff, float sigma,
                                               const double2 *__restrict__ cpart, int Pa, int Pp,
                                               float *__restrict__ bias, float *__restrict__ rscale,
                                               float *__restrict__ colmean, double *__restrict__ cst,
                                               double *__restrict__ scal)
{
    __shared__ double red[16];
    const int tid = threadIdx.x;
    // eight partial sums per thread (eight loads in flight), added in a fixed order
    double p[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    int s8 = tid;
    for (; s8 + 7 * 1024 < S; s8 += 8 * 1024)
#pragma unroll
        for (int q = 0; q < 8; ++q) p[q] += sumW[s8 + q * 1024];
#pragma unroll
    for (int q = 0; q < 8; ++q)
        if (s8 + q * 1024 < S) p[q] += sumW[s8 + q * 1024];
    double acc = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
    acc = wave_sum(acc);
    if ((tid & 63) == 0) red[tid >> 6] = acc;
    __syncthreads();
    double SW = 0.0;
    for (int k = 0; k < 16; ++k) SW += red[k];
    double phi0 = 1.0;
    if (diff == EMC_DIFF_TRUE_POISSON) {
        if (fluence > 0.0) phi0 = fluence;
        else if (SW > 0.0 && I > 0 && sumK_total > 0.0) phi0 = (sumK_total / I) / (SW / S);  // else undefined: 1
    }
    const double B0 = (diff == EMC_DIFF_TRUE_POISSON && S > 0) ? phi0 * SW / S : 0.0;
    if (blockIdx.x == 0 && tid == 0) {
        scal[SC_PHI0] = phi0;
        scal[SC_LOGPHI0] = log(phi0);
        scal[SC_SUMW] = SW;
        scal[SC_B0] = B0;
    }
    const double inv2s2 = 1.0 / (2.0 * (double)sigma * (double)sigma);
    // 256 elements per workgroup: the column sums' 32 loads a pixel then come from many compute units
    if (tid >= 256) return;
    const int t0 = blockIdx.x * 256 + tid, stride = gridDim.x * 256;
    for (int s = t0; s < Sp; s += stride) {
        float b = 0.0f, rs = 0.0f;
        if (s < S) {
            if (diff == EMC_DIFF_TRUE_POISSON) b = (float)((double)logw[s] - phi0 * sumW[s] + B0);
            else {
                b = logw[s];
                rs = ns[s] > 0 ? (float)(inv2s2 / (double)ns[s]) : 0.0f;
            }
        }
        bias[s] = b;
        rscale[s] = rs;
    }
    if (!cpart) {  // no centring: the pattern constants are the shift alone
        for (int i = t0; i < I; i += stride) cst[i] = -B0;
        return;
    }
    // column mean of log(phi0 W) over rotations (invalid samples count as 0)
    const double lp = log(phi0);
    for (int j = t0; j < Pp; j += stride) {
        double a = 0.0, n = 0.0;
        if (j < Pa)
#pragma unroll 16
            for (int r = 0; r < kColParts; ++r) {
                const double2 v = cpart[(size_t)r * Pp + j];
                a += v.x;
                n += v.y;
            }
        colmean[j] = j < Pa && S > 0 ? (float)((a + n * lp) / S) : 0.0f;
    }
}

}  // namespace

hipError_t launch_rotmat(const float *q, const float *w, int S, int Sp, float *rotm, float *logw,
                         hipStream_t st)
{
    hipLaunchKernelGGL(k_rotmat, dim3((Sp + 255) / 256), dim3(256), 0, st, q, w, S, Sp, rotm, logw);
    return hipGetLastError();
}

hipError_t launch_fill_f32(float *p, float v, int64_t n, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    const int64_t blocks = std::min<int64_t>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(k_fill<float>, dim3((unsigned)blocks), dim3(256), 0, st, p, v, n);
    return hipGetLastError();
}

hipError_t launch_fill_f64(double *p, double v, int64_t n, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    const int64_t blocks = std::min<int64_t>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(k_fill<double>, dim3((unsigned)blocks), dim3(256), 0, st, p, v, n);
    return hipGetLastError();
}

hipError_t launch_fill_i32(int32_t *p, int32_t v, int64_t n, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    const int64_t blocks = std::min<int64_t>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(k_fill<int32_t>, dim3((unsigned)blocks), dim3(256), 0, st, p, v, n);
    return hipGetLastError();
}

hipError_t launch_export(const float *a, const float *b, int64_t N3, int64_t o, int n, float *out, hipStream_t st)
{
    hipLaunchKernelGGL(k_export, dim3(std::min((n + 255) / 256, 128)), dim3(256), 0, st, a, b, N3, o, n, out);
    return hipGetLastError();
}

int64_t quad_model_len(int L) { return 8 * quad_blocks(L) * quad_blocks(L) * quad_blocks(L); }
int64_t colp_len(int S, int Pp) { return (int64_t)((S + kStatsG - 1) / kStatsG) * Pp; }
int64_t colpart_len(int Pp) { return (int64_t)kColParts * Pp; }

// The FP32 path's operands come from the statistics pass when one chunk covers every rotation.
static bool f32_slices_kept(const emc_ctx *c) { return !c->mfma && c->chunk >= c->S; }

template <int INTERP>
static void slice_stats_interp(const emc_ctx *c, hipStream_t st)
{
    const int nblk = (c->S + kStatsG - 1) / kStatsG, nall = c->chunkp / kStatsG;  // with the padding rows
    const bool poisson = c->opt.diff == EMC_DIFF_TRUE_POISSON;
    const auto run = [&](auto kernel, float2 *colp, float *out0, float *out1) {
        hipLaunchKernelGGL(kernel, dim3(out1 ? nall : nblk), dim3(256), 0, st, c->model, c->modelq, c->L, c->rotm, c->S, c->axyz, c->Pa,
                           c->Pp, (int)c->opt.diff, c->sumW, c->ns, colp, out0, out1, c->scal);
    };
    if (c->chi2_mfma) run(k_slice_stats<INTERP, KEEP_W>, nullptr, c->lw32, nullptr);
    else if (c->mfma) run(k_slice_stats<INTERP, KEEP_LOG>, c->colp, c->lw32, nullptr);
    else if (f32_slices_kept(c) && poisson) run(k_slice_stats<INTERP, KEEP_LOG>, nullptr, c->A0, nullptr);
    else if (f32_slices_kept(c)) run(k_slice_stats<INTERP, KEEP_WA>, nullptr, c->A0, c->A1);
    else run(k_slice_stats<INTERP, KEEP_NONE>, nullptr, nullptr, nullptr);
}

hipError_t launch_slice_stats(const emc_ctx *c, hipStream_t st)
{
    if (c->opt.interp == EMC_INTERP_NEAREST) {
        slice_stats_interp<EMC_INTERP_NEAREST>(c, st);
    } else {
        const int64_t n3 = quad_model_len(c->L);
        hipLaunchKernelGGL(k_quad_model, dim3((unsigned)std::min<int64_t>((n3 + 255) / 256, 4096)), dim3(256), 0, st,
                           c->model, c->L, c->modelq);
        slice_stats_interp<EMC_INTERP_TRILINEAR>(c, st);
    }
    if (c->mfma && !c->chi2_mfma)
        hipLaunchKernelGGL(k_colsum_part, dim3((c->Pa + 255) / 256, kColParts), dim3(256), 0, st, c->colp,
                           (c->S + kStatsG - 1) / kStatsG, c->Pa, c->Pp, c->colpart);
    return hipGetLastError();
}

hipError_t launch_bias(const emc_ctx *c, float sigma, hipStream_t st)
{
    const int nb = std::max(1, std::min((std::max(c->Sp, c->Pp) + 255) / 256, kBiasGroups));
    hipLaunchKernelGGL(k_bias, dim3(nb), dim3(1024), 0, st, c->sumW, c->ns, c->logw, c->S, c->Sp, c->I,
                       c->sumK_total, c->opt.fluence, c->opt.diff, sigma,
                       c->mfma && !c->chi2_mfma ? c->colpart : nullptr, c->Pa, c->Pp, c->bias, c->rscale, c->colmean,
                       c->cst, c->scal);
    return hipGetLastError();
}

template <int INTERP>
static hipError_t slice_f32_interp(const emc_ctx *c, int s0, int cs, hipStream_t st)
{
    const dim3 grid(c->chunkp), blk(256);
    switch (c->opt.diff) {
    case EMC_DIFF_TRUE_POISSON:
        hipLaunchKernelGGL((k_slice_f32<INTERP, EMC_DIFF_TRUE_POISSON>), grid, blk, 0, st, c->model, c->L,
                           c->rotm, s0, cs, c->axyz, c->Pa, c->Pp, c->scal, c->A0, c->A1);
        break;
    case EMC_DIFF_POISSON:
        hipLaunchKernelGGL((k_slice_f32<INTERP, EMC_DIFF_POISSON>), grid, blk, 0, st, c->model, c->L,
                           c->rotm, s0, cs, c->axyz, c->Pa, c->Pp, c->scal, c->A0, c->A1);
        break;
    case EMC_DIFF_ABSOLUTE:
        hipLaunchKernelGGL((k_slice_f32<INTERP, EMC_DIFF_ABSOLUTE>), grid, blk, 0, st, c->model, c->L,
                           c->rotm, s0, cs, c->axyz, c->Pa, c->Pp, c->scal, c->A0, c->A1);
        break;
    default:
        hipLaunchKernelGGL((k_slice_f32<INTERP, EMC_DIFF_RELATIVE>), grid, blk, 0, st, c->model, c->L,
                           c->rotm, s0, cs, c->axyz, c->Pa, c->Pp, c->scal, c->A0, c->A1);
        break;
    }
    return hipGetLastError();
}

hipError_t launch_slice_f32(const emc_ctx *c, int s0, int cs, hipStream_t st)
{
    if (f32_slices_kept(c)) {
        const int64_t n = (int64_t)c->chunkp * c->Pp / 4;
        if (c->opt.diff == EMC_DIFF_TRUE_POISSON)
            hipLaunchKernelGGL(k_log_phi0, dim3((unsigned)std::min<int64_t>((n + 255) / 256, 8192)), dim3(256), 0, st, c->A0,
                               cs, c->chunkp, c->Pa, c->Pp, c->scal);
        return hipGetLastError();
    }
    return c->opt.interp == EMC_INTERP_NEAREST ? slice_f32_interp<EMC_INTERP_NEAREST>(c, s0, cs, st)
                                               : slice_f32_interp<EMC_INTERP_TRILINEAR>(c, s0, cs, st);
}

hipError_t launch_slice_bf16(const emc_ctx *c, int s0, int cs, hipStream_t st)
{
    const int gx = (c->Pp / 4 + 255) / 256, nsplit = (c->chunkp + kSplitRows - 1) / kSplitRows;
    const int nconst = s0 == 0 ? (c->I + 3) / 4 : 0;  // the constants go with the first chunk
    const auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(gx * nsplit + nconst), dim3(256), 0, st, c->lw32, s0, cs, c->Pa, c->Pp, c->colmean,
                           c->scal, c->Lh, c->Lm, c->Ll, gx, nsplit, c->K16, c->k_split ? c->K16lo : nullptr, c->K8, c->I,
                           c->cst);
    };
    if (c->la_terms == 3) run(k_split_bf16<3>);
    else run(k_split_bf16<2>);
    return hipGetLastError();
}

hipError_t launch_expand(const emc_ctx *c, int s0, int cs, float *out, hipStream_t st)
{
    if (cs <= 0) return hipSuccess;
    if (c->opt.interp == EMC_INTERP_NEAREST)
        hipLaunchKernelGGL(k_expand<EMC_INTERP_NEAREST>, dim3(cs), dim3(256), 0, st, c->model, c->L, c->rotm, s0,
                           c->coords, c->P, out);
    else
        hipLaunchKernelGGL(k_expand<EMC_INTERP_TRILINEAR>, dim3(cs), dim3(256), 0, st, c->model, c->L, c->rotm,
                           s0, c->coords, c->P, out);
    return hipGetLastError();
}

}  // namespace emc
