// FP32 contractions (precision FP32): FP32 operands, products and accumulation.
//
//   logL   : R[s,i] = sum_j f(A0[s,j], A1[s,j], K[i,j]) then the epilogue
//              TRUE_POISSON  f = A0*K              R = acc + bias_s            (emc_cuda.cu:218-238 form)
//              chi^2 kinds   f = A1*(A0-K)^2      R = log w_s - acc * rscale_s (emc_cuda.cu:160-216, 270-275)
//              scaled chi^2  f = A1*(A0-K/phi)^2  with 1/phi[s,i] per output element (emc_cuda.cu:164-165,
//                                                 182-183, 201-205 with scaling != 1)
//   M-step : U[s,j] = sum_i P[s,i] KT[j,i]                                    (emc_atomic.cu:88-132)
//
// All are "NT" products (reduction index contiguous in both operands).
//
// Plain products (k_gemm_f32m: Poisson logits, the scaling sums, U) run on the matrix cores'
// v_mfma_f32_32x32x2_f32, which adds its two products by fused multiply-adds in ascending k (checked on the
// device, 204,800 of 204,800 random elements): the same chain, so the same bits, as a thread's fmaf loop.
// Bound by the f32 matrix rate (152 TFLOP/s reached by a large library product here).  Operands go into LDS
// by DMA, 32 k (one 128-byte row line) per stage, laid out and swizzled as in gemm_small.hip; the
// instruction takes k from lanes 0-31 and k + 1 from lanes 32-63, so a lane reads two single floats per four k.
// Four wavefronts, each 32 TM x 32 TN.  6,300 x 4,001 x 3,200 logits: 1.38 ms; 1.89 on the vector ALU (128 x 128 tiles,
// 8 x 8 per thread).
//
// The chi^2 kinds' weighted squared difference is no product: vector ALU (three operations per element), 64 x 64
// or 32 x 64 tile, 256 threads, 4 x 4 or 2 x 4 outputs per thread, BK = 16, operands staged transposed in LDS
// so each thread reads quads of A and B per k; global loads for tile k+1 are issued before the FMAs of tile k.
#include <algorithm>

#include "gemm_tile.h"

namespace emc {
namespace {

constexpr int BK = 16;
typedef float f32x4 __attribute__((ext_vector_type(4)));

enum { F_CHI2 = 1, F_CHI2S = 3 };

template <int TM, int TN>
__global__ __launch_bounds__(256) void k_gemm_f32m(const float *__restrict__ A, int64_t lda, const float *__restrict__ B,
                                                   int64_t ldb, int Kd, float *__restrict__ C, int64_t ldc, int m_valid,
                                                   int n_valid, const float *__restrict__ bias,
                                                   const double *__restrict__ gate, double gate_thr)
{
    if (gate && *gate <= gate_thr) return;  // the sparse M-step runs instead
    constexpr int TILE_M = 64 * TM, TILE_N = 64 * TN, KB = 32;
    constexpr int STAGE = (TILE_M + TILE_N) * KB * 4, ST = 3;
    constexpr int LPW = (TILE_M + TILE_N) / 8 / 4;  // DMA instructions per wavefront and stage (8 rows each)
    constexpr int AHEAD = (ST - 2) * LPW;
    static_assert(AHEAD < 16);
    constexpr uint32_t kVm0 = 0x0F70;  // s_waitcnt encoding: vmcnt(0), lgkmcnt and expcnt not waited
    __shared__ __attribute__((aligned(1024))) unsigned char smem[ST * STAGE];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m0 = blockIdx.y * TILE_M, n0 = blockIdx.x * TILE_N;
    if (m0 >= m_valid || n0 >= n_valid) return;  // a tile of padding
    const int fr = lane & 31, fh = lane >> 5;
    const int wm = (wave >> 1) * 32 * TM, wn = (wave & 1) * 32 * TN;

    // DMA instruction g of the stage: rows 8 g .. 8 g + 7 of A, then of B; lane l writes chunk l & 7 of row
    // 8 g + l / 8, which holds logical chunk (l & 7) ^ ((row >> 1) & 7)
    const int lr = lane >> 3, c_even = (lane & 7) ^ (lr >> 1);
    const uint32_t offA = (uint32_t)(lr * (int)lda * 4 + c_even * 16), offB = (uint32_t)(lr * (int)ldb * 4 + c_even * 16);
    const uint32_t flip = (c_even & 4) ? (uint32_t)-64 : 64u;  // odd row groups: chunk ^ 4
    const unsigned char *src[LPW];
#pragma unroll
    for (int q = 0; q < LPW; ++q) {
        const int g = wave * LPW + q;
        src[q] = reinterpret_cast<const unsigned char *>(g < TILE_M / 8 ? A + (int64_t)(m0 + g * 8) * lda
                                                                        : B + (int64_t)(n0 + (g - TILE_M / 8) * 8) * ldb);
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    auto issue = [&](int step, int stage) {
#pragma unroll
        for (int q = 0; q < LPW; ++q) {
            const int g = wave * LPW + q;
            lds_dma16((g < TILE_M / 8 ? offA : offB) + ((g & 1) ? flip : 0u), src[q] + (int64_t)step * (KB * 4),
                      lds0 + stage * STAGE + g * 1024);
        }
    };
    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    const int sw = (fr >> 1) & 7;
    // the two k of this lane's half in the four k of chunk q: 4 q + fh and 4 q + 2 + fh
    struct Frag {
        float a[TM][2], b[TN][2];
    };
    auto rd = [&](Frag &f, int stage, int q) {
        const float *ra = reinterpret_cast<const float *>(smem + stage * STAGE + (wm + fr) * 128 + (q ^ sw) * 16) + fh;
        const float *rb = reinterpret_cast<const float *>(smem + stage * STAGE + (TILE_M + wn + fr) * 128 + (q ^ sw) * 16) + fh;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int i = 0; i < TM; ++i) f.a[i][t] = ra[i * 32 * 32 + 2 * t];
#pragma unroll
            for (int j = 0; j < TN; ++j) f.b[j][t] = rb[j * 32 * 32 + 2 * t];
        }
    };
    auto step_mm = [&](int stage) {
        Frag f[2];
        rd(f[0], stage, 0);
#pragma unroll
        for (int q = 0; q < 8; ++q) {  // the next chunk's reads fly while this one multiplies
            if (q + 1 < 8) rd(f[(q + 1) & 1], stage, q + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(f[q & 1].a[i][t], f[q & 1].b[j][t], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // step k is in stage k % ST; past the last step the loads fetch it again (into a stage nothing reads), so
    // the number of loads in flight is the same in every step
    const int nk = Kd / KB;
#pragma unroll
    for (int s = 0; s < ST - 1; ++s) issue(min(s, nk - 1), s);
    int st = 0;
    for (int k = 0; k < nk; ++k) {
        __builtin_amdgcn_s_waitcnt(kVm0 | AHEAD);  // this wavefront's loads of step k
        __syncthreads();                           // every wavefront's, and the last reads of step k - 1's stage
        issue(min(k + ST - 1, nk - 1), st == 0 ? ST - 1 : st - 1);
        step_mm(st);
        st = st + 1 == ST ? 0 : st + 1;
    }
    __builtin_amdgcn_s_waitcnt(kVm0);  // no load is left to write LDS

    // accumulator layout: lane holds column lane % 32 of each 32 x 32 tile, rows 8*(r/4) + 4*(lane/32) + r%4
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = m0 + wm + i * 32 + 8 * (r >> 2) + 4 * fh + (r & 3);
            if (m >= m_valid) continue;
            const float add = bias ? bias[m] : 0.0f;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = n0 + wn + j * 32 + fr;
                if (n < n_valid) C[(size_t)m * ldc + n] = bias ? acc[i][j][r] + add : acc[i][j][r];
            }
        }
}

// Elements the busiest of 256 CUs computes with bm x bn tiles.
double busiest(int m_valid, int n_valid, int bm, int bn)
{
    const int64_t t = (int64_t)((m_valid + bm - 1) / bm) * ((n_valid + bn - 1) / bn);
    return (double)((t + 255) / 256) * bm * bn;
}

// C [M][N] = A [M][Kd] . B [N][Kd]^T (+ bias per row).  M a multiple of 256, N of 128, Kd of 128.  64 x 128 or 64 x 64
// tiles by what the busiest CU computes; per element they cost about the same.  Measured (logL, us; 128 x 128 /
// 64 x 128 / 64 x 64): 1,380 x 500 x 768 78/45/30, 3,240 x 1,000 x 768 83/73/79, 3,240 x 1,500 x 1,792 236/206/172,
// 6,300 x 4,001 x 3,200 1443/1385/1368 (121 TFLOP/s), 10,860 x 4,000 x 3,200 2270/2318/2364.
hipError_t run_f32(const float *A, int64_t lda, const float *B, int64_t ldb, int M, int N, int Kd, float *C, int64_t ldc,
                   int m_valid, int n_valid, const float *bias, const double *gate, double gate_thr, hipStream_t st)
{
    if (M % 256 || N % 128 || Kd % 32 || lda >= (1 << 25) || ldb >= (1 << 25)) return hipErrorInvalidValue;
    if (busiest(m_valid, n_valid, 64, 128) <= 1.01 * busiest(m_valid, n_valid, 64, 64))
        hipLaunchKernelGGL((k_gemm_f32m<1, 2>), dim3(N / 128, M / 64), dim3(256), 0, st, A, lda, B, ldb, Kd, C, ldc, m_valid,
                           n_valid, bias, gate, gate_thr);
    else
        hipLaunchKernelGGL((k_gemm_f32m<1, 1>), dim3(N / 64, M / 64), dim3(256), 0, st, A, lda, B, ldb, Kd, C, ldc, m_valid,
                           n_valid, bias, gate, gate_thr);
    return hipGetLastError();
}

// RT x 4 outputs per thread, tiles of 16 RT x 64.
template <int EPI, int RT>
__global__ __launch_bounds__(256) void k_gemm_chi2(const float *__restrict__ A0, const float *__restrict__ A1,
                                                   int lda, const float *__restrict__ B, int ldb, int Kd,
                                                   float *__restrict__ C, int64_t ldc, int m_valid, int n_valid,
                                                   const float *__restrict__ bias, const float *__restrict__ rscale,
                                                   const float *__restrict__ iphi = nullptr)
{
    constexpr int CT = 4, BMT = 16 * RT, BNT = 16 * CT;
    constexpr int AC = BMT * 4;  // 16-byte chunks of an A tile (row = idx / 4); the B tile has 256
    __shared__ float As[2][BK][BMT + 4];
    __shared__ float Bs[BK][BNT + 4];
    const int tid = threadIdx.x;
    const int m0 = blockIdx.y * BMT, n0 = blockIdx.x * BNT;
    if (m0 >= m_valid || n0 >= n_valid) return;  // a tile of padding
    const int tx = tid & 15, ty = tid >> 4;
    const int row = tid >> 2, kq = (tid & 3) * 4;
    f32x4 ra[2], rb;
    auto gload = [&](int k0) {
        if (AC == 256 || tid < AC) {
            ra[0] = *reinterpret_cast<const f32x4 *>(A0 + (size_t)(m0 + row) * lda + k0 + kq);
            ra[1] = *reinterpret_cast<const f32x4 *>(A1 + (size_t)(m0 + row) * lda + k0 + kq);
        }
        rb = *reinterpret_cast<const f32x4 *>(B + (size_t)(n0 + row) * ldb + k0 + kq);
    };
    auto sstore = [&]() {
        if (AC == 256 || tid < AC)
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int q = 0; q < 4; ++q) As[a][kq + q][row] = ra[a][q];
#pragma unroll
        for (int q = 0; q < 4; ++q) Bs[kq + q][row] = rb[q];
    };

    float acc[RT][CT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[i][j] = 0.0f;
    // scaled chi^2: this thread's block of 1/phi
    float ip[EPI == F_CHI2S ? RT : 1][EPI == F_CHI2S ? CT : 1];
    if (EPI == F_CHI2S) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < CT; ++j) {
                const int m = m0 + ty * RT + i, n = n0 + tx * CT + j;
                ip[i][j] = (m < m_valid && n < n_valid) ? iphi[(size_t)m * ldc + n] : 1.0f;
            }
    }

    const int nk = Kd / BK;
    gload(0);
    sstore();
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
        if (kt + 1 < nk) gload((kt + 1) * BK);
#pragma unroll 4
        for (int k = 0; k < BK; ++k) {
            float a0[RT], a1[RT], b[CT];
            if constexpr (RT == 2) {
                const float2 x = *reinterpret_cast<const float2 *>(&As[0][k][ty * 2]);
                const float2 y = *reinterpret_cast<const float2 *>(&As[1][k][ty * 2]);
                a0[0] = x.x; a0[1] = x.y;
                a1[0] = y.x; a1[1] = y.y;
            } else {
                const f32x4 x = *reinterpret_cast<const f32x4 *>(&As[0][k][ty * 4]);
                const f32x4 y = *reinterpret_cast<const f32x4 *>(&As[1][k][ty * 4]);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    a0[q] = x[q];
                    a1[q] = y[q];
                }
            }
            const f32x4 z = *reinterpret_cast<const f32x4 *>(&Bs[k][tx * 4]);
#pragma unroll
            for (int q = 0; q < 4; ++q) b[q] = z[q];
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < CT; ++j) {
                    const float d = EPI == F_CHI2S ? __builtin_fmaf(-b[j], ip[EPI == F_CHI2S ? i : 0][EPI == F_CHI2S ? j : 0], a0[i])
                                                   : a0[i] - b[j];
                    acc[i][j] = __builtin_fmaf(a1[i] * d, d, acc[i][j]);
                }
        }
        __syncthreads();
        if (kt + 1 < nk) {
            sstore();
            __syncthreads();
        }
    }

#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const int m = m0 + ty * RT + i, n = n0 + tx * CT;
        if (m >= m_valid) continue;
        const float add = bias[m], mul = -rscale[m];
        float v[CT];
#pragma unroll
        for (int j = 0; j < CT; ++j) v[j] = __builtin_fmaf(acc[i][j], mul, add);
        float *dst = C + (size_t)m * ldc + n;
        if (n + 3 < n_valid) {
            *reinterpret_cast<f32x4 *>(dst) = f32x4{v[0], v[1], v[2], v[3]};
        } else {
#pragma unroll
            for (int j = 0; j < CT; ++j)
                if (n + j < n_valid) dst[j] = v[j];
        }
    }
}

template <int EPI, int RT>
hipError_t launch_chi2(const emc_ctx *c, int s0, int cs, hipStream_t st)
{
    hipLaunchKernelGGL((k_gemm_chi2<EPI, RT>), dim3(c->Ip / 64, c->chunkp / (16 * RT)), dim3(256), 0, st, c->A0, c->A1,
                       c->Pp, c->K32, c->Pp, c->Pp, c->R + (size_t)s0 * c->Ip, (int64_t)c->Ip, cs, c->I, c->bias + s0,
                       c->rscale + s0, EPI == F_CHI2S ? c->iphi + (size_t)s0 * c->Ip : nullptr);
    return hipGetLastError();
}

// 64 x 64 tiles, or 32 x 64 where the busiest CU then has clearly less.  Measured (scaled, us; 128 x 128 with 8 x 8
// outputs per thread, as at first / 64 x 64 / 32 x 64): 420 x 64 x 512 206/80/57, 1,380 x 1,000 x 3,200 1253/496/432,
// 3,240 x 1,500 x 1,792 832/619/648, 6,300 x 100 x 3,200 1253/484/488, 6,300 x 4,001 x 3,200 5920/5101/5493.
template <int EPI>
hipError_t run_chi2(const emc_ctx *c, int s0, int cs, hipStream_t st)
{
    if (busiest(cs, c->I, 64, 64) <= 1.05 * busiest(cs, c->I, 32, 64)) return launch_chi2<EPI, 4>(c, s0, cs, st);
    return launch_chi2<EPI, 2>(c, s0, cs, st);
}

}  // namespace

// Logits of rotations [s0, s0+cs): A rows are the chunk buffer (chunkp rows), output rows go to
// R[s0 + r].  bias / rscale are indexed by the chunk-local row through pointer offsets.
hipError_t launch_logl_f32(const emc_ctx *c, int s0, int cs, hipStream_t st)
{
    if (c->opt.diff == EMC_DIFF_TRUE_POISSON)
        return run_f32(c->A0, c->Pp, c->K32, c->Pp, c->chunkp, c->Ip, c->Pp, c->R + (size_t)s0 * c->Ip, c->Ip, cs, c->I,
                       c->bias + s0, nullptr, 0.0, st);
    return c->opt.scaling ? run_chi2<F_CHI2S>(c, s0, cs, st) : run_chi2<F_CHI2>(c, s0, cs, st);
}

// U rows for rotations [s0, s0+cs): A = responsibilities (FP32, in R), B = counts^T.
hipError_t launch_mstep_f32(const emc_ctx *c, int s0, int cs, const double *gate, double gate_thr, hipStream_t st)
{
    const float *A = (c->opt.scaling ? c->Pphi : c->R) + (size_t)s0 * c->Ip;  // P / phi or P
    return run_f32(A, c->Ip, c->KT32, c->Ip, c->chunkp, c->Pp, c->Ip, c->U, c->Pp, cs, c->Pp, nullptr, gate, gate_thr, st);
}

namespace {

// Operands of the scaling sums from the chunk's slices (A0 = W on valid pixels, else 0).
__global__ void k_scale_operands(const float *__restrict__ A0, int64_t n, float *__restrict__ Am,
                                 float *__restrict__ AWm)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x) {
        const float w = A0[t];
        const bool in = w > 1.0e-10f;  // emc_cuda.cu:444
        Am[t] = in ? 1.0f : 0.0f;
        AWm[t] = in ? w : 0.0f;
    }
}

// 1/phi = (sum K W) / (sum K^2); rows [0, cs) of the chunk, patterns [0, I).  A pattern with no
// photon on the slice's support (either sum 0) keeps phi = 1.
__global__ void k_iphi(float *__restrict__ sumK2, const float *__restrict__ sumKW, int cs, int I, int64_t ld)
{
    const int64_t n = (int64_t)cs * ld;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x) {
        if ((int)(t % ld) >= I) continue;
        const float a = sumK2[t], b = sumKW[t];
        sumK2[t] = (a > 0.0f && b > 0.0f) ? b / a : 1.0f;
    }
}

__global__ void k_pscale(const float *__restrict__ P, const float *__restrict__ iphi, int64_t n,
                         float *__restrict__ Pphi)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x)
        Pphi[t] = P[t] * iphi[t];
}

__global__ void k_square(const float *__restrict__ K, int64_t n, float *__restrict__ K2)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x)
        K2[t] = K[t] * K[t];
}

unsigned grid_for(int64_t n) { return (unsigned)std::min<int64_t>((n + 255) / 256, 8192); }

}  // namespace

hipError_t launch_scaling_f32(const emc_ctx *c, int s0, int cs, hipStream_t st)
{
    const int64_t na = (int64_t)c->chunkp * c->Pp;
    hipLaunchKernelGGL(k_scale_operands, dim3(grid_for(na)), dim3(256), 0, st, c->A0, na, c->Am, c->AWm);
    float *sK2 = c->iphi + (size_t)s0 * c->Ip, *sKW = c->R + (size_t)s0 * c->Ip;  // R rows are free until the logits
    hipError_t e = run_f32(c->Am, c->Pp, c->K2, c->Pp, c->chunkp, c->Ip, c->Pp, sK2, c->Ip, cs, c->Ip, nullptr, nullptr, 0.0, st);
    if (e == hipSuccess)
        e = run_f32(c->AWm, c->Pp, c->K32, c->Pp, c->chunkp, c->Ip, c->Pp, sKW, c->Ip, cs, c->Ip, nullptr, nullptr, 0.0, st);
    if (e != hipSuccess) return e;
    const int64_t no = (int64_t)cs * c->Ip;
    hipLaunchKernelGGL(k_iphi, dim3(grid_for(no)), dim3(256), 0, st, sK2, sKW, cs, c->I, (int64_t)c->Ip);
    return hipGetLastError();
}

hipError_t launch_pscale_f32(const emc_ctx *c, hipStream_t st)
{
    const int64_t n = (int64_t)c->Sp * c->Ip;
    hipLaunchKernelGGL(k_pscale, dim3(grid_for(n)), dim3(256), 0, st, c->R, c->iphi, n, c->Pphi);
    return hipGetLastError();
}

hipError_t launch_square_counts(const emc_ctx *c, hipStream_t st)
{
    const int64_t n = (int64_t)c->Ip * c->Pp;
    hipLaunchKernelGGL(k_square, dim3(grid_for(n)), dim3(256), 0, st, c->K32, n, c->K2);
    return hipGetLastError();
}

}  // namespace emc
