// MFMA contractions for CDNA4 (gfx950): C[m, n] = sum_k sum_{(a,b)} A_a[m, k] B_b[n, k]
// with A and B given as BF16 terms whose sum carries the operand (A_0 = hi, A_1 = next 8 bits, ...)
// and FP32 accumulation in the matrix cores.  Here are the launchers (which kernel a shape gets, the logL's bands and
// stores) and the kernels that stage operands through registers: 128 x 128 tiles (mfma_tile = 1, and the fused scatter) and
// 256-row tiles (mfma_staging = 1).  The default kernels, staged by DMA, are in gemm_dma.hip and gemm_small.hip.
//
//   logL   : A = centred log-slices (NA = 2 or 3 terms) [rows = rotations], B = counts
//            [rows = patterns] (NB = 1, or 2 when a count exceeds 256), k = active pixels.
//            Epilogue: R[s, i] = acc + bias_s.
//   M-step : A = responsibilities hi+lo [rows = rotations], B = counts^T [rows = pixels],
//            k = patterns.  Epilogue: store U, or scatter U straight into the model (fused).
//
// Term pairs (a, b) with a + b < NA (max(NA, NB) in the DMA kernels) are accumulated (the dropped pairs are below
// 2^-8NA of the product).  The 128 x 128 kernel: macro tile, 256 threads = 4 wavefronts of 64 lanes, each wave a
// 64 x 64 block of 2 x 2 v_mfma_f32_32x32x16_bf16 tiles; BK = 64; operands staged in LDS with
// rows padded to 72 BF16 (144 B) so the 16-byte fragment reads of 16 lanes hit 64 distinct
// banks; the next k-tile is fetched into registers while the current one is multiplied.
// The fused-scatter epilogue stages the accumulators through LDS, 64 rows at a time.
#include <algorithm>
#include <type_traits>

#include "../emc_internal.h"
#include "gemm_tile.h"
#include "geom.h"

namespace emc {
namespace {

constexpr int BM = 128, BN = 128, BK = 64, LDK = BK + 8;

__device__ __forceinline__ void scatter_one(const EpiArgs &e, const float *m, float Ts, int j, float u)
{
    if (!(u >= 0.0f) || j >= e.Pa) return;
    float ux, uy, uz;
    rot_point(m, e.axyz[j], e.axyz[e.Pp + j], e.axyz[2 * e.Pp + j], model_c(e.L), ux, uy, uz);
    const int L = e.L;
    if (e.interp == EMC_INTERP_NEAREST) {
        const int vx = nearest(ux), vy = nearest(uy), vz = nearest(uz);
        if (vx >= 0 && vx < L && vy >= 0 && vy < L && vz >= 0 && vz < L) {
            const size_t v = ((size_t)vz * L + vy) * L + vx;
            atomicAdd(e.Mnum + v, u);
            atomicAdd(e.Wt + v, Ts);
        }
    } else {
        int bx, by, bz;
        float fx, fy, fz;
        if (!tri_axis(ux, L, bx, fx) || !tri_axis(uy, L, by, fy) || !tri_axis(uz, L, bz, fz)) return;
        const float g[2][3] = {{1.0f - fx, 1.0f - fy, 1.0f - fz}, {fx, fy, fz}};
        const size_t base = ((size_t)bz * L + by) * L + bx;
        for (int dz = 0; dz < 2; ++dz)
            for (int dy = 0; dy < 2; ++dy)
                for (int dx = 0; dx < 2; ++dx) {
                    const float w = g[dx][0] * g[dy][1] * g[dz][2];
                    const size_t v = base + ((size_t)dz * L + dy) * L + dx;
                    atomicAdd(e.Mnum + v, w * u);
                    atomicAdd(e.Wt + v, w * Ts);
                }
    }
}

template <int NA, int NB, int EPI>
__global__ __launch_bounds__(256) void k_gemm_mfma(const bf16_t *__restrict__ A0, const bf16_t *__restrict__ A1,
                                                   const bf16_t *__restrict__ A2, int64_t lda,
                                                   const bf16_t *__restrict__ B0, const bf16_t *__restrict__ B1,
                                                   int64_t ldb, int Kd, EpiArgs e)
{
    if (e.gate && *e.gate <= e.gate_thr) return;
    constexpr int kTileBytes = (NA + NB) * BM * LDK * 2;
    static_assert(kTileBytes >= 64 * (BN + 4) * 4, "LDS too small for the epilogue staging");
    __shared__ __attribute__((aligned(16))) unsigned char smem[kTileBytes];
    bf16_t(*As)[BM][LDK] = reinterpret_cast<bf16_t(*)[BM][LDK]>(smem);
    bf16_t(*Bs)[BN][LDK] = reinterpret_cast<bf16_t(*)[BN][LDK]>(smem + NA * BM * LDK * 2);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;

    // 128 rows x 64 k x 2 B = 1024 chunks of 16 B per operand term; 4 per thread
    const int lrow = tid >> 3, lcol = (tid & 7) * 8;
    const bf16_t *ga[NA], *gb[NB];
    ga[0] = A0 + (size_t)(m0 + lrow) * lda + lcol;
    if (NA > 1) ga[1] = A1 + (size_t)(m0 + lrow) * lda + lcol;
    if (NA > 2) ga[NA - 1] = A2 + (size_t)(m0 + lrow) * lda + lcol;
    gb[0] = B0 + (size_t)(n0 + lrow) * ldb + lcol;
    if (NB > 1) gb[NB - 1] = B1 + (size_t)(n0 + lrow) * ldb + lcol;

    u32x4 ra[NA][4], rb[NB][4];
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int h = 0; h < 4; ++h) ra[a][h] = *reinterpret_cast<const u32x4 *>(ga[a] + (size_t)32 * h * lda);
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int h = 0; h < 4; ++h) rb[b][h] = *reinterpret_cast<const u32x4 *>(gb[b] + (size_t)32 * h * ldb);

    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    const int nk = Kd / BK;
    const int fr = lane & 31, fk = (lane >> 5) * 8;
    for (int kt = 0; kt < nk; ++kt) {
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int h = 0; h < 4; ++h) *reinterpret_cast<u32x4 *>(&As[a][lrow + 32 * h][lcol]) = ra[a][h];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int h = 0; h < 4; ++h) *reinterpret_cast<u32x4 *>(&Bs[b][lrow + 32 * h][lcol]) = rb[b][h];
        __syncthreads();
        if (kt + 1 < nk) {
            const int k1 = (kt + 1) * BK;
#pragma unroll
            for (int a = 0; a < NA; ++a)
#pragma unroll
                for (int h = 0; h < 4; ++h)
                    ra[a][h] = *reinterpret_cast<const u32x4 *>(ga[a] + (size_t)32 * h * lda + k1);
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int h = 0; h < 4; ++h)
                    rb[b][h] = *reinterpret_cast<const u32x4 *>(gb[b] + (size_t)32 * h * ldb + k1);
        }
#pragma unroll
        for (int kk = 0; kk < BK; kk += 16) {
            bf16x8 fa[NA][2], fb[NB][2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
#pragma unroll
                for (int a = 0; a < NA; ++a)
                    fa[a][t] = *reinterpret_cast<const bf16x8 *>(&As[a][wm + t * 32 + fr][kk + fk]);
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    fb[b][t] = *reinterpret_cast<const bf16x8 *>(&Bs[b][wn + t * 32 + fr][kk + fk]);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int a = NA - 1; a >= 0; --a)
#pragma unroll
                        for (int b = NB - 1; b >= 0; --b)
                            if (a + b < NA)
                                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a][i], fb[b][j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }

    // accumulator layout: lane holds column n = lane%32 of each 32x32 tile and rows
    // 8*(r/4) + 4*(lane/32) + r%4, r = 0..15
    if (EPI != EPI_SCATTER) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + wm + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (m >= e.m_valid) continue;
                const float add = EPI == EPI_LOGL ? e.bias[m] : 0.0f;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int n = n0 + wn + j * 32 + (lane & 31);
                    if (n < e.n_valid) e.C[(size_t)m * e.ldc + n] = acc[i][j][r] + add;
                }
            }
        return;
    }

    // fused scatter: stage one 64-row half of the tile in LDS, then every thread scatters a
    // strided share of it (one compact loop instead of 64 unrolled scatter bodies)
    float(*Cs)[BN + 4] = reinterpret_cast<float(*)[BN + 4]>(smem);
    for (int half = 0; half < 2; ++half) {
        if ((wave >> 1) == half) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        Cs[i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)][wn + j * 32 + (lane & 31)] = acc[i][j][r];
        }
        __syncthreads();
        for (int row = wave; row < 64; row += 4) {
            const int m = m0 + half * 64 + row;
            if (m >= e.m_valid) continue;
            const double Td = e.T[m];
            if (!(Td > 1e-10)) continue;
            float rm[9];
#pragma unroll
            for (int k = 0; k < 9; ++k) rm[k] = e.rotm[12 * (size_t)m + k];
            for (int col = lane; col < BN; col += 64) scatter_one(e, rm, (float)Td, n0 + col, Cs[row][col]);
        }
        __syncthreads();
    }
}

template <int NA, int NB, int EPI>
hipError_t run(dim3 grid, hipStream_t st, const bf16_t *A0, const bf16_t *A1, const bf16_t *A2, int64_t lda,
               const bf16_t *B0, const bf16_t *B1, int64_t ldb, int Kd, const EpiArgs &e)
{
    hipLaunchKernelGGL((k_gemm_mfma<NA, NB, EPI>), grid, dim3(256), 0, st, A0, A1, A2, lda, B0, B1, ldb, Kd, e);
    return hipGetLastError();
}

// ---- 256-row variant ------------------------------------------------------------------------
// 256 x BN2 macro tile, 512 threads = 8 wavefronts (4 along M x 2 along N), each wave a 64 x BN2/2
// block of 2 x (BN2/64) 32x32 tiles, so every A fragment (NA terms) feeds BN2/64 MFMAs and every
// B fragment NA * 2.  BK = 32; two LDS stages (rows padded to 40 BF16 = 80 B: the 16-byte
// fragment reads of 16 lanes cover all 64 banks once), one barrier per k-step; the global loads
// run two k-steps ahead through two register sets (one step ahead left the load latency exposed:
// 6.15 -> 5.6 ms at the 64^3 / 25,680 / 20,000 logL shape).
// Workgroups are renumbered so that each XCD (round-robin dispatch: workgroup b runs on XCD b % 8)
// works on a contiguous band of tiles, which share A row panels in that XCD's L2.
constexpr int BK2 = 32, LDK2 = BK2 + 8;
constexpr int kTileRows = 1;  // default row panels per group of consecutive tiles

// Counts stored as bytes (exact to 255) widen to BF16 on the way to LDS: 8 bytes -> 8 BF16.
__device__ __forceinline__ u32x4 widen_u8x8(u32x2 v)
{
    u32x4 o;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t w = v[k >> 1] >> ((k & 1) * 16);
        const uint32_t f0 = __builtin_bit_cast(uint32_t, (float)(w & 0xffu));
        const uint32_t f1 = __builtin_bit_cast(uint32_t, (float)((w >> 8) & 0xffu));
        o[k] = (f0 >> 16) | (f1 & 0xffff0000u);  // integers < 256 have zero low mantissa bits
    }
    return o;
}

template <int NA, int EPI, int BN2, bool BU8>
__global__ __launch_bounds__(512) void k_gemm_mfma2(const bf16_t *__restrict__ A0, const bf16_t *__restrict__ A1,
                                                    const bf16_t *__restrict__ A2, int64_t lda,
                                                    const void *__restrict__ Bv, int64_t ldb, int Kd, int ntn,
                                                    int n_base, int gm, EpiArgs e)
{
    if (e.gate && *e.gate <= e.gate_thr) return;
    constexpr int TN = BN2 / 64;                       // 32-wide tiles per wave along N
    constexpr int BCH = BN2 * (BK2 / 8) / 512;         // 16-byte B chunks per thread per stage
    constexpr int STAGE = (NA * BM2 + BN2) * LDK2;     // BF16 elements per stage
    __shared__ __attribute__((aligned(16))) bf16_t smem[2 * STAGE];

    // XCD-aware renumbering (bijective for any grid size), then tiles in groups of gm row panels:
    // consecutive tiles t walk the gm rows of a group fastest, so the workgroups an XCD runs at
    // once share gm A panels and (their count / gm) B panels in its L2
    const int nwg = gridDim.x, b = blockIdx.x;
    const int base = nwg / 8, rem = nwg % 8, xcd = b % 8, loc = b / 8;
    const int t = xcd * base + min(xcd, rem) + loc;
    const int ntm = nwg / ntn, gi = t / (gm * ntn), gr = t % (gm * ntn);
    const int rows = min(gm, ntm - gi * gm);
    const int m0 = (gi * gm + gr % rows) * BM2, n0 = n_base + (gr / rows) * BN2;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * (BN2 / 2);
    // One 16-byte chunk per thread and 128-row half: k offset lcol of row lrow.  Lanes 4q..4q+3
    // hold the four chunks of one row, and the two rows of a lane octet are 4 apart (rows 8k + j
    // and 8k + j + 4): with 80-byte LDS rows the octet's stores then fall on 8 distinct 16-byte
    // bank groups (adjacent rows would share one).
    const int lrow = ((tid >> 5) << 3) + ((tid >> 3) & 3) + (((tid >> 2) & 1) << 2), lcol = (tid & 3) * 8;

    const bf16_t *ga[NA];
    ga[0] = A0 + (size_t)(m0 + lrow) * lda + lcol;
    if (NA > 1) ga[1] = A1 + (size_t)(m0 + lrow) * lda + lcol;
    if (NA > 2) ga[NA - 1] = A2 + (size_t)(m0 + lrow) * lda + lcol;
    // B element size 1 (bytes) or 2 (BF16); one chunk = 8 consecutive k
    const unsigned char *gb = reinterpret_cast<const unsigned char *>(Bv) + ((size_t)(n0 + lrow) * ldb + lcol) * (BU8 ? 1 : 2);

    // two register sets: the global loads run two k-steps ahead of the multiplication
    u32x4 ra[2][NA][2], rb[2][BCH];
    u32x2 rb8[2][BCH];
    auto gload = [&](int set, int k0) {
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int h = 0; h < 2; ++h) ra[set][a][h] = *reinterpret_cast<const u32x4 *>(ga[a] + (size_t)128 * h * lda + k0);
#pragma unroll
        for (int h = 0; h < BCH; ++h) {
            if (BU8) rb8[set][h] = *reinterpret_cast<const u32x2 *>(gb + (size_t)128 * h * ldb + k0);
            else rb[set][h] = *reinterpret_cast<const u32x4 *>(gb + ((size_t)128 * h * ldb + k0) * 2);
        }
    };
    auto sstore = [&](int set, int stage) {
        bf16_t *S = smem + stage * STAGE;
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                *reinterpret_cast<u32x4 *>(S + ((size_t)a * BM2 + lrow + 128 * h) * LDK2 + lcol) = ra[set][a][h];
#pragma unroll
        for (int h = 0; h < BCH; ++h)
            *reinterpret_cast<u32x4 *>(S + ((size_t)NA * BM2 + lrow + 128 * h) * LDK2 + lcol) =
                BU8 ? widen_u8x8(rb8[set][h]) : rb[set][h];
    };

    f32x16 acc[2][TN];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    const int fr = lane & 31, fk = (lane >> 5) * 8;
    auto compute = [&](int stage) {
        const bf16_t *S = smem + stage * STAGE;
#pragma unroll
        for (int kk = 0; kk < BK2; kk += 16) {
            bf16x8 fa[NA][2], fb[TN];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int a = 0; a < NA; ++a)
                    fa[a][i] = *reinterpret_cast<const bf16x8 *>(S + ((size_t)a * BM2 + wm + i * 32 + fr) * LDK2 + kk + fk);
#pragma unroll
            for (int j = 0; j < TN; ++j)
                fb[j] = *reinterpret_cast<const bf16x8 *>(S + ((size_t)NA * BM2 + wn + j * 32 + fr) * LDK2 + kk + fk);
#pragma unroll
            for (int a = NA - 1; a >= 0; --a)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a][i], fb[j], acc[i][j], 0, 0, 0);
        }
    };

    // Step k is multiplied from LDS stage k % 2 while the loads of step k + 2 are in flight into
    // register set k % 2 (stored at the end of step k - 1) and those of step k + 1 land in set
    // (k + 1) % 2, which is written to the other stage at the end of step k.  The loop is unrolled
    // by two so every set and stage index is a constant.
    // The loads are unconditional (past the last step they re-read it) so the compiler can count
    // the loads in flight and wait for one register set only, and a scheduling barrier keeps them
    // at the top of the step (the scheduler otherwise sinks them below the multiplications).
    const int nk = Kd / BK2;
    gload(0, 0);
    gload(1, min(1, nk - 1) * BK2);
    sstore(0, 0);
    __syncthreads();
    int kt = 0;
    for (; kt + 1 < nk; kt += 2) {
        gload(0, min(kt + 2, nk - 1) * BK2);
        __builtin_amdgcn_sched_barrier(0);  // keep the loads ahead of the multiplications
        compute(0);
        sstore(1, 1);
        __syncthreads();
        gload(1, min(kt + 3, nk - 1) * BK2);
        __builtin_amdgcn_sched_barrier(0);
        compute(1);
        sstore(0, 0);  // past the last step: a copy of it that nothing reads
        __syncthreads();
    }
    if (kt < nk) {  // odd step count: the last step was stored in stage 0
        compute(0);
        __syncthreads();  // the epilogue reuses the LDS
    }

    if constexpr (EPI == EPI_LOGL) {
        float *bias_l = reinterpret_cast<float *>(reinterpret_cast<unsigned char *>(smem) + 48 * BN2);
        if (tid < BM2) bias_l[tid] = m0 + tid < e.m_valid ? e.bias[m0 + tid] : 0.0f;
        __syncthreads();
        logl_epilogue<4, TN, BN2>(acc, e, m0, n0, wm, wn, smem, bias_l);
    } else {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + wm + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (m >= e.m_valid) continue;
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const int n = n0 + wn + j * 32 + (lane & 31);
                    if (n < e.n_valid) {
                        float *cp = e.C + (size_t)m * e.ldc + n;
                        *cp = e.accumulate ? *cp + acc[i][j][r] : acc[i][j][r];
                    }
                }
            }
    }
}

template <int NA, int EPI, int BN2, bool BU8>
hipError_t run2(int ntm, int ntn, int n_base, hipStream_t st, const bf16_t *A0, const bf16_t *A1, const bf16_t *A2,
                int64_t lda, const void *B, int64_t ldb, int Kd, const EpiArgs &e)
{
    const int gm = std::max(1, std::min(e.tile_rows > 0 ? e.tile_rows : kTileRows, ntm));
    hipLaunchKernelGGL((k_gemm_mfma2<NA, EPI, BN2, BU8>), dim3(ntm * ntn), dim3(512), 0, st, A0, A1, A2, lda, B, ldb,
                       Kd, ntn, n_base, gm, e);
    return hipGetLastError();
}

// Large-tile kernel for a single-term B operand (BF16, or bytes when B8 is given).  One or two A
// terms: 256-wide column tiles, plus one 128-wide launch for the remainder when N % 256 = 128;
// three A terms: 128-wide tiles (LDS).
template <int EPI, bool U8>
hipError_t run_large_t(int M, int N, hipStream_t st, int na, const bf16_t *A0, const bf16_t *A1, const bf16_t *A2,
                       int64_t lda, const void *B, int64_t ldb, int Kd, const EpiArgs &e)
{
    const int ntm = M / BM2;
    if (na == 3) return run2<3, EPI, 128, U8>(ntm, N / 128, 0, st, A0, A1, A2, lda, B, ldb, Kd, e);
    const int n256 = N / 256;
    hipError_t err = hipSuccess;
    if (na == 1) {
        if (n256 > 0) err = run2<1, EPI, 256, U8>(ntm, n256, 0, st, A0, A1, A2, lda, B, ldb, Kd, e);
        if (err == hipSuccess && N % 256)
            err = run2<1, EPI, 128, U8>(ntm, 1, n256 * 256, st, A0, A1, A2, lda, B, ldb, Kd, e);
        return err;
    }
    if (n256 > 0) err = run2<2, EPI, 256, U8>(ntm, n256, 0, st, A0, A1, A2, lda, B, ldb, Kd, e);
    if (err == hipSuccess && N % 256) err = run2<2, EPI, 128, U8>(ntm, 1, n256 * 256, st, A0, A1, A2, lda, B, ldb, Kd, e);
    return err;
}

template <int EPI>
hipError_t run_large(int M, int N, hipStream_t st, int na, const bf16_t *A0, const bf16_t *A1, const bf16_t *A2,
                     int64_t lda, const bf16_t *B16, const uint8_t *B8, int64_t ldb, int Kd, const EpiArgs &e)
{
    if (B8) return run_large_t<EPI, true>(M, N, st, na, A0, A1, A2, lda, B8, ldb, Kd, e);
    return run_large_t<EPI, false>(M, N, st, na, A0, A1, A2, lda, B16, ldb, Kd, e);
}

}  // namespace

static GemmTile logl_tile(const emc_ctx *c) { return pick_tile(c->chunkp, c->Ip, c->la_terms, c->k_split ? 2 : 1); }

int logl_band_rows(const emc_ctx *c) { return tile_rows_of(logl_tile(c)); }

bool logl_band_pass(const emc_ctx *c) { return logl_tile(c) == kTile64; }

bool logl_fuses_softmax(const emc_ctx *c)
{
    return c->mfma && !c->chi2_mfma && c->opt.mfma_tile == 0 && !(c->k_split && logl_band_pass(c));
}

static int bands_of(const emc_ctx *c, int band_rows)
{
    return (int)((int64_t)((c->S + c->chunk - 1) / c->chunk) * (c->chunkp / band_rows));
}

int softmax_fused_bands(const emc_ctx *c) { return bands_of(c, logl_band_rows(c)); }

int softmax_fused_bands_max(const emc_ctx *c)
{
    return bands_of(c, std::min(tile_rows_of(pick_tile(c->chunkp, c->Ip, c->la_terms, 1)),
                                tile_rows_of(pick_tile(c->chunkp, c->Ip, c->la_terms, 2))));
}

bool logl_skips_stores(const emc_ctx *c)
{
    // the softmax's 8-row groups must not straddle a band (chunks of a multiple of 8 rotations); three-term
    // slices and two-term counts keep every logit, which a caller may read after an iteration
    return c->skip_logits && logl_fuses_softmax(c) && c->la_terms == 2 && !c->k_split && c->opt.mfma_staging == 0 &&
           c->chunk % 8 == 0;
}

// One contraction by the kernel of its tile (with more terms than one launch of the larger tiles takes, the
// leading term of B first and the other added).
static hipError_t contract(int epi, const Contraction &g, hipStream_t st)
{
    if (g.tile == kTile64) return run_small(epi, g, st);
    if (g.na < 3 || g.nb == 1) return run_dma(epi, g, st);
    Contraction h = g;  // (0, 0), (1, 0) and (2, 0), stored; then (0, 1) and (1, 1)
    h.nb = 1;
    hipError_t err = run_dma(EPI_STORE, h, st);
    if (err != hipSuccess) return err;
    h = g;
    h.na = 2;
    h.nb = 1;
    h.B[0] = g.B[1];
    h.split = h.e.accumulate = true;
    return run_dma(epi, h, st);
}

hipError_t launch_logl_mfma(const emc_ctx *c, int s0, int cs, hipStream_t st)
{
    Contraction g;
    EpiArgs &e = g.e;
    e.tile_rows = c->opt.tile_rows;
    e.C = c->R + (size_t)s0 * c->Ip;
    e.ldc = c->Ip;
    e.m_valid = cs;
    e.n_valid = c->I;
    e.bias = c->bias + s0;
    const bf16_t *A1 = c->la_terms == 3 ? c->Lm : c->Ll;
    const bf16_t *A2 = c->Ll;
    if (c->opt.mfma_tile != 0) {
        const dim3 grid(c->Ip / BN, c->chunkp / BM);
        if (c->la_terms == 3) {
            if (c->k_split) return run<3, 2, EPI_LOGL>(grid, st, c->Lh, A1, A2, c->Pp, c->K16, c->K16lo, c->Pp, c->Pp, e);
            return run<3, 1, EPI_LOGL>(grid, st, c->Lh, A1, A2, c->Pp, c->K16, nullptr, c->Pp, c->Pp, e);
        }
        if (c->k_split) return run<2, 2, EPI_LOGL>(grid, st, c->Lh, A1, nullptr, c->Pp, c->K16, c->K16lo, c->Pp, c->Pp, e);
        return run<2, 1, EPI_LOGL>(grid, st, c->Lh, A1, nullptr, c->Pp, c->K16, nullptr, c->Pp, c->Pp, e);
    }
    // band partials in c->part: pm (floats) [bands][I] then ps (doubles) [bands][I]
    if (logl_fuses_softmax(c)) {
        e.pm = reinterpret_cast<float *>(c->part);
        e.ps = c->part + (int64_t)softmax_fused_bands(c) * c->I;
    }
    e.band0 = (int64_t)(s0 / c->chunk) * (c->chunkp / logl_band_rows(c));
    e.ldp = c->I;
    if (logl_skips_stores(c)) {
        // the running maxima start at -inf with the pass's first chunk and carry over the others
        e.runmax = c->runmax;
        e.skipped = c->scal + SC_SKIPPED;
        e.blk = c->blk;
        if (s0 == 0) {
            hipError_t err = launch_fill_i32(c->runmax, kOrdNegInf, c->I, st);
            if (err == hipSuccess) err = launch_fill_f64(e.skipped, 0.0, 1, st);
            if (err != hipSuccess) return err;
        }
    }
    g.tile = logl_tile(c);
    if (g.tile >= kTile256x128 && c->opt.mfma_staging == 1 && !c->k_split)
        return run_large<EPI_LOGL>(c->chunkp, c->Ip, st, c->la_terms, c->Lh, A1, A2, c->Pp, c->K16, c->K8, c->Pp,
                                   c->Pp, e);
    g.na = c->la_terms;
    g.nb = c->k_split ? 2 : 1;
    g.A[0] = c->Lh;
    g.A[1] = A1;
    if (g.na == 3) g.A[2] = A2;
    g.B[0] = c->K16;
    if (c->k_split) g.B[1] = c->K16lo;
    g.lda = g.ldb = g.K = c->Pp;
    g.M = c->chunkp;
    g.N = c->Ip;
    return contract(EPI_LOGL, g, st);
}

hipError_t launch_gemm_store_mfma(const emc_ctx *c, int na, const bf16_t *A0, const bf16_t *A1, const bf16_t *A2, int nb,
                                  const bf16_t *B0, const bf16_t *B1, const uint8_t *B8, float *C, bool accumulate,
                                  hipStream_t st)
{
    if (na < 1 || na > 3 || nb < 1 || nb > 2 || c->chunkp % BM2 || c->Ip % 128 || c->Pp % BK2) return hipErrorInvalidValue;
    Contraction g;
    g.e.tile_rows = c->opt.tile_rows;
    g.e.C = C;
    g.e.ldc = c->Ip;
    g.e.m_valid = c->chunkp;
    g.e.n_valid = c->Ip;
    g.e.accumulate = accumulate;
    g.two_sums = nb == 2;
    g.tile = g.two_sums && na < 3 ? pick_tile_two(c->chunkp, c->Ip, na) : pick_tile(c->chunkp, c->Ip, na, nb);
    if (g.tile >= kTile256x128 && c->opt.mfma_staging == 1 && nb == 1)
        return run_large<EPI_STORE>(c->chunkp, c->Ip, st, na, A0, A1, A2, c->Pp, B0, B8, c->Pp, c->Pp, g.e);
    g.na = na;
    g.nb = nb;
    g.A[0] = A0;
    g.A[1] = A1;
    g.A[2] = A2;
    g.B[0] = B0;
    g.B[1] = B1;
    g.lda = g.ldb = g.K = c->Pp;
    g.M = c->chunkp;
    g.N = c->Ip;
    return contract(EPI_STORE, g, st);
}

hipError_t launch_mstep_mfma(const emc_ctx *c, int s0, int cs, bool fused, const double *gate, double gate_thr,
                             hipStream_t st)
{
    EpiArgs e{};
    e.tile_rows = c->opt.tile_rows;
    e.gate = fused ? nullptr : gate;
    e.gate_thr = gate_thr;
    e.C = c->U;
    e.ldc = c->Pp;
    e.m_valid = fused ? cs : c->chunkp;
    e.n_valid = c->Pp;
    e.T = c->T + s0;
    e.rotm = c->rotm + 12 * (size_t)s0;
    e.axyz = c->axyz;
    e.Pp = c->Pp;
    e.Pa = c->Pa;
    e.L = c->L;
    e.interp = c->opt.interp;
    e.Mnum = c->Mnum;
    e.Wt = c->Wt;
    const dim3 grid(c->Pp / BN, c->chunkp / BM);
    const bf16_t *Ah = c->Ph + (size_t)s0 * c->Ip, *Al = c->Pl + (size_t)s0 * c->Ip;
    if (fused) {
        if (c->k_split) return run<2, 2, EPI_SCATTER>(grid, st, Ah, Al, nullptr, c->Ip, c->KT16, c->KT16lo, c->Ip, c->Ip, e);
        return run<2, 1, EPI_SCATTER>(grid, st, Ah, Al, nullptr, c->Ip, c->KT16, nullptr, c->Ip, c->Ip, e);
    }
    if (c->opt.mfma_tile == 1) {
        if (c->k_split) return run<2, 2, EPI_STORE>(grid, st, Ah, Al, nullptr, c->Ip, c->KT16, c->KT16lo, c->Ip, c->Ip, e);
        return run<2, 1, EPI_STORE>(grid, st, Ah, Al, nullptr, c->Ip, c->KT16, nullptr, c->Ip, c->Ip, e);
    }
    const GemmTile tile = pick_tile(c->chunkp, c->Pp, 2, c->k_split ? 2 : 1);
    if (tile >= kTile256x128 && c->opt.mfma_staging == 1 && !c->k_split)
        return run_large<EPI_STORE>(c->chunkp, c->Pp, st, 2, Ah, Al, nullptr, c->Ip, c->KT16, c->KT8, c->Ip, c->Ip, e);
    Contraction g;
    g.tile = tile;
    g.e = e;
    g.na = 2;
    g.nb = c->k_split ? 2 : 1;
    g.A[0] = Ah;
    g.A[1] = Al;
    g.B[0] = c->KT16;
    if (c->k_split) g.B[1] = c->KT16lo;
    g.lda = g.ldb = g.K = c->Ip;
    g.M = c->chunkp;
    g.N = c->Pp;
    return contract(EPI_STORE, g, st);
}

}  // namespace emc
