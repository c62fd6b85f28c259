// MFMA contractions whose operands go from global memory straight into LDS (gfx950's vector-memory DMA
// path, global_load_lds_dwordx4): C[m, n] = sum_k sum_{a + b < max(NA, NB)} A_a[m, k] B_b[n, k] with NA and
// NB BF16 terms per operand and FP32 accumulation.
//
// Tile 256 x BN (BN = 320, 256 or 128), 8 wavefronts (4 along M x 2 along N), each a 64 x BN/2 block of
// 2 x TN v_mfma_f32_32x32x16_bf16 tiles; BK = 32; or 128 x 128, 4 wavefronts.  LDS rows are 64 B (32 BF16) without padding; the four
// 16-byte chunks of row r sit at chunk ^ lds_swz(r), which spreads the fragment reads of 8 (or 16)
// consecutive rows over distinct bank groups.  No register staging and no LDS store instructions.
//
// What bounds it: the matrix cores at the clock the chip holds under them (1.33 PFLOP/s executed at
// 25,856 x 20,224 x 3,200, the rate the vendor library reaches on the plain product), then the latency
// of a step's loads at the step's barrier.  Three operand stages where they fit (loads two steps
// ahead), else two (NA + NB = 4: 64 KB a stage; a step multiplies three term pairs there, so one step
// of cover lasts as long as one and a half of the two-pair kernel).
//
// The two-term x one-term product against the register-staged kernel, logL at 25,856 x 20,224 x 3,200:
// 5.70 vs 5.90 ms and 5.86 vs 6.28 ms on two boxes, bit-identical results.
#include "gemm_tile.h"

namespace emc {
namespace {

constexpr int BK2 = 32;
constexpr int kTileRows = 1;  // default row panels per group of consecutive tiles

__device__ __forceinline__ int lds_swz(int r) { return ((r >> 2) & 1) | ((((r >> 1) ^ (r >> 3)) & 1) << 1); }

template <int NA, int NB, int WGM, int TN>
struct Cfg {
    static constexpr int BM = 64 * WGM, BN = 64 * TN;
    static constexpr int OPA = BM * BK2 * 2, OPB = BN * BK2 * 2;  // bytes of one operand term per stage
    static constexpr int STAGE = NA * OPA + NB * OPB;
    // stages in LDS; the 128-row tiles run two workgroups per CU
    static constexpr int ST = 3 * STAGE <= (WGM == 4 ? 159744 : 73728) ? 3 : 2;
    static constexpr int NG = STAGE / 1024;                         // DMA instructions per step (16 rows each)
    static constexpr int LPW = (NG + 2 * WGM - 1) / (2 * WGM);      // per wave (the last ones may repeat one)
    static constexpr int NT = NA > NB ? NA : NB;                    // term pairs a + b < NT are multiplied
    static_assert(STAGE % 1024 == 0 && LPW < 16 && ST * STAGE <= 159744);
};

// SPLIT, logL: the logits of two-term counts; with NB = 1 the sums of the leading count terms are in C already.
// SPLIT, store: two sums (Contraction::two_sums).  In one chain the low term's products, 2^-8 of the others and less,
// would each be rounded to the high sum's size: chi^2 log-sum-exps at 64^3, 6,300 x 2,000 were 4 % (absolute, two-term) to
// 20 % (scaled, normalised patterns, three-term) further from 64 bits so.
template <int EPI, int NA, int NB, int WGM, int TN, bool SPLIT>
__global__ __launch_bounds__(128 * WGM, EPI == EPI_STORE && SPLIT ? 2 : 1) void k_dma(const bf16_t *__restrict__ A0, const bf16_t *__restrict__ A1,
                                             const bf16_t *__restrict__ A2, int64_t lda,
                                             const bf16_t *__restrict__ B0, const bf16_t *__restrict__ B1, int64_t ldb,
                                             int N, int Kd, int ntn, int gm, EpiArgs e)
{
    static_assert(EPI == EPI_LOGL || EPI == EPI_STORE, "logL or store epilogue");
    if (e.gate && *e.gate <= e.gate_thr) return;  // the sparse M-step runs instead
    using C = Cfg<NA, NB, WGM, TN>;
    constexpr int BM = C::BM, BN = C::BN, ST = C::ST, LPW = C::LPW;
    constexpr uint32_t kVm0 = 0x0F70;  // s_waitcnt encoding: vmcnt(0), lgkmcnt and expcnt not waited
    __shared__ __attribute__((aligned(1024))) unsigned char smem[ST * C::STAGE];
    __shared__ float bias_s[BM];
    __shared__ int32_t rm_s[BN];

    // XCD-aware tile order (workgroup b runs on XCD b % 8): XCD x takes its contiguous share of the tiles,
    // in groups of gm row panels, except that a last row band holding padded rows is left to the end of
    // every XCD's share (its ntn tiles split over the XCDs): the waves of its padded rows skip their
    // products, so those tiles cost about half, and each XCD's final, partly filled round is made of them.
    const int nwg = gridDim.x, b = blockIdx.x;
    const int base = nwg / 8, rem = nwg % 8, xcd = b % 8, loc = b / 8;
    const int ntm = nwg / ntn;
    int m0, n0;
    if (e.m_valid < ntm * BM && ntm > 1 && ntn >= 8) {  // then every XCD has room for its share
        const int pc = ntn / 8 + (xcd < ntn % 8 ? 1 : 0), pstart = xcd * (ntn / 8) + min(xcd, ntn % 8);
        const int fc = base + (xcd < rem ? 1 : 0) - pc, fstart = xcd * base + min(xcd, rem) - pstart;
        if (loc < fc) {
            const int t = fstart + loc, gi = t / (gm * ntn), gr = t % (gm * ntn);
            const int rows = min(gm, ntm - 1 - gi * gm);
            m0 = (gi * gm + gr % rows) * BM;
            n0 = (gr / rows) * BN;
        } else {
            m0 = (ntm - 1) * BM;
            n0 = (pstart + loc - fc) * BN;
        }
    } else {
        const int t = xcd * base + min(xcd, rem) + loc;
        const int gi = t / (gm * ntn), gr = t % (gm * ntn);
        const int rows = min(gm, ntm - gi * gm);
        m0 = (gi * gm + gr % rows) * BM;
        n0 = (gr / rows) * BN;
    }

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * (BN / 2);
    const bool live = m0 + wm < e.m_valid;  // a wave whose 64 rows are all padding multiplies nothing
    // DMA instruction q of this wave: one operand term, its rows 16 rb .. 16 rb + 15; lane l fetches logical
    // chunk (l & 3) ^ lds_swz(l / 4) of row 16 rb + l / 4 (the swizzle uses the row's low four bits).  A
    // tile past N (N a multiple of 128, BN = 256) reads its last rows again: its columns are not stored.
    const int lr = lane >> 2, lc = ((lane & 3) ^ lds_swz(lr)) * 16;
    const uint32_t offA = (uint32_t)(lr * (int)lda * 2 + lc), offB = (uint32_t)(lr * (int)ldb * 2 + lc);
    const unsigned char *src[LPW];
#pragma unroll
    for (int q = 0; q < LPW; ++q) {
        const int g = min(wave * LPW + q, C::NG - 1);
        const bool isa = g < NA * (BM / 16);
        const int ga = g / (BM / 16), gb = (g - NA * (BM / 16)) / (BN / 16);
        const bf16_t *op = isa ? (ga == 0 ? A0 : ga == 1 ? A1 : A2) : (gb == 0 ? B0 : B1);
        const int row = isa ? m0 + g % (BM / 16) * 16 : min(n0 + (g - NA * (BM / 16)) % (BN / 16) * 16, N - 16);
        src[q] = reinterpret_cast<const unsigned char *>(op + (int64_t)row * (isa ? lda : ldb));
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    auto issue = [&](int step, int stage) {
#pragma unroll
        for (int q = 0; q < LPW; ++q) {
            const int g = min(wave * LPW + q, C::NG - 1);
            lds_dma16(g < NA * (BM / 16) ? offA : offB, src[q] + (int64_t)step * (BK2 * 2), lds0 + stage * C::STAGE + g * 1024);
        }
    };

    constexpr bool TWO = EPI == EPI_STORE && SPLIT;  // the products with B1 are summed in acc1
    f32x16 acc[2][TN], acc1[2][TN];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = acc1[i][j][r] = 0.0f;
    const int fr = lane & 31, sw = lds_swz(fr & 15), c0 = lane >> 5;
    struct Frag {
        bf16x8 a[NA][2], b[NB][TN];
    };
    auto rd = [&](Frag &F, int stage, int kk) {  // fragments of k-half kk (0 or 16) of a stage
        const unsigned char *S = smem + stage * C::STAGE;
        const int co = ((c0 + kk / 8) ^ sw) * 16;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int a = 0; a < NA; ++a)
                F.a[a][i] = *reinterpret_cast<const bf16x8 *>(S + a * C::OPA + (wm + i * 32 + fr) * 64 + co);
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int t = 0; t < NB; ++t)
                F.b[t][j] = *reinterpret_cast<const bf16x8 *>(S + NA * C::OPA + t * C::OPB + (wn + j * 32 + fr) * 64 + co);
    };
    auto mm = [&](const Frag &F) {  // low terms first, as in the register-staged kernels
#pragma unroll
        for (int a = NA - 1; a >= 0; --a)
#pragma unroll
            for (int t = NB - 1; t >= 0; --t)
                if (a + t < C::NT)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < TN; ++j) {
                            f32x16 &to = TWO && t == 1 ? acc1[i][j] : acc[i][j];
                            to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(F.a[a][i], F.b[t][j], to, 0, 0, 0);
                        }
    };

    const int nk = Kd / BK2;
    constexpr bool kOneFrag = NA + NB == 4 && TN == 5;  // two sets of fragments beside 160 accumulators do not fit
    Frag F0, F1;
    const float bv = EPI == EPI_LOGL && tid < BM && m0 + tid < e.m_valid ? e.bias[m0 + tid] : 0.0f;
    // running maxima of the tile's columns for the store skipping, read now (kept in LDS): a value
    // read earlier is still a lower bound of the pattern's largest logit when the epilogue uses it
    const int32_t rv = EPI == EPI_LOGL && e.runmax && tid < BN && n0 + tid < e.n_valid ? e.runmax[n0 + tid] : kOrdNegInf;
    issue(0, 0);
    if (nk > 1) issue(1, 1);
    if (nk > 1) __builtin_amdgcn_s_waitcnt(kVm0 | LPW);
    else __builtin_amdgcn_s_waitcnt(kVm0);
    if (tid < BM) bias_s[tid] = bv;
    if (tid < BN) rm_s[tid] = rv;
    __syncthreads();
    // the k loop; a wave of padded rows (LIVE false) only issues its share of the loads and keeps
    // the barriers.  Each step reads the fragments of its second k-half while the first half
    // multiplies, and those of the next step's first half (after the barrier) while the second does.
    auto kloop = [&](auto live_tag) {
        constexpr bool LIVE = decltype(live_tag)::value;
        if (LIVE) rd(F0, 0, 0);
        if constexpr (ST == 3) {
            // stage of step k: k % 3.  The loads of step k + 2 go to the stage of step k - 1, whose reads
            // all completed before the barrier in step k - 1.  The barrier in step k follows the wait for
            // this wave's loads of step k + 1 (issued in step k - 1): LPW newer instructions may remain.
            int k = 0;
            for (; k + 2 < nk; ++k) {
                if (LIVE) rd(F1, k % ST, 16);
                issue(k + 2, (k + 2) % ST);
                __builtin_amdgcn_sched_barrier(0);
                if (LIVE) mm(F0);
                __builtin_amdgcn_s_waitcnt(kVm0 | LPW);
                __syncthreads();
                if (LIVE) rd(F0, (k + 1) % ST, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (LIVE) mm(F1);
            }
            if (k + 1 < nk) {
                if (LIVE) rd(F1, k % ST, 16);
                __builtin_amdgcn_sched_barrier(0);
                if (LIVE) mm(F0);
                __builtin_amdgcn_s_waitcnt(kVm0);
                __syncthreads();
                if (LIVE) rd(F0, (k + 1) % ST, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (LIVE) mm(F1);
                ++k;
            }
            if (LIVE) {
                rd(F1, k % ST, 16);
                mm(F0);
                mm(F1);
            }
        } else {
            // stage of step k: k % 2.  The barrier in step k follows this wave's wait for its loads of step
            // k + 1 (issued in step k - 1) and every wave's last fragment read of step k, so the loads
            // of step k + 2 may then overwrite its stage.
            if constexpr (kOneFrag) {  // the other wavefront of the SIMD covers the fragment reads
                for (int k = 0; k < nk; ++k) {
                    if (LIVE) {
                        mm(F0);
                        rd(F0, k & 1, 16);
                    }
                    if (k + 1 < nk) {
                        __builtin_amdgcn_s_waitcnt(kVm0);
                        __syncthreads();
                        if (k + 2 < nk) issue(k + 2, k & 1);
                    }
                    if (LIVE) {
                        mm(F0);
                        if (k + 1 < nk) rd(F0, (k + 1) & 1, 0);
                    }
                }
                return;
            }
            for (int k = 0; k < nk; ++k) {
                if (LIVE) rd(F1, k & 1, 16);
                __builtin_amdgcn_sched_barrier(0);
                if (LIVE) mm(F0);
                if (k + 1 < nk) {
                    __builtin_amdgcn_s_waitcnt(kVm0);
                    __syncthreads();
                    if (k + 2 < nk) issue(k + 2, k & 1);
                    if (LIVE) rd(F0, (k + 1) & 1, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (LIVE) mm(F1);
            }
        }
    };
    if (live) kloop(std::true_type{});
    else kloop(std::false_type{});
    __syncthreads();  // the epilogue reuses the LDS
    if constexpr (TWO)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] += acc1[i][j][r];
    if constexpr (EPI == EPI_LOGL && SPLIT && NB == 1) {  // the sums of the term pairs an earlier launch left in C
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + wm + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (m >= e.m_valid) continue;
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const int n = n0 + wn + j * 32 + (lane & 31);
                    if (n < e.n_valid) acc[i][j][r] += e.C[(size_t)m * e.ldc + n];
                }
            }
        __syncthreads();  // packed columns may land on another wave's rows
    }
    if constexpr (EPI == EPI_LOGL) {
        logl_epilogue<WGM, TN, BN, SPLIT>(acc, e, m0, n0, wm, wn, smem, bias_s, e.runmax ? rm_s : nullptr);
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

template <int EPI, int NA, int NB, int WGM, int TN, bool SPLIT>
hipError_t launch(const Contraction &g, hipStream_t st)
{
    const int ntm = g.M / (64 * WGM), ntn = (g.N + 64 * TN - 1) / (64 * TN);
    const int gm = std::max(1, std::min(g.e.tile_rows > 0 ? g.e.tile_rows : kTileRows, ntm));
    hipLaunchKernelGGL((k_dma<EPI, NA, NB, WGM, TN, SPLIT>), dim3(ntm * ntn), dim3(128 * WGM), 0, st, g.A[0], g.A[1], g.A[2], g.lda, g.B[0],
                       g.B[1], g.ldb, g.N, g.K, ntn, gm, g.e);
    return hipGetLastError();
}

template <int EPI, int NA, int NB, bool SPLIT = false>
hipError_t pick(const Contraction &g, hipStream_t st)
{
    constexpr bool kWide = !(EPI == EPI_STORE && SPLIT);  // twice the accumulators of 256 x 256 do not fit the registers
    switch (g.tile) {
    case kTile256:
        if constexpr (kWide) return launch<EPI, NA, NB, 4, 4, SPLIT>(g, st);
        break;
    case kTile256x320:
        if constexpr (kWide && NA == 2 && !(SPLIT && NB == 1)) return launch<EPI, NA, NB, 4, 5, SPLIT>(g, st);
        break;
    case kTile256x128: return launch<EPI, NA, NB, 4, 2, SPLIT>(g, st);
    case kTile128: return launch<EPI, NA, NB, 2, 2, SPLIT>(g, st);
    case kTile64: break;
    }
    return hipErrorInvalidValue;
}

}  // namespace

// The CUs take a launch in rounds of the tiles they hold at once: 256 of the 256-row tiles, whose last round
// costs a whole one, and two 128-row tiles per CU, whose tail shortens (a lone workgroup on a CU runs
// faster).  Costs in rounds of the 256 x 256 tile.  Measured (logL, 64^3, 3,200 pixels, us; 64 / 128 / 256 x 128 /
// 256 x 256 tiles; one-term counts with two-term slices, then two-term counts, then three-term slices):
//   1,380 x 1,000   40/61/84/128      46/89/106/199     49/89/130/196
//   6,300 x 1,000   134/107/98/136    171/146/118/209   195/145/159/220
//   6,300 x 2,000   224/194/196/146   291/267/242/226   341/272/324/229
//   6,300 x 3,000   325/266/283/274   440/384/341/427   510/373/447/438
//   6,300 x 4,000   435/392/381/296   605/527/490/450   679/517/622/459
//   25,680 x 4,000  1713/1518/1377/1039
// 256 x 320 tiles (two-term slices), against the best of the others, one-term then two-term counts:
//   6,300 x 2,000 173/146 258/226   6,300 x 3,000 190/266 280/341   6,300 x 4,000 338/296 518/450
//   10,860 x 4,000 544/460 801/705   25,680 x 4,000 1078/1039 1592/1798   6,300 x 3,001 (12,928 pixels) 689/1097 1073/1492
// and at 32^3 (768 pixels) 3,240 x 1,000: 31/29/35/53, 33/37/43/74, 36/36/49/73; 1,380 x 500: 14/27/35/52.
constexpr int64_t kSmallTiles = 56;  // up to this many 256 x 256 tiles' worth: 64 x 64 tiles
GemmTile pick_tile(int64_t rows, int64_t cols, int na, int nb)
{
    const auto tiles = [&](int64_t bm, int64_t bn) { return (rows + bm - 1) / bm * ((cols + bn - 1) / bn); };
    if (tiles(256, 256) <= kSmallTiles) return kTile64;
    const auto rounds = [](int64_t t) { return (double)((t + 255) / 256); };
    const double t256 = rounds(tiles(256, 256));
    const double t2x1 = rounds(tiles(256, 128)) * (nb == 2 ? 0.53 : na == 3 ? 0.71 : 0.65);
    const double t128 = std::max(0.66, (double)tiles(128, 128) / 512.0 * (na + nb == 4 ? 0.74 : 0.80));
    const double t320 = na == 2 ? rounds(tiles(256, 320)) * (nb == 2 ? 1.16 : 1.27) : 1e9;
    if (t320 < t256 && t320 < t2x1 && t320 < t128) return kTile256x320;
    return t256 <= t2x1 && t256 <= t128 ? kTile256 : t2x1 <= t128 ? kTile256x128 : kTile128;
}

// Two sums: the tiles whose two sets of accumulators fit the registers, by the costs above.  An iteration of scaled
// chi^2 at 64^3, us, on 128 x 128 tiles / by this rule: 6,300 x 1,000 1,101/1,051, x 2,000 1,477/1,377, x 4,000 2,323/2,126,
// 10,860 x 4,000 3,809/3,566, not scaled 6,300 x 3,000 1,649/1,683.  With one sum on any tile 6,300 x 4,000 is 2,105, with a
// launch per term, the second adding to what the first stored, 2,350.
GemmTile pick_tile_two(int64_t rows, int64_t cols, int na)
{
    const auto tiles = [&](int64_t bm, int64_t bn) { return (rows + bm - 1) / bm * ((cols + bn - 1) / bn); };
    if (tiles(256, 256) <= kSmallTiles) return kTile64;
    const double t2x1 = (double)((tiles(256, 128) + 255) / 256) * 0.53;
    const double t128 = std::max(0.66, (double)tiles(128, 128) / 512.0 * (na == 2 ? 0.74 : 0.80));
    return t2x1 <= t128 ? kTile256x128 : kTile128;
}

hipError_t run_dma(int epi, const Contraction &g, hipStream_t st)
{
    if (g.M % BM2 || g.N % 128 || g.K % BK2 || g.N < 128 || g.lda >= (1 << 26) || g.ldb >= (1 << 26))
        return hipErrorInvalidValue;
    const int k = g.na * 4 + g.nb;
    if (epi == EPI_LOGL) {
        if (k == 9 && g.split) return pick<EPI_LOGL, 2, 1, true>(g, st);
        if (k == 9) return pick<EPI_LOGL, 2, 1>(g, st);
        if (k == 10) return pick<EPI_LOGL, 2, 2, true>(g, st);
        if (k == 13) return pick<EPI_LOGL, 3, 1>(g, st);
    } else {
        if (k == 5) return pick<EPI_STORE, 1, 1>(g, st);
        if (k == 9) return pick<EPI_STORE, 2, 1>(g, st);
        if (k == 6 && g.two_sums) return pick<EPI_STORE, 1, 2, true>(g, st);
        if (k == 10 && g.two_sums) return pick<EPI_STORE, 2, 2, true>(g, st);
        if (k == 10) return pick<EPI_STORE, 2, 2>(g, st);
        if (k == 13) return pick<EPI_STORE, 3, 1>(g, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace emc
