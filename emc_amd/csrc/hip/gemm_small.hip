// MFMA contractions of small shapes: the 256-row tiles of gemm_dma.hip would leave most of the 256 CUs
// idle (420 rotations x 64 patterns are two of them: 33 us, all latency), so the tile is 64 x 64, one
// 32 x 32 block per wavefront.  Each element's products are added in the order of the larger tiles
// (k ascending, low terms first; two sums where those have two), so the results do not depend on the tile; only the
// logits of three-term slices with two-term counts do, in which the larger tiles add the low counts' products last.
//
// Bound by the latency of the loads along k: the operands go into LDS by DMA (gemm_dma.hip), 64 k at a time,
// kST stages deep, so kST - 1 blocks are in flight, with one barrier per block.  A DMA instruction
// fetches 8 rows of 128 bytes (fragments loaded straight from global memory touch 32 lines per
// instruction: 17.5 us for the 420 x 64 x 512 logL; staged, see kSmallTiles).  LDS rows are 128 B; the eight
// 16-byte chunks of row r sit at chunk ^ ((r >> 1) & 7): 16 consecutive rows fall on distinct banks.
#include "gemm_tile.h"

namespace emc {
namespace {

constexpr int SM = 64, SN = 64, SK = 64;
constexpr int kTerm = 64 * SK * 2;  // LDS bytes of one operand term per stage

// TWO: the products with B[0] and with B[1] are summed apart and added at the end, as two launches of the large
// tiles' store epilogue would (the second adding to the first).
template <int EPI, int NA, int NB, bool TWO, bool DEEP>
__global__ __launch_bounds__(256) void k_small(const bf16_t *__restrict__ A0, const bf16_t *__restrict__ A1,
                                               const bf16_t *__restrict__ A2, int64_t lda,
                                               const bf16_t *__restrict__ B0, const bf16_t *__restrict__ B1,
                                               int64_t ldb, int Kd, EpiArgs e)
{
    if (e.gate && *e.gate <= e.gate_thr) return;  // the sparse M-step runs instead
    constexpr int NT = NA > NB ? NA : NB;         // term pairs a + b < NT are multiplied
    __shared__ float red[4][32];
    __shared__ uint32_t kept_s[2];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * SM, n0 = blockIdx.x * SN;
    if (n0 >= e.n_valid) return;  // a tile of padding (never read)
    if (m0 >= e.m_valid) {
        if (EPI == EPI_LOGL && e.pm && wave == 0 && n0 + lane < e.n_valid)  // k_sm_band reads every group's
            e.pm[(e.band0 + m0 / SM) * e.ldp + n0 + lane] = -1.0e10f;
        return;
    }
    const int fr = lane & 31, fh = lane >> 5;
    const int mw = m0 + (wave >> 1) * 32, nw = n0 + (wave & 1) * 32;
    constexpr int NTERM = NA + NB, STAGE = NTERM * kTerm;
    // stages: two workgroups per CU, or one with as many as its LDS holds
    constexpr int kST = DEEP ? (NTERM <= 2 ? 8 : NTERM == 3 ? 6 : NTERM == 4 ? 4 : 3) : NTERM <= 3 ? 3 : 2;
    constexpr int LPW = NTERM * 2;  // DMA instructions per wavefront and stage (8 rows each; 8 per term)
    constexpr int AHEAD = (kST - (DEEP ? 3 : 2)) * LPW, FIRST = (kST - 2) * LPW;
    static_assert(AHEAD >= 0 && FIRST < 64);
    // s_waitcnt encoding: vmcnt in bits 3:0 and 15:14, lgkmcnt and expcnt not waited
    constexpr uint32_t kVmAhead = 0x0F70 | (AHEAD & 15) | ((AHEAD >> 4) << 14), kVm0 = 0x0F70;
    constexpr uint32_t kVmFirst = 0x0F70 | (FIRST & 15) | ((FIRST >> 4) << 14);
    __shared__ __attribute__((aligned(1024))) unsigned char smem[kST * STAGE];
    // DMA instruction q of this wavefront: rows 8 rb .. 8 rb + 7 of one term; lane l writes chunk l & 7 of row
    // 8 rb + l / 8, which holds logical chunk (l & 7) ^ ((row >> 1) & 7)
    const int lr = lane >> 3;
    const unsigned char *src[LPW];
    uint32_t off[2];  // lane offsets for operand A and B, even rb (odd rb: chunk ^ 4, 64 bytes away)
    const int c_even = (lane & 7) ^ (lr >> 1);
    off[0] = (uint32_t)(lr * (int)lda * 2 + c_even * 16);
    off[1] = (uint32_t)(lr * (int)ldb * 2 + c_even * 16);
    const uint32_t flip = (c_even & 4) ? (uint32_t)-64 : 64u;
#pragma unroll
    for (int q = 0; q < LPW; ++q) {
        const int g = __builtin_amdgcn_readfirstlane(wave) * LPW + q, t = g >> 3, row = (g & 7) * 8;
        const bf16_t *op = t < NA ? (t == 0 ? A0 : t == 1 ? A1 : A2) : (t == NA ? B0 : B1);
        src[q] = reinterpret_cast<const unsigned char *>(op + (t < NA ? (int64_t)(m0 + row) * lda : (int64_t)(n0 + row) * ldb));
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    auto issue = [&](int step, int stage) {
#pragma unroll
        for (int q = 0; q < LPW; ++q) {
            const int g = __builtin_amdgcn_readfirstlane(wave) * LPW + q;
            lds_dma16(off[(g >> 3) < NA ? 0 : 1] + ((g & 1) ? flip : 0u), src[q] + (int64_t)step * (SK * 2),
                      lds0 + stage * STAGE + g * 1024);
        }
    };
    f32x16 acc, acc1;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = acc1[r] = 0.0f;
    const int sw = (fr >> 1) & 7;
    struct Frags {
        bf16x8 a[NA][4], b[NB][4];
    };
    auto fetch = [&](int stage, Frags &f) {
        const unsigned char *S = smem + stage * STAGE;
        const unsigned char *ra = S + ((wave >> 1) * 32 + fr) * 128, *rb = S + NA * kTerm + ((wave & 1) * 32 + fr) * 128;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int co = ((2 * t + fh) ^ sw) * 16;
#pragma unroll
            for (int a = 0; a < NA; ++a) f.a[a][t] = *reinterpret_cast<const bf16x8 *>(ra + a * kTerm + co);
#pragma unroll
            for (int b = 0; b < NB; ++b) f.b[b][t] = *reinterpret_cast<const bf16x8 *>(rb + b * kTerm + co);
        }
    };
    auto multiply = [&](const Frags &f) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int a = NA - 1; a >= 0; --a)
#pragma unroll
                for (int b = NB - 1; b >= 0; --b)
                    if (a + b < NT) {
                        f32x16 &to = TWO && b == 1 ? acc1 : acc;
                        to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[a][t], f.b[b][t], to, 0, 0, 0);
                    }
    };
    // step k is in stage k % kST.  Past the last step the loads fetch it again (into a stage nothing reads),
    // so the number of loads in flight is the same in every step.
    const int nk = Kd / SK;
#pragma unroll
    for (int s = 0; s < kST - 1; ++s) issue(min(s, nk - 1), s);
    if constexpr (DEEP) {
        // step k multiplies the fragments read in step k - 1, while those of step k + 1 are read
        Frags f[2];
        __builtin_amdgcn_s_waitcnt(kVmFirst);  // this wavefront's loads of step 0
        __syncthreads();
        fetch(0, f[0]);
        int st = 0;
        auto step = [&](int k, const Frags &now, Frags &next) {
            __builtin_amdgcn_s_waitcnt(kVmAhead);  // of step k + 1
            __syncthreads();                       // every wavefront's, and the last reads of step k - 1's stage
            issue(min(k + kST - 1, nk - 1), st == 0 ? kST - 1 : st - 1);
            st = st + 1 == kST ? 0 : st + 1;
            fetch(st, next);
            multiply(now);
        };
        for (int k = 0; k < nk; k += 2) {
            step(k, f[0], f[1]);
            if (k + 1 < nk) step(k + 1, f[1], f[0]);
        }
    } else {
        Frags f;
        int st = 0;
        for (int k = 0; k < nk; ++k) {
            __builtin_amdgcn_s_waitcnt(kVmAhead);  // this wavefront's loads of step k
            __syncthreads();                       // every wavefront's, and the last reads of step k - 1's stage
            issue(min(k + kST - 1, nk - 1), st == 0 ? kST - 1 : st - 1);
            fetch(st, f);
            multiply(f);
            st = st + 1 == kST ? 0 : st + 1;
        }
    }
    __builtin_amdgcn_s_waitcnt(kVm0);  // no load is left to write LDS
    if constexpr (TWO)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] += acc1[r];

    // accumulator layout: lane holds column lane % 32, rows 8*(r/4) + 4*(lane/32) + r%4, r = 0..15
    const int n = nw + fr;
    const bool nok = n < e.n_valid;
    if constexpr (EPI == EPI_STORE) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = mw + 8 * (r >> 2) + 4 * fh + (r & 3);
            if (m >= e.m_valid || !nok) continue;
            float *cp = e.C + (size_t)m * e.ldc + n;
            *cp = e.accumulate ? *cp + acc[r] : acc[r];
        }
        return;
    }
    // logL: the bias, the maxima of the tile's 64 rows (e.pm; k_sm_band forms the sums, from the stored logits) and
    // the store skipping by the rules of the larger tiles' epilogue (every logit that is stored is stored in place)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int m = mw + 8 * (r >> 2) + 4 * fh + (r & 3);
        acc[r] = m < e.m_valid ? acc[r] + e.bias[m] : -INFINITY;
    }
    bool kept = true;
    if (e.pm) {
        float mx = -1.0e10f;
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, acc[r]);
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        if (lane < 32) red[wave][lane] = mx;
        __syncthreads();
        mx = fmaxf(red[wave & 1][fr], red[2 + (wave & 1)][fr]);
        if (wave < 2) {  // the upper wavefronts read the running maxima: the lower ones take their choice
            const bool keep = !(e.runmax && nok && (double)mx < (double)float_of_ord(e.runmax[n]) - kSkipStoreNats);
            const uint64_t kb = __ballot(keep);
            if (lane == 0) kept_s[wave] = (uint32_t)kb;
        }
        __syncthreads();
        const uint32_t kept_m = kept_s[wave & 1];
        kept = (kept_m >> fr) & 1u;
        const int64_t orow = (e.band0 + m0 / SM) * e.ldp;
        if (wave < 2 && lane < 32 && nok) {
            e.pm[orow + n] = mx;
            if (e.blk) e.blk[orow + n] = (int16_t)(kept ? -2 : -1);
            if (e.runmax && mx == mx) atomicMax(e.runmax + n, ord_of(mx));
        }
        if (e.runmax && wave < 2) {
            const int cnt = __popc(~kept_m & (uint32_t)__ballot(nok));
            if (lane == 0 && cnt > 0) atomicAdd(e.skipped, (double)cnt);
        }
    }
    if (kept && nok)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = mw + 8 * (r >> 2) + 4 * fh + (r & 3);
            if (m < e.m_valid) e.C[(size_t)m * e.ldc + n] = acc[r];
        }
}

// Up to one tile per CU: a workgroup has the CU to itself, all of its LDS for stages, and reads the next step's
// fragments while it multiplies (three-term slices, 1,000 x 777 x 1,664: 22.4 us with two stages, 21 with four, 17
// with the fragments ahead too; 420 x 64 x 512 8.2 both ways).  With more tiles two workgroups share a CU and hide each
// other's waits: 3,240 x 1,000 x 896 two-term counts 30 us, one workgroup with four stages 46.
constexpr int64_t kDeepTiles = 256;

template <int EPI, int NA, int NB, bool TWO = false>
hipError_t launch(const Contraction &g, hipStream_t st)
{
    const dim3 grid((g.N + SN - 1) / SN, g.M / SM);
    const bool deep = (int64_t)grid.x * grid.y <= kDeepTiles;
    const auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, g.A[0], g.A[1], g.A[2], g.lda, g.B[0], g.B[1], g.ldb, g.K, g.e);
    };
    if (deep) run(k_small<EPI, NA, NB, TWO, true>);
    else run(k_small<EPI, NA, NB, TWO, false>);
    return hipGetLastError();
}

}  // namespace

hipError_t run_small(int epi, const Contraction &g, hipStream_t st)
{
    if (g.M % SM || g.N % SN || g.K % SK) return hipErrorInvalidValue;
    const int k = g.na * 4 + g.nb;
    if (epi == EPI_LOGL) {
        if (k == 9) return launch<EPI_LOGL, 2, 1>(g, st);
        if (k == 10) return launch<EPI_LOGL, 2, 2>(g, st);
        if (k == 13) return launch<EPI_LOGL, 3, 1>(g, st);
        if (k == 14) return launch<EPI_LOGL, 3, 2>(g, st);
    } else if (g.two_sums && g.nb == 2) {
        if (g.na == 1) return launch<EPI_STORE, 1, 2, true>(g, st);
        if (g.na == 2) return launch<EPI_STORE, 2, 2, true>(g, st);
        if (g.na == 3) return launch<EPI_STORE, 3, 2, true>(g, st);
    } else {
        if (k == 5) return launch<EPI_STORE, 1, 1>(g, st);
        if (k == 9) return launch<EPI_STORE, 2, 1>(g, st);
        if (k == 10) return launch<EPI_STORE, 2, 2>(g, st);
        if (k == 13) return launch<EPI_STORE, 3, 1>(g, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace emc
