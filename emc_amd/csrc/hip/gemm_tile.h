// Device code shared by the MFMA contraction kernels (gemm_mfma.hip, gemm_dma.hip, gemm_small.hip):
// fragment types, the epilogue's arguments and the logL epilogue of the tiles of 128 and 256 rows.
#pragma once

#include <algorithm>
#include <type_traits>

#include "../emc_internal.h"

namespace emc {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

enum { EPI_LOGL = 0, EPI_STORE = 1, EPI_SCATTER = 2 };

struct EpiArgs {
    float *C;            // logits / U output
    int64_t ldc;
    int m_valid, n_valid;
    const float *bias;   // [rows] (logL)
    // fused scatter
    const double *T;     // [rows] slice sums
    const float *rotm;   // [rows][12]
    const float *axyz;   // [3][Pp]
    int Pp, Pa, L, interp;
    float *Mnum, *Wt;
    // softmax partials of the logL epilogue: per band (the tile's rows) and pattern, the band
    // maximum pm and (not from 64-row tiles) sum of exp(R - pm) ps; band = band0 + m-tile
    float *pm;
    double *ps;
    int64_t band0, ldp;
    // the DMA logL kernel's store skipping (null: every logit is stored): per pattern the running
    // maximum of the band maxima (ord_of form), and the count of columns left out
    int32_t *runmax;
    double *skipped;
    int16_t *blk;  // [band][ldp] where each column's logits went (null: every logit in place)
    // device-side choice between this kernel and the sparse M-step: the whole grid returns at
    // once when *gate <= gate_thr (the responsibilities' non-zero count is small)
    const double *gate;
    double gate_thr;
    bool accumulate;  // store epilogue (and the logL's where split names it): C += acc instead of C = acc
    int tile_rows;    // row panels per group of consecutive tiles (0 = kTileRows; not 64 x 64 tiles)
};

constexpr int BM2 = 256;  // rows of the large tiles

// One DMA load of 16 bytes per lane, from base + off (lane offset), into LDS at the wave-uniform byte
// address lds (lane l lands at lds + 16 l).  Written as inline asm: with the builtin, the compiler's
// LDS-DMA tracking puts a vmcnt(0) in front of every LDS read, which would wait for the loads of later
// stages too; the kernel waits with explicit vmcnt counts instead.  The instruction has no register result;
// the s_nop is the one wait state required between writing M0 and an LDS DMA.  M0 is a reserved register to
// the compiler; the kernels' code uses it nowhere else (clang warns about the clobber, silenced here).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_dma16(uint32_t off, const void *base, uint32_t lds)
{
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds)
                 : "memory", "m0");
}
#pragma clang diagnostic pop

// Order-preserving integer form of a float (signed compare = float compare, NaN aside), for the
// running per-pattern maxima kept with integer atomicMax; kOrdNegInf is the form of -inf.
__device__ __forceinline__ int32_t ord_of(float x)
{
    const int32_t b = __float_as_int(x);
    return b >= 0 ? b : b ^ 0x7fffffff;
}
__device__ __forceinline__ float float_of_ord(int32_t k) { return __int_as_float(k >= 0 ? k : k ^ 0x7fffffff); }
constexpr int32_t kOrdNegInf = (int32_t)0x807fffff;

// A band's logits of a pattern are not stored when the band's largest one lies more than this many
// nats below a largest logit already found for the pattern: every responsibility in the band is then
// below exp(-128) of the pattern's largest one, and the softmax, which treats every band more than
// kSkipApplyNats below the pattern's lse as -inf, computes P = 0 there from the band maxima alone.
constexpr double kSkipStoreNats = 128.0;

// logL epilogue of the tiles of 256 and 128 rows (WGM = 4 or 2 waves along M x 2 along N, each a 64-row
// by BN2/2-column block of 2 x TN 32x32 tiles).  Accumulator layout: lane holds column lane % 32
// of each 32x32 tile and rows 8*(r/4) + 4*(lane/32) + r%4, r = 0..15.  R = acc + bias_s.  The
// softmax partials of this band, the tile's rows (e.pm and e.ps: these kernels run only with
// the softmax fused) restate k_sm_partial's rules: column maxima from the -1e10 floor, over the lane
// pair, then over the row-waves through LDS; then the sums of exp(R - max), where a term with
// R - max <= -1e10 (or not a number) adds nothing.  With one-term counts each lane sums its 32 terms of a
// column in FP32 on the hardware exp2 (the exponent floored at -1e10, whose exp2 is 0) and the lane and wave
// partials are added in FP64; with two-term counts (SPLIT) every term is an expf and is added in FP64, as in
// k_sm_partial, which forms these sums where the tile is 64 x 64.
// The logits are stored after the maxima are known.  Without e.blk every logit is stored in place
// (row-major R).  With e.blk (the iteration's store skipping): a column whose band maximum lies
// kSkipStoreNats below rmk[column of the tile] (running maxima read when the workgroup started:
// lower bounds of the pattern's largest logit) is not stored; in a 256 x 256 tile inside the valid rows and
// columns the kept columns are packed, in column order, as blocks of 256 consecutive floats (the
// column's rows) in the tile's own rows of R (block k in row m0 + k, columns n0 .. n0 + 255), so the
// HBM writes are whole lines however few columns are kept; the other tiles store their kept columns
// in place.  e.blk[band][pattern] records the block (>= 0), -2 (in place) or -1 (not stored); every
// band maximum is merged into e.runmax, and e.skipped counts the columns left out.
// A tile inside the valid rows and columns (every tile but the last row band and column tile) takes
// a path without bounds checks.  lds: 48 BN2 + 1056 bytes, free (the main loop's stages).  bias_lds:
// the tile's row biases, copied to LDS by the kernel (0 past m_valid), so no vector-memory wait
// holds up the logit stores (on gfx9 a wait for a load also waits for every store issued before it)
// and no bias stays in registers between the passes.
template <int WGM, int TN, int BN2, bool SPLIT, bool kFull>
__device__ __forceinline__ void logl_epi(const f32x16 (&acc)[2][TN], const EpiArgs &e, int m0, int n0, int wm, int wn,
                                         void *lds, const float *bias_lds, const int32_t *rmk)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    wm = __builtin_amdgcn_readfirstlane(wm);
    wn = __builtin_amdgcn_readfirstlane(wn);
    const int hr = 4 * (lane >> 5), cl = lane & 31;
    const uint32_t lo = (uint32_t)(hr * e.ldc + cl);  // lane offset from a row's base
    // bias of accumulator row r of tile i; -inf past m_valid (adds to neither the maximum nor the sum)
    auto bias = [&](int i, int r) {
        const int mt = wm + i * 32 + 8 * (r >> 2) + (r & 3) + hr;
        return kFull || m0 + mt < e.m_valid ? bias_lds[mt] : -INFINITY;
    };
    float cmax[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) cmax[j] = -1.0e10f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float add = bias(i, r);
#pragma unroll
            for (int j = 0; j < TN; ++j) cmax[j] = fmaxf(cmax[j], acc[i][j][r] + add);
        }
    constexpr int BM = 64 * WGM;
    auto over_waves = [&](const auto *x, int c, auto op) {  // row-waves combined pairwise, in order
        if constexpr (WGM == 4) return op(op(x[c], x[BN2 + c]), op(x[2 * BN2 + c], x[3 * BN2 + c]));
        else return op(x[c], x[BN2 + c]);
    };
    auto fmx = [](float a, float b) { return fmaxf(a, b); };
    float *red = reinterpret_cast<float *>(lds);            // [WGM][BN2] maxima
    double *reds = reinterpret_cast<double *>(lds) + 2 * BN2;  // [WGM][BN2] sums (after the maxima)
    int *cnt = reinterpret_cast<int *>(reinterpret_cast<unsigned char *>(lds) + 48 * BN2 + 1024);  // [2 TN]
    const int wrow = wave >> 1, half = wn / (BN2 / 2);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        cmax[j] = fmaxf(cmax[j], __shfl_xor(cmax[j], 32, 64));
        if (lane < 32) red[wrow * BN2 + wn + j * 32 + lane] = cmax[j];
    }
    __syncthreads();
    bool keep[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int c = wn + j * 32 + cl;
        cmax[j] = over_waves(red, c, fmx);
        keep[j] = !(rmk && (double)cmax[j] < (double)float_of_ord(rmk[c]) - kSkipStoreNats);
        if (!kFull) keep[j] = keep[j] && n0 + c < e.n_valid;
    }
    const bool compact = kFull && e.blk && BN2 == 256 && BM == 256;  // a block is 256 floats of the tile's row
    // kept columns of each group of 32 (the same in every row-wave: keep depends on the column only)
    uint32_t km[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) km[j] = (uint32_t)__ballot(keep[j]);
    if (compact && wrow == 0 && lane == 0)
#pragma unroll
        for (int j = 0; j < TN; ++j) cnt[half * TN + j] = __popc(km[j]);
    if (rmk && wrow == 0) {  // the columns left out, counted once (row-wave 0, lanes 0-31)
        int nskip = 0;
#pragma unroll
        for (int j = 0; j < TN; ++j) nskip += __popc(~km[j] & (uint32_t)__ballot(n0 + wn + j * 32 + cl < e.n_valid));
        if (lane == 0 && nskip > 0) atomicAdd(e.skipped, (double)nskip);
    }
    constexpr float kLog2e = 1.4426950408889634f;
    std::conditional_t<SPLIT, double, float> fs[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) fs[j] = 0;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float add = bias(i, r);
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const float d = fmaxf((acc[i][j][r] + add) - cmax[j], -1.0e10f);
                if constexpr (SPLIT) fs[j] += (double)expf(d);
                else fs[j] += __builtin_amdgcn_exp2f(d * kLog2e);
            }
        }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        double s = (double)fs[j];
        s += __shfl_xor(s, 32, 64);
        if (lane < 32) reds[wrow * BN2 + wn + j * 32 + lane] = s;
    }
    __syncthreads();  // also publishes the kept-column counts
    const int64_t orow = (e.band0 + m0 / BM) * e.ldp;  // this band's row of pm, ps and blk
    if (compact) {
        int off = 0;  // blocks of the groups before (half, j) in column order
#pragma unroll
        for (int g = 0; g < 2 * TN; ++g) off += g < half * TN ? cnt[g] : 0;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int rank = off + __popc(km[j] & ((1u << cl) - 1u));
            off += __popc(km[j]);
            if (wrow == 0 && lane < 32) e.blk[orow + n0 + wn + j * 32 + cl] = (int16_t)(keep[j] ? rank : -1);
            if (!keep[j]) continue;
            float *blk = e.C + (size_t)(m0 + rank) * e.ldc + n0;
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g) {  // rows 8 g + hr + 0..3 of tile i: 16 contiguous bytes
                    const int mr = wm + i * 32 + 8 * g + hr;
                    const float4 v = make_float4(acc[i][j][4 * g] + bias(i, 4 * g), acc[i][j][4 * g + 1] + bias(i, 4 * g + 1),
                                                 acc[i][j][4 * g + 2] + bias(i, 4 * g + 2),
                                                 acc[i][j][4 * g + 3] + bias(i, 4 * g + 3));
                    *reinterpret_cast<float4 *>(blk + mr) = v;
                }
        }
    } else {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            if (e.blk && wrow == 0 && lane < 32 && n0 + wn + j * 32 + cl < e.n_valid)
                e.blk[orow + n0 + wn + j * 32 + cl] = (int16_t)(keep[j] ? -2 : -1);
            if (!keep[j]) continue;
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int mt = wm + i * 32 + 8 * (r >> 2) + (r & 3);  // tile row of lanes 0-31
                    if (!kFull && m0 + mt + hr >= e.m_valid) continue;
                    float *row = e.C + (size_t)(m0 + mt) * e.ldc + (n0 + wn);
                    row[lo + j * 32] = acc[i][j][r] + bias(i, r);
                }
        }
    }
    for (int c = tid; c < BN2; c += 128 * WGM) {
        const int n = n0 + c;
        if (n >= e.n_valid) continue;
        const float mx = over_waves(red, c, fmx);
        double sm = reds[c];
#pragma unroll
        for (int w = 1; w < WGM; ++w) sm += reds[w * BN2 + c];
        e.pm[orow + n] = mx;
        e.ps[orow + n] = sm;
        if (e.runmax && mx == mx) atomicMax(e.runmax + n, ord_of(mx));
    }
}

template <int WGM, int TN, int BN2, bool SPLIT = false>
__device__ __forceinline__ void logl_epilogue(const f32x16 (&acc)[2][TN], const EpiArgs &e, int m0, int n0, int wm, int wn,
                                              void *lds, const float *bias_lds, const int32_t *rmk = nullptr)
{
    if (m0 + 64 * WGM <= e.m_valid && n0 + BN2 <= e.n_valid)
        logl_epi<WGM, TN, BN2, SPLIT, true>(acc, e, m0, n0, wm, wn, lds, bias_lds, rmk);
    else logl_epi<WGM, TN, BN2, SPLIT, false>(acc, e, m0, n0, wm, wn, lds, bias_lds, rmk);
}

// The contraction C [M][N] (row stride e.ldc) = sum over the term pairs (a, b), a + b < max(na, nb), of
// A[a] [M][K] . B[b] [N][K]^T with FP32 accumulation (na <= 3 and nb <= 2 BF16 terms).  M is a multiple
// of 256, N of 128, K of 128.
enum GemmTile { kTile64, kTile128, kTile256x128, kTile256, kTile256x320 };

struct Contraction {
    GemmTile tile = kTile256;
    int na = 1, nb = 1;
    const bf16_t *A[3] = {nullptr, nullptr, nullptr}, *B[2] = {nullptr, nullptr};
    int64_t lda = 0, ldb = 0;
    int M = 0, N = 0, K = 0;
    bool split = false;     // run_dma's logits: two-term counts' (the last of the launches that take them, where several do)
    bool two_sums = false;  // nb = 2, store epilogue: the products of the two B terms summed apart, then added
    EpiArgs e{};
};

// Tile for a contraction of this many rows, columns and terms, and its rows (the logL epilogue's maxima are over these).
GemmTile pick_tile(int64_t rows, int64_t cols, int na, int nb);
GemmTile pick_tile_two(int64_t rows, int64_t cols, int na);  // two_sums
inline int tile_rows_of(GemmTile t) { return t == kTile64 ? 64 : t == kTile128 ? 128 : 256; }
// epi: EPI_LOGL or EPI_STORE.  run_small: kTile64; run_dma: the others, na + nb <= 4.
hipError_t run_small(int epi, const Contraction &g, hipStream_t st);
hipError_t run_dma(int epi, const Contraction &g, hipStream_t st);

}  // namespace emc
