// Responsibilities: per-pattern log-sum-exp over rotations and P = exp(R - lse).
//
// Restates cuda_max_vector + cuda_respons_max_expf + the host log/add + cuda_norm_respons_sumexpf
// (emc_cuda.cu:1041-1056, 1175-1217, 1253-1272; main.cpp:367-392) as three streaming passes over
// the logits R[S][I] (row = rotation, so a pattern is a column):
//   1. partial: each thread owns one pattern column over a band of rotation rows and keeps an
//      online (max, sum of exp) pair; exp is FP32, the sum FP64.  Reads are coalesced rows.
//   2. final:   combine the bands per pattern in FP64 -> lse'_i; per-block partial sums of lse'.
//   3. apply:   P = exp(R - lse'_i) written either in place (FP32 path) or as a BF16 hi+lo pair
//      (MFMA path), plus per-band row sums of P (T_s partials), reduced in FP64, and (MFMA path)
//      the count of non-zero P, which picks the dense or the sparse form of the M-step.
// The reference's -1e10 floor on the max and on R - max is kept.
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

// Partials of the 256-row bands where the logL ran on 64-row tiles with one-term counts, whose epilogue wrote the maxima
// of the 64-row groups (gm, [4 groups per band][I]): the sums of exp(R - max) in the order and arithmetic of the 256-row
// tiles' epilogue (32 rows of a column in FP32, on the hardware exp2, the pairs and the groups of 64 rows in
// FP64), so the partials are those of the 256-row tiles bit for bit (128-row tiles have bands of 128 rows, and two-term
// counts on 64-row tiles take k_sm_partial: other sums, to rounding the same).  A group whose logits were left out (gblk, null: none) adds
// nothing: its terms are below exp(-128) of the pattern's sum.  Bands count from each chunk's first rotation.
// One workgroup takes 32 columns, a thread 32 rows of one; all latency: 5.5 us at
// 3,880 x 777, 10.5 when the logits were read after the group's record.
__global__ __launch_bounds__(256) void k_sm_band(const float *__restrict__ R, int64_t ldr, int S, int I, int chunk, int bpc,
                                                 const float *__restrict__ gm, const int16_t *__restrict__ gblk,
                                                 float *__restrict__ pm, double *__restrict__ ps)
{
    __shared__ double red[4][32];
    constexpr float kLog2e = 1.4426950408889634f;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, hr = 4 * (lane >> 5);
    const int band = blockIdx.y, i = blockIdx.x * 32 + (lane & 31), ic = min(i, I - 1);
    const int l0 = (band % bpc) * 256 + 64 * w, s0 = (band / bpc) * chunk + l0;  // this wave's group of 64 rows
    const int rows = min(min(chunk, S - (band / bpc) * chunk) - l0, 64);
    float fs = 0.0f, mx = -1.0e10f, v[32], m4[4];
    int kept = -2;
    if (rows > 0) {  // every load in flight at once (the logits of a left-out group are old ones, not used)
        if (gblk) kept = gblk[(size_t)(4 * band + w) * I + ic];
#pragma unroll
        for (int k = 0; k < 32; ++k) {
            const int r = 32 * (k >> 4) + 8 * ((k >> 2) & 3) + (k & 3) + hr;
            v[k] = R[(size_t)(s0 + min(r, rows - 1)) * ldr + ic];
        }
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) m4[g] = gm[(size_t)(4 * band + g) * I + ic];
#pragma unroll
    for (int g = 0; g < 4; ++g) mx = fmaxf(mx, m4[g]);
    if (rows > 0 && kept != -1)
#pragma unroll
        for (int k = 0; k < 32; ++k) {
            const int r = 32 * (k >> 4) + 8 * ((k >> 2) & 3) + (k & 3) + hr;
            fs += __builtin_amdgcn_exp2f(fmaxf((r < rows ? v[k] : -INFINITY) - mx, -1.0e10f) * kLog2e);
        }
    double s = (double)fs;
    s += __shfl_xor(s, 32, 64);
    if (lane < 32) red[w][lane] = s;
    __syncthreads();
    if (threadIdx.x < 32 && i < I) {
        pm[(size_t)band * I + i] = mx;
        ps[(size_t)band * I + i] = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
    }
}

constexpr int kPartialRows = 8;
__global__ __launch_bounds__(256) void k_sm_partial(const float *__restrict__ R, int64_t ldr, int S, int I,
                                                    int rows_per_band, float *__restrict__ pm,
                                                    double *__restrict__ ps)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int band = blockIdx.y;
    if (i >= I) return;
    const int r0 = band * rows_per_band, r1 = min(S, r0 + rows_per_band);
    float m = -1.0e10f;
    double sum = 0.0;
    const float *col = R + i;
    for (int s = r0; s < r1; s += kPartialRows) {  // the rows' loads in flight together
        float v[kPartialRows];
#pragma unroll
        for (int q = 0; q < kPartialRows; ++q) v[q] = col[(size_t)min(s + q, r1 - 1) * ldr];
#pragma unroll
        for (int q = 0; q < kPartialRows; ++q) {
            if (s + q >= r1) break;
            const bool up = v[q] > m;
            const float d = up ? m - v[q] : v[q] - m;
            const double ex = (double)expf(d);
            if (up) {
                sum = sum * ex + 1.0;
                m = v[q];
            } else if (d > -1.0e10f) {
                sum += ex;
            }
        }
    }
    pm[(size_t)band * I + i] = m;
    ps[(size_t)band * I + i] = sum;
}

// lse_i = m_i + log sum_b ps_b exp(pm_b - m_i) over the bands.  Eight lanes per pattern take every
// eighth band and combine over a fixed butterfly (deterministic); 32 patterns per workgroup.
constexpr int kFinalPat = 32;
__global__ __launch_bounds__(256) void k_sm_final(const float *__restrict__ pm, const double *__restrict__ ps,
                                                  int nbands, int I, double *__restrict__ lse,
                                                  double *__restrict__ blk_sum, double *__restrict__ scal)
{
    __shared__ double red[4];
    const int g = threadIdx.x & 7;
    const int i = blockIdx.x * kFinalPat + (threadIdx.x >> 3);
    float m = -1.0e10f;
    if (i < I)
        for (int b = g; b < nbands; b += 8) m = fmaxf(m, pm[(size_t)b * I + i]);
    m = fmaxf(m, __shfl_xor(m, 1, 64));
    m = fmaxf(m, __shfl_xor(m, 2, 64));
    m = fmaxf(m, __shfl_xor(m, 4, 64));
    double sum = 0.0;
    if (i < I)
        for (int b = g; b < nbands; b += 8) {
            const double sb = ps[(size_t)b * I + i];
            if (sb > 0.0) sum += sb * exp((double)pm[(size_t)b * I + i] - (double)m);
        }
    sum += __shfl_xor(sum, 1, 64);
    sum += __shfl_xor(sum, 2, 64);
    sum += __shfl_xor(sum, 4, 64);
    double l = 0.0;
    if (i < I && g == 0) {
        l = (double)m + log(sum);
        if (!isfinite(l)) scal[SC_NONFINITE] = 1.0;
        lse[i] = l;
    }
    l = wave_sum(l);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = l;
    __syncthreads();
    if (threadIdx.x == 0) blk_sum[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// Deterministic sum of n doubles by one workgroup of 1,024 threads (the value in thread 0).
__device__ __forceinline__ double block_sum(const double *__restrict__ x, int n, double *red)
{
    // eight partial sums per thread (eight loads in flight), added in a fixed order
    double p[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    int k = threadIdx.x;
    for (; k + 7 * 1024 < n; k += 8 * 1024)
#pragma unroll
        for (int q = 0; q < 8; ++q) p[q] += x[k + q * 1024];
#pragma unroll
    for (int q = 0; q < 8; ++q)
        if (k + q * 1024 < n) p[q] += x[k + q * 1024];
    double a = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
    a = wave_sum(a);
    __syncthreads();  // an earlier sum's partials are read
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
    __syncthreads();
    double t = 0.0;
    for (int k = 0; k < 16; ++k) t += red[k];
    return t;
}

// The E-step's last sums in one launch (each was a launch of its own, about 5 us of the smallest problems'
// 200): workgroup 0 the non-zero responsibilities, workgroup 1 the total log-likelihood (log-sum-exps
// and pattern constants), the others T_s = sum over column blocks of the partial row sums, in order.
__global__ __launch_bounds__(1024) void k_sm_sums(const double *__restrict__ nz, int nnz, const double *__restrict__ blk,
                                                  int nblk, const double *__restrict__ cst, int I,
                                                  const double *__restrict__ Tpart, int ncb, int S, int Sp,
                                                  double *__restrict__ T, double *__restrict__ scal)
{
    __shared__ double red[16];
    if (blockIdx.x == 0) {
        const double t = block_sum(nz, nnz, red);
        if (threadIdx.x == 0) scal[SC_NNZ] = t;
        return;
    }
    if (blockIdx.x == 1) {
        const double t = block_sum(blk, nblk, red) + block_sum(cst, I, red);
        if (threadIdx.x == 0) scal[SC_TOTAL] = t;
        return;
    }
    const int s = (blockIdx.x - 2) * 1024 + threadIdx.x;
    if (s >= Sp) return;
    double t = 0.0;
    if (s < S)
        for (int b = 0; b < ncb; ++b) t += Tpart[(size_t)b * S + s];
    T[s] = t;
}

constexpr int kApplyRows = 8;    // rotation rows per workgroup (the block reads of k_sm_apply assume 8)

// Two floats to a packed BF16 pair (a in the low half), round to nearest even: gfx950's
// two-source v_cvt_pk_bf16_f32, which rounds as f2bf_dev does.  Written as asm because the compiler
// emits one single-source conversion per value and merges the halves with extra instructions.
// The s_nop is the wait state gfx950 requires between a transcendental VALU instruction (the
// v_exp_f32 that produces p) and a VALU instruction that reads its result, and between a write with
// a destination select and its reader: the compiler inserts these for the instructions it emits but
// not in front of inline asm, and without it the conversion can read a stale value when scheduled
// right after the exp.
__device__ __forceinline__ uint32_t pk_bf16(float a, float b)
{
    uint32_t r;
    asm("s_nop 0\n\tv_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
constexpr int kApplyCols = 1024; // pattern columns per workgroup (4 per thread)

// OUT = 0: P in place (FP32), and P * iphi to Pphi when iphi is given; pdirty says which 256-pattern segments
// hold a non-zero.  OUT = 1: BF16 hi/lo pair, of P * iphi when iphi is given (the
// M-step's P/phi under intensity scaling; the slice sums T stay sums of P).
// OUT = 1 skips the store of a wave's 256-pattern row segment when every value in it is zero and
// pdirty says the segment already holds only zeros (P is mostly zeros once the posteriors are
// sharp); pdirty is then updated to whether the segment holds a non-zero value.
// pm (the logL epilogue's band maxima, [band][I], band of row s = (s / chunk) bpc + (s % chunk) / brows;
// null without them): a pattern's logits in a band whose maximum lies more than kSkipApplyNats below
// its lse are not read and count as -inf, which gives the P = 0 that they give (exp of less than -110
// is 0 in FP32).  blk (the skipping logL pass's record, [band][I]; null when every logit is in
// place): -1 = the band's logits of the pattern were not stored (they are negligible: the pass
// leaves out only bands more than 128 below a maximum of the pattern, so pm marks them too), -2 = in
// place, k >= 0 = the 256 logits of the band are the row brow0 + k of R from the pattern's 256-column
// tile on (brow0 = the band's first row).
constexpr double kSkipApplyNats = 110.0;
template <int OUT>
__global__ __launch_bounds__(256) void k_sm_apply(float *__restrict__ R, int64_t ldr, int S, int I,
                                                  const double *__restrict__ lse, bf16_t *__restrict__ Ph,
                                                  bf16_t *__restrict__ Pl, double *__restrict__ Tpart,
                                                  double *__restrict__ nnz, const float *__restrict__ iphi,
                                                  uint8_t *__restrict__ pdirty, int nseg, const float *__restrict__ pm,
                                                  const int16_t *__restrict__ blk, int chunk, int bpc, int brows,
                                                  float *__restrict__ Pphi)
{
    static_assert(kApplyRows == 8, "8 rows: two per wave in the row sums, 8 floats per block read");
    constexpr float kLog2e = 1.4426950408889634f;
    int nz = 0;  // entries of non-zero P (OUT = 1: hi or lo term; for the choice of the M-step)
    // per-thread row sums: each is a float (a float sum of the thread's four values, or one value),
    // kept as such and widened when the row sums are formed
    __shared__ float rs[kApplyRows][256];
    const int c0 = blockIdx.x * kApplyCols + threadIdx.x * 4;
    const int r0 = blockIdx.y * kApplyRows;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int seg = (blockIdx.x * kApplyCols) / 256 + wave;  // this wave's 256 patterns
    const bool seg_live = seg * 256 < I;                      // uniform over the wave
    // lse as a float pair: x - lh is exact wherever p is not negligible (x and lse within a factor
    // of 2, Sterbenz), so exp((x - lh) - ll) carries the double-precision argument to float rounding
    // (a column past I gets lh = +inf: its p is exp2(-inf) = 0 without a select per element)
    // The thread's four patterns' lse, band maxima and block records are read with one vector load
    // each (lse always: c0 is a multiple of 4 and lse holds Ip >= I rounded up to 4 entries; the
    // [band][I] rows of pm and blk when I is a multiple of 4), element by element otherwise: the
    // short workgroups of this kernel are bound by the vector-memory data path.
    double lv[4];
    if (c0 < I) {
        const double2 a = *reinterpret_cast<const double2 *>(lse + c0), b = *reinterpret_cast<const double2 *>(lse + c0 + 2);
        lv[0] = a.x; lv[1] = a.y; lv[2] = b.x; lv[3] = b.y;
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) lv[k] = 0.0;
    }
    float lh[4], ll[4];
    bool neg[4];  // this band's logits of pattern c0 + k are negligible (not read)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const double l = (c0 + k < I) ? lv[k] : 0.0;
        lh[k] = (c0 + k < I) ? (float)l : INFINITY;
        ll[k] = (c0 + k < I) ? (float)(l - (double)lh[k]) : 0.0f;
        neg[k] = false;
    }
    int code[4] = {-2, -2, -2, -2};
    int brow0 = 0, b0 = 0;
    bool one_band = false;
    if (OUT == 1 && pm) {
        const int rl = min(r0 + kApplyRows - 1, S - 1);
        b0 = (r0 / chunk) * bpc + (r0 % chunk) / brows;
        const int b1 = (rl / chunk) * bpc + (rl % chunk) / brows;
        // the workgroup's rows lie in one band (always, when blk is given), or in two smaller ones of the same 256 rows of a
        // chunk, taken as one: the sparse form, which adds each P in FP64, must not depend on the tile's rows
        one_band = b0 == b1 || (!blk && r0 / chunk == rl / chunk && (r0 % chunk) / 256 == (rl % chunk) / 256);
        if (one_band) {
            brow0 = (r0 / chunk) * chunk + ((r0 % chunk) / brows) * brows;
            float pv[4];
            int cv[4] = {-2, -2, -2, -2};
            const size_t o = (size_t)b0 * I + c0;
            if ((I & 3) == 0 && c0 < I) {  // uniform layout test; then c0 + 3 < I
                const float4 v = *reinterpret_cast<const float4 *>(pm + o);
                pv[0] = v.x; pv[1] = v.y; pv[2] = v.z; pv[3] = v.w;
                if (blk) {
                    const uint2 w = *reinterpret_cast<const uint2 *>(blk + o);
                    cv[0] = (int16_t)(w.x & 0xffffu); cv[1] = (int16_t)(w.x >> 16);
                    cv[2] = (int16_t)(w.y & 0xffffu); cv[3] = (int16_t)(w.y >> 16);
                }
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    pv[k] = c0 + k < I ? pm[o + k] : 0.0f;
                    if (blk && c0 + k < I) cv[k] = blk[o + k];
                }
            }
            if (b1 != b0)
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (c0 + k < I) pv[k] = fmaxf(pv[k], pm[(size_t)b1 * I + c0 + k]);
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (c0 + k < I) {
                    neg[k] = (double)pv[k] < lv[k] - kSkipApplyNats;
                    code[k] = cv[k];
                    neg[k] = neg[k] || code[k] == -1;
                }
        }
    }
    // segment flags (a segment past the last reads the last; rows past S read row S - 1: not used):
    // the same 8 bytes for the whole wavefront, so lane rr loads row rr's and the others take it by
    // readlane
    int flag[kApplyRows];
    const int segc = OUT == 1 ? min(seg, nseg - 1) : 0;
    {
        const int fv = OUT == 1 && lane < kApplyRows ? (int)pdirty[(size_t)min(r0 + lane, S - 1) * nseg + segc] : 0;
#pragma unroll
        for (int rr = 0; rr < kApplyRows; ++rr) flag[rr] = __builtin_amdgcn_readlane(fv, rr);
    }

    // Sparse form: when at most kSparseMax of the workgroup's patterns have a band that is not
    // negligible, one thread per such pattern computes its 8 values (the others are exactly 0), the
    // values go to LDS, and the P row segments that have to be written are assembled from there.
    constexpr int kSparseMax = 256;
    __shared__ int16_t amap[kApplyCols];               // local pattern -> its slot, -1 if negligible
    __shared__ int16_t alist[kSparseMax];              // slot -> local pattern
    __shared__ uint32_t aval[kSparseMax][kApplyRows];  // hi | lo << 16 per slot and row
    __shared__ int wcnt[4];
    __shared__ uint32_t nzf[kApplyRows];               // bit g: segment g of the row holds a non-zero
    bool sparse = false;
    if (OUT == 1 && pm && !iphi && one_band) {  // uniform over the workgroup
        bool act[4];
        int below = 0, wc = 0;
        const uint64_t lt = (1ull << lane) - 1ull;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            act[k] = c0 + k < I && !neg[k];
            const uint64_t bal = __ballot(act[k]);
            wc += __popcll(bal);
            below += __popcll(bal & lt);
        }
        if (lane == 0) wcnt[wave] = wc;
        if (threadIdx.x < kApplyRows) nzf[threadIdx.x] = 0u;
        __syncthreads();
        const int total = wcnt[0] + wcnt[1] + wcnt[2] + wcnt[3];
        sparse = total <= kSparseMax;
        if (sparse) {
            int slot = below;
            for (int w = 0; w < wave; ++w) slot += wcnt[w];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                amap[4 * threadIdx.x + k] = (int16_t)(act[k] ? slot : -1);
                if (act[k]) alist[slot++] = (int16_t)(4 * threadIdx.x + k);
            }
            __syncthreads();
            float ts[kApplyRows];
#pragma unroll
            for (int rr = 0; rr < kApplyRows; ++rr) ts[rr] = 0.0f;
            if (threadIdx.x < total) {
                const int lp = alist[threadIdx.x], n = blockIdx.x * kApplyCols + lp;
                const double l = lse[n];
                const float lhn = (float)l, lln = (float)(l - (double)lhn);
                const int cd = blk ? (int)blk[(size_t)b0 * I + n] : -2;
                float x[kApplyRows];
                if (cd >= 0) {
                    const float *b = R + (size_t)(brow0 + cd) * ldr + (n & ~255) + (r0 - brow0);
                    const float4 a0 = *reinterpret_cast<const float4 *>(b), a1 = *reinterpret_cast<const float4 *>(b + 4);
                    x[0] = a0.x; x[1] = a0.y; x[2] = a0.z; x[3] = a0.w;
                    x[4] = a1.x; x[5] = a1.y; x[6] = a1.z; x[7] = a1.w;
                } else {
#pragma unroll
                    for (int rr = 0; rr < kApplyRows; ++rr) x[rr] = R[(size_t)min(r0 + rr, S - 1) * ldr + n];
                }
#pragma unroll
                for (int rr = 0; rr < kApplyRows; ++rr) {
                    const float p = r0 + rr < S ? __builtin_amdgcn_exp2f(((x[rr] - lhn) - lln) * kLog2e) : 0.0f;
                    ts[rr] = p;
                    // the dense form's rounding: hi = bf16(p), lo = bf16(p - hi), one conversion each
                    const uint32_t h = pk_bf16(p, 0.0f) & 0xffffu;
                    const uint32_t lo = pk_bf16(p - __builtin_bit_cast(float, h << 16), 0.0f) & 0xffffu;
                    aval[threadIdx.x][rr] = h | (lo << 16);
                    if (h != 0u) {
                        ++nz;
                        atomicOr(&nzf[rr], 1u << (lp >> 8));
                    }
                }
            }
#pragma unroll
            for (int rr = 0; rr < kApplyRows; ++rr) rs[rr][threadIdx.x] = ts[rr];
        }
    }
    if (!sparse) {
        // every row's logits are loaded before the first is used, so the wave waits for memory once
        // rather than once per row (rows past S read row S - 1: not used)
        float xv[kApplyRows][4];
        const bool in_place = code[0] == -2 && code[1] == -2 && code[2] == -2 && code[3] == -2;
        const bool read = !(neg[0] && neg[1] && neg[2] && neg[3]);
#pragma unroll
        for (int rr = 0; rr < kApplyRows; ++rr) {
            const size_t sc = (size_t)min(r0 + rr, S - 1);
            float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (c0 < I && read && in_place) v = *reinterpret_cast<const float4 *>(R + sc * ldr + c0);
            xv[rr][0] = v.x;
            xv[rr][1] = v.y;
            xv[rr][2] = v.z;
            xv[rr][3] = v.w;
        }
        if (!in_place)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (neg[k]) continue;
                if (code[k] >= 0) {  // 8 consecutive floats of the pattern's block
                    const float *b = R + (size_t)(brow0 + code[k]) * ldr + ((c0 + k) & ~255) + (r0 - brow0);
                    const float4 a0 = *reinterpret_cast<const float4 *>(b), a1 = *reinterpret_cast<const float4 *>(b + 4);
                    xv[0][k] = a0.x; xv[1][k] = a0.y; xv[2][k] = a0.z; xv[3][k] = a0.w;
                    xv[4][k] = a1.x; xv[5][k] = a1.y; xv[6][k] = a1.z; xv[7][k] = a1.w;
                } else {
#pragma unroll
                    for (int rr = 0; rr < kApplyRows; ++rr) xv[rr][k] = R[(size_t)min(r0 + rr, S - 1) * ldr + c0 + k];
                }
            }
#pragma unroll
        for (int rr = 0; rr < kApplyRows; ++rr) {
            const int s = r0 + rr;
            float acc = 0.0f;
            uint2 hv = make_uint2(0u, 0u), lv = make_uint2(0u, 0u);
            int any_nz = 0;
            if (s < S && c0 < I) {
                float *src = R + (size_t)s * ldr + c0;
                const float x[4] = {neg[0] ? -INFINITY : xv[rr][0], neg[1] ? -INFINITY : xv[rr][1],
                                    neg[2] ? -INFINITY : xv[rr][2], neg[3] ? -INFINITY : xv[rr][3]};
                // exp(d) = 2^(d log2 e) on the hardware exp2: relative error about |d| 6e-8, below the
                // 2^-16 of the BF16 pair P is stored as
                float p[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) p[k] = __builtin_amdgcn_exp2f(((x[k] - lh[k]) - ll[k]) * kLog2e);
                acc = (p[0] + p[1]) + (p[2] + p[3]);
                if (OUT == 0) {
                    *reinterpret_cast<float4 *>(src) = make_float4(p[0], p[1], p[2], p[3]);
                    if (iphi) {
                        const size_t o = (size_t)s * ldr + c0;
                        const float4 f = *reinterpret_cast<const float4 *>(iphi + o);
                        *reinterpret_cast<float4 *>(Pphi + o) = make_float4(p[0] * f.x, p[1] * f.y, p[2] * f.z, p[3] * f.w);
                    }
                    const int mine = (p[0] != 0.0f) + (p[1] != 0.0f) + (p[2] != 0.0f) + (p[3] != 0.0f);
                    nz += mine;
                    any_nz = mine != 0;
                } else {
                    const size_t o = (size_t)s * ldr + c0;
                    float q[4] = {p[0], p[1], p[2], p[3]};
                    if (iphi) {
                        const float4 f = *reinterpret_cast<const float4 *>(iphi + o);
                        q[0] *= f.x; q[1] *= f.y; q[2] *= f.z; q[3] *= f.w;
                    }
                    // hi of a pair in one v_cvt_pk_bf16_f32; its two values back as floats by a shift
                    // and a mask; lo = bf16(q - hi).  q >= 0, so (hi | lo) != 0 exactly when hi != 0.
                    const uint32_t h01 = pk_bf16(q[0], q[1]), h23 = pk_bf16(q[2], q[3]);
                    const uint32_t l01 = pk_bf16(q[0] - __builtin_bit_cast(float, h01 << 16),
                                                 q[1] - __builtin_bit_cast(float, h01 & 0xffff0000u));
                    const uint32_t l23 = pk_bf16(q[2] - __builtin_bit_cast(float, h23 << 16),
                                                 q[3] - __builtin_bit_cast(float, h23 & 0xffff0000u));
                    const int mine = ((h01 & 0xffffu) != 0) + ((h01 >> 16) != 0) + ((h23 & 0xffffu) != 0) +
                                     ((h23 >> 16) != 0);
                    nz += mine;
                    hv = make_uint2(h01, h23);
                    lv = make_uint2(l01, l23);
                    any_nz = mine != 0;
                }
            }
            if (OUT == 0 && s < S && seg_live) {
                const bool seg_nz = __any(any_nz) != 0;
                if (lane == 0) pdirty[(size_t)s * nseg + seg] = seg_nz ? 1 : 0;
            }
            if (OUT == 1 && s < S && seg_live) {  // s and seg_live are uniform over the wave
                const bool seg_nz = __any(any_nz) != 0;
                const size_t fo = (size_t)s * nseg + seg;
                const bool dirty = flag[rr] != 0;
                if ((seg_nz || dirty) && c0 < I) {
                    const size_t o = (size_t)s * ldr + c0;
                    *reinterpret_cast<uint2 *>(Ph + o) = hv;
                    *reinterpret_cast<uint2 *>(Pl + o) = lv;
                }
                if (lane == 0 && dirty != seg_nz) pdirty[fo] = seg_nz ? 1 : 0;
            }
            rs[rr][threadIdx.x] = acc;
        }
    }
    // row sums over the workgroup's 1,024 patterns through LDS: wave w adds rows 2w and 2w + 1 (one
    // per 32-lane half, eight values a lane, then five shuffle steps), in a fixed order
    __shared__ int nzw[4];
    nz = wave_sum(nz);
    if (lane == 0) nzw[wave] = nz;
    __syncthreads();
    {
        const int row = 2 * wave + (lane >> 5), part = lane & 31;
        double t = 0.0;
#pragma unroll
        for (int q = 0; q < 8; ++q) t += (double)rs[row][part + 32 * q];
#pragma unroll
        for (int o = 16; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
        if (part == 0 && r0 + row < S) Tpart[(size_t)blockIdx.x * S + r0 + row] = t;
    }
    if (sparse) {  // the P row segments that hold a non-zero or held one, assembled from the slots
#pragma unroll
        for (int rr = 0; rr < kApplyRows; ++rr) {
            const int s = r0 + rr;
            if (s >= S || !seg_live) continue;
            const bool seg_nz = (nzf[rr] >> wave) & 1u;
            const bool dirty = flag[rr] != 0;
            if ((seg_nz || dirty) && c0 < I) {
                uint32_t v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int a = amap[4 * threadIdx.x + k];
                    v[k] = a >= 0 ? aval[a][rr] : 0u;
                }
                const size_t o = (size_t)s * ldr + c0;
                *reinterpret_cast<uint2 *>(Ph + o) =
                    make_uint2((v[0] & 0xffffu) | (v[1] << 16), (v[2] & 0xffffu) | (v[3] << 16));
                *reinterpret_cast<uint2 *>(Pl + o) =
                    make_uint2((v[0] >> 16) | (v[1] & 0xffff0000u), (v[2] >> 16) | (v[3] & 0xffff0000u));
            }
            if (lane == 0 && dirty != seg_nz) pdirty[(size_t)s * nseg + seg] = seg_nz ? 1 : 0;
        }
    }
    // per-workgroup non-zero count, summed by one deterministic pass afterwards
    if (threadIdx.x == 0)
        nnz[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = (double)(nzw[0] + nzw[1] + nzw[2] + nzw[3]);
}

}  // namespace

// Partials layout inside c->part:  pm (float, nb*I) | ps (double, nb*I) | blk (double) | Tpart |
// non-zero counts (one per apply workgroup).
// nb = the partial pass's band count, or (MFMA logL with fused partials) one band per logl_band_rows rows; after
// 64-row tiles the bands of 256 rows have theirs in the place of ps.
int softmax_bands(int S, int I)
{
    return std::max(1, std::min((S + 63) / 64, 4096 / std::max(1, (I + 255) / 256) + 1));
}

int64_t softmax_part_len(int S, int I, int fused_bands)
{
    const int64_t nb = std::max(softmax_bands(S, I), fused_bands);
    const int ncb = (I + kApplyCols - 1) / kApplyCols;
    return nb * I /*pm as floats packed in doubles: over-allocate*/ + nb * I + (I + kFinalPat - 1) / kFinalPat + 1 +
           (int64_t)ncb * S + (int64_t)ncb * ((S + kApplyRows - 1) / kApplyRows) + 16;
}

__global__ void k_mark_dirty(uint8_t *__restrict__ d, int64_t n)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x)
        d[t] = 1;
}

hipError_t launch_mark_p_dirty(const emc_ctx *c, hipStream_t st)
{
    if (!c->pdirty) return hipSuccess;
    const int64_t n = (int64_t)c->Sp * p_segments(c);
    hipLaunchKernelGGL(k_mark_dirty, dim3((unsigned)std::min<int64_t>((n + 255) / 256, 4096)), dim3(256), 0, st,
                       c->pdirty, n);
    return hipGetLastError();
}

hipError_t launch_sm_sums(const emc_ctx *c, const double *nz, int nnz, const double *blk, int nblk, const double *Tpart,
                          int ncb, hipStream_t st)
{
    const int nT = Tpart ? (c->Sp + 1023) / 1024 : 0;
    hipLaunchKernelGGL(k_sm_sums, dim3(2 + nT), dim3(1024), 0, st, nz, nnz, blk, nblk, c->cst, c->I, Tpart, ncb, c->S, c->Sp,
                       c->T, c->scal);
    return hipGetLastError();
}

hipError_t launch_softmax(const emc_ctx *c, hipStream_t st)
{
    const int S = c->S, I = c->I;
    const int ncol = (I + 255) / 256;
    const int nfin = (I + kFinalPat - 1) / kFinalPat;
    const bool fused = logl_fuses_softmax(c);  // the logL epilogue wrote the band partials
    const int nb = fused ? softmax_fused_bands(c) : softmax_bands(S, I);
    const int rows = (S + nb - 1) / nb;
    double *base = c->part;
    float *pm = reinterpret_cast<float *>(base);
    double *ps = base + (int64_t)nb * I;
    double *blk = ps + (int64_t)nb * I;
    double *Tpart = blk + nfin + 1;
    if (!fused)
        hipLaunchKernelGGL(k_sm_partial, dim3(ncol, nb), dim3(256), 0, st, c->R, (int64_t)c->Ip, S, I, rows, pm, ps);
    const int16_t *gblk = fused && c->logits_partial ? c->blk : nullptr;
    if (fused && logl_band_pass(c)) {  // pm: maxima of 64-row groups; the bands' partials take the place of ps
        const int bands = nb / 4;
        float *bm = reinterpret_cast<float *>(ps + (int64_t)bands * I);
        hipLaunchKernelGGL(k_sm_band, dim3((I + 31) / 32, bands), dim3(256), 0, st, c->R, (int64_t)c->Ip, S, I, c->chunk,
                           c->chunkp / 256, pm, gblk, bm, ps);
        hipLaunchKernelGGL(k_sm_final, dim3(nfin), dim3(256), 0, st, bm, ps, bands, I, c->lse, blk, c->scal);
    } else {
        hipLaunchKernelGGL(k_sm_final, dim3(nfin), dim3(256), 0, st, pm, ps, nb, I, c->lse, blk, c->scal);
    }
    const int ncb = (I + kApplyCols - 1) / kApplyCols;
    const dim3 ga(ncb, (S + kApplyRows - 1) / kApplyRows);
    double *nzpart = Tpart + (int64_t)ncb * S;  // one non-zero count per apply workgroup
    if (c->mfma)
        hipLaunchKernelGGL(k_sm_apply<1>, ga, dim3(256), 0, st, c->R, (int64_t)c->Ip, S, I, c->lse, c->Ph, c->Pl,
                           Tpart, nzpart, c->opt.scaling ? c->iphi : nullptr, c->pdirty, p_segments(c),
                           fused ? pm : nullptr, gblk, c->chunk,
                           c->chunkp / logl_band_rows(c), logl_band_rows(c), nullptr);
    else
        hipLaunchKernelGGL(k_sm_apply<0>, ga, dim3(256), 0, st, c->R, (int64_t)c->Ip, S, I, c->lse, nullptr, nullptr,
                           Tpart, nzpart, c->opt.scaling ? c->iphi : nullptr, c->pdirty, p_segments(c), nullptr, nullptr, 1,
                           1, 1, c->Pphi);
    return launch_sm_sums(c, nzpart, (int)(ga.x * ga.y), blk, nfin, Tpart, ncb, st);
}

}  // namespace emc
