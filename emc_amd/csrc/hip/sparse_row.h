// One row of the sparse M-step sum: out[j] = sum_n p_n K[pat(n), j] over the non-zero entries n of
// a row of responsibilities stored as BF16 hi + lo (p_n = hi + lo).  Device code shared by the
// dense-layout and the per-cell (grouped) M-steps; one 256-thread workgroup per row.
//
// The row is scanned 32 entries per thread and step (two 16-byte loads of hi per thread in flight;
// lo only beside a non-zero hi, which is exact for the split lo = bf16(p - hi)).  A step with no
// non-zero hi in the whole workgroup ends after one barrier; otherwise its non-zero entries are
// compacted into an LDS list in ascending order (wave scans and a block prefix sum keep the order,
// so the result is deterministic), in as many batches as the list needs, and each full list (and
// the last) has its count rows added to registers, PX pixels per thread and pass.  Counts as
// bytes (KT 0), BF16 (KT 1) or BF16 hi + lo (KT 2); NPASS chunks of PX pixels per thread (Pp <=
// 256 * PX * NPASS).  FP32 accumulation, one fused multiply-add per entry and pixel, in ascending entry order: the
// chain of the dense FP32 contraction without its zero entries.
// KT 3 is the FP32 precision: the row is float (ph; pl unused) and so are the counts.
#pragma once

#include "../emc_internal.h"

namespace emc {

namespace sparse_row_detail {
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
constexpr int kCap = 2048;        // LDS list entries per batch
constexpr int kPer = 32;          // consecutive entries per thread and step
constexpr int kStep = 256 * kPer; // entries scanned per step
static_assert(256 % kPer == 0, "a thread's entries lie in one 256-entry segment");

__device__ __forceinline__ float half16(const u32x4 &v, int k) { return bf2f((bf16_t)(v[k >> 1] >> (16 * (k & 1)))); }
// N 32-bit words from p (aligned to them, at most 16 bytes)
template <int N>
__device__ __forceinline__ void load_words(const void *__restrict__ p, uint32_t (&w)[N])
{
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    static_assert(N == 1 || N == 2 || N % 4 == 0);
    if constexpr (N == 1) {
        w[0] = *reinterpret_cast<const uint32_t *>(p);
    } else if constexpr (N == 2) {
        const u32x2 v = *reinterpret_cast<const u32x2 *>(p);
        w[0] = v[0];
        w[1] = v[1];
    } else {
#pragma unroll
        for (int k = 0; k < N; k += 4) {
            const u32x4 v = reinterpret_cast<const u32x4 *>(p)[k / 4];
#pragma unroll
            for (int q = 0; q < 4; ++q) w[k + q] = v[q];
        }
    }
}
__device__ __forceinline__ bool nonzero(const u32x4 &v) { return (v[0] | v[1] | v[2] | v[3]) != 0u; }
}  // namespace sparse_row_detail

// n entries of the row; pat == nullptr: entry n is pattern n.  Pp is a multiple of 16 and at most
// 256 * PX * NPASS; the row holds a multiple of 8 readable entries (padding entries are 0) and starts
// 16-byte aligned.  seg (or nullptr): one flag per 256 entries of the row, 0 where those entries are
// known to be zero (their loads are skipped).
template <int KT, int NPASS, int PX = 16>
__device__ __forceinline__ void sparse_row(const void *__restrict__ ph, const bf16_t *__restrict__ pl, int n,
                                           const int32_t *__restrict__ pat, const void *__restrict__ Kv,
                                           const bf16_t *__restrict__ Klo, int Pp, float *__restrict__ out,
                                           const uint8_t *__restrict__ seg = nullptr)
{
    using namespace sparse_row_detail;
    constexpr int E = KT == 3 ? 4 : 8;  // entries per 16-byte load
    constexpr int kV = kPer / E;        // loads per thread and step
    auto load16 = [&](int i) {
        return *reinterpret_cast<const u32x4 *>(reinterpret_cast<const unsigned char *>(ph) + (size_t)i * (16 / E));
    };
    // entry k of a load: its bits (0: not listed) and value
    auto bits_of = [&](const u32x4 &h, const u32x4 &l, int k) -> uint32_t {
        return KT == 3 ? h[k & 3] << 1 : ((h[(k >> 1) & 3] | l[(k >> 1) & 3]) >> (16 * (k & 1))) & 0xffffu;
    };
    auto value_of = [&](const u32x4 &h, const u32x4 &l, int k) {
        return KT == 3 ? __uint_as_float(h[k & 3]) : half16(h, k & 7) + half16(l, k & 7);
    };
    __shared__ int li[kCap];
    __shared__ float lp[kCap];
    __shared__ int wsum[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nch = Pp / PX;
    constexpr int kAhead = PX == 16 ? 4 : 8;
    float acc[NPASS][PX];
#pragma unroll
    for (int q = 0; q < NPASS; ++q)
#pragma unroll
        for (int k = 0; k < PX; ++k) acc[q][k] = 0.0f;

    auto accumulate = [&](int cnt) {
#pragma unroll
        for (int q = 0; q < NPASS; ++q) {
            const int pc = tid + q * 256;
            if (pc >= nch) break;
            // unrolled so that the count-row loads of several entries are in flight together (the
            // sums still add the entries in list order)
#pragma unroll kAhead
            for (int e = 0; e < cnt; ++e) {
                const size_t row = (size_t)li[e] * Pp + PX * (size_t)pc;
                const float p = lp[e];
                if constexpr (KT == 0) {
                    uint32_t v[PX / 4];
                    load_words(reinterpret_cast<const uint8_t *>(Kv) + row, v);
#pragma unroll
                    for (int k = 0; k < PX; ++k)
                        acc[q][k] = __builtin_fmaf(p, (float)((v[k >> 2] >> (8 * (k & 3))) & 0xffu), acc[q][k]);
                } else if constexpr (KT == 3) {
                    uint32_t v[PX];
                    load_words(reinterpret_cast<const float *>(Kv) + row, v);
#pragma unroll
                    for (int k = 0; k < PX; ++k) acc[q][k] = __builtin_fmaf(p, __uint_as_float(v[k]), acc[q][k]);
                } else {
                    uint32_t v[PX / 2], vl[PX / 2];
                    load_words(reinterpret_cast<const bf16_t *>(Kv) + row, v);
                    if (KT == 2) load_words(Klo + row, vl);
#pragma unroll
                    for (int k = 0; k < PX; ++k) {
                        float x = bf2f((bf16_t)(v[k >> 1] >> (16 * (k & 1))));
                        if (KT == 2) x += bf2f((bf16_t)(vl[k >> 1] >> (16 * (k & 1))));
                        acc[q][k] = __builtin_fmaf(p, x, acc[q][k]);
                    }
                }
            }
        }
    };

    int m = 0;  // entries in the list (the same in every thread)
    for (int i0 = 0; i0 < n; i0 += kStep) {
        const int ib = i0 + tid * kPer;  // kPer divides 256: the thread's entries share one flag
        const bool live = ib < n && (!seg || seg[ib >> 8] != 0);
        u32x4 h[kV], l[kV];
        bool any = false;
#pragma unroll
        for (int v = 0; v < kV; ++v) {
            h[v] = u32x4{0u, 0u, 0u, 0u};
            l[v] = u32x4{0u, 0u, 0u, 0u};
            if (live && ib + E * v < n) h[v] = load16(ib + E * v);
            any |= nonzero(h[v]);
        }
        if (!__syncthreads_or(any)) continue;
        int cnt = 0;
#pragma unroll
        for (int v = 0; v < kV; ++v) {
            if (KT != 3 && nonzero(h[v])) l[v] = *reinterpret_cast<const u32x4 *>(pl + ib + E * v);
#pragma unroll
            for (int k = 0; k < E; ++k) cnt += (bits_of(h[v], l[v], k) != 0u && ib + E * v + k < n) ? 1 : 0;
        }
        int incl = cnt;  // inclusive scan over the wave
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int t = __shfl_up(incl, o, 64);
            if (lane >= o) incl += t;
        }
        if (lane == 63) wsum[wave] = incl;
        __syncthreads();
        int woff = 0;
        for (int w = 0; w < wave; ++w) woff += wsum[w];
        const int step_total = wsum[0] + wsum[1] + wsum[2] + wsum[3];
        const int rank0 = woff + incl - cnt;  // rank of this thread's first entry within the step
        // the step's entries with rank in [base, base + take) fill the list from position m
        for (int base = 0;;) {  // block-uniform loop
            const int take = min(kCap - m, step_total - base);
            int rank = rank0;
#pragma unroll
            for (int v = 0; v < kV; ++v)
#pragma unroll
                for (int k = 0; k < E; ++k)
                    if (bits_of(h[v], l[v], k) != 0u && ib + E * v + k < n) {
                        const int q = rank - base;
                        if (q >= 0 && q < take) {
                            li[m + q] = pat ? pat[ib + E * v + k] : ib + E * v + k;
                            lp[m + q] = value_of(h[v], l[v], k);
                        }
                        ++rank;
                    }
            m += take;
            base += take;
            __syncthreads();
            if (base >= step_total) break;
            accumulate(m);  // the list is full
            __syncthreads();
            m = 0;
        }
    }
    accumulate(m);

#pragma unroll
    for (int q = 0; q < NPASS; ++q) {
        const int pc = tid + q * 256;
        if (pc >= nch) break;
#pragma unroll
        for (int k = 0; k < PX; k += 4)
            *reinterpret_cast<float4 *>(out + PX * pc + k) = make_float4(acc[q][k], acc[q][k + 1], acc[q][k + 2], acc[q][k + 3]);
    }
}

}  // namespace emc
