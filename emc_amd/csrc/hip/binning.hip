// Maximize, scatter half, binned: deterministic insertion without atomics.
//
// The geometry of insertion (which voxels a rotated pixel touches, with which trilinear weights)
// depends only on the rotation list, the detector coordinates and the mask, not on the
// iteration.  Once per geometry the valid (rotation s, active pixel j) pairs are sorted by the
// model brick (kBrick^3 voxels) that holds their base voxel, per rotation chunk, with a stable
// radix sort (rocPRIM), so each brick lists its pairs in (s, j) order; each brick's list is cut
// into units of at most kUnit pairs, and inside a unit the pairs are ranked once more by base
// voxel (a 16-bit permutation, the start of each base voxel's run, and for trilinear the pairs'
// fractions in base-voxel order, laid out for coalesced reads).  Per pair the iteration then reads
// 4 bytes of list (the packed pair), 2 of permutation and 12 of fractions.  Every iteration:
//   1. one workgroup per unit reads its pairs in (s, j) order, where the reads of U are runs of
//      consecutive pixels, and writes U and T_s into LDS at the pair's position in base-voxel order;
//   2. every thread sums an equal share of the positions into per-base-voxel corner sums (the
//      pieces of a voxel's run that crosses threads are added in thread order);
//   3. the corner sums of up to kUnitsPerBlock units of one brick (a block) are added in order, then every
//      voxel of the halo brick ((kBrick+1)^3) gathers them in a fixed order, and the halo brick is stored as
//      the block's partial (no atomics).  A workgroup takes a block's units in turn or, where the blocks
//      are few, one unit each, and a pass over the blocks adds them: the same sums in the same order;
//   4. a grouping pass sums the partials of up to kGroup consecutive blocks of one brick (left out where no brick
//      has more than kDirect), and a last pass gives every model voxel the sum, in order, of the groups
//      of the (at most 8) bricks whose halo covers it.
// No sum depends on scheduling, so repeated runs give bit-identical models.  This replaces the 16
// global atomics per (s, j) of the reference's insert_slices_kernel (emc_atomic.cu:33-85,
// 183-200); the skip rules (T_s > 1e-10, emc_atomic.cu:190; U >= 0, emc_atomic.cu:56) and the
// bounds are the same as in the atomic form.
#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include <rocprim/device/device_radix_sort.hpp>

#include "../emc_internal.h"
#include "geom.h"

namespace emc {
namespace {

constexpr int kBrick = 8;
constexpr int kBrick3 = kBrick * kBrick * kBrick;  // base voxels of a brick
constexpr int kUnit = 4096;                        // pairs of a unit (positions fit 16 bits)
constexpr int kUnitsPerBlock = 4;                  // units of a block
// Up to this many units a chunk take a workgroup each (their corner sums, 32 KB a unit, go through memory; with more of
// them the chip's 512 workgroup slots are filled by the blocks).  Insertion kernel and the pass over the units, us,
// against a workgroup per block: 24^3 / 420 rotations (60 units) 21 / 36, 32^3 / 3,240 (700) 41 / 56, 45^3 nearest,
// 1,000 a chunk (400) 26 / 33.
constexpr int kSplitUnits = 1024;
constexpr int kVbeg = 520;                         // run starts per unit: kBrick3 + 1, padded to 16 bytes
constexpr int kGroup = 32;                         // blocks whose partials one grouping workgroup sums
constexpr int kDirect = 8;                         // up to this many blocks per brick: no grouping pass (a launch;
                                                   // at 12 the last pass takes longer by as much)
constexpr int kHalo = kBrick + 1;
constexpr int kHalo3 = kHalo * kHalo * kHalo;      // voxels a brick's pairs reach
constexpr int kThreads = 512;  // 8 waves; with 67 KB of LDS and 128 registers two workgroups (16 waves) fit a CU
// Threads of a workgroup of the last pass: all latency for few voxels, so spread over the chip (32^3: 12.1 us with 512,
// 10.8 with 128); larger models read the partials of a brick from fewer places (128^3: 38 us with 512, 49 with 128).
inline int reduce_threads(int64_t voxels) { return voxels < 256 * kThreads ? 128 : kThreads; }
constexpr int kPer = kUnit / kThreads;  // positions per thread in step 2

struct BinGeom {
    int L, nb, S, Pa, Pp, chunk, interp, jbits;
};

__device__ __forceinline__ void unpack(uint32_t p, int jbits, int &s, int &j)
{
    s = (int)(p >> jbits);
    j = (int)(p & ((1u << jbits) - 1u));
}

// Voxel cell of active pixel j under rotation s (nearest: the voxel; trilinear: the base corner and
// the fractions); false when out of bounds (emc_atomic.cu:67-69 for nearest).
__device__ __forceinline__ bool item_cell(const float *__restrict__ rotm, const float *__restrict__ axyz,
                                          const BinGeom &g, int s, int j, int &bx, int &by, int &bz, float &fx,
                                          float &fy, float &fz)
{
    float m[9];
    load_rot(rotm, s, m);
    float ux, uy, uz;
    rot_point(m, axyz[j], axyz[g.Pp + j], axyz[2 * g.Pp + j], model_c(g.L), ux, uy, uz);
    if (g.interp == EMC_INTERP_NEAREST) {
        bx = nearest(ux);
        by = nearest(uy);
        bz = nearest(uz);
        fx = fy = fz = 0.0f;
        return bx >= 0 && bx < g.L && by >= 0 && by < g.L && bz >= 0 && bz < g.L;
    }
    return tri_axis(ux, g.L, bx, fx) && tri_axis(uy, g.L, by, fy) && tri_axis(uz, g.L, bz, fz);
}

// Sort key of every pair (chunk-major brick; invalid pairs get invalid_key) and its packed value
// s << jbits | j, in (s, j) order.
__global__ void k_bin_keys(const float *__restrict__ rotm, const float *__restrict__ axyz, BinGeom g, int64_t n,
                           uint32_t invalid_key, uint32_t *__restrict__ keys, uint32_t *__restrict__ vals)
{
    for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < n; idx += (int64_t)gridDim.x * blockDim.x) {
        const int s = (int)(idx / g.Pa), j = (int)(idx % g.Pa);
        int bx, by, bz;
        float fx, fy, fz;
        uint32_t key = invalid_key;
        if (item_cell(rotm, axyz, g, s, j, bx, by, bz, fx, fy, fz)) {
            const int brick = ((bz / kBrick) * g.nb + by / kBrick) * g.nb + bx / kBrick;
            key = (uint32_t)((s / g.chunk) * g.nb * g.nb * g.nb + brick);
        }
        keys[idx] = key;
        vals[idx] = ((uint32_t)s << g.jbits) | (uint32_t)j;
    }
}

__global__ void k_bin_count(const uint32_t *__restrict__ keys, int64_t n, uint32_t nkeys, int32_t *__restrict__ counts)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t k = keys[t];
        if (k < nkeys && (t == 0 || keys[t - 1] != k)) counts[2 * k] = (int32_t)t;              // first position
        if (k < nkeys && (t == n - 1 || keys[t + 1] != k)) counts[2 * k + 1] = (int32_t)(t + 1);  // end
    }
}

__global__ void k_iota(uint32_t *__restrict__ v, int64_t n)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x)
        v[t] = (uint32_t)t;
}

// Second sort key of the pairs of unit u: u * kBrick3 + the base voxel's index inside the brick.
__global__ __launch_bounds__(kThreads) void k_unit_keys(const int32_t *__restrict__ units,
                                                        const uint32_t *__restrict__ vals,
                                                        const float *__restrict__ rotm,
                                                        const float *__restrict__ axyz, BinGeom g,
                                                        uint32_t *__restrict__ keys)
{
    const int u = blockIdx.x;
    const int begin = units[4 * u + 1], end = units[4 * u + 2];
    for (int t = begin + threadIdx.x; t < end; t += kThreads) {
        int s, j;
        unpack(vals[t], g.jbits, s, j);
        int bx = 0, by = 0, bz = 0;
        float fx, fy, fz;
        item_cell(rotm, axyz, g, s, j, bx, by, bz, fx, fy, fz);  // valid: only valid pairs are listed
        const int lv = ((bz % kBrick) * kBrick + by % kBrick) * kBrick + bx % kBrick;
        keys[t] = (uint32_t)u * kBrick3 + (uint32_t)lv;
    }
}

// Per unit: each pair's position in base-voxel order (a stable order, so (s, j) order within a base
// voxel), stored at the pair's place in (s, j) order; the start of each base voxel's run
// (kBrick3 + 1 entries); for trilinear, the fractions of the pair at base-voxel position k, stored
// at frac[(u * 3 + axis) * kUnit + (k % kPer) * kThreads + k / kPer], where the insertion's thread
// k / kPer reads them in step (k % kPer) of its share, all lanes of a wave on consecutive words.
__global__ __launch_bounds__(kThreads) void k_unit_perm(const int32_t *__restrict__ units,
                                                        const uint32_t *__restrict__ skeys,
                                                        const uint32_t *__restrict__ spos,
                                                        const uint32_t *__restrict__ vals,
                                                        const float *__restrict__ rotm, const float *__restrict__ axyz,
                                                        BinGeom g, uint16_t *__restrict__ inv,
                                                        uint16_t *__restrict__ vbeg, float *__restrict__ frac)
{
    const int u = blockIdx.x;
    const int begin = units[4 * u + 1], end = units[4 * u + 2];
    for (int t = begin + threadIdx.x; t < end; t += kThreads) {
        const int k = t - begin;
        inv[spos[t]] = (uint16_t)k;
        if (frac) {
            int s, j, bx, by, bz;
            float f[3];
            unpack(vals[spos[t]], g.jbits, s, j);
            item_cell(rotm, axyz, g, s, j, bx, by, bz, f[0], f[1], f[2]);
            for (int a = 0; a < 3; ++a) frac[((size_t)u * 3 + a) * kUnit + (k % kPer) * kThreads + k / kPer] = f[a];
        }
    }
    for (int lv = threadIdx.x; lv <= kBrick3; lv += kThreads) {
        const uint32_t key = (uint32_t)u * kBrick3 + (uint32_t)lv;
        int lo = begin, hi = end;  // first position with skeys >= key
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (skeys[mid] < key) lo = mid + 1;
            else hi = mid;
        }
        vbeg[(size_t)u * kVbeg + lv] = (uint16_t)(lo - begin);
    }
}

// Steps 1-3 for one block: consecutive units of one brick, one after the other, whose corner sums accumulate in
// LDS; the block's halo brick is stored as its partial
// (part: [block - first block of the chunk][2][kHalo3], numerator then weight).  SPLIT: one unit (u0 + blockIdx.x)
// a workgroup, whose corner sums are stored as they are for k_bin_units.
// Step 1 writes U (or -1: skipped) and T_s into LDS at the pair's position in base-voxel order.  Step 2
// gives every thread the same share of the unit, kPer consecutive positions, with the trilinear
// fractions read from the precomputed coalesced planes (a thread per base voxel would wait on the
// brick's heaviest voxel: at 64^3 / 25,680 the slowest thread of a unit would sum 2.5 times the
// mean, up to 32 times).  A base voxel's run that crosses a thread boundary is summed piecewise: a
// piece that continues into the next thread is handed over as a tail, and the thread holding the
// run's last position adds the pieces in thread order.  Corner c = dx + 2 dy + 4 dz, weights
// (1-f or f) per axis.  LDS layouts avoid bank conflicts: position k sits at k ^ ((k >> 6) % kPer) (a
// thread's kPer positions are consecutive, so the 64 lanes of a read fall on 64 banks), the
// corner sums are corner-major, the tails value-major.
//
// What bounds it: memory, 22 bytes a pair with U, and the latency of list -> U, which the list read one unit ahead
// halves, and the vector units at the runs' ends, where the lanes part.  64^3 / 25,680: 820 -> 609 us with the list
// ahead and the swizzle above (k ^ ((k >> 3) & 7) before, which left eight lanes on each bank), 594 with only the last
// run of a thread looked at for a tail (3.1 TB/s).  The corner sums added by LDS atomics (one instruction for three): 1,110 us.  Forming the fractions here instead of reading them: 985 us (the vector units,
// then); U, T and the fractions one unit ahead too: 17 to 31 registers spilled, 856 us.
__device__ __forceinline__ int rswz(int k) { return k ^ ((k >> 6) & (kPer - 1)); }

// The corner sums of a block -> its halo brick: each voxel adds those of the base voxels below it, in corner order.
template <int NC>
__device__ __forceinline__ void gather_halo(const float (*cM)[kBrick3], const float (*cW)[kBrick3], float *pM, float *pW)
{
    for (int hv = threadIdx.x; hv < kHalo3; hv += kThreads) {
        const int hx = hv % kHalo, hy = (hv / kHalo) % kHalo, hz = hv / (kHalo * kHalo);
        float sm = 0.0f, sw = 0.0f;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int bx = hx - (c & 1), by = hy - ((c >> 1) & 1), bz = hz - (c >> 2);
            if (bx < 0 || by < 0 || bz < 0 || bx >= kBrick || by >= kBrick || bz >= kBrick) continue;
            const int lb = (bz * kBrick + by) * kBrick + bx;
            sm += cM[c][lb];
            sw += cW[c][lb];
        }
        pM[hv] = sm;
        pW[hv] = sw;
    }
}

template <int INTERP, bool SPLIT>
__global__ __launch_bounds__(kThreads, 4) void k_insert_binned(const int32_t *__restrict__ blocks, int u0,
                                                               const int32_t *__restrict__ units,
                                                               const uint32_t *__restrict__ vals,
                                                               const uint16_t *__restrict__ inv,
                                                               const uint16_t *__restrict__ vbeg,
                                                               const float *__restrict__ frac,
                                                               const float *__restrict__ U, int s0,
                                                               const double *__restrict__ T, BinGeom g,
                                                               float *__restrict__ part)
{
    constexpr int NC = INTERP == EMC_INTERP_NEAREST ? 1 : 8;
    constexpr int kBuf = 2 * kUnit > 2 * NC * kThreads ? 2 * kUnit : 2 * NC * kThreads;
    __shared__ float buf[kBuf];  // a unit's U (-1: skipped) and T_s by base-voxel position, then the tails
    __shared__ uint16_t svb[kBrick3 + 1];
    __shared__ __attribute__((aligned(16))) float cM[NC][kBrick3], cW[NC][kBrick3];
    __shared__ int tail_lv[kThreads];
    float(*sv)[kUnit] = reinterpret_cast<float(*)[kUnit]>(buf);
    float(*tail)[kThreads] = reinterpret_cast<float(*)[kThreads]>(buf);  // [2 NC][kThreads]
    const int b = blockIdx.x;
    const int ub = SPLIT ? u0 + b : blocks[4 * b + 1], ue = SPLIT ? ub + 1 : blocks[4 * b + 2];
    const int tid = threadIdx.x;
    for (int k = tid; k < NC * kBrick3 / 4; k += kThreads) {
        reinterpret_cast<float4 *>(&cM[0][0])[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        reinterpret_cast<float4 *>(&cW[0][0])[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    // the pairs of a unit, read one unit ahead (past the end of a unit: a valid pair, not stored)
    uint32_t pv[kPer];
    uint16_t pos[kPer];
    int begin = units[4 * ub + 1], n = units[4 * ub + 2] - begin;
    auto load_pairs = [&] {
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            const int k = begin + min(tid + q * kThreads, n - 1);
            pv[q] = vals[k];
            pos[q] = inv[k];
        }
    };
    load_pairs();
    for (int u = ub; u < ue; ++u) {
        const int k0 = tid * kPer, k1 = min(n, k0 + kPer);
        // 1. U and T_s by base-voxel position, from the pairs in (s, j) order
        double Td[kPer];
        float val[kPer];
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            int s, j;
            unpack(pv[q], g.jbits, s, j);
            Td[q] = T[s];
            val[q] = U[(size_t)(s - s0) * g.Pp + j];
        }
        // this thread's fractions (used after the barriers)
        float fr[kPer][3];
        if constexpr (INTERP == EMC_INTERP_TRILINEAR) {
#pragma unroll
            for (int i = 0; i < kPer; ++i)
#pragma unroll
                for (int a = 0; a < 3; ++a) fr[i][a] = frac[((size_t)u * 3 + a) * kUnit + i * kThreads + tid];
        }
        __syncthreads();  // the previous unit's tails and run starts are consumed
        for (int k = tid; k <= kBrick3; k += kThreads) svb[k] = vbeg[(size_t)u * kVbeg + k];
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            if (tid + q * kThreads >= n) break;
            const int p = rswz(pos[q]);
            sv[0][p] = (Td[q] > 1e-10 && val[q] >= 0.0f) ? val[q] : -1.0f;  // emc_atomic.cu:190, :56
            sv[1][p] = (float)Td[q];
        }
        if (u + 1 < ue) {  // the next unit's pairs
            begin = units[4 * (u + 1) + 1];
            n = units[4 * (u + 1) + 2] - begin;
            load_pairs();
        }
        __syncthreads();
        // 2. positions [k0, k1); lv = the base voxel of the current run
        int lv = 0;
        if (k0 < k1) {  // the voxel whose run holds k0: the last lv with svb[lv] <= k0
            int lo = 0, hi = kBrick3 - 1;
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (svb[mid] <= k0) lo = mid;
                else hi = mid - 1;
            }
            lv = lo;
        }
        float acc[2 * NC], own[2 * NC];
#pragma unroll
        for (int c = 0; c < 2 * NC; ++c) acc[c] = own[c] = 0.0f;
        // in: svb[lv] <= k0 < end; a run that began before k0 is the first one, and only the last may go on past k1
        int own_lv = -1, my_tail = -1;
        bool left = k0 < k1 && svb[lv] < k0;
        int end = k0 < k1 ? svb[lv + 1] : 0;
        auto close_run = [&] {
            if (left) {  // this thread holds the run's last position: adds the pieces later
#pragma unroll
                for (int c = 0; c < 2 * NC; ++c) own[c] = acc[c];
                own_lv = lv;
                left = false;
            } else {  // the whole run: only this thread touches lv in this unit
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    cM[c][lv] += acc[c];
                    cW[c][lv] += acc[NC + c];
                }
            }
        };
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int k = k0 + i;
            if (k >= k1) break;
            if (k >= end) {
                close_run();
#pragma unroll
                for (int c = 0; c < 2 * NC; ++c) acc[c] = 0.0f;
                do {  // skip base voxels without pairs
                    ++lv;
                    end = svb[lv + 1];
                } while (end <= k);
            }
            const int p = rswz(k);
            const float v = sv[0][p];
            if (v < 0.0f) continue;
            const float Ts = sv[1][p];
            if constexpr (INTERP == EMC_INTERP_NEAREST) {
                acc[0] += v;
                acc[1] += Ts;
            } else {
                const float gw[2][3] = {{1.0f - fr[i][0], 1.0f - fr[i][1], 1.0f - fr[i][2]},
                                        {fr[i][0], fr[i][1], fr[i][2]}};
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    const float w = gw[c & 1][0] * gw[(c >> 1) & 1][1] * gw[c >> 2][2];
                    acc[c] += w * v;
                    acc[NC + c] += w * Ts;
                }
            }
        }
        if (k0 < k1) {
            if (end > k1) my_tail = lv;  // continues into the next thread: acc is handed over
            else close_run();
        }
        __syncthreads();  // the staging is consumed: the tails take its space
        tail_lv[tid] = my_tail;
        if (my_tail >= 0)
#pragma unroll
            for (int c = 0; c < 2 * NC; ++c) tail[c][tid] = acc[c];
        __syncthreads();
        if (own_lv >= 0) {  // the pieces of earlier threads, in thread order, then this thread's
            int t0 = tid;
            while (t0 > 0 && tail_lv[t0 - 1] == own_lv) --t0;
            float sum[2 * NC];
#pragma unroll
            for (int c = 0; c < 2 * NC; ++c) sum[c] = 0.0f;
            for (int t = t0; t < tid; ++t)
#pragma unroll
                for (int c = 0; c < 2 * NC; ++c) sum[c] += tail[c][t];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                cM[c][own_lv] += sum[c] + own[c];
                cW[c][own_lv] += sum[NC + c] + own[NC + c];
            }
        }
    }
    __syncthreads();
    if constexpr (SPLIT) {  // the unit's corner sums, [2][NC][kBrick3]
        float4 *out = reinterpret_cast<float4 *>(part + (size_t)b * 2 * NC * kBrick3);
        for (int k = tid; k < NC * kBrick3 / 4; k += kThreads) {
            out[k] = reinterpret_cast<const float4 *>(&cM[0][0])[k];
            out[NC * kBrick3 / 4 + k] = reinterpret_cast<const float4 *>(&cW[0][0])[k];
        }
    } else {
        gather_halo<NC>(cM, cW, part + (size_t)b * 2 * kHalo3, part + (size_t)b * 2 * kHalo3 + kHalo3);
    }
}

// Step 3 where every unit had a workgroup of its own: the block's units [ub, ue) added in order, then its halo brick.
template <int NC>
__global__ __launch_bounds__(kThreads) void k_bin_units(const int32_t *__restrict__ blocks, int u0,
                                                        const float *__restrict__ usum, float *__restrict__ part)
{
    __shared__ __attribute__((aligned(16))) float cs[2][NC][kBrick3];
    const int b = blockIdx.x, ub = blocks[4 * b + 1] - u0, nu = blocks[4 * b + 2] - u0 - ub;
    constexpr int kQuads = 2 * NC * kBrick3 / 4;
    const float4 *in = reinterpret_cast<const float4 *>(usum) + (size_t)ub * kQuads;
#pragma unroll 4
    for (int k = threadIdx.x; k < kQuads; k += kThreads) {
        float4 v[kUnitsPerBlock];
#pragma unroll
        for (int u = 0; u < kUnitsPerBlock; ++u) v[u] = in[(size_t)min(u, nu - 1) * kQuads + k];
        float4 a = v[0];
#pragma unroll
        for (int u = 1; u < kUnitsPerBlock; ++u)
            if (u < nu) a = make_float4(a.x + v[u].x, a.y + v[u].y, a.z + v[u].z, a.w + v[u].w);
        reinterpret_cast<float4 *>(&cs[0][0][0])[k] = a;
    }
    __syncthreads();
    gather_halo<NC>(cs[0], cs[1], part + (size_t)b * 2 * kHalo3, part + (size_t)b * 2 * kHalo3 + kHalo3);
}

// Step 4a: group g sums the partials of its blocks [gu0, gu1) (consecutive blocks of one brick), in
// block order.  groups: [g][4] = key, first block, end block, 0 (blocks relative to the chunk).
__global__ __launch_bounds__(kThreads) void k_bin_group(const int32_t *__restrict__ groups,
                                                        const float *__restrict__ part, float *__restrict__ gpart)
{
    const int gi = blockIdx.x;
    const int u0 = groups[4 * gi + 1], u1 = groups[4 * gi + 2];
    float *out = gpart + (size_t)gi * 2 * kHalo3;
    for (int e = threadIdx.x; e < 2 * kHalo3; e += kThreads) {
        float acc = 0.0f;
        int u = u0;
        for (; u + 4 <= u1; u += 4) {  // four independent loads, added in order
            const float a = part[(size_t)u * 2 * kHalo3 + e], b = part[(size_t)(u + 1) * 2 * kHalo3 + e];
            const float c = part[(size_t)(u + 2) * 2 * kHalo3 + e], d = part[(size_t)(u + 3) * 2 * kHalo3 + e];
            acc += a;
            acc += b;
            acc += c;
            acc += d;
        }
        for (; u < u1; ++u) acc += part[(size_t)u * 2 * kHalo3 + e];
        out[e] = acc;
    }
}

// Step 4b: every voxel adds the groups of the bricks whose halo covers it: its own brick and, on
// a brick's low face, the neighbour below on that axis (whose halo index there is kBrick); in a
// fixed order.  gbeg: [key - key0] first group of each brick of the chunk (kBricks + 1 entries);
// without a grouping pass, blocks and their partials take the place of the groups.
__global__ __launch_bounds__(kThreads) void k_insert_reduce(const float *__restrict__ gpart,
                                                            const int32_t *__restrict__ gbeg, BinGeom g,
                                                            float *__restrict__ Mnum, float *__restrict__ Wt,
                                                            bool first, bool direct)
{
    const int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int L = g.L;
    if (v >= (int64_t)L * L * L) return;
    const int x = (int)(v % L), y = (int)((v / L) % L), z = (int)(v / ((int64_t)L * L));
    const int bx = x / kBrick, by = y / kBrick, bz = z / kBrick;
    const int lx = x % kBrick, ly = y % kBrick, lz = z % kBrick;
    const int nx = (lx == 0 && bx > 0) ? 2 : 1, ny = (ly == 0 && by > 0) ? 2 : 1, nz = (lz == 0 && bz > 0) ? 2 : 1;
    float sm = 0.0f, sw = 0.0f;
    for (int dz = 0; dz < nz; ++dz)
        for (int dy = 0; dy < ny; ++dy)
            for (int dx = 0; dx < nx; ++dx) {
                const int key = ((bz - dz) * g.nb + (by - dy)) * g.nb + (bx - dx);
                const int hv = ((dz ? kBrick : lz) * kHalo + (dy ? kBrick : ly)) * kHalo + (dx ? kBrick : lx);
                const int g1 = gbeg[key + 1];
                int gi = gbeg[key];
                float bm = 0.0f, bw = 0.0f;  // blocks of one brick first, as the grouping pass adds them
                float &am = direct ? bm : sm, &aw = direct ? bw : sw;
                for (; gi + 4 <= g1; gi += 4) {  // independent loads, added in order
                    float a[4], w[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        a[q] = gpart[(size_t)(gi + q) * 2 * kHalo3 + hv];
                        w[q] = gpart[(size_t)(gi + q) * 2 * kHalo3 + kHalo3 + hv];
                    }
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        am += a[q];
                        aw += w[q];
                    }
                }
                for (; gi < g1; ++gi) {
                    am += gpart[(size_t)gi * 2 * kHalo3 + hv];
                    aw += gpart[(size_t)gi * 2 * kHalo3 + kHalo3 + hv];
                }
                if (direct) {
                    sm += bm;
                    sw += bw;
                }
            }
    if (first) {  // the pass's first rotation chunk: the sums start here (no separate zero fill)
        Mnum[v] = sm;
        Wt[v] = sw;
    } else {
        Mnum[v] += sm;
        Wt[v] += sw;
    }
}

BinGeom geom_of(const emc_ctx *c)
{
    BinGeom g;
    g.L = c->L;
    g.nb = (c->L + kBrick - 1) / kBrick;
    g.S = c->S;
    g.Pa = c->Pa;
    g.Pp = c->Pp;
    g.chunk = c->chunk;
    g.interp = c->opt.interp;
    int jb = 1;
    while ((1 << jb) < c->Pa) ++jb;
    g.jbits = jb;
    return g;
}

}  // namespace

// Builds the pair lists, units, groups and their device tables.  Allocates (setup time only).
hipError_t build_bins(emc_ctx *c, std::string &err)
{
    hipStream_t st = c->stream;
    const BinGeom g = geom_of(c);
    const int64_t n = (int64_t)c->S * c->Pa;
    if (n >= ((int64_t)1 << 31) || ((int64_t)c->S << g.jbits) > ((int64_t)1 << 32)) {
        err = "binned insertion supports S * active pixels < 2^31 and S * 2^ceil(log2 P_act) <= 2^32 "
              "(use insert = ATOMIC)";
        return hipErrorInvalidValue;
    }
    const int nch = (c->S + c->chunk - 1) / c->chunk;
    const uint32_t nbr = (uint32_t)g.nb * g.nb * g.nb;
    const uint32_t nkeys = (uint32_t)nch * nbr;
    int max_brick_blocks = 0, max_units = 0;
    int end_bit = 1;
    while (end_bit < 32 && ((uint64_t)1 << end_bit) <= nkeys) ++end_bit;
    uint32_t *kin = nullptr, *vin = nullptr, *kout = nullptr, *pout = nullptr;
    void *tmp = nullptr;
    int32_t *cnt = nullptr;
    size_t tmp_bytes = 0;
    hipError_t e = hipSuccess;
    auto chk = [&](hipError_t r) {
        if (e == hipSuccess) e = r;
    };
    auto release = [](auto *&p) {
        if (p) (void)hipFree(p);
        p = nullptr;
    };
    release(c->bin_vals);
    release(c->bin_perm);
    release(c->bin_vbeg);
    release(c->bin_frac);
    release(c->bin_units);
    release(c->bin_blocks);
    release(c->bin_groups);
    release(c->bin_gbeg);
    release(c->bin_part);
    release(c->bin_gpart);
    chk(hipMalloc((void **)&kin, sizeof(uint32_t) * n));
    chk(hipMalloc((void **)&vin, sizeof(uint32_t) * n));
    chk(hipMalloc((void **)&kout, sizeof(uint32_t) * n));
    chk(hipMalloc((void **)&c->bin_vals, sizeof(uint32_t) * n));
    chk(hipMalloc((void **)&cnt, sizeof(int32_t) * 2 * (size_t)nkeys));
    const int grid1 = (int)std::min<int64_t>((n + 255) / 256, 65536);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_bin_keys, dim3(grid1), dim3(256), 0, st, c->rotm, c->axyz, g, n, nkeys, kin, vin);
        chk(hipGetLastError());
    }
    if (e == hipSuccess)
        chk(rocprim::radix_sort_pairs(nullptr, tmp_bytes, kin, kout, vin, c->bin_vals, (size_t)n, 0, end_bit, st));
    if (e == hipSuccess) chk(hipMalloc(&tmp, std::max<size_t>(tmp_bytes, 16)));
    if (e == hipSuccess)
        chk(rocprim::radix_sort_pairs(tmp, tmp_bytes, kin, kout, vin, c->bin_vals, (size_t)n, 0, end_bit, st));
    if (e == hipSuccess) chk(hipMemsetAsync(cnt, 0, sizeof(int32_t) * 2 * (size_t)nkeys, st));
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_bin_count, dim3(grid1), dim3(256), 0, st, kout, n, nkeys, cnt);
        chk(hipGetLastError());
    }
    std::vector<int32_t> h(2 * (size_t)nkeys, 0);
    if (e == hipSuccess) chk(hipMemcpyAsync(h.data(), cnt, sizeof(int32_t) * h.size(), hipMemcpyDeviceToHost, st));
    if (e == hipSuccess) chk(hipStreamSynchronize(st));
    // units (key, begin, end, 0): at most kUnit pairs, key order (chunk-major); blocks (key, first
    // unit, end unit, 0): at most kUnitsPerBlock consecutive units of one brick, one insertion
    // workgroup each, numbered per chunk (unit indices global); groups (key, first block, end
    // block, 0): at most kGroup consecutive blocks of one brick, numbered per chunk, with each
    // brick's first group in gbeg
    std::vector<int32_t> units, blocks, groups, gbeg, bbeg;  // bbeg: each brick's first block
    c->bin_chunk_blocks.assign(nch + 1, 0);
    c->bin_chunk_units.assign(nch + 1, 0);
    c->bin_chunk_groups.assign(nch + 1, 0);
    int max_blocks = 0, max_groups = 0;
    for (int ch = 0; ch < nch && e == hipSuccess; ++ch) {
        const int b_first = (int)(blocks.size() / 4), g_first = (int)(groups.size() / 4);
        for (uint32_t br = 0; br < nbr; ++br) {
            const uint32_t k = (uint32_t)ch * nbr + br;
            gbeg.push_back((int32_t)(groups.size() / 4) - g_first);
            const int32_t kb = h[2 * k], ke = h[2 * k + 1];
            const int ub = (int)(units.size() / 4);
            for (int32_t t = kb; t < ke; t += kUnit) {
                units.push_back((int32_t)k);
                units.push_back(t);
                units.push_back(std::min(ke, t + kUnit));
                units.push_back(0);
            }
            const int ue = (int)(units.size() / 4);
            const int bb = (int)(blocks.size() / 4) - b_first;
            for (int u = ub; u < ue; u += kUnitsPerBlock) {
                blocks.push_back((int32_t)k);
                blocks.push_back(u);
                blocks.push_back(std::min(ue, u + kUnitsPerBlock));
                blocks.push_back(0);
            }
            const int be = (int)(blocks.size() / 4) - b_first;
            max_brick_blocks = std::max(max_brick_blocks, be - bb);
            bbeg.push_back(bb);
            for (int bl = bb; bl < be; bl += kGroup) {
                groups.push_back((int32_t)k);
                groups.push_back(bl);
                groups.push_back(std::min(be, bl + kGroup));
                groups.push_back(0);
            }
        }
        gbeg.push_back((int32_t)(groups.size() / 4) - g_first);
        bbeg.push_back((int32_t)(blocks.size() / 4) - b_first);
        c->bin_chunk_blocks[ch + 1] = (int)(blocks.size() / 4);
        c->bin_chunk_groups[ch + 1] = (int)(groups.size() / 4);
        c->bin_chunk_units[ch + 1] = (int)(units.size() / 4);
        max_units = std::max(max_units, c->bin_chunk_units[ch + 1] - c->bin_chunk_units[ch]);
        max_blocks = std::max(max_blocks, c->bin_chunk_blocks[ch + 1] - c->bin_chunk_blocks[ch]);
        max_groups = std::max(max_groups, c->bin_chunk_groups[ch + 1] - c->bin_chunk_groups[ch]);
    }
    const uint32_t n_units = (uint32_t)(units.size() / 4);
    c->bin_direct = max_brick_blocks <= kDirect;
    const bool split = max_units <= kSplitUnits;
    if (c->bin_direct) gbeg = bbeg;
    if (e == hipSuccess && n_units > 0) {
        chk(hipMalloc((void **)&c->bin_units, sizeof(int32_t) * units.size()));
        chk(hipMalloc((void **)&c->bin_blocks, sizeof(int32_t) * blocks.size()));
        chk(hipMalloc((void **)&c->bin_groups, sizeof(int32_t) * groups.size()));
        chk(hipMalloc((void **)&c->bin_gbeg, sizeof(int32_t) * gbeg.size()));
        chk(hipMalloc((void **)&c->bin_part, sizeof(float) * 2 * kHalo3 * (size_t)max_blocks));
        // Kept from one build to the next while it is large enough (it is at most 32 MB): freeing and allocating it again
        // made a new mask or new rotations 0.2 to 0.3 ms slower (32^3 / 3,240: 1.9 -> 2.2 ms).
        const size_t usum =
            split ? sizeof(float) * 2 * kBrick3 * (c->opt.interp == EMC_INTERP_NEAREST ? 1 : 8) * (size_t)max_units : 0;
        if (!split || usum > c->bin_usum_bytes) {
            release(c->bin_usum);
            c->bin_usum_bytes = 0;
            if (split) chk(hipMalloc((void **)&c->bin_usum, usum));
            if (c->bin_usum) c->bin_usum_bytes = usum;
        }
        if (!c->bin_direct) chk(hipMalloc((void **)&c->bin_gpart, sizeof(float) * 2 * kHalo3 * (size_t)max_groups));
        chk(hipMalloc((void **)&c->bin_perm, sizeof(uint16_t) * n));
        chk(hipMalloc((void **)&c->bin_vbeg, sizeof(uint16_t) * kVbeg * (size_t)n_units));
        if (c->opt.interp == EMC_INTERP_TRILINEAR)
            chk(hipMalloc((void **)&c->bin_frac, sizeof(float) * 3 * kUnit * (size_t)n_units));
        if (e == hipSuccess)
            chk(hipMemcpy(c->bin_units, units.data(), sizeof(int32_t) * units.size(), hipMemcpyHostToDevice));
        if (e == hipSuccess)
            chk(hipMemcpy(c->bin_blocks, blocks.data(), sizeof(int32_t) * blocks.size(), hipMemcpyHostToDevice));
        if (e == hipSuccess)
            chk(hipMemcpy(c->bin_groups, groups.data(), sizeof(int32_t) * groups.size(), hipMemcpyHostToDevice));
        if (e == hipSuccess) chk(hipMemcpy(c->bin_gbeg, gbeg.data(), sizeof(int32_t) * gbeg.size(), hipMemcpyHostToDevice));
        // within each unit, rank the pairs by base voxel (stable: then by (s, j))
        const uint64_t nkeys2 = (uint64_t)n_units * kBrick3;
        int end_bit2 = 1;
        while (end_bit2 < 32 && ((uint64_t)1 << end_bit2) <= nkeys2) ++end_bit2;
        if (nkeys2 >= ((uint64_t)1 << 32)) chk(hipErrorInvalidValue);
        // pairs outside every unit (no valid voxel) keep the largest key and stay at the end
        const uint32_t sentinel = (uint32_t)(((uint64_t)1 << end_bit2) - 1);
        if (e == hipSuccess) chk(hipMemsetD32Async((hipDeviceptr_t)kin, (int)sentinel, (size_t)n, st));
        if (e == hipSuccess) {
            hipLaunchKernelGGL(k_unit_keys, dim3(n_units), dim3(kThreads), 0, st, c->bin_units, c->bin_vals, c->rotm,
                               c->axyz, g, kin);
            chk(hipGetLastError());
        }
        if (e == hipSuccess) {
            hipLaunchKernelGGL(k_iota, dim3(grid1), dim3(256), 0, st, vin, n);
            chk(hipGetLastError());
        }
        chk(hipMalloc((void **)&pout, sizeof(uint32_t) * n));
        size_t tmp2 = 0;
        if (e == hipSuccess)
            chk(rocprim::radix_sort_pairs(nullptr, tmp2, kin, kout, vin, pout, (size_t)n, 0, end_bit2, st));
        if (e == hipSuccess && tmp2 > tmp_bytes) {
            (void)hipFree(tmp);
            tmp = nullptr;
            chk(hipMalloc(&tmp, tmp2));
            tmp_bytes = tmp2;
        }
        if (e == hipSuccess)
            chk(rocprim::radix_sort_pairs(tmp, tmp_bytes, kin, kout, vin, pout, (size_t)n, 0, end_bit2, st));
        if (e == hipSuccess) {
            hipLaunchKernelGGL(k_unit_perm, dim3(n_units), dim3(kThreads), 0, st, c->bin_units, kout, pout, c->bin_vals,
                               c->rotm, c->axyz, g, c->bin_perm, c->bin_vbeg, c->bin_frac);
            chk(hipGetLastError());
        }
        if (e == hipSuccess) chk(hipStreamSynchronize(st));
    }
    (void)hipFree(kin);
    (void)hipFree(vin);
    (void)hipFree(kout);
    (void)hipFree(pout);
    (void)hipFree(tmp);
    (void)hipFree(cnt);
    if (e != hipSuccess && err.empty()) err = std::string("build_bins: ") + hipGetErrorString(e);
    c->bins_valid = e == hipSuccess;
    return e;
}

hipError_t launch_insert_binned(const emc_ctx *c, int s0, int cs, hipStream_t st)
{
    (void)cs;
    const int k = s0 / c->chunk;
    const int b0 = c->bin_chunk_blocks[k], b1 = c->bin_chunk_blocks[k + 1];
    const int g0 = c->bin_chunk_groups[k], g1 = c->bin_chunk_groups[k + 1];
    if (b1 <= b0) {  // no pairs in this chunk; the first chunk still starts the sums at zero
        hipError_t e = hipSuccess;
        if (k == 0) e = launch_fill_f32(c->Mnum, 0.0f, c->N3, st);
        if (e == hipSuccess && k == 0) e = launch_fill_f32(c->Wt, 0.0f, c->N3, st);
        return e;
    }
    const BinGeom g = geom_of(c);
    const int32_t *blocks = c->bin_blocks + 4 * (size_t)b0;
    const int u0 = c->bin_chunk_units[k], nu = c->bin_chunk_units[k + 1] - u0;
    const bool split = c->bin_usum != nullptr, nearest = c->opt.interp == EMC_INTERP_NEAREST;
    const auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(split ? nu : b1 - b0), dim3(kThreads), 0, st, blocks, u0, c->bin_units, c->bin_vals,
                           c->bin_perm, c->bin_vbeg, c->bin_frac, c->U, s0, c->T, g, split ? c->bin_usum : c->bin_part);
    };
    const auto add_units = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(b1 - b0), dim3(kThreads), 0, st, blocks, u0, c->bin_usum, c->bin_part);
    };
    if (split && nearest) {
        run(k_insert_binned<EMC_INTERP_NEAREST, true>);
        add_units(k_bin_units<1>);
    } else if (split) {
        run(k_insert_binned<EMC_INTERP_TRILINEAR, true>);
        add_units(k_bin_units<8>);
    } else {
        run(nearest ? k_insert_binned<EMC_INTERP_NEAREST, false> : k_insert_binned<EMC_INTERP_TRILINEAR, false>);
    }
    if (!c->bin_direct)
        hipLaunchKernelGGL(k_bin_group, dim3(g1 - g0), dim3(kThreads), 0, st, c->bin_groups + 4 * (size_t)g0, c->bin_part,
                           c->bin_gpart);
    const int nbr = g.nb * g.nb * g.nb;
    const int rt = reduce_threads(c->N3);
    hipLaunchKernelGGL(k_insert_reduce, dim3((unsigned)((c->N3 + rt - 1) / rt)), dim3(rt), 0, st,
                       c->bin_direct ? c->bin_part : c->bin_gpart, c->bin_gbeg + (size_t)k * (nbr + 1), g, c->Mnum,
                       c->Wt, k == 0, c->bin_direct);
    return hipGetLastError();
}

}  // namespace emc
