// Maximize, contraction half, sparse form: U[s, j] = sum_i P[s, i] K[i, j] over the patterns whose
// responsibility for rotation s is non-zero (emc_atomic.cu:88-132 computes the same sums densely).
//
// Once the model has formed, a pattern keeps its responsibility on a handful of rotations and
// exp() underflows to exactly 0 everywhere else (at 64^3 / 25,680 / 20,000 about 0.02 % of P is
// non-zero from the fifth iteration on), so the dense contraction multiplies almost only zeros.
// One workgroup per rotation row (sparse_row.h): the row of P is scanned, its non-zero entries are
// compacted in pattern order and their count rows summed.  Same operands as the dense path
// (P = hi + lo; counts as bytes, or BF16 [+ lo] above 255; both float at precision FP32, whose dense chain it
// repeats without the zeros, bit for bit) with FP32 accumulation: only the order of the sum over patterns differs.
// FP32 at 6,300 x 4,001 x 3,200 with a formed model: 43 us; the dense contraction took 1.76 ms on the vector ALU.
#include "../emc_internal.h"
#include "sparse_row.h"

namespace emc {
namespace {

template <int KT, int NPASS, int PX>
__global__ __launch_bounds__(256) void k_mstep_sparse(const void *__restrict__ Ph, const bf16_t *__restrict__ Pl,
                                                      int64_t ldp, int s0, int I, const void *__restrict__ Kv,
                                                      const bf16_t *__restrict__ Klo, int Pp,
                                                      const double *__restrict__ gate, double gate_thr,
                                                      float *__restrict__ U, const uint8_t *__restrict__ pdirty,
                                                      int nseg)
{
    if (gate && *gate > gate_thr) return;  // the dense contraction runs instead
    const size_t o = (size_t)(s0 + blockIdx.x) * ldp;
    sparse_row<KT, NPASS, PX>(reinterpret_cast<const unsigned char *>(Ph) + o * (KT == 3 ? 4 : 2), KT == 3 ? nullptr : Pl + o,
                          I, nullptr, Kv, Klo, Pp, U + (size_t)blockIdx.x * Pp,
                          pdirty ? pdirty + (size_t)(s0 + blockIdx.x) * nseg : nullptr);
}

}  // namespace

template <int NPASS, int PX>
static void launch_np(const emc_ctx *c, int s0, int cs, const double *gate, double gate_thr, hipStream_t st)
{
    const dim3 grid(cs), blk(256);
    if (!c->mfma)
        hipLaunchKernelGGL((k_mstep_sparse<3, NPASS, PX>), grid, blk, 0, st, c->opt.scaling ? c->Pphi : c->R, nullptr,
                           (int64_t)c->Ip, s0, c->I, c->K32, nullptr, c->Pp, gate, gate_thr, c->U, c->pdirty, p_segments(c));
    else if (c->K8)
        hipLaunchKernelGGL((k_mstep_sparse<0, NPASS, PX>), grid, blk, 0, st, c->Ph, c->Pl, (int64_t)c->Ip, s0, c->I, c->K8,
                           nullptr, c->Pp, gate, gate_thr, c->U, c->pdirty, p_segments(c));
    else if (c->k_split)  // K16lo is kept allocated after a pattern set that needed it: key on k_split
        hipLaunchKernelGGL((k_mstep_sparse<2, NPASS, PX>), grid, blk, 0, st, c->Ph, c->Pl, (int64_t)c->Ip, s0, c->I, c->K16,
                           c->K16lo, c->Pp, gate, gate_thr, c->U, c->pdirty, p_segments(c));
    else
        hipLaunchKernelGGL((k_mstep_sparse<1, NPASS, PX>), grid, blk, 0, st, c->Ph, c->Pl, (int64_t)c->Ip, s0, c->I, c->K16,
                           nullptr, c->Pp, gate, gate_thr, c->U, c->pdirty, p_segments(c));
}

hipError_t launch_mstep_sparse(const emc_ctx *c, int s0, int cs, const double *gate, double gate_thr, hipStream_t st)
{
    if (c->Pp > kSparseMaxPp || c->Pp % 16 != 0) return hipErrorInvalidValue;
    // Pixels per thread so that most of the 256 threads have some: 3,240 x 1,000 x 896 with two-term counts 52 us at
    // 16 (56 threads), 39 at 4; 45^3 (1,664) 46 us for four chunks both at 16 and 8.
    if (c->Pp <= 1024) launch_np<1, 4>(c, s0, cs, gate, gate_thr, st);
    else if (c->Pp <= 2048) launch_np<1, 8>(c, s0, cs, gate, gate_thr, st);
    else if (c->Pp <= 4096) launch_np<1, 16>(c, s0, cs, gate, gate_thr, st);
    else launch_np<kSparseMaxPp / 4096, 16>(c, s0, cs, gate, gate_thr, st);
    return hipGetLastError();
}

}  // namespace emc
