// SageAttention forward for gfx950, pipelined kernel under an additive mask tensor together with the causal flag: the instances of
// attn_fast_kernel.h that add -1e6 to what the causal mask hides (attn_fwd_fast_addmask.hip holds those without the flag).
// Before, the general kernel served these calls: B2 H32/8 M1717 N1717 D64 bf16 603 -> 151 us, B4 H2 M2224 D128 246 -> 87 us, B4 H8/1
// M1856 D128 with a row of entries per sequence 157 -> 75 us.
#include "attn_fast_kernel.h"

namespace sage {
namespace attn {
namespace {

template <int D, typename VT, typename MT>
int launch_additive(const AttnArgs& a, hipStream_t stream) {
    AttnArgs b = a;
    const int nq2 = (a.M + kFastRows - 1) / kFastRows;
    b.total_wg = (int)((int64_t)a.total_wg / a.nq * nq2);
    b.causal = 0;  // (the limits of the walk and of the rows, not the score registers of hidden keys: see c_first)
    b.mask_causal = b.longest_first = 1;
    dim3 grid((unsigned)b.total_wg), block(kFastThreads);
    hipLaunchKernelGGL((sage_attn_fwd_fast_kernel<D, VT, true, 1, MT, false, true>), grid, block, 0, stream, b, nq2);
    return check_launch("sage_attn_fwd_fast_kernel (additive mask and causal)");
}

template <int D, typename VT>
int launch_additive_mt(const AttnArgs& a, hipStream_t stream) {
    if (a.mask_dt == SAGE_F32) return launch_additive<D, VT, float>(a, stream);
    return a.mask_dt == SAGE_BF16 ? launch_additive<D, VT, __bf16>(a, stream) : launch_additive<D, VT, _Float16>(a, stream);
}

}  // namespace

int launch_fast_additive_causal(const AttnArgs& a, int head_dim, int v_dtype, hipStream_t stream) {
    if (head_dim == 128)
        return v_dtype == SAGE_BF16 ? launch_additive_mt<128, __bf16>(a, stream) : launch_additive_mt<128, _Float16>(a, stream);
    return v_dtype == SAGE_BF16 ? launch_additive_mt<64, __bf16>(a, stream) : launch_additive_mt<64, _Float16>(a, stream);
}

}  // namespace attn
}  // namespace sage
