// Backward of bitfield-masked attention at head dims 33 to 64: dK/dV and dQ of small problems in one launch.
#include "bwd_kernels.h"

namespace bam {

template <typename T, int D, int BIAS_FORM>
static int launch_both_m(const AttnParams& kv, const AttnParams& p, hipStream_t stream) {
    const int dkdv_blocks = kv.num_kt * kv.B * kv.Hkv, blocks = dkdv_blocks + p.num_m * p.B * p.Hq;
    if (p.mask_mode == MASK_INDEXED)
        hipLaunchKernelGGL((bwd_both_kernel<T, D, MASK_INDEXED, BIAS_FORM>), dim3(blocks), dim3(DKDV_THREADS), 0, stream, kv, p, dkdv_blocks);
    else if (p.mask_mode == MASK_DENSE)
        hipLaunchKernelGGL((bwd_both_kernel<T, D, MASK_DENSE, BIAS_FORM>), dim3(blocks), dim3(DKDV_THREADS), 0, stream, kv, p, dkdv_blocks);
    else
        hipLaunchKernelGGL((bwd_both_kernel<T, D, MASK_BITFIELD, BIAS_FORM>), dim3(blocks), dim3(DKDV_THREADS), 0, stream, kv, p, dkdv_blocks);
    return (int)hipGetLastError();
}
template <typename T, int D>
static int launch_both_t(const AttnParams& kv, const AttnParams& p, hipStream_t stream) {
    return p.bias == nullptr ? launch_both_m<T, D, BIAS_NONE>(kv, p, stream) : launch_both_m<T, D, BIAS_TILES>(kv, p, stream);
}

// Both kernels keep one workgroup of eight waves on a unit, so their workgroups share the units as they come free.  Worth it wherever dQ
// runs with two streams, by the end of a launch (a fifth of it where there are two workgroups a unit) and by the launch that
// dQ's delta costs its workgroups 2 us each for; beyond, dQ's smaller workgroups fill the units by themselves.  Step, us, two launches ->
// the pre-pass and one, D 64: 2 x 283 tokens, 6 / 2 heads 64.4 -> 55.4; 2048, 16 heads 110.8 -> 93.7; 4096, 8 heads 163.5 -> 137.6;
// 8192, 6 / 1 heads 311.7 -> 283.0; 2 x 2048, 16 heads, with a bias 160.2 -> 151.5; a bool mask, 2048, 16 heads 99.3 -> 82.0; 2048, 32 / 8
// heads (parts) 149.6 -> 145.2, nothing hidden 141.1 -> 142.4.  D 32, where three workgroups of either kernel fit a unit and two of this one:
// 2 x 2048, 16 heads 108.3 -> 111.4, 4096, 32 / 8 heads 254.8 -> 262.4: not there.
bool both_in_one_launch(const AttnParams& p) {
    if (p.D != 64 || !two_streams(p) || p.rows != nullptr) return false;
    if (p.Sq > MAX_SLICE_LIST * 32 || p.Sk > MAX_LIST * DQ_KT || dkdv_far(p)) return false;  // (walked in passes)
    return p.bias == nullptr ? p.lse_scaled != nullptr : p.bias_sm == 0 && p.bias_vec;
}

int launch_bwd_both(const AttnParams& kv, const AttnParams& p, int dtype, hipStream_t stream) {
    return dtype == 1 ? launch_both_t<BF16, 64>(kv, p, stream) : launch_both_t<F16, 64>(kv, p, stream);
}

}  // namespace bam
