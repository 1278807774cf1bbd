// Backward of bitfield-masked attention at head dims above 32: dK/dV and dQ of small problems in one launch.
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
// the pre-pass and one, D 64: 2 x 283 tokens, 6 / 2 heads replayed as a graph 57.7 -> 46.6, but the same 87 where the host that issues the launches
// is what is waited for (64.4 -> 55.4 with a quicker one); 2048, 16 heads 110.8 -> 93.7; 4096, 8 heads 163.5 -> 137.6;
// 8192, 6 / 1 heads 311.7 -> 283.0; 2 x 2048, 16 heads, with a bias 160.2 -> 151.5; a bool mask, 2048, 16 heads 99.3 -> 82.0; 2048, 32 / 8
// heads (parts) 149.6 -> 145.2, nothing hidden 141.1 -> 142.4.  D 32, where three workgroups of either kernel fit a unit and two of this one:
// 2 x 2048, 16 heads 108.3 -> 111.4, 4096, 32 / 8 heads 254.8 -> 262.4: not there.
// Above head dim 64 the two launches hand dS over: the host waits for the plan's count to size that workspace, dQ waits for the last
// of dK/dV, and dS goes through memory; one launch computes S and dP again instead.  With no more workgroups than units (256) both
// kernels take the time of the longer one: faster whatever the mask, D 128: 1024, 8 heads 101.1 -> 83.6 (the host's wait); 2048, 8
// heads 135.0 -> 103.7, nothing hidden 152.6 -> 125.7, with a bias 150.7 -> 117.4; 16384, 1 head 755.9 -> 550.3; a bool mask, 1024, 8
// heads 86.4 -> 70.7; D 80, 1024, 16 heads 101.5 -> 81.7.  Up to two rounds (512) where the count, waited for, leaves the lists
// uneven: 4096, 8 heads, pairs of 0.52 of the tiles 240.2 -> 203.3, 0.54 235.7 -> 230.1, 0.73 268.4 -> 272.2; 3000, 10 / 2 heads 0.51
// 197.8 -> 167.6, 8 heads 0.65 189.5 -> 177.8; 8192, 4 heads, D 80 366.5 -> 314.6; 4096, 6 / 1 heads (parts) 233.7 -> 183.7; 2048, 16
// heads, nothing hidden 180.2 -> 188.9.  Beyond: 2048, 24 heads 166.9 -> 170.7, 20 heads 157.0 -> 153.9.  The line at 768
// keys is not one of speed: below it one launch would be as good (4 x 283, 16 / 4 heads 100.7 -> 79.0, the host's wait ahead of the
// launches).  The tests of the hand-over (a limit or a failing allocation of its workspace, the same bits in runs of heads) hold calls
// of up to 640 keys to asking for a workspace.
bool both_in_one_launch(const AttnParams& p, int64_t dkdv_blocks, int64_t pairs) {
    if (p.D < 64 || !two_streams(p) || p.rows != nullptr) return false;
    if (p.D > 64) {
        const int64_t blocks = (int64_t)p.num_m * p.B * p.Hq + dkdv_blocks;
        const bool few_pairs = pairs > 0 && 3 * pairs <= 2 * (int64_t)p.B * p.num_kt * ((p.Sq + 31) / 32);
        if (p.ds_ws != nullptr || !one_launch_sizes(p.Sq, p.Sk, p.B, p.Hq) || blocks > (few_pairs ? 512 : 256)) return false;
    }
    if (p.Sq > MAX_SLICE_LIST * 32 || p.Sk > MAX_LIST * DQ_KT || dkdv_far(p)) return false;  // (walked in passes)
    return p.bias == nullptr ? p.D > 64 || p.lse_scaled != nullptr : p.bias_sm == 0 && p.bias_vec;
}

int launch_bwd_both(const AttnParams& kv, const AttnParams& p, int dtype, hipStream_t stream) {
    if (dtype == 1)
        return p.D == 128  ? launch_both_t<BF16, 128>(kv, p, stream)
               : p.D == 96 ? launch_both_t<BF16, 96>(kv, p, stream)
                           : launch_both_t<BF16, 64>(kv, p, stream);
    return p.D == 128  ? launch_both_t<F16, 128>(kv, p, stream)
           : p.D == 96 ? launch_both_t<F16, 96>(kv, p, stream)
                       : launch_both_t<F16, 64>(kv, p, stream);
}

}  // namespace bam
