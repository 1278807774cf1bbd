// Backward of bitfield-masked attention: delta pre-pass and the dK/dV instantiations for sequences of up to 131072
// rows, with their dispatch.
#include "bwd_kernels.h"

namespace bam {

int launch_bwd_dkdv_long(const AttnParams& p, int dtype, hipStream_t stream);  // bwd_long.hip

template <typename T, int D>
static int launch_pre_t(const AttnParams& p, hipStream_t stream) {
    const int64_t threads = (int64_t)p.B * p.Sq * p.Hq * (LDS_COLS<D> / 8);
    const int64_t blocks = (threads + 255) / 256;
    hipLaunchKernelGGL((bwd_preprocess_kernel<T, D>), dim3((unsigned)blocks), dim3(256), 0, stream, p);
    return (int)hipGetLastError();
}
// dK / dV (blockIdx.y) = the sum of the parts, in their order; four columns per thread.  Bound by its launch where the
// parts are small (4 to 6 us), else by reading them, mostly from the last-level cache: 49 MB 9.6 us, 67 MB 12.0 (5 to 5.7 TB/s).
template <typename T>
__global__ __launch_bounds__(256) void sum_parts_kernel(const AttnParams p, const float* parts_dk, const float* parts_dv, int parts) {
    const unsigned quads = (unsigned)p.d / 4u;
    const unsigned item = blockIdx.x * 256u + threadIdx.x;  // (b, key, kv head, quad); the host keeps it below 2^31
    if (item >= (unsigned)p.B * (unsigned)p.Sk * (unsigned)p.Hkv * quads) return;
    const unsigned row = item / quads, c = 4u * (item - row * quads);
    const unsigned bs = row / (unsigned)p.Hkv, h = row - bs * (unsigned)p.Hkv;
    const unsigned b = bs / (unsigned)p.Sk, s = bs - b * (unsigned)p.Sk;
    const float* src = (blockIdx.y ? parts_dv : parts_dk) + (int64_t)row * parts * p.d + c;
    f32x4 x = *(const f32x4*)src;
    for (int j = 1; j < parts; ++j) x += *(const f32x4*)(src + (int64_t)j * p.d);
    const Tensor4 t = blockIdx.y ? p.dv : p.dk;
    const int64_t at = (int64_t)b * t.sb + (int64_t)s * t.ss + (int64_t)h * t.sh + c;
    if (p.grad_typed) {
        *(u32x2*)((unsigned short*)t.ptr + at) = u32x2{T::pack2(x[0], x[1]), T::pack2(x[2], x[3])};
    } else {
        f32x4* dst = (f32x4*)((float*)t.ptr + at);
        *dst = *dst + x;
    }
}
int launch_sum_parts(const AttnParams& p, const float* parts_dk, const float* parts_dv, int parts, int dtype, hipStream_t stream) {
    const int64_t items = (int64_t)p.B * p.Sk * p.Hkv * (p.d / 4);
    const dim3 grid((unsigned)((items + 255) / 256), 2);
    if (dtype == 1)
        hipLaunchKernelGGL((sum_parts_kernel<BF16>), grid, dim3(256), 0, stream, p, parts_dk, parts_dv, parts);
    else
        hipLaunchKernelGGL((sum_parts_kernel<F16>), grid, dim3(256), 0, stream, p, parts_dk, parts_dv, parts);
    return (int)hipGetLastError();
}
template <typename T, int D>
static int launch_dkdv_t(const AttnParams& p, hipStream_t stream) {
    return p.bias != nullptr ? launch_dkdv_b<T, D, true, false>(p, stream) : launch_dkdv_b<T, D, false, false>(p, stream);
}

int launch_bwd_preprocess(const AttnParams& p, int dtype, hipStream_t stream) { BAM_DISPATCH(launch_pre_t) }
int launch_bwd_dkdv(const AttnParams& p, int dtype, hipStream_t stream) {
    if (p.Sq > MAX_SLICE_LIST * 32 || dkdv_far(p)) return launch_bwd_dkdv_long(p, dtype, stream);
    BAM_DISPATCH(launch_dkdv_t)
}

}  // namespace bam
