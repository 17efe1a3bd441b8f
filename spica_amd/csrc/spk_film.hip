// spk_film.hip -- film read-back: the compensated float32 sums resolved on the device.
//
// A film pixel is four float4 (sums of L and L^2 with their Kahan compensations).  Bound: the
// copy to the host.  Resolving there moved 64 bytes a pixel over PCIe and then ran one scalar
// loop over fresh host pages; here a pixel crosses as the 12 bytes (image) or 56 bytes (film)
// the caller asked for, already in place.  One thread a pixel: the kernels read 16-byte vectors
// and take microseconds.  Measured: a 1920x1080 sphere-field image of 32 samples 77.2 -> 31.6 ms (the
// read-back was 47 ms of it), 256x256 of 64 samples 3.75 -> 3.33 ms.  These kernels keep single-precision subnormals (the
// stage kernels flush theirs), so the results equal the host's conversion bit for bit.
#include "spk_internal.h"

namespace spk {

namespace {

// The Kahan compensation holds the negated lost low-order part.
__device__ __forceinline__ double comp_sum(float s, float c) { return (double)s - (double)c; }

__global__ __launch_bounds__(256) void k_resolve_film(const float4* __restrict__ sum, const float4* __restrict__ c,
                                                      const float4* __restrict__ sq, const float4* __restrict__ sqc,
                                                      uint32_t n, double* out_sum, double* out_sq, double* out_count) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const float4 s = sum[i];
    if (out_sum) {
        const float4 k = c[i];
        double* o = out_sum + 3 * (size_t)i;
        o[0] = comp_sum(s.x, k.x);
        o[1] = comp_sum(s.y, k.y);
        o[2] = comp_sum(s.z, k.z);
    }
    if (out_sq) {
        const float4 q = sq[i], k = sqc[i];
        double* o = out_sq + 3 * (size_t)i;
        o[0] = comp_sum(q.x, k.x);
        o[1] = comp_sum(q.y, k.y);
        o[2] = comp_sum(q.z, k.z);
    }
    if (out_count) out_count[i] = (double)s.w;
}

__global__ __launch_bounds__(256) void k_resolve_image(const float4* __restrict__ sum, const float4* __restrict__ c,
                                                       uint32_t n, float* __restrict__ rgb) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const float4 s = sum[i], k = c[i];
    const double w = (double)s.w + 1e-12;
    float* o = rgb + 3 * (size_t)i;
    o[0] = (float)(comp_sum(s.x, k.x) / w);
    o[1] = (float)(comp_sum(s.y, k.y) / w);
    o[2] = (float)(comp_sum(s.z, k.z) / w);
}

}  // namespace

int launch_resolve_film(const RenderBufs& b, size_t off, uint32_t n, double* out_sum, double* out_sq, double* out_count,
                        hipStream_t st) {
    hipLaunchKernelGGL(k_resolve_film, dim3((n + 255) / 256), dim3(256), 0, st, (const float4*)b.film_sum + off,
                       (const float4*)b.film_c + off, (const float4*)b.film_sq + off, (const float4*)b.film_sqc + off, n,
                       out_sum, out_sq, out_count);
    SPK_CHECK_HIP(hipGetLastError());
    return SPK_OK;
}

int launch_resolve_image(const RenderBufs& b, size_t off, uint32_t n, float* rgb, hipStream_t st) {
    hipLaunchKernelGGL(k_resolve_image, dim3((n + 255) / 256), dim3(256), 0, st, (const float4*)b.film_sum + off,
                       (const float4*)b.film_c + off, n, rgb);
    SPK_CHECK_HIP(hipGetLastError());
    return SPK_OK;
}

}  // namespace spk
