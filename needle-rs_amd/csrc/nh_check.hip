// Device functions of the forward run alone over given operands, for checks.
// (A file of its own: kernels added beside the forward's move its code, 0.2 %
// of a 300-token prompt.)
#include "nh_forward.h"
#include "nh_internal.h"
#include "nh_mix8.h"

namespace nh {

// Both passes of the layer kernel over given operands (nh_debug_mix8): the
// factor into fragment order, x as each pass reads it.
__global__ __launch_bounds__(MIX_T) void k_mix8(const uint16_t* __restrict__ factor, const float* __restrict__ x,
                                                float* __restrict__ yt, float* __restrict__ yn) {
    __shared__ alignas(16) uint16_t kf[HADA_N];
    __shared__ alignas(16) float A[HADA_N], B[HADA_NB * BT_PITCH], C[HADA_N];
    const int t = threadIdx.x;
    for (int e = t; e < HADA_N; e += MIX_T) {
        const int st = e & 7, lane = (e >> 3) & 63, tile = e >> 9;
        kf[e] = factor[(4 * st + lane / 16) * HADA_NB + tile * 16 + lane % 16];
        A[mix_in(e)] = x[e];
    }
    __syncthreads();
    const uint4* f = reinterpret_cast<const uint4*>(kf);
    mix8_t(t, f, A, B);
    __syncthreads();
    auto at = [](int e) { return (e >> 5) * BT_PITCH + (e & 3) * 8 + ((e & 31) >> 2); };
    for (int e = t; e < HADA_N; e += MIX_T) yt[e] = B[at(e)];
    __syncthreads();
    for (int e = t; e < HADA_N; e += MIX_T) B[at(e)] = x[e];
    __syncthreads();
    mix8_n(t, B, f, C, HADA_NB);
    __syncthreads();
    for (int e = t; e < HADA_N; e += MIX_T) yn[e] = C[e];
}

hipError_t fwd_mix8(const uint16_t* factor, const float* x, float* yt, float* yn, hipStream_t s) {
    hipLaunchKernelGGL(k_mix8, dim3(1), dim3(MIX_T), 0, s, factor, x, yt, yn);
    return hipGetLastError();
}

}  // namespace nh
