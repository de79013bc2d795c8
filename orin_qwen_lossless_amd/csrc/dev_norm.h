// The RMS norm of one row of 2048 elements by 256 threads, eight consecutive elements each, shared by the glue kernel
// (kernels_moe.hip) and the router GEMV that forms its own input (kernels_compat.hip).
#pragma once

#include "dev_common.h"

namespace bf16n {
namespace dev {

constexpr int NORM8_N = 2048, NORM8_THREADS = NORM8_N / 8;

// eight BF16 values <-> floats
__device__ __forceinline__ void unpack8(const uint4 v, float (&f)[8]) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        f[2 * i] = __uint_as_float(w[i] << 16);
        f[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
    }
}
__device__ __forceinline__ uint4 pack8(const float (&f)[8]) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        w[i] = f32_to_bf16_rne(f[2 * i]) | ((uint32_t) f32_to_bf16_rne(f[2 * i + 1]) << 16);
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// bf16(v * rsqrt(mean(v^2) + eps) * gamma) of this thread's eight elements; wave_sq: NORM8_THREADS / 64 floats of LDS
// (one barrier inside)
__device__ __forceinline__ uint4 norm8_row(const float (&v)[8], const uint16_t * gamma, float eps, float * wave_sq) {
    float sq = 0.f;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        sq = fmaf(v[i], v[i], sq);
    }
    sq = wave_sum(sq);
    if ((threadIdx.x & 63) == 0) {
        wave_sq[threadIdx.x >> 6] = sq;
    }
    __syncthreads();
    const float total = ((wave_sq[0] + wave_sq[1]) + wave_sq[2]) + wave_sq[3];
    const float scale = 1.0f / sqrtf(total / (float) NORM8_N + eps);
    float g[8] = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f};
    if (gamma) {
        unpack8(*(const uint4 *) (gamma + 8 * threadIdx.x), g);
    }
    float o[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        o[i] = v[i] * scale * g[i];
    }
    return pack8(o);
}

} // namespace dev
} // namespace bf16n
