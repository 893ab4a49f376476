// Instances of the half-entry segment kernel (vqk_half.h) and the kernels that
// split its inputs.
#include "vqk_half.h"

#include "vqk_internal.h"

namespace vqk {

int launch_half(const HalfParams &p, int bits, dim3 grid, hipStream_t st) {
    if (bits != 14) return set_error(VQK_ENOTIMPL, "no half-entry segment kernel for bits=%d", bits);
    return launch_with_lds<k_half<14>>(grid, dim3(64 * kHalfWaves), half_lds(14), st, p);
}

// x -> fp16 half columns [2][n / 2]: columns 0..3 and 4..7 of every 8
__global__ void __launch_bounds__(256) k_x_split(const void *x, int x_type, int64_t n8, u32x2 *out) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n8) return;
    const u32x4 v = load8_act(x, x_type, i * 8);
    out[i] = u32x2{v[0], v[1]};
    out[n8 + i] = u32x2{v[2], v[3]};
}

int launch_x_split(const void *x, int x_type, int64_t n, uint16_t *out, hipStream_t st) {
    hipLaunchKernelGGL(k_x_split, dim3(unsigned((n / 8 + 255) / 256)), dim3(256), 0, st, x, x_type, n / 8,
                       reinterpret_cast<u32x2 *>(out));
    return hip_status(hipGetLastError(), "activation split launch");
}

// fp16(silu(g0 + g1) * (u0 + u1)) as half columns [2][n / 2]
struct SwigluArgs {
    const float *g0, *g1, *u0, *u1;
    int64_t n8;
    u32x2 *out;
};
__global__ void __launch_bounds__(256) k_swiglu_split(const SwigluArgs p) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= p.n8) return;
    f32x4 v[4][2];
    const float *src[4] = {p.g0, p.g1, p.u0, p.u1};
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) v[s][h] = reinterpret_cast<const f32x4 *>(src[s])[2 * i + h];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint32_t q[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float g = v[0][h][c] + v[1][h][c], u = v[2][h][c] + v[3][h][c];
            q[c] = f32_to_h(g / (1.f + __expf(-g)) * u);
        }
        p.out[h * p.n8 + i] = u32x2{q[0] | (q[1] << 16), q[2] | (q[3] << 16)};
    }
}

int launch_swiglu_split(const float *g0, const float *g1, const float *u0, const float *u1, int64_t n,
                        uint16_t *out, hipStream_t st) {
    const SwigluArgs a{g0, g1, u0, u1, n / 8, reinterpret_cast<u32x2 *>(out)};
    hipLaunchKernelGGL(k_swiglu_split, dim3(unsigned((n / 8 + 255) / 256)), dim3(256), 0, st, a);
    return hip_status(hipGetLastError(), "SwiGLU split launch");
}

}  // namespace vqk
