// The last pass of a linear layer: out = cast(float(y) + bias), y the layer's
// product in f32 or bf16.
//
// Bound by its bytes (and, for a few rows, by the launch).  As three torch
// passes (to f32, add, to the output type) the f32 product went through
// memory four times: 512 x 8960 from bf16 to bf16 took 20 us for 18 MB that
// one pass reads and writes in 4.  One thread takes 8 values of a row (16
// bytes of bf16); rows whose start or length is not a multiple of 8 take the
// same kernel one value at a time.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "../../include/vramc_rans.h"

namespace {

constexpr int kFinishThreads = 256;

template <typename T, int V>
struct alignas(sizeof(T) * V) Vec {
    T v[V];
};

template <typename Y, typename O, int V>
__global__ void __launch_bounds__(kFinishThreads)
    linear_finish_kernel(const Y* __restrict__ y, int64_t ld, const float* __restrict__ bias,
                         O* __restrict__ out, int64_t rows, int cols) {
    const int c = (blockIdx.x * kFinishThreads + threadIdx.x) * V;
    if (c >= cols) return;
    Vec<float, V> b = {};
    if (bias) b = *reinterpret_cast<const Vec<float, V>*>(bias + c);
    for (int64_t r = blockIdx.y; r < rows; r += gridDim.y) {
        const auto in = *reinterpret_cast<const Vec<Y, V>*>(y + r * ld + c);
        Vec<O, V> o;
#pragma unroll
        for (int i = 0; i < V; i++) {
            const float f = (float)in.v[i];
            o.v[i] = (O)(bias ? f + b.v[i] : f);
        }
        *reinterpret_cast<Vec<O, V>*>(out + r * cols + c) = o;
    }
}

template <typename Y, typename O>
int finish(const void* y, int64_t ld, const float* bias, void* out, int64_t rows, int cols,
           hipStream_t stream) {
    const bool wide = cols % 8 == 0 && ld % 8 == 0 && (uintptr_t)y % 32 == 0 &&
                      (uintptr_t)out % 32 == 0 && (uintptr_t)bias % 32 == 0;
    const int per = kFinishThreads * (wide ? 8 : 1);
    const dim3 grid((cols + per - 1) / per, (unsigned)(rows < 32768 ? rows : 32768));
    const auto* yp = static_cast<const Y*>(y);
    auto* op = static_cast<O*>(out);
    if (wide)
        hipLaunchKernelGGL((linear_finish_kernel<Y, O, 8>), grid, dim3(kFinishThreads), 0, stream,
                           yp, ld, bias, op, rows, cols);
    else
        hipLaunchKernelGGL((linear_finish_kernel<Y, O, 1>), grid, dim3(kFinishThreads), 0, stream,
                           yp, ld, bias, op, rows, cols);
    return (int)hipGetLastError();
}

template <typename Y>
int finish_to(const void* y, int64_t ld, const float* bias, void* out, int out_dtype, int64_t rows,
              int cols, hipStream_t stream) {
    switch (out_dtype) {
        case RANS_X_F32: return finish<Y, float>(y, ld, bias, out, rows, cols, stream);
        case RANS_X_BF16: return finish<Y, __bf16>(y, ld, bias, out, rows, cols, stream);
        case RANS_X_F16: return finish<Y, _Float16>(y, ld, bias, out, rows, cols, stream);
        default: return RANS_EARG;
    }
}

}  // namespace

extern "C" int rans_linear_finish(const void* y, int y_dtype, int64_t ld, const float* bias,
                                  void* out, int out_dtype, int64_t rows, int cols,
                                  hipStream_t stream) {
    if (!y || !out || rows <= 0 || cols <= 0 || ld < cols) return RANS_EARG;
    if (y_dtype == RANS_X_F32)
        return finish_to<float>(y, ld, bias, out, out_dtype, rows, cols, stream);
    if (y_dtype == RANS_X_BF16)
        return finish_to<__bf16>(y, ld, bias, out, out_dtype, rows, cols, stream);
    return RANS_EARG;
}
