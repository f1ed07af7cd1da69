// silu(gate) * up of a gated MLP whose two projections are one matrix product: the rows hold gate | up.
#include "ckv_common.h"

namespace ckv {
namespace {

// One row is the ordinary case (a decoding step), so it is bound by its launch and one trip to memory: two launches with the row of
// silu(gate) between them took 4.8 + 3.9 us for 14336 columns in bfloat16 and 14.6 + 11.6 for 512 rows, this one 4.0 and 10.2 (5.7
// TB/s).  A thread has 16 bytes where the rows are made of those, else an element.
template <typename T, int kPer>
__global__ void __launch_bounds__(64) gated_silu_kernel(const T* gate_up, T* out, int64_t rows, int64_t inter, int64_t row_stride) {
    struct alignas(sizeof(T) * kPer) Piece {
        T v[kPer];
    };
    const int64_t col = ((int64_t)blockIdx.x * 64 + threadIdx.x) * kPer;
    if (col >= inter) return;
    for (int64_t row = blockIdx.y; row < rows; row += gridDim.y) {
        const T* from = gate_up + row * row_stride + col;
        const Piece gate = *reinterpret_cast<const Piece*>(from), up = *reinterpret_cast<const Piece*>(from + inter);
        Piece o;
#pragma unroll
        for (int i = 0; i < kPer; i++) o.v[i] = gated(gate.v[i], up.v[i]);
        *reinterpret_cast<Piece*>(out + row * inter + col) = o;
    }
}

template <typename T>
int run_gated(const void* gate_up, void* out, int64_t rows, int64_t inter, int64_t row_stride, hipStream_t stream) {
    constexpr int kPer = 16 / (int)sizeof(T);
    const bool pieces = inter % kPer == 0 && row_stride % kPer == 0 &&
                        ((reinterpret_cast<uintptr_t>(gate_up) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    const int64_t cols = pieces ? inter / kPer : inter, blocks = (cols + 63) / 64;
    if (blocks > 0x7fffffff) return CKV_ERR_UNSUPPORTED;
    const dim3 grid((unsigned)blocks, (unsigned)(rows < 65535 ? rows : 65535));
    if (pieces)
        hipLaunchKernelGGL((gated_silu_kernel<T, kPer>), grid, dim3(64), 0, stream, (const T*)gate_up, (T*)out, rows, inter, row_stride);
    else
        hipLaunchKernelGGL((gated_silu_kernel<T, 1>), grid, dim3(64), 0, stream, (const T*)gate_up, (T*)out, rows, inter, row_stride);
    CKV_HIP_TRY(hipGetLastError());
    return CKV_OK;
}

}  // namespace
}  // namespace ckv

extern "C" int ckv_gated_silu(const void* gate_up, void* out, int64_t rows, int64_t inter, int64_t row_stride, int32_t dtype, void* stream_) {
    using namespace ckv;
    if (rows < 0 || inter <= 0 || row_stride < 2 * inter) return CKV_ERR_SHAPE;
    if (dtype != CKV_F32 && dtype != CKV_F16 && dtype != CKV_BF16) return CKV_ERR_DTYPE;
    if (rows == 0) return CKV_OK;
    if (!gate_up || !out) return CKV_ERR_NULL;
    hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
    switch (dtype) {
        case CKV_F32: return run_gated<float>(gate_up, out, rows, inter, row_stride, stream);
        case CKV_F16: return run_gated<__half>(gate_up, out, rows, inter, row_stride, stream);
        default: return run_gated<__hip_bfloat16>(gate_up, out, rows, inter, row_stride, stream);
    }
}
