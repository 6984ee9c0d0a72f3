// Re-lays a row-major fp8 weight matrix into MFMA operand order (weight_layout.h), once per layer
// after loading.  One thread moves one 16-byte chunk; consecutive threads write consecutive chunks
// of the destination, so the writes are contiguous and the reads are 16-byte pieces of 16
// neighbouring rows.
//
// A plain matrix is re-laid in place: unit u (16 rows x K) holds the same bytes in both orders, so a workgroup takes them
// into its registers, waits for everyone and writes them back - half the bytes of re-laying into a second matrix and
// copying that back.  A gated unit takes rows from both halves of the matrix, so that form stays out of place.
#include <hip/hip_runtime.h>

#include "fp8_device.h"
#include "launch.h"
#include "weight_layout.h"

namespace phyai {

__global__ __launch_bounds__(256) void weight_to_operand_order_kernel(const uint4* __restrict__ w, uint4* __restrict__ out,
                                                                      uint32_t N, uint32_t K, int gated, uint64_t chunks) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;   // destination chunk
    if (i >= chunks) return;
    const uint32_t steps = K >> 7;
    const uint32_t r = (uint32_t)(i & 15), c = (uint32_t)((i >> 4) & 7);
    const uint64_t us = i >> 7;                                     // u * steps + s
    const uint32_t u = (uint32_t)(us / steps), s = (uint32_t)(us % steps);
    uint32_t row;
    if (gated) row = ((r >> 1) & 1) * (N >> 1) + 8 * u + 2 * (r >> 2) + (r & 1);
    else row = 16 * u + r;
    out[i] = w[((uint64_t)row * K + ((uint64_t)s << 7) + (c << 4)) >> 4];
}

// CHUNKS 16-byte chunks per thread: K <= 1024 * CHUNKS.
template <int CHUNKS>
__global__ __launch_bounds__(1024) void weight_to_operand_order_inplace_kernel(v4i* __restrict__ w, uint32_t K) {
    v4i* unit = w + (size_t)blockIdx.x * K;   // 16 rows of K / 16 chunks
    v4i v[CHUNKS];
#pragma unroll
    for (int j = 0; j < CHUNKS; ++j) {
        const uint32_t t = j * 1024 + threadIdx.x, i = t < K ? t : K - 1;   // destination chunk: K step i / 128, chunk (i / 16) % 8 of row i % 16
        v[j] = unit[(i & 15) * (K >> 4) + (i >> 7) * 8 + ((i >> 4) & 7)];
    }
    // every chunk is in a register before one is overwritten: a barrier alone would let loads be in flight across it
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
#pragma unroll
    for (int j = 0; j < CHUNKS; ++j) {
        const uint32_t i = j * 1024 + threadIdx.x;
        if (i < K) unit[i] = v[j];
    }
}

int launch_weight_to_operand_order_inplace(void* w, int64_t N, int64_t K, hipStream_t st) {
    const dim3 grid((unsigned)(N / 16));
    v4i* p = static_cast<v4i*>(w);
    const uint32_t k = (uint32_t)K;
    if (K <= 1024) hipLaunchKernelGGL((weight_to_operand_order_inplace_kernel<1>), grid, dim3(1024), 0, st, p, k);
    else if (K <= 2048) hipLaunchKernelGGL((weight_to_operand_order_inplace_kernel<2>), grid, dim3(1024), 0, st, p, k);
    else if (K <= 4096) hipLaunchKernelGGL((weight_to_operand_order_inplace_kernel<4>), grid, dim3(1024), 0, st, p, k);
    else if (K <= 8192) hipLaunchKernelGGL((weight_to_operand_order_inplace_kernel<8>), grid, dim3(1024), 0, st, p, k);
    else if (K <= 16384) hipLaunchKernelGGL((weight_to_operand_order_inplace_kernel<16>), grid, dim3(1024), 0, st, p, k);
    else return -2;
    return 0;
}

int launch_weight_to_operand_order(const void* w, int64_t N, int64_t K, int gated, void* out, hipStream_t st) {
    const uint64_t chunks = (uint64_t)N * (uint64_t)K / 16;
    const uint64_t blocks = (chunks + 255) / 256;
    if (blocks > 0x7FFFFFFFull) return -2;
    hipLaunchKernelGGL(weight_to_operand_order_kernel, dim3((unsigned)blocks), dim3(256), 0, st,
                       static_cast<const uint4*>(w), static_cast<uint4*>(out), (uint32_t)N, (uint32_t)K, gated, chunks);
    return 0;
}

}  // namespace phyai
