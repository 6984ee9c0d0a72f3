// Re-lays a row-major fp8 weight matrix into MFMA operand order (weight_layout.h), once per layer
// after loading.  One thread moves CHUNKS 16-byte chunks; consecutive threads write consecutive chunks
// of the destination, so the writes are contiguous and the reads are 16-byte pieces of 16
// neighbouring rows.  Bound by bytes (6.8 TB/s).  Two chunks where the source is a second matrix below 20 MB, whose workgroups
// would be few (us, start of a load with the copy in front of it, 1 / 2 / 4: 4096 x 2688 15.2 / 11.1 / 14.8, 5504 x 2688 16.8 / 14.0 / 17.8,
// 8192 x 2048 18.3 / 15.6 / 18.9), otherwise four (2 / 4: 14336 x 2048 23.6 / 24.1 with the copy; without one 13.7 / 13.2, 10240 x
// 2048 8.31 / 8.26, 11776 x 2048 gated 11.6 / 10.6, 2048 x 16384 14.0 / 13.6, 32768 x 2048 26.1 / 24.9, 16384 x 8192 level), as where
// large matrices are re-laid by halves (a whole load of 16384 x 2048 39.6 / 37.4, 24576 x 2048 55.7 / 54.0, 32768 x 2048 72.6 /
// 71.9).
//
// A plain matrix is re-laid in place: unit u (16 rows x K) holds the same bytes in both orders, so a workgroup takes them
// into its registers, waits for everyone and writes them back - half the bytes of re-laying into a second matrix and
// copying that back.  A gated unit takes rows from both halves of the matrix and goes through a second one, three quarters of
// it where the matrix is large (phyai_host_relay_gated).
#include <hip/hip_runtime.h>

#include "fp8_device.h"
#include "host_entry.h"
#include "launch.h"
#include "weight_layout.h"

namespace phyai {

constexpr int64_t kFewChunks = 20 << 20;   // bytes of a matrix below which a thread moves two chunks, not four

// The launch's own status.  hipGetLastError() may return an older error of the thread, and a caller that went another way for
// it would re-lay the matrix a second time.
template <class T> struct AsIs { typedef T type; };
template <class... P>
static bool launched(void (*kernel)(P...), unsigned blocks, unsigned threads, hipStream_t st, typename AsIs<P>::type... a) {
    void* args[] = {&a...};
    return hipLaunchKernel(reinterpret_cast<const void*>(kernel), dim3(blocks), dim3(threads), args, 0, st) == hipSuccess;
}

// Chunks [first * K, first * K + chunks) of the destination, i.e. units from `first` on (a unit is K chunks).  Gated: gate rows
// from `gate`, up rows from `up`, both counted from column 0; plain: rows of the matrix at `gate`.
template <int CHUNKS>
__global__ __launch_bounds__(256) void weight_to_operand_order_kernel(const v4i* gate, const v4i* up, v4i* out,
                                                                      uint32_t first, uint32_t K, int gated, uint32_t chunks) {
    const uint32_t steps = K >> 7;
    v4i v[CHUNKS];
#pragma unroll
    for (int j = 0; j < CHUNKS; ++j) {
        const uint32_t t = blockIdx.x * (256 * CHUNKS) + j * 256 + threadIdx.x, i = t < chunks ? t : chunks - 1;
        const uint32_t r = i & 15, c = (i >> 4) & 7, us = i >> 7;   // us = u * steps + s
        const uint32_t u = first + us / steps, s = us % steps;
        const uint32_t row = gated ? 8 * u + 2 * (r >> 2) + (r & 1) : 16 * u + r;
        v[j] = (gated && (r & 2) ? up : gate)[(size_t)row * (K >> 4) + s * 8 + c];
    }
#pragma unroll
    for (int j = 0; j < CHUNKS; ++j) {
        const uint32_t i = blockIdx.x * (256 * CHUNKS) + j * 256 + threadIdx.x;
        if (i < chunks) out[(size_t)first * K + i] = v[j];
    }
}

// The up half of a gated matrix, `half` chunks from chunk `half` on, and its first `kept` chunks behind it.
__global__ __launch_bounds__(256) void weight_save_kernel(const v4i* __restrict__ w, v4i* __restrict__ saved, uint32_t half, uint32_t kept) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t i = blockIdx.x * 1024 + j * 256 + threadIdx.x;
        if (i < half + kept) saved[i] = w[i < half ? half + i : i - half];
    }
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
    const unsigned units = (unsigned)(N / 16);
    v4i* p = static_cast<v4i*>(w);
    const uint32_t k = (uint32_t)K;
    bool ok;
    if (K <= 1024) ok = launched(weight_to_operand_order_inplace_kernel<1>, units, 1024, st, p, k);
    else if (K <= 2048) ok = launched(weight_to_operand_order_inplace_kernel<2>, units, 1024, st, p, k);
    else if (K <= 4096) ok = launched(weight_to_operand_order_inplace_kernel<4>, units, 1024, st, p, k);
    else if (K <= 8192) ok = launched(weight_to_operand_order_inplace_kernel<8>, units, 1024, st, p, k);
    else if (K <= 16384) ok = launched(weight_to_operand_order_inplace_kernel<16>, units, 1024, st, p, k);
    else return -2;
    return ok ? 0 : -3;
}

template <int CHUNKS>
static bool launch_units(const v4i* gate, const v4i* up, v4i* out, uint32_t first, uint32_t end, uint32_t K, int gated, hipStream_t st) {
    const uint32_t chunks = (end - first) * K;
    return launched(weight_to_operand_order_kernel<CHUNKS>, (chunks + 256 * CHUNKS - 1) / (256 * CHUNKS), 256, st, gate, up, out, first, K, gated, chunks);
}

int launch_weight_to_operand_order(const void* w, int64_t N, int64_t K, int gated, void* out, hipStream_t st) {
    if (N * K > 0x7FFFFFFFll) return -2;
    const v4i* rows = static_cast<const v4i*>(w);
    const auto launch = N * K < kFewChunks ? launch_units<2> : launch_units<4>;
    return launch(rows, rows + N / 2 * K / 16, static_cast<v4i*>(out), 0, (uint32_t)(N / 16), (uint32_t)K, gated, st) ? 0 : -3;
}

}  // namespace phyai

// The gated form in place, for the host extension beside this library (no part of the C interface): w as
// phyai_fp8_weight_to_operand_order() takes it, scratch of 3/4 N * K bytes.  -2: not for this form or not launched, the matrix is
// as it was; -3: half of it is re-laid.
//
// Saving the whole matrix and re-laying from there moves every byte four times.  The upper half of the units needs less: it
// overwrites the up half of the matrix and reads the upper gate rows, which are still in place.  So the up half and the
// lower gate rows are saved, the upper units go first and the lower ones, all of whose rows are saved, after them: 3.5 times,
// for one more launch.  us, event-timed in a stream, whole copy / this: 32768 x 2048 43.8 / 39.4, 4096 x 16384 43.3 / 39.6, 32768 x 1024
// 26.5 / 23.6, 16384 x 2048 25.4 / 23.3; at 10 and 17 MB between 4 % ahead and 2 % behind, so from 32 MB on.  (Going on by
// halves saves bytes and loses more in launches: 42.6 with one more, 44.9 with two.)
extern "C" int phyai_host_relay_gated(void* w, int64_t N, int64_t K, void* scratch, void* stream) {
    using namespace phyai;
    if (N <= 0 || K <= 0 || N % 32 != 0 || K % 128 != 0 || N > 0x7FFFFFFFll || K > 0x7FFFFFFFll) return -2;
    if (N * K < (1ll << 25) || N * K > 0x7FFFFFFFll || ((reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(scratch)) & 15) != 0) return -2;
    hipStream_t st = static_cast<hipStream_t>(stream);
    v4i *m = static_cast<v4i*>(w), *up = static_cast<v4i*>(scratch);
    const uint32_t k = (uint32_t)K, units = (uint32_t)(N / 16), half = (uint32_t)(N / 2 * K / 16);
    const uint32_t middle = units / 2, kept = middle * 8 * (k / 16);   // (N % 32 == 0: units is even)
    if (!launched(weight_save_kernel, (half + kept + 1023) / 1024, 256, st, m, up, half, kept)) return -2;
    if (!launch_units<4>(m, up, m, middle, units, k, 1, st)) return -2;
    return launch_units<4>(up + half, up, m, 0, middle, k, 1, st) ? 0 : -3;
}
