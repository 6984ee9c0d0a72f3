// Activation / weight quantizers for gfx950.
//
// One workgroup per row.  Each thread keeps its slice of the row in registers
// (CHUNKS x 8 bf16 = CHUNKS 128-bit loads), so the row is read from HBM once:
// pass 1 reduces |x| to the row maximum across the wavefront (cross-lane
// shuffles) and then across wavefronts through LDS; pass 2 divides, converts to
// e4m3fn and stores 8 codes per 64-bit store.
#include "fp8_device.h"
#include "launch.h"
#include "quant_device.h"

namespace phyai {

template <int THREADS>
__device__ __forceinline__ uint32_t block_max_u32(uint32_t v, uint32_t* smem) {
    v = wave_max_u32(v);
    if constexpr (THREADS > kWave) {
        constexpr int NW = THREADS / kWave;
        const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
        if (lane == 0) smem[wave] = v;
        __syncthreads();
        uint32_t r = smem[0];
#pragma unroll
        for (int i = 1; i < NW; ++i) r = smem[i] > r ? smem[i] : r;
        v = r;
    }
    return v;
}

// A tensor that is far larger than the caches and read once is loaded without keeping its lines
// in L2 (from 100 MB, long rows only: 13056 x 16384 119.9 -> 111.9 us; at 6528 x 2048 it would
// cost 10 %).  The codes are stored normally: streaming them out as well makes this kernel
// faster (816 x 16384: 12.0 -> 9.2 us) but the GEMM that reads them next slower by more.
// Same box, alternating builds.
__device__ __forceinline__ uint4 nt_load16(const uint16_t* p) {
    const v4i v = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(p));
    return make_uint4((uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]);
}

template <int THREADS, int CHUNKS, int MODE, bool STREAM_IN>
__global__ __launch_bounds__(THREADS) void quant_rows_reg_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, int K, int ldq, uint8_t* __restrict__ xq,
    float* __restrict__ scale) {
    __shared__ uint32_t smem[THREADS / kWave];
    const int64_t row = blockIdx.x;
    const uint16_t* xr = x + row * ldx;
    uint4 v[CHUNKS];
    uint32_t m = 0;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int k = (c * THREADS + threadIdx.x) * 8;
        v[c] = make_uint4(0, 0, 0, 0);
        if (k < K) v[c] = STREAM_IN ? nt_load16(xr + k) : *reinterpret_cast<const uint4*>(xr + k);
        m = absmax8(v[c], m);
    }
    m = block_max_u32<THREADS>(m, smem);
    const float s = scale_from_amax_bits<MODE>(m);
    if (threadIdx.x == 0) scale[row] = s;
    const RowDivisor d = make_divisor<MODE>(s);
    uint8_t* qr = xq + row * (int64_t)ldq;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int k = (c * THREADS + threadIdx.x) * 8;
        if (k < K) *reinterpret_cast<uint2*>(qr + k) = encode8<MODE>(v[c], d);
        else if (MODE != QUANT_WEIGHT && k < ldq) *reinterpret_cast<uint2*>(qr + k) = make_uint2(0, 0);   // (weights have no padding)
    }
}

// Rows too long for the register-resident form: two passes over global memory
// (the second one hits L2).
template <int MODE>
__global__ __launch_bounds__(256) void quant_rows_loop_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, int K, int ldq, uint8_t* __restrict__ xq,
    float* __restrict__ scale) {
    __shared__ uint32_t smem[256 / kWave];
    const int64_t row = blockIdx.x;
    const uint16_t* xr = x + row * ldx;
    uint32_t m = 0;
    for (int k = threadIdx.x * 8; k < K; k += 256 * 8)
        m = absmax8(*reinterpret_cast<const uint4*>(xr + k), m);
    m = block_max_u32<256>(m, smem);
    const float s = scale_from_amax_bits<MODE>(m);
    if (threadIdx.x == 0) scale[row] = s;
    const RowDivisor d = make_divisor<MODE>(s);
    uint8_t* qr = xq + row * (int64_t)ldq;
    for (int k = threadIdx.x * 8; k < ldq; k += 256 * 8)
        *reinterpret_cast<uint2*>(qr + k) = k < K ? encode8<MODE>(*reinterpret_cast<const uint4*>(xr + k), d) : make_uint2(0, 0);
}

// Static per-tensor quantizer: clamp(fp32(x)/s, +-448) -> e4m3fn, NaN elements to NaN codes as torch.clamp lets them
// through.  Bound by its bytes: a wavefront takes 2048 elements of one row, four loads in flight per lane and no index
// division (one per 8 elements took as long as the bytes: the linear 10143 x 512 x 2944 41.7 -> 34.5 us with both).
__global__ __launch_bounds__(256) void quant_static_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, int M, int K, int ldq, const float* __restrict__ input_scale, uint8_t* __restrict__ xq) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= M) return;
    const uint16_t* xr = x + row * ldx;
    uint8_t* qr = xq + row * (int64_t)ldq;
    const StaticDivisor d = make_static_divisor(*input_scale);
    uint4 v[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int k = blockIdx.y * 2048 + (c * 64 + lane) * 8;
        if (k < K) v[c] = *reinterpret_cast<const uint4*>(xr + k);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int k = blockIdx.y * 2048 + (c * 64 + lane) * 8;
        if (k < K)
            *reinterpret_cast<uint2*>(qr + k) =
                __builtin_expect(!d.fast || any_nan_or_inf(v[c]), 0) ? encode8_static_exact(v[c], d.s) : encode8_static_fast(v[c], d);
        else if (k < ldq) *reinterpret_cast<uint2*>(qr + k) = make_uint2(0, 0);
    }
}

__global__ __launch_bounds__(256) void debug_cast_kernel(const float* __restrict__ v, int64_t n,
                                                         uint8_t* __restrict__ codes) {
    for (int64_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        codes[i] = (uint8_t)(e4m3_pack2(v[i], 0.0f) & 0xFFu);
}

template <int MODE>
static int launch_quant_rows(const void* x, int64_t M, int64_t K, int64_t ld, void* xq, int64_t ldq,
                             float* scale, hipStream_t st) {
    if (M == 0) return 0;
    const uint16_t* xp = static_cast<const uint16_t*>(x);
    uint8_t* qp = static_cast<uint8_t*>(xq);
    const dim3 grid((unsigned)M);
    const int k = (int)K;
    const bool stream_in = M * K * 2 >= ((int64_t)100 << 20);   // only long rows get that large in practice
#define PHYAI_QL(T, C)                                                                                             \
    do {                                                                                                           \
        if (T * C >= 1024 && stream_in)                                                                            \
            hipLaunchKernelGGL((quant_rows_reg_kernel<T, C, MODE, (T * C >= 1024)>), grid, dim3(T), 0, st, xp, ld, k, (int)ldq, qp, scale); \
        else                                                                                                       \
            hipLaunchKernelGGL((quant_rows_reg_kernel<T, C, MODE, false>), grid, dim3(T), 0, st, xp, ld, k, (int)ldq, qp, scale);   \
    } while (0)
    // One load per thread where there are few rows: a row is then one trip to memory and a reduction.  Many rows fill the chip
    // either way, and two wavefronts wait for each other less than four (us, 256 threads / 128: 816 x 2048 3.25 / 3.28, 3264 x 2048
    // 6.2 / 5.9, 13056 x 2048 13.9 / 13.4).  Long rows: 512 threads instead of 256 (50 x 16384 3.9 / 3.5, 816 x 16384
    // 9.5 / 9.3, 3264 x 16384 25.7 - 27.4 / 24.3 - 27.0, 13056 x 16384 95.0 / 94.1); 1024 are
    // slower again with many of them (58.4 at 13056 x 8192, where 512 take 49).  Up to K = 5632 for few rows only (50 x 8192 2.8 / 2.6, 256 x
    // 5120 3.15 / 2.98, 777 x 5504 4.4 / 4.2): with many the second half of a workgroup waits for a short rest of the row (1600 x
    // 4304 5.7 / 6.1, 3264 x 4608 9.3 / 9.4, 4800 x 4608 13.9 / 14.5, 8000 x 5120 22.9 / 23.6; level at K = 5632, and beyond, where it
    // has half a row, 1600 x 7168 7.55 / 7.17, 4800 x 8064 22.6 / 22.1, 13056 x 8192 51.8 / 51.2).
    if (K <= 512) PHYAI_QL(64, 1);
    else if (K <= 1024) PHYAI_QL(128, 1);
    else if (K <= 2048 && M >= 2048) PHYAI_QL(128, 2);
    else if (K <= 2048) PHYAI_QL(256, 1);
    else if (K <= 4096) PHYAI_QL(256, 2);
    else if (K <= 5632 && M >= 1536) PHYAI_QL(256, 4);
    else if (K <= 8192) PHYAI_QL(512, 2);
    else if (K <= 16384) PHYAI_QL(512, 4);
    else if (K <= 32768) PHYAI_QL(256, 16);
    else hipLaunchKernelGGL((quant_rows_loop_kernel<MODE>), grid, dim3(256), 0, st, xp, ld, k, (int)ldq, qp, scale);
#undef PHYAI_QL
    return 0;
}

int launch_quant_rowwise(const void* x, int64_t M, int64_t K, int64_t ldx, void* xq, int64_t ldq, float* xs,
                         hipStream_t st) {
    return launch_quant_rows<QUANT_ACT_DYNAMIC>(x, M, K, ldx, xq, ldq, xs, st);
}
int launch_weight_quant(const void* w, int64_t N, int64_t K, int64_t ldw, void* wq, float* ws,
                        hipStream_t st) {
    return launch_quant_rows<QUANT_WEIGHT>(w, N, K, ldw, wq, K, ws, st);
}
// ---- RMSNorm / adaptive RMSNorm + quantizer ----------------------------------------------
template <int THREADS>
__device__ __forceinline__ float block_sum_f32(float v, float* smem) {
    v = wave_sum_f32(v);
    if constexpr (THREADS > kWave) {
        constexpr int NW = THREADS / kWave;
        const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
        if (lane == 0) smem[wave] = v;
        __syncthreads();
        float r = smem[0];
#pragma unroll
        for (int i = 1; i < NW; ++i) r += smem[i];
        v = r;
    }
    return v;
}

__device__ __forceinline__ void unpack8(uint4 q, float* f) {
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[2 * i] = bf16_bits_to_f32(w[i] & 0xFFFFu);
        f[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
    }
}

// Eight values rounded to bf16: four hardware converts instead of some fifty instructions.  They differ from
// f32_to_bf16_bits in the bits of a NaN only, so where a NaN may be among them that form is taken.
__device__ __forceinline__ uint4 round8_bf16(const float* o) {
    uint4 b = make_uint4(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]), pack_bf16x2(o[4], o[5]), pack_bf16x2(o[6], o[7]));
    if (__builtin_expect(any_nan_or_inf(b), 0)) {
        b.x = f32_to_bf16_bits(o[0]) | (f32_to_bf16_bits(o[1]) << 16);
        b.y = f32_to_bf16_bits(o[2]) | (f32_to_bf16_bits(o[3]) << 16);
        b.z = f32_to_bf16_bits(o[4]) | (f32_to_bf16_bits(o[5]) << 16);
        b.w = f32_to_bf16_bits(o[6]) | (f32_to_bf16_bits(o[7]) << 16);
    }
    return b;
}

// One workgroup per row, the row in registers: sum of squares (fp32), normalise, affine, round to
// bf16 - the tensor the reference's norm kernel would have written - and, on those bf16 values,
// the per-token quantizer (row absmax, scale, codes) of quant_rows_reg_kernel.  Its arithmetic takes as long as its bytes: the
// affine part is asked for together with the row, the rows per modulation row are divided by in 32 bits, and values are rounded by
// the hardware (us, before / with all three, plain and adaptive: 3264 x 2048 8.9 / 8.1 and 9.8 / 8.8, 13056 x 2048 21.5 / 18.8 and 23.5 /
// 21.2, 4800 x 4096 16.3 / 13.4 and 16.9 / 14.6, 816 x 2048 4.4 / 4.2 and 4.7 / 4.4).
template <int THREADS, int CHUNKS, bool ADAPTIVE>
__global__ __launch_bounds__(THREADS) void norm_quant_kernel(
    const uint16_t* __restrict__ a_x, int64_t a_ldx, int a_D, int a_group, const uint16_t* __restrict__ a_mod,
    int64_t a_ld_mod, const uint16_t* __restrict__ a_weight, float a_eps, int a_gemma, uint8_t* __restrict__ a_xq,
    float* __restrict__ a_scale, uint16_t* __restrict__ a_out, int64_t a_ldo, uint16_t* __restrict__ a_gate,
    int64_t a_ld_gate, int64_t a_ldq) {
    // scalar arguments in the order the kernel needs them (the first 16 dwords are preloaded)
    NormQuantArgs p;
    p.x = a_x; p.ldx = a_ldx; p.D = a_D; p.eps = a_eps; p.weight = a_weight; p.gemma = a_gemma; p.mod = a_mod;
    p.ld_mod = a_ld_mod; p.group = a_group; p.out = a_out; p.ldo = a_ldo; p.gate = a_gate; p.ld_gate = a_ld_gate;
    p.xq = a_xq; p.ldq = a_ldq; p.scale = a_scale;
    __shared__ float ssum[THREADS / kWave];
    __shared__ uint32_t smax[THREADS / kWave];
    const int64_t row = blockIdx.x;
    const uint16_t* xr = p.x + row * p.ldx;
    const int64_t mrow = ADAPTIVE ? (int64_t)((uint32_t)row / (uint32_t)p.group) : 0;   // (M < 2^31)
    const uint16_t* mr = ADAPTIVE ? p.mod + mrow * p.ld_mod : nullptr;
    float xf[CHUNKS][8];
    uint4 affine[CHUNKS][ADAPTIVE ? 2 : 1];   // weight, or scale and shift: asked for with the row, not after its sum is there
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int k = (c * THREADS + threadIdx.x) * 8;
        uint4 v = make_uint4(0, 0, 0, 0);
        if (k < p.D) {
            v = *reinterpret_cast<const uint4*>(xr + k);
            affine[c][0] = *reinterpret_cast<const uint4*>((ADAPTIVE ? mr : p.weight) + k);
            if constexpr (ADAPTIVE) affine[c][1] = *reinterpret_cast<const uint4*>(mr + p.D + k);
        }
        unpack8(v, xf[c]);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += xf[c][e] * xf[c][e];
    }
    ss = block_sum_f32<THREADS>(ss, ssum);
    const float rstd = 1.0f / sqrtf(ss / (float)p.D + p.eps);

    uint4 ob[CHUNKS];
    uint32_t m = 0;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int k = (c * THREADS + threadIdx.x) * 8;
        ob[c] = make_uint4(0, 0, 0, 0);
        if (k < p.D) {
            float o[8];
            if constexpr (ADAPTIVE) {
                float sc[8], sh[8];
                unpack8(affine[c][0], sc);
                unpack8(affine[c][1], sh);
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = (xf[c][e] * rstd) * (1.0f + sc[e]) + sh[e];
                if (p.gate != nullptr && (uint32_t)row == (uint32_t)mrow * (uint32_t)p.group)
                    *reinterpret_cast<uint4*>(p.gate + mrow * p.ld_gate + k) =
                        *reinterpret_cast<const uint4*>(mr + 2 * p.D + k);
            } else {
                float w[8];
                unpack8(affine[c][0], w);
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = (xf[c][e] * rstd) * (p.gemma ? w[e] + 1.0f : w[e]);
            }
            ob[c] = round8_bf16(o);
            if (p.out != nullptr) *reinterpret_cast<uint4*>(p.out + row * p.ldo + k) = ob[c];
        }
        m = absmax8(ob[c], m);
    }
    if (p.xq == nullptr) return;
    m = block_max_u32<THREADS>(m, smax);
    const float s = scale_from_amax_bits<QUANT_ACT_DYNAMIC>(m);
    if (threadIdx.x == 0) p.scale[row] = s;
    const RowDivisor d = make_divisor<QUANT_ACT_DYNAMIC>(s);
    uint8_t* qr = p.xq + row * p.ldq;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int k = (c * THREADS + threadIdx.x) * 8;
        if (k < p.D) *reinterpret_cast<uint2*>(qr + k) = encode8<QUANT_ACT_DYNAMIC>(ob[c], d);
        else if (k < p.ldq) *reinterpret_cast<uint2*>(qr + k) = make_uint2(0, 0);
    }
}

// Rows too long for registers (D > 8192, the reference's two-pass kernels): the row is read again
// for every pass - sum of squares, then the bf16 result and its absmax, then the codes.
template <bool ADAPTIVE>
__global__ __launch_bounds__(256) void norm_quant_loop_kernel(
    const uint16_t* __restrict__ a_x, int64_t a_ldx, int a_D, int a_group, const uint16_t* __restrict__ a_mod,
    int64_t a_ld_mod, const uint16_t* __restrict__ a_weight, float a_eps, int a_gemma, uint8_t* __restrict__ a_xq,
    float* __restrict__ a_scale, uint16_t* __restrict__ a_out, int64_t a_ldo, uint16_t* __restrict__ a_gate,
    int64_t a_ld_gate, int64_t a_ldq) {
    // scalar arguments in the order the kernel needs them (the first 16 dwords are preloaded)
    NormQuantArgs p;
    p.x = a_x; p.ldx = a_ldx; p.D = a_D; p.eps = a_eps; p.weight = a_weight; p.gemma = a_gemma; p.mod = a_mod;
    p.ld_mod = a_ld_mod; p.group = a_group; p.out = a_out; p.ldo = a_ldo; p.gate = a_gate; p.ld_gate = a_ld_gate;
    p.xq = a_xq; p.ldq = a_ldq; p.scale = a_scale;
    __shared__ float ssum[256 / kWave];
    __shared__ uint32_t smax[256 / kWave];
    const int64_t row = blockIdx.x;
    const uint16_t* xr = p.x + row * p.ldx;
    float ss = 0.f;
    for (int k = threadIdx.x * 8; k < p.D; k += 256 * 8) {
        float f[8];
        unpack8(*reinterpret_cast<const uint4*>(xr + k), f);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += f[e] * f[e];
    }
    ss = block_sum_f32<256>(ss, ssum);
    const float rstd = 1.0f / sqrtf(ss / (float)p.D + p.eps);
    const int64_t mrow = ADAPTIVE ? row / p.group : 0;
    const uint16_t* mr = ADAPTIVE ? p.mod + mrow * p.ld_mod : nullptr;
    auto result8 = [&](int k) -> uint4 {
        float f[8], o[8];
        unpack8(*reinterpret_cast<const uint4*>(xr + k), f);
        if constexpr (ADAPTIVE) {
            float sc[8], sh[8];
            unpack8(*reinterpret_cast<const uint4*>(mr + k), sc);
            unpack8(*reinterpret_cast<const uint4*>(mr + p.D + k), sh);
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = (f[e] * rstd) * (1.0f + sc[e]) + sh[e];
        } else {
            float w[8];
            unpack8(*reinterpret_cast<const uint4*>(p.weight + k), w);
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = (f[e] * rstd) * (p.gemma ? w[e] + 1.0f : w[e]);
        }
        return round8_bf16(o);
    };
    uint32_t m = 0;
    for (int k = threadIdx.x * 8; k < p.D; k += 256 * 8) {
        const uint4 b = result8(k);
        if (p.out != nullptr) *reinterpret_cast<uint4*>(p.out + row * p.ldo + k) = b;
        if constexpr (ADAPTIVE) {
            if (p.gate != nullptr && row % p.group == 0)
                *reinterpret_cast<uint4*>(p.gate + mrow * p.ld_gate + k) = *reinterpret_cast<const uint4*>(mr + 2 * p.D + k);
        }
        m = absmax8(b, m);
    }
    if (p.xq == nullptr) return;
    m = block_max_u32<256>(m, smax);
    const float s = scale_from_amax_bits<QUANT_ACT_DYNAMIC>(m);
    if (threadIdx.x == 0) p.scale[row] = s;
    const RowDivisor d = make_divisor<QUANT_ACT_DYNAMIC>(s);
    uint8_t* qr = p.xq + row * p.ldq;
    for (int k = threadIdx.x * 8; k < p.ldq; k += 256 * 8)
        *reinterpret_cast<uint2*>(qr + k) = k < p.D ? encode8<QUANT_ACT_DYNAMIC>(result8(k), d) : make_uint2(0, 0);
}

template <bool ADAPTIVE>
static int launch_norm_quant_t(const NormQuantArgs& a, int64_t M, hipStream_t st) {
    const dim3 grid((unsigned)M);
#define PHYAI_NQ_ARGS a.x, a.ldx, a.D, a.group, a.mod, a.ld_mod, a.weight, a.eps, a.gemma, a.xq, a.scale, a.out, a.ldo, a.gate, a.ld_gate, a.ldq
#define PHYAI_NQ(T, C) hipLaunchKernelGGL((norm_quant_kernel<T, C, ADAPTIVE>), grid, dim3(T), 0, st, PHYAI_NQ_ARGS)
    if (a.D <= 512) PHYAI_NQ(64, 1);
    else if (a.D <= 1024) PHYAI_NQ(128, 1);
    else if (a.D <= 2048) PHYAI_NQ(256, 1);
    else if (a.D <= 4096) PHYAI_NQ(256, 2);
    else if (a.D <= 8192) PHYAI_NQ(256, 4);
    else hipLaunchKernelGGL((norm_quant_loop_kernel<ADAPTIVE>), grid, dim3(256), 0, st, PHYAI_NQ_ARGS);
#undef PHYAI_NQ
#undef PHYAI_NQ_ARGS
    return 0;
}

int launch_norm_quant(const NormQuantArgs& a, int64_t M, bool adaptive, hipStream_t st) {
    if (M == 0) return 0;
    return adaptive ? launch_norm_quant_t<true>(a, M, st) : launch_norm_quant_t<false>(a, M, st);
}

int launch_quant_static(const void* x, int64_t M, int64_t K, int64_t ldx, const float* input_scale,
                        void* xq, int64_t ldq, hipStream_t st) {
    if (M == 0) return 0;
    // (M < 2^31; the grid's x covers the rows)
    hipLaunchKernelGGL(quant_static_kernel, dim3((unsigned)((M + 3) / 4), (unsigned)((K + 2047) / 2048)), dim3(256), 0, st,
                       static_cast<const uint16_t*>(x), ldx, (int)M, (int)K, (int)ldq, input_scale, static_cast<uint8_t*>(xq));
    return 0;
}
int launch_debug_cast(const float* v, int64_t n, void* codes, hipStream_t st) {
    if (n == 0) return 0;
    int blocks = (int)((n + 255) / 256);
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(debug_cast_kernel, dim3(blocks), dim3(256), 0, st, v, n,
                       static_cast<uint8_t*>(codes));
    return 0;
}

}  // namespace phyai
