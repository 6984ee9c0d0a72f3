// Small-M linear that quantizes its own rows, for what gemm_skinny_fused.hip does not take: K that is no multiple of
// 128, K up to 16384, activations with one static scale.  One launch instead of quantizer + GEMM where selfq_max_k says.
//
// What bounds these calls is the host: a launch costs it 3.3 us (2.5 us of it inside the runtime), and for a few token
// rows neither the quantizer nor the GEMM lasts as long.  So the quantizer's launch goes, at the price of every workgroup
// converting the rows it multiplies (4 or 8 rows x K, at most 2.7 us at K = 8192) beside the weights it streams.
//
//  * a workgroup (8 wavefronts) owns 16 NT weight rows x 4 RG token rows over the whole K; wavefront w takes the
//    128-byte K steps w, w + 8, ... as in the other weight-streaming kernels, so sums come out in the same order;
//  * the bf16 rows stay in registers from their arrival until their conversion (the row maximum needs all of K first):
//    128 registers per lane at K = 16384 with 8 rows, which leaves room for five K steps of weights in flight (selfq_window);
//  * weights go straight into registers in both layouts: operand order in 1 KB runs; row-major with 64 contiguous bytes
//    per row, which a CU pulls at 62 GB/s against 110 - enough beside the conversions, and it needs no LDS staging;
//  * WINDOW steps of weights are in flight ahead of the MFMAs, the first ones requested right behind the rows;
//  * K steps past the end and the ragged end of the last one multiply codes that are zero (their weight addresses are
//    clamped into the row), so the loop over the steps is straight-line code.
//
// SCALE: where the row scales come from - found here (own), handed over as row maxima by the kernel that wrote the rows
// (see AmaxOut in gemm_skinny_fused.hip), or one static scale for all rows.  Codes are those of the stand-alone
// quantizers, bit for bit.
#pragma once

#include "fp8_device.h"
#include "launch.h"
#include "quant_device.h"
#include "weight_layout.h"

namespace phyai {

constexpr int SELFQ_OWN = SELFQ_FROM_ROWS, SELFQ_HANDED = SELFQ_FROM_MAXIMA, SELFQ_STATIC = SELFQ_FROM_SCALAR;
constexpr int SQ_WAVES = 8, SQ_THREADS = SQ_WAVES * kWave;
// K steps per wavefront that exist as kernels (a step more than needed is work on zeros, so the list is dense)
constexpr int kSelfqSteps[] = {1, 2, 4, 6, 8, 12, 16};
constexpr int selfq_prev_steps(int steps) {
    int prev = 0;
    for (int s : kSelfqSteps)
        if (s < steps) prev = s;
    return prev;
}
// Longest K that a workgroup of 4 rg rows and nt weight tiles is taken for: where this one launch stops being ahead of
// quantizer + GEMM.  What decides is nt: the rows leave the fewer registers for weights in flight the longer K is
// (selfq_window: nt = 4 holds 3 steps at K = 6016, nt = 1 all 6), and a row-major tile is pulled in 64-byte pieces.
// Below, one launch / two launches in us, in a graph over 600 MB of weights and called eagerly (a launch costs the host
// 3.3 us), accepted where the product of the two ratios is below one - measured at M = 1 ... 128, N = 256 ... 16384:
//   operand order  nt = 1  15 x  1024 x 16384  10.3 / 14.3, 10.6 / 14.5     4 x 256 x 16384   7.2 /  9.4,  7.3 / 10.1
//                  nt = 2  15 x  4096 x 12160  13.7 / 14.1, 13.6 / 14.0    15 x 4096 x 16384 18.2 / 17.5, 18.1 / 17.4
//                  nt = 4  15 x  5552 x  4096 ratios 1.06, 0.91            15 x 5552 x  6016 12.9 / 11.6, 12.7 / 11.3
//                  nt = 8  M x N x 2048 one scale 1.02, 0.76               M x N x 2176 1.23, 1.01
//   row-major      nt = 1  15 x  1024 x  8192   8.8 /  9.1,  8.9 /  9.8    15 x 1024 x 10240 11.5 / 11.3, 11.6 / 11.4
//                  nt = 2, 8 rows  M x N x 3088 ratios 1.02, 0.76          15 x 4096 x  4224 10.5 /  8.3, 10.7 / 10.0
//                  nt = 4  M x N x 2032 ratios 0.86, 0.80                  15 x 5552 x  2064 10.1 /  7.8, 10.2 / 10.0
//                  nt = 8  M x N x 1040 ratios 1.05, 0.72 (one scale: 1552 1.07, 0.80)   M x N x 1168 1.29, 0.89
// With one scale 8 rows in operand order stop at 8192 (M x N x 10240 1.07, 1.01 with nt = 1): its quantizer is cheaper.
constexpr int selfq_max_k(int rg, int nt, bool operand, bool one_scale) {
    if (operand) return nt >= 8 ? 2048 : nt == 4 ? 4096 : rg == 1 ? 16384 : one_scale ? 8192 : nt == 2 ? 12288 : 16384;
    return nt >= 8 ? (one_scale ? 1600 : 1088) : nt == 4 ? 2048 : nt == 2 && rg == 2 ? 4096 : 8192;
}
// Shapes that exist as kernels: those that some K is taken for, less what gemm_skinny_fused.hip serves first - its own
// maxima up to K = 4096 in operand order, where only grids of four tiles beyond K = 2048 are left to this kernel, and
// handed-over maxima up to K = 1024 in operand order, where only grids of eight are.
constexpr bool selfq_exists(int rg, int nt, int steps, bool operand, int scale) {
    if (1024 * selfq_prev_steps(steps) >= selfq_max_k(rg, nt, operand, scale == SELFQ_STATIC)) return false;
    if (operand && scale == SELFQ_OWN && steps <= 4) return steps == 4 && nt == 4;
    if (operand && scale == SELFQ_HANDED && steps == 1) return nt == 8;
    return true;
}
// steps of weights in flight: what a wavefront's 256 registers leave beside the rows, the sums and about 80 for the
// conversions and addresses
constexpr int selfq_window(int rg, int nt, int steps) {
    const int w = (176 - steps * rg * 4 - nt * 6) / (nt * 8);
    return w < 1 ? 1 : (w < steps ? w : steps);
}

template <int RG, int NT, int STEPS, int EPI, bool OPERAND, int SCALE>
__global__ __launch_bounds__(SQ_THREADS) void gemm_fp8_selfq_kernel(
    const uint8_t* __restrict__ a_w, const uint8_t* __restrict__ a_x, int K, int N, int M, int ldx_bytes,
    const void* __restrict__ a_handed, int a_parts, const float* __restrict__ a_w_scale,
    const uint16_t* __restrict__ a_bias, uint16_t* __restrict__ a_out, int64_t a_ldo, const ResidualArgs a_res,
    uint16_t* __restrict__ a_amax_out) {
    constexpr bool GATED = epi_is_gated(EPI);
    constexpr int ROWS = 4 * RG, COLS_PER_TILE = GATED ? 8 : 16;
    constexpr int WINDOW = selfq_window(RG, NT, STEPS), PREV = selfq_prev_steps(STEPS);
    constexpr int SLICES = STEPS < 4 ? STEPS : 4;     // code blocks (8 rows x 128 bytes) of a wavefront
    constexpr int PER_WAVE = SLICES * 1024 > NT * 1024 ? SLICES * 1024 : NT * 1024;
    constexpr bool MAKES_AMAX = EPI != EPI_NONE;
    static_assert(SCALE == SELFQ_OWN || EPI == EPI_NONE, "handed-over and static scales: plain projections");
    __shared__ __attribute__((aligned(1024))) uint8_t smem[SQ_WAVES * PER_WAVE];
    __shared__ uint32_t amax_tbl[SCALE == SELFQ_OWN ? SQ_WAVES * ROWS : 1];
    __shared__ uint32_t amax_made[MAKES_AMAX ? ROWS : 1];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q = lane >> 4;
    const int xr = lane >> 4, xc = lane & 15;         // row loads: 16 lanes per row, 8 elements per lane
    const int half_n = N / 2, n_out_total = GATED ? half_n : N;
    const int col0 = blockIdx.x * (COLS_PER_TILE * NT), m_base = blockIdx.y * ROWS;
    const int total_steps = (K + 127) >> 7;

    // ---- the rows of this wavefront's K steps (rows past M repeat the last one) --------------------------------
    uint4 xv[STEPS][RG];
    const uint8_t* xp[RG];
#pragma unroll
    for (int i = 0; i < RG; ++i) {
        const int r = m_base + 4 * i + xr;
        xp[i] = a_x + (size_t)(r < M ? r : M - 1) * (uint32_t)ldx_bytes;
    }
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        int at = (j * SQ_WAVES + wave) * 256 + xc * 16;
        if (j >= PREV) at = at < 2 * K ? at : 2 * K - 16;
#pragma unroll
        for (int i = 0; i < RG; ++i) xv[j][i] = *reinterpret_cast<const uint4*>(xp[i] + at);
    }
    uint4 am[SCALE == SELFQ_HANDED ? 4 : 1];
    if constexpr (SCALE == SELFQ_HANDED) {   // 64 slots of 8 rows per load: lane l takes 8 slots of row l / 8
        const int r = m_base + (lane >> 3);
        const uint8_t* at = static_cast<const uint8_t*>(a_handed) + (size_t)(r < M ? r : M - 1) * (kRowAmaxSlots * 2) + (lane & 7) * 16;
#pragma unroll
        for (int a = 0; a < 4; ++a) am[a] = *reinterpret_cast<const uint4*>(at + (64 * a < a_parts ? a : 0) * 128);
    }
    float s_static = 1.0f;
    if constexpr (SCALE == SELFQ_STATIC) s_static = *static_cast<const float*>(a_handed);
    __builtin_amdgcn_sched_barrier(0);

    // ---- the first weights ------------------------------------------------------------------------------------
    const uint8_t* wp[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        if constexpr (OPERAND) {
            const uint32_t units = (uint32_t)N >> 4, u = blockIdx.x * NT + nt;
            wp[nt] = a_w + (size_t)(u < units ? u : units - 1) * (uint32_t)total_steps * kOperandStepBytes + lane * 16;
        } else {
            int wr;
            if constexpr (GATED) {   // the row order of a gated tile, see gemm_skinny_fused.hip
                const int g = col0 + nt * 8 + 2 * (l16 >> 2) + (l16 & 1);
                wr = ((l16 & 2) ? half_n : 0) + (g < half_n ? g : half_n - 1);
            } else {
                const int r = col0 + nt * 16 + l16;
                wr = r < N ? r : N - 1;
            }
            wp[nt] = a_w + (size_t)wr * (uint32_t)K;
        }
    }
    v4i wlo[WINDOW][NT], whi[WINDOW][NT];
    auto request = [&](int j) {
        const int s = j * SQ_WAVES + wave;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            if constexpr (OPERAND) {
                const uint8_t* at = wp[nt] + (size_t)(j < PREV || s < total_steps ? s : total_steps - 1) * kOperandStepBytes;
                wlo[j % WINDOW][nt] = *reinterpret_cast<const v4i*>(at);
                whi[j % WINDOW][nt] = *reinterpret_cast<const v4i*>(at + 1024);
            } else {
                int lo = s * 128 + q * 16, hi = lo + 64;
                if (j >= PREV) { lo = lo < K ? lo : K - 16; hi = hi < K ? hi : K - 16; }
                wlo[j % WINDOW][nt] = *reinterpret_cast<const v4i*>(wp[nt] + lo);
                whi[j % WINDOW][nt] = *reinterpret_cast<const v4i*>(wp[nt] + hi);
            }
        }
    };
#pragma unroll
    for (int j = 0; j < WINDOW; ++j) request(j);
    __builtin_amdgcn_sched_barrier(0);

    // ---- row scales -------------------------------------------------------------------------------------------
#pragma unroll
    for (int j = PREV; j < STEPS; ++j) {
        const uint32_t keep = (j * SQ_WAVES + wave) * 128 + xc * 8 < K ? ~0u : 0u;
#pragma unroll
        for (int i = 0; i < RG; ++i) { xv[j][i].x &= keep; xv[j][i].y &= keep; xv[j][i].z &= keep; xv[j][i].w &= keep; }
    }
    // A row with an Inf or NaN has that scale: its products are NaN through x * rcp(s) as through the division, so the
    // whole output row is, and no second form of the conversion is needed here, where the codes themselves go nowhere.
    float s_row = 1.0f, r_row = 1.0f;   // own: lane l <-> row l; handed over: lanes 8 r .. 8 r + 7 <-> row r
    if constexpr (SCALE == SELFQ_OWN) {
#pragma unroll
        for (int i = 0; i < RG; ++i) {
            uint32_t m2 = 0;
#pragma unroll
            for (int j = 0; j < STEPS; ++j) m2 = absmax8_pk(xv[j][i], m2);
            uint32_t v = absmax_finish(m2), o;
            o = dpp_move_u32<0xB1>(v);  v = o > v ? o : v;      // the 16 lanes of a row
            o = dpp_move_u32<0x4E>(v);  v = o > v ? o : v;
            o = dpp_move_u32<0x141>(v); v = o > v ? o : v;
            o = dpp_move_u32<0x140>(v); v = o > v ? o : v;
            if (xc == 0) amax_tbl[wave * ROWS + 4 * i + xr] = v;
        }
    }
    if constexpr (MAKES_AMAX) {
        if (tid < ROWS) amax_made[tid] = 0u;
    }
    if constexpr (SCALE == SELFQ_OWN) {
        __syncthreads();
        if (lane < ROWS) {
            uint32_t a = amax_tbl[lane];
#pragma unroll
            for (int w = 1; w < SQ_WAVES; ++w) a = amax_tbl[w * ROWS + lane] > a ? amax_tbl[w * ROWS + lane] : a;
            s_row = scale_from_amax_bits<QUANT_ACT_DYNAMIC>(a);
        }
    } else if constexpr (SCALE == SELFQ_HANDED) {
        uint32_t m2 = 0;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const int e0 = 64 * a + 8 * (lane & 7);   // this lane's first slot of the load
            const uint32_t w[4] = {am[a].x, am[a].y, am[a].z, am[a].w};
            uint32_t k[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                k[i] = w[i] & ((e0 + 2 * i < a_parts ? 0x7FFFu : 0u) | (e0 + 2 * i + 1 < a_parts ? 0x7FFF0000u : 0u));
            m2 = absmax8_pk(make_uint4(k[0], k[1], k[2], k[3]), m2);
        }
        uint32_t v = absmax_finish(m2), o;
        o = dpp_move_u32<0xB1>(v);  v = o > v ? o : v;          // the 8 lanes of a row
        o = dpp_move_u32<0x4E>(v);  v = o > v ? o : v;
        o = dpp_move_u32<0x141>(v); v = o > v ? o : v;
        s_row = scale_from_amax_bits<QUANT_ACT_DYNAMIC>(v);
    } else {
        s_row = s_static;
    }
    if constexpr (SCALE != SELFQ_STATIC) r_row = biased_reciprocal(s_row);
    auto of_row = [&](float v, int row) -> float {
        if constexpr (SCALE == SELFQ_STATIC) return v;
        const int src = SCALE == SELFQ_HANDED ? 8 * row : row;
        return __uint_as_float((uint32_t)__builtin_amdgcn_ds_bpermute(src << 2, (int)__float_as_uint(v)));
    };
    const float sa = of_row(s_row, l16 & (ROWS - 1));
    const StaticDivisor ds = make_static_divisor(s_static);
    RowDivisor dv[RG];
#pragma unroll
    for (int i = 0; i < RG; ++i) {
        dv[i].s = 1.0f;   // (not used: every row takes the reciprocal)
        dv[i].r = of_row(r_row, 4 * i + xr);
        dv[i].fast = true;
    }

    // ---- column operands and residual of the epilogue -------------------------------------------------------------
    const int e_nt = wave < NT ? wave : 0, e_m = m_base + l16, e_n = col0 + e_nt * COLS_PER_TILE + (GATED ? 2 : 4) * q;
    const bool e_live = wave < NT && l16 < ROWS && e_m < M && e_n < n_out_total;
    const int e_n_safe = e_live ? e_n : 0;
    v4f sw4 = {0.f, 0.f, 0.f, 0.f}, su4 = {0.f, 0.f, 0.f, 0.f};
    uint2 bw2 = make_uint2(0, 0), bu2 = make_uint2(0, 0), res2 = make_uint2(0, 0), gate2 = make_uint2(0, 0);
    if constexpr (GATED) {
        const float2 sg = *reinterpret_cast<const float2*>(a_w_scale + e_n_safe), su = *reinterpret_cast<const float2*>(a_w_scale + half_n + e_n_safe);
        sw4 = v4f{sg.x, sg.y, 0.f, 0.f};
        su4 = v4f{su.x, su.y, 0.f, 0.f};
        if (a_bias) {
            bw2.x = *reinterpret_cast<const uint32_t*>(a_bias + e_n_safe);
            bu2.x = *reinterpret_cast<const uint32_t*>(a_bias + half_n + e_n_safe);
        }
    } else {
        sw4 = *reinterpret_cast<const v4f*>(a_w_scale + e_n_safe);
        if (a_bias) bw2 = *reinterpret_cast<const uint2*>(a_bias + e_n_safe);
    }
    if constexpr (EPI == EPI_NONE) {
        if (a_res.residual != nullptr && e_live) {
            res2 = *reinterpret_cast<const uint2*>(a_res.residual + (int64_t)e_m * a_res.ld_res + e_n);
            gate2 = *reinterpret_cast<const uint2*>(a_res.gate + (int64_t)(e_m / a_res.gate_group) * a_res.ld_gate + e_n);
        }
    }

    // ---- codes, MFMAs -----------------------------------------------------------------------------------------------
    uint8_t* mine = smem + wave * PER_WAVE;
    const int xl = l16 & (ROWS - 1), xswz = (xl >> 1) & 7;
    const int rd_lo = xl * 128 + ((q ^ xswz) << 4), rd_hi = xl * 128 + (((4 + q) ^ xswz) << 4);
    v4f acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = v4f{0.f, 0.f, 0.f, 0.f};
    if (SCALE == SELFQ_STATIC && __builtin_expect(!ds.fast, 0)) {
        // a scale at the ends of the fp32 range: the division, step by step
#pragma nounroll
        for (int s = wave; s < total_steps; s += SQ_WAVES) {
#pragma unroll
            for (int i = 0; i < RG; ++i) {
                const int at = s * 256 + xc * 16, r = 4 * i + xr;
                uint4 v = *reinterpret_cast<const uint4*>(xp[i] + (at < 2 * K ? at : 2 * K - 16));
                if (at >= 2 * K) v = make_uint4(0, 0, 0, 0);
                uint2 c = encode8_static_exact(v, ds.s);
                if (at >= 2 * K) c = make_uint2(0, 0);   // (0 / 0)
                *reinterpret_cast<uint2*>(mine + r * 128 + (((xc >> 1) ^ ((r >> 1) & 7)) << 4) + (xc & 1) * 8) = c;
            }
            const v4i lo = *reinterpret_cast<const v4i*>(mine + rd_lo), hi = *reinterpret_cast<const v4i*>(mine + rd_hi);
            v8i xb;
#pragma unroll
            for (int e = 0; e < 4; ++e) { xb[e] = lo[e]; xb[4 + e] = hi[e]; }
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                int w_lo = OPERAND ? s * (int)kOperandStepBytes : s * 128 + q * 16, w_hi = OPERAND ? w_lo + 1024 : w_lo + 64;
                if (!OPERAND) { w_lo = w_lo < K ? w_lo : K - 16; w_hi = w_hi < K ? w_hi : K - 16; }
                const v4i a = *reinterpret_cast<const v4i*>(wp[nt] + w_lo), b = *reinterpret_cast<const v4i*>(wp[nt] + w_hi);
                v8i wb;
#pragma unroll
                for (int e = 0; e < 4; ++e) { wb[e] = a[e]; wb[4 + e] = b[e]; }
                acc[nt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wb, xb, acc[nt], 0, 0, 0, 0, 0, 0);
            }
        }
    } else
#pragma unroll
    for (int j0 = 0; j0 < STEPS; j0 += SLICES) {
#pragma unroll
        for (int j = j0; j < j0 + SLICES && j < STEPS; ++j)
#pragma unroll
            for (int i = 0; i < RG; ++i) {
                const int r = 4 * i + xr;
                uint2 c;
                if constexpr (SCALE == SELFQ_STATIC) {
                    // (a NaN makes its output row NaN; which of the 8 elements it is does not matter here)
                    c = encode8_static_fast(xv[j][i], ds);
                    if (absmax_finish(absmax8_pk(xv[j][i], 0u)) > 0x7F80u) c = make_uint2(0x7F7F7F7Fu, 0x7F7F7F7Fu);
                }
                else c = encode8<QUANT_ACT_DYNAMIC>(xv[j][i], dv[i]);
                *reinterpret_cast<uint2*>(mine + (j - j0) * 1024 + r * 128 + (((xc >> 1) ^ ((r >> 1) & 7)) << 4) + (xc & 1) * 8) = c;
            }
#pragma unroll
        for (int j = j0; j < j0 + SLICES && j < STEPS; ++j) {
            const v4i lo = *reinterpret_cast<const v4i*>(mine + (j - j0) * 1024 + rd_lo), hi = *reinterpret_cast<const v4i*>(mine + (j - j0) * 1024 + rd_hi);
            v8i xb;
#pragma unroll
            for (int e = 0; e < 4; ++e) { xb[e] = lo[e]; xb[4 + e] = hi[e]; }
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                v8i wb;
#pragma unroll
                for (int e = 0; e < 4; ++e) { wb[e] = wlo[j % WINDOW][nt][e]; wb[4 + e] = whi[j % WINDOW][nt][e]; }
                acc[nt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wb, xb, acc[nt], 0, 0, 0, 0, 0, 0);
            }
            if (j + WINDOW < STEPS) request(j + WINDOW);
        }
        __builtin_amdgcn_sched_barrier(0);   // (conversions of later steps hoisted up here would spill)
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the sums below overwrite this wavefront's codes

    // ---- the eight wavefronts' sums, in wavefront order; epilogue as in gemm_skinny_fused.hip ---------------------
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) reinterpret_cast<v4f*>(mine)[nt * kWave + lane] = acc[nt];
    __syncthreads();
    if (wave < NT) {
        auto part = [&](int w) { return reinterpret_cast<const v4f*>(smem + w * PER_WAVE)[e_nt * kWave + lane]; };
        v4f g = part(0);
#pragma unroll
        for (int w = 1; w < SQ_WAVES; ++w) g += part(w);
        const float bwf[4] = {bf16_bits_to_f32(bw2.x & 0xFFFFu), bf16_bits_to_f32(bw2.x >> 16), bf16_bits_to_f32(bw2.y & 0xFFFFu),
                              bf16_bits_to_f32(bw2.y >> 16)};
        uint32_t p0, p1 = 0;
        if constexpr (GATED) {
            const float buf[2] = {bf16_bits_to_f32(bu2.x & 0xFFFFu), bf16_bits_to_f32(bu2.x >> 16)};
            float vf[2];
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                float v = __builtin_fmaf(g[r], sa * sw4[r], bwf[r]);
                float up = __builtin_fmaf(g[2 + r], sa * su4[r], buf[r]);
                round_bf16_pair(v, up);
                vf[r] = apply_act<EPI>(v) * up;
            }
            p0 = pack_bf16x2(vf[0], vf[1]);
            if (e_live) *reinterpret_cast<uint32_t*>(a_out + (int64_t)e_m * a_ldo + e_n) = p0;
        } else {
            float vf[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float v = __builtin_fmaf(g[r], sa * sw4[r], bwf[r]);
                if constexpr (EPI != EPI_NONE) v = apply_act<EPI>(round_bf16(v));
                vf[r] = v;
            }
            if constexpr (EPI == EPI_NONE) {
                if (a_res.residual != nullptr) addcmul4(vf, res2, gate2);
            }
            p0 = pack_bf16x2(vf[0], vf[1]);
            p1 = pack_bf16x2(vf[2], vf[3]);
            if (e_live) *reinterpret_cast<uint2*>(a_out + (int64_t)e_m * a_ldo + e_n) = make_uint2(p0, p1);
        }
        if constexpr (MAKES_AMAX) {
            if (a_amax_out != nullptr && e_live) {
                const u16x2_t m = __builtin_elementwise_max(__builtin_bit_cast(u16x2_t, p0 & 0x7FFF7FFFu), __builtin_bit_cast(u16x2_t, p1 & 0x7FFF7FFFu));
                atomicMax(&amax_made[l16], absmax_finish(__builtin_bit_cast(uint32_t, m)));
            }
        }
    }
    if constexpr (MAKES_AMAX) {
        if (a_amax_out != nullptr) {
            __syncthreads();
            if (tid < ROWS && m_base + tid < M) a_amax_out[(size_t)(m_base + tid) * kRowAmaxSlots + blockIdx.x] = (uint16_t)amax_made[tid];
        }
    }
}

template <int RG, int NT, int STEPS, int EPI, bool OPERAND, int SCALE>
static int selfq_launch_layout(const GemmProblem& g, const SelfqPlan& pl, const void* handed, hipStream_t st) {
    if constexpr ((OPERAND && EPI != EPI_NONE) || !selfq_exists(RG, NT, STEPS, OPERAND, SCALE)) {
        return -2;
    } else {
        hipLaunchKernelGGL((gemm_fp8_selfq_kernel<RG, NT, STEPS, EPI, OPERAND, SCALE>), dim3(pl.tiles, pl.msplit), dim3(SQ_THREADS), 0, st, g.w,
                           reinterpret_cast<const uint8_t*>(g.x_bf16), g.K, g.N, g.M, (int)(g.ldx * 2), handed, g.amax_parts, g.w_scale, g.bias,
                           g.out, g.ldo, residual_of(g), EPI != EPI_NONE ? g.amax_out : nullptr);
        return 0;
    }
}

template <int RG, int NT, int STEPS, int EPI, int SCALE>
static int selfq_launch(const GemmProblem& g, const SelfqPlan& pl, const void* handed, hipStream_t st) {
    return g.weight_layout == W_ROW_MAJOR ? selfq_launch_layout<RG, NT, STEPS, EPI, false, SCALE>(g, pl, handed, st)
                                          : selfq_launch_layout<RG, NT, STEPS, EPI, true, SCALE>(g, pl, handed, st);
}

template <int RG, int STEPS, int EPI, int SCALE>
static int selfq_launch_nt(const GemmProblem& g, const SelfqPlan& pl, const void* handed, hipStream_t st) {
    switch (pl.nt) {
    case 1: return selfq_launch<RG, 1, STEPS, EPI, SCALE>(g, pl, handed, st);
    case 2: return selfq_launch<RG, 2, STEPS, EPI, SCALE>(g, pl, handed, st);
    case 4: return selfq_launch<RG, 4, STEPS, EPI, SCALE>(g, pl, handed, st);
    case 8: return selfq_launch<RG, 8, STEPS, EPI, SCALE>(g, pl, handed, st);
    default: return -2;
    }
}

template <int STEPS, int EPI, int SCALE>
static int selfq_launch_rg(const GemmProblem& g, const SelfqPlan& pl, const void* handed, hipStream_t st) {
    return pl.rg == 1 ? selfq_launch_nt<1, STEPS, EPI, SCALE>(g, pl, handed, st) : selfq_launch_nt<2, STEPS, EPI, SCALE>(g, pl, handed, st);
}

template <int SCALE>
static int selfq_launch_plain(const GemmProblem& g, const SelfqPlan& pl, const void* handed, hipStream_t st) {
    switch (pl.steps) {
    case 1: return selfq_launch_rg<1, EPI_NONE, SCALE>(g, pl, handed, st);
    case 2: return selfq_launch_rg<2, EPI_NONE, SCALE>(g, pl, handed, st);
    case 4: return selfq_launch_rg<4, EPI_NONE, SCALE>(g, pl, handed, st);
    case 6: return selfq_launch_rg<6, EPI_NONE, SCALE>(g, pl, handed, st);
    case 8: return selfq_launch_rg<8, EPI_NONE, SCALE>(g, pl, handed, st);
    case 12: return selfq_launch_rg<12, EPI_NONE, SCALE>(g, pl, handed, st);
    case 16: return selfq_launch_rg<16, EPI_NONE, SCALE>(g, pl, handed, st);
    default: return -2;
    }
}

}  // namespace phyai
