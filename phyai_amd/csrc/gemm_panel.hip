// Linears of more than 48 token rows, up to 1024 of K and few enough output tiles that gemm_skinny_fused.hip and gemm_selfq.h
// do not take, in ONE launch: a workgroup quantizes the 16 token rows it multiplies into LDS, all of K, and multiplies from there.
//
// What bounds these calls is not bytes or operations (400 x 2560 x 1024: 1.1 us of either) but the two kernels' dependent
// trips to memory and the quantizer's own node and launch: 7.6 us in a graph (now 6.7), and called eagerly two launches, which
// cost the host 6 us (the call takes 1.27 - 1.45 times as long as one launch's: 400 x 2560 x 1024, 1000 x 1024 x 512,
// 100 x 1536 x 656).  Here a workgroup asks for rows, weights, scales and bias
// at once and waits for them once (for a gated residual and its gate once more, behind the MFMAs):
//
//  * four wavefronts own 64 NT weight rows x 16 token rows over the whole K; wavefront w converts four of the rows for all
//    of them (one barrier) and multiplies 16 NT weight rows, whose whole K is in flight in registers from the first
//    instructions on, behind the bf16 rows;
//  * the price is that every workgroup of a row converts it again: 16 x K elements at 4 (row scales) to 7 (one static scale,
//    whose division is exact for any fp32) instructions each.  Larger panels (32 or 64 rows) convert longer in one go and
//    were slower throughout; from K = 1536 on (16 steps) the conversions and the weights no longer in flight at once cost
//    what the launch saves (400 x 1024 x 2048 one scale 8.8 us in two launches, 9.1 in one);
//  * codes lie in K-step blocks of 16 rows x 128 bytes with the chunks of a row rotated, as in the other kernels.
//
// Codes are those of the stand-alone quantizers and sums come in the order of the GEMM kernel that the shape would run
// (BY_WAVES: weight streaming's eight sums of one K step each, added in turn; otherwise K ascending), so results are the
// same bits.  Measured in graphs over weight sets beyond the Infinity Cache, two launches / one, us, row scales | one scale:
//   400 x 2560 x 1024   7.6 / 6.7 | 7.8 / 7.0       400 x 1024 x 1024  6.6 / 5.3 | 6.8 / 5.7      544 x 1536 x 768 7.2 / 5.8 | 7.3 / 6.1
//   400 x  512 x  512   5.4 / 3.6 | 5.5 / 3.7      1000 x 1024 x  512  6.6 / 5.0 | 6.6 / 5.3      200 x 4096 x 512 6.4 / 4.9 | 6.7 / 5.1
#include <stdlib.h>

#include "fp8_device.h"
#include "launch.h"
#include "quant_device.h"
#include "tuning.h"
#include "weight_layout.h"

namespace phyai {

constexpr int PN_WAVES = 4, PN_THREADS = PN_WAVES * kWave;
constexpr int PN_ROWS = 16, PN_STEPS = 8;   // K <= 1024: as many K steps as weight streaming has wavefronts

template <int NT, bool OPERAND, bool STATIC, bool BY_WAVES>
__global__ __launch_bounds__(PN_THREADS) __attribute__((amdgpu_waves_per_eu(2)))
void gemm_fp8_panel_kernel(const uint8_t* __restrict__ a_w, const uint8_t* __restrict__ a_x, int K, int N, int M, int ldx_bytes, int n_tiles,
                           int m_tiles, const float* __restrict__ a_x_scale, const float* __restrict__ a_w_scale,
                           const uint16_t* __restrict__ a_bias, uint16_t* __restrict__ a_out, int64_t a_ldo, const ResidualArgs a_res) {
    __shared__ __attribute__((aligned(1024))) uint8_t panel[PN_STEPS * PN_ROWS * 128];
    __shared__ float row_scale[PN_ROWS];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q = lane >> 4;
    // tiles column after column, cut into eight equal runs, one per XCD: its L2 holds the run's weights once
    const int xcd = blockIdx.x & 7, total = n_tiles * m_tiles;
    const int e = ((xcd * total) >> 3) + (blockIdx.x >> 3);
    if (e >= (((xcd + 1) * total) >> 3)) return;
    const int tile_n = e / m_tiles, m_base = (e - tile_n * m_tiles) * PN_ROWS, col0 = (tile_n * PN_WAVES + wave) * (16 * NT);
    const int steps = (K + 127) >> 7;

    // ---- rows 4 wave .. 4 wave + 3 of the panel (rows past M repeat the last one): 16 lanes per row, 8 elements per lane and step
    const int xr = lane >> 4, xc = lane & 15, r = wave * 4 + xr;
    const uint8_t* xp = a_x + (size_t)(m_base + r < M ? m_base + r : M - 1) * (uint32_t)ldx_bytes + xc * 16;
    uint4 xv[PN_STEPS];
#pragma unroll
    for (int s = 0; s < PN_STEPS; ++s) {
        xv[s] = make_uint4(0, 0, 0, 0);
        if (s < steps && (OPERAND || s * 128 + xc * 8 < K)) xv[s] = *reinterpret_cast<const uint4*>(xp + s * 256);
    }
    float s_static = 1.0f;
    if constexpr (STATIC) s_static = *a_x_scale;
    __builtin_amdgcn_sched_barrier(0);

    // ---- column operands of the epilogue, the weights ------------------------------------------------------------------------
    v4f sw[NT];
    uint2 bw[NT];
    const uint8_t* wp[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int n = col0 + nt * 16 + 4 * q, n_safe = n < N ? n : 0;
        sw[nt] = *reinterpret_cast<const v4f*>(a_w_scale + n_safe);
        bw[nt] = make_uint2(0, 0);
        if (a_bias) bw[nt] = *reinterpret_cast<const uint2*>(a_bias + n_safe);
        if constexpr (OPERAND) {
            const uint32_t units = (uint32_t)N >> 4, u = (uint32_t)(tile_n * PN_WAVES + wave) * NT + nt;
            wp[nt] = a_w + (size_t)(u < units ? u : units - 1) * (uint32_t)steps * kOperandStepBytes + lane * 16;
        } else {
            const int row = col0 + nt * 16 + l16;
            wp[nt] = a_w + (size_t)(row < N ? row : N - 1) * (uint32_t)K;
        }
    }
    v4i wlo[PN_STEPS][NT], whi[PN_STEPS][NT];
#pragma unroll
    for (int s = 0; s < PN_STEPS; ++s) {
        if (s >= steps) break;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            if constexpr (OPERAND) {
                wlo[s][nt] = *reinterpret_cast<const v4i*>(wp[nt] + s * (int)kOperandStepBytes);
                whi[s][nt] = *reinterpret_cast<const v4i*>(wp[nt] + s * (int)kOperandStepBytes + 1024);
            } else {
                // (past the end of the row: its last chunk again, multiplied by zero codes)
                const int lo = s * 128 + q * 16, hi = lo + 64;
                wlo[s][nt] = *reinterpret_cast<const v4i*>(wp[nt] + (lo < K ? lo : K - 16));
                whi[s][nt] = *reinterpret_cast<const v4i*>(wp[nt] + (hi < K ? hi : K - 16));
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- codes -----------------------------------------------------------------------------------------------------------------
    {
        const StaticDivisor ds = make_static_divisor(s_static);
        RowDivisor d = {s_static, 1.0f, true};
        uint32_t m2 = 0, o;
#pragma unroll
        for (int s = 0; s < PN_STEPS; ++s) m2 = absmax8_pk(xv[s], m2);
        uint32_t v = absmax_finish(m2);
        bool odd = false;   // one static scale: NaNs or huge values, or a scale at the ends of the fp32 range
        if constexpr (STATIC) {
            odd = __builtin_amdgcn_ballot_w64(v >= kStaticPlainBf16) != 0 || !ds.fast;
        } else {
            o = dpp_move_u32<0xB1>(v);  v = o > v ? o : v;      // the 16 lanes of a row
            o = dpp_move_u32<0x4E>(v);  v = o > v ? o : v;
            o = dpp_move_u32<0x141>(v); v = o > v ? o : v;
            o = dpp_move_u32<0x140>(v); v = o > v ? o : v;
            d.s = scale_from_amax_bits<QUANT_ACT_DYNAMIC>(v);
            d.r = biased_reciprocal(d.s);
        }
        if (xc == 0) row_scale[r] = d.s;
        uint8_t* to = panel + r * 128 + (((xc >> 1) ^ ((r >> 1) & 7)) << 4) + (xc & 1) * 8;
        if (STATIC && __builtin_expect(odd, 0)) {
#pragma unroll
            for (int s = 0; s < PN_STEPS; ++s) {
                uint2 c = encode8_static_exact(xv[s], d.s);
                if (s * 128 + xc * 8 >= K) c = make_uint2(0, 0);   // (0 / 0)
                *reinterpret_cast<uint2*>(to + s * (PN_ROWS * 128)) = c;
            }
        } else {
#pragma unroll
            for (int s = 0; s < PN_STEPS; ++s) {
                uint2 c;
                if constexpr (STATIC) c = encode8_static_plain(xv[s], ds);
                else c = encode8<QUANT_ACT_DYNAMIC>(xv[s], d);   // (a row with an Inf or a NaN: codes of NaN throughout)
                if (s < steps) *reinterpret_cast<uint2*>(to + s * (PN_ROWS * 128)) = c;
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();

    // ---- MFMAs: the weight block is the first operand, so a lane owns four columns of one token row ----------------------------
    const int swz = (l16 >> 1) & 7;
    const int rd_lo = l16 * 128 + ((q ^ swz) << 4), rd_hi = l16 * 128 + (((4 + q) ^ swz) << 4);
    auto join = [](v4i lo, v4i hi) {
        v8i f;
#pragma unroll
        for (int i = 0; i < 4; ++i) { f[i] = lo[i]; f[4 + i] = hi[i]; }
        return f;
    };
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    v4f acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = zero;
#pragma unroll
    for (int s = 0; s < PN_STEPS; ++s) {
        if (s >= steps) break;
        const uint8_t* blk = panel + s * (PN_ROWS * 128);
        const v8i xb = join(*reinterpret_cast<const v4i*>(blk + rd_lo), *reinterpret_cast<const v4i*>(blk + rd_hi));
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const v8i wb = join(wlo[s][nt], whi[s][nt]);
            if constexpr (BY_WAVES) {
                const v4f part = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wb, xb, zero, 0, 0, 0, 0, 0, 0);
                acc[nt] = s == 0 ? part : acc[nt] + part;
            } else {
                acc[nt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wb, xb, acc[nt], 0, 0, 0, 0, 0, 0);
            }
        }
    }
    if constexpr (BY_WAVES) {
        if (steps < PN_STEPS) {   // (a wavefront without a step adds a zero: the sign of a zero sum)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) acc[nt] += zero;
        }
    }

    // ---- epilogue --------------------------------------------------------------------------------------------------------------
    const int m = m_base + l16;
    const float sa = row_scale[l16];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int n = col0 + nt * 16 + 4 * q;
        if (m >= M || n >= N) continue;
        const float bwf[4] = {bf16_bits_to_f32(bw[nt].x & 0xFFFFu), bf16_bits_to_f32(bw[nt].x >> 16), bf16_bits_to_f32(bw[nt].y & 0xFFFFu),
                              bf16_bits_to_f32(bw[nt].y >> 16)};
        float vf[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) vf[i] = __builtin_fmaf(acc[nt][i], sa * sw[nt][i], bwf[i]);
        if (a_res.residual != nullptr)
            addcmul4(vf, *reinterpret_cast<const uint2*>(a_res.residual + (int64_t)m * a_res.ld_res + n),
                     *reinterpret_cast<const uint2*>(a_res.gate + (int64_t)(m / a_res.gate_group) * a_res.ld_gate + n));
        *reinterpret_cast<uint2*>(a_out + (int64_t)m * a_ldo + n) = make_uint2(pack_bf16x2(vf[0], vf[1]), pack_bf16x2(vf[2], vf[3]));
    }
}

// Where one launch is ahead: workgroups of 64 columns up to 512 of them (two per CU at once), of 128 columns up to 512 again.
// A third round eats it: 513 - 768 workgroups of 128 columns 0.98 (K = 512) to 0.83 (K = 1024) of the speed of two launches.
// Row-major weights cost more the longer K is: K = 768 0.75 - 1.22 of the speed of two launches, 896 0.68 - 0.92 (why is not
// known: eight lanes to a row with the halves exchanged between lanes, i.e. 128-byte pieces, is level, and K steps in another
// order per wavefront 5 - 10 % worse), so K < 768 there, with 64 columns up to 768 workgroups.
// Over 520 linears drawn from what the rule
// takes (M = 49 - 11000, N = 16 - 23000), two launches took 1.4 to 1.5 times as long in the geometric mean, 1.01 at the least
// (89 x 6016 x 640 row-major).
PanelPlan panel_plan(int M, int N, int K, int epilogue, int64_t ldo, int weight_layout) {
    PanelPlan pl = {};
    if (const char* e = tuning_env("PHYAI_FP8_FUSED")) { if (atoi(e) == 0) return pl; }
    for (const char* kernel : {"PHYAI_FP8_BIG", "PHYAI_FP8_TILE", "PHYAI_FP8_SKINNY_PLAN"})   // (a tuning run that names a kernel gets it)
        if (tuning_env(kernel)) return pl;
    if (M <= 48 || K % 16 != 0 || K > PN_STEPS * 128 || N % 16 != 0 || ldo % 4 != 0 || epilogue != EPI_NONE) return pl;
    const bool operand = weight_layout != W_ROW_MAJOR;
    if (!operand && K >= 768) return pl;
    const int64_t m_tiles = ((int64_t)M + PN_ROWS - 1) / PN_ROWS;
    for (int nt = 1; nt <= (operand ? 2 : 1); ++nt) {
        const int64_t n_tiles = ((int64_t)N + 64 * nt - 1) / (64 * nt);
        if (m_tiles * n_tiles > (operand ? 512 : 768)) continue;
        pl.nt = nt; pl.n_tiles = (int)n_tiles; pl.m_tiles = (int)m_tiles;
        break;
    }
    return pl;
}

template <int NT, bool OPERAND, bool STATIC>
static int panel_launch(const GemmProblem& g, const PanelPlan& pl, bool by_waves, hipStream_t st) {
    const dim3 grid(8 * (unsigned)((pl.n_tiles * pl.m_tiles + 7) / 8));   // (eight runs of tiles)
    const uint8_t* x = reinterpret_cast<const uint8_t*>(g.x_bf16);
    const int ldx_bytes = (int)(g.ldx * 2);
    if (by_waves)
        hipLaunchKernelGGL((gemm_fp8_panel_kernel<NT, OPERAND, STATIC, true>), grid, dim3(PN_THREADS), 0, st, g.w, x, g.K, g.N, g.M, ldx_bytes,
                           pl.n_tiles, pl.m_tiles, g.x_scale, g.w_scale, g.bias, g.out, g.ldo, residual_of(g));
    else
        hipLaunchKernelGGL((gemm_fp8_panel_kernel<NT, OPERAND, STATIC, false>), grid, dim3(PN_THREADS), 0, st, g.w, x, g.K, g.N, g.M, ldx_bytes,
                           pl.n_tiles, pl.m_tiles, g.x_scale, g.w_scale, g.bias, g.out, g.ldo, residual_of(g));
    return 0;
}

int launch_gemm_panel(const GemmProblem& g, const PanelPlan& pl, bool by_waves, hipStream_t st) {
    const bool operand = g.weight_layout != W_ROW_MAJOR, one_scale = g.x_scale_is_scalar != 0;
    if (pl.nt == 2) return one_scale ? panel_launch<2, true, true>(g, pl, by_waves, st) : panel_launch<2, true, false>(g, pl, by_waves, st);
    if (pl.nt != 1) return -2;
    if (operand) return one_scale ? panel_launch<1, true, true>(g, pl, by_waves, st) : panel_launch<1, true, false>(g, pl, by_waves, st);
    return one_scale ? panel_launch<1, false, true>(g, pl, by_waves, st) : panel_launch<1, false, false>(g, pl, by_waves, st);
}

}  // namespace phyai
