// Self-quantizing small-M linears (gemm_selfq.h): plan, dispatch and the plain kernels that find their own row maxima.
#include "gemm_selfq.h"
#include "tuning.h"
#include <stdlib.h>

namespace phyai {

static int sq_ceil_div(int a, int b) { return (a + b - 1) / b; }

// Up to 48 token rows - 128 with one static scale, which spares the tables and their barriers - whose workgroups (4 or 8
// rows, as few weight tiles each as keeps the grid within the 256 CUs) run in one round: with a second round the repeated
// conversions (rows x K elements, 5.5 / 64 cycles each) cost more than the quantizer's launch.  Activation epilogues
// exist for row-major weights up to K = 2048 (gemm_skinny_fused.hip serves the rest of what an MLP's first projection is).
SelfqPlan selfq_plan(int M, int N, int K, int epilogue, int64_t ldo, int weight_layout, int source) {
    SelfqPlan pl = {0, 0, 0, 0, 0};
    if (const char* e = tuning_env("PHYAI_FP8_FUSED")) { if (atoi(e) == 0) return pl; }
    if (M < 1 || M > (source == SELFQ_FROM_SCALAR ? 128 : 48) || K % 16 != 0 || K > 16384 || ldo % 4 != 0) return pl;
    const bool gated = epi_is_gated(epilogue), plain = epilogue == EPI_NONE;
    if (!plain && (weight_layout != W_ROW_MAJOR || K > 2048 || source != SELFQ_FROM_ROWS)) return pl;
    const int cols = gated ? N / 2 : N;
    if (cols % 8 != 0) return pl;
    const int per_wave = sq_ceil_div(sq_ceil_div(K, 128), SQ_WAVES);
    int steps = 0;
    for (int s : kSelfqSteps)
        if (s >= per_wave) { steps = s; break; }
    const int rg = M <= 4 ? 1 : 2, msplit = sq_ceil_div(M, 4 * rg), per_tile = gated ? 8 : 16;
    for (int nt = 1; nt <= 8; nt *= 2) {
        const int tiles = sq_ceil_div(cols, per_tile * nt);
        if ((int64_t)tiles * msplit > 256) continue;
        const bool operand = weight_layout != W_ROW_MAJOR;
        if (K > selfq_max_k(rg, nt, operand, source == SELFQ_FROM_SCALAR)) break;
        if (!selfq_exists(rg, nt, steps, operand, source)) continue;
        pl.rg = rg; pl.nt = nt; pl.steps = steps; pl.tiles = tiles; pl.msplit = msplit;
        break;
    }
    return pl;
}

int launch_selfq_own(const GemmProblem& g, const SelfqPlan& pl, hipStream_t st) { return selfq_launch_plain<SELFQ_OWN>(g, pl, nullptr, st); }

int launch_gemm_selfq(const GemmProblem& g, const SelfqPlan& pl, int source, hipStream_t st) {
    if (pl.rg == 0) return -2;
    if (source == SELFQ_FROM_SCALAR) return launch_selfq_static(g, pl, st);
    if (source == SELFQ_FROM_MAXIMA) return launch_selfq_handed(g, pl, st);
    return g.epilogue == EPI_NONE ? launch_selfq_own(g, pl, st) : launch_selfq_own_act(g, pl, st);
}

}  // namespace phyai
