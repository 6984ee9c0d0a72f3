// Self-quantizing small-M linears (gemm_selfq.h) with an activation epilogue.
#include "gemm_selfq.h"

namespace phyai {

template <int EPI>
static int launch_act(const GemmProblem& g, const SelfqPlan& pl, hipStream_t st) {
    if (g.weight_layout != W_ROW_MAJOR || (g.amax_out != nullptr && pl.tiles > kRowAmaxSlots)) return -2;
    switch (pl.steps) {
    case 1: return selfq_launch_rg<1, EPI, SELFQ_OWN>(g, pl, nullptr, st);
    case 2: return selfq_launch_rg<2, EPI, SELFQ_OWN>(g, pl, nullptr, st);
    default: return -2;
    }
}

int launch_selfq_own_act(const GemmProblem& g, const SelfqPlan& pl, hipStream_t st) {
    switch (g.epilogue) {
    case EPI_GEGLU_TANH: return launch_act<EPI_GEGLU_TANH>(g, pl, st);
    case EPI_GEGLU_ERF: return launch_act<EPI_GEGLU_ERF>(g, pl, st);
    case EPI_SWIGLU: return launch_act<EPI_SWIGLU>(g, pl, st);
    case EPI_GELU_TANH: return launch_act<EPI_GELU_TANH>(g, pl, st);
    case EPI_GELU_ERF: return launch_act<EPI_GELU_ERF>(g, pl, st);
    default: return -2;
    }
}

}  // namespace phyai
