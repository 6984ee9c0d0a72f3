// Self-quantizing small-M linears (gemm_selfq.h) with one static activation scale.
#include "gemm_selfq.h"

namespace phyai {

int launch_selfq_static(const GemmProblem& g, const SelfqPlan& pl, hipStream_t st) {
    if (g.epilogue != EPI_NONE || !g.x_scale_is_scalar) return -2;
    return selfq_launch_plain<SELFQ_STATIC>(g, pl, g.x_scale, st);
}

}  // namespace phyai
