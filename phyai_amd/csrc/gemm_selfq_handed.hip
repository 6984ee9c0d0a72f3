// Self-quantizing small-M linears (gemm_selfq.h) on rows whose maxima their producer left.
#include "gemm_selfq.h"

namespace phyai {

int launch_selfq_handed(const GemmProblem& g, const SelfqPlan& pl, hipStream_t st) {
    if (g.epilogue != EPI_NONE || g.amax_in == nullptr || g.amax_parts < 1 || g.amax_parts > kRowAmaxSlots) return -2;
    return selfq_launch_plain<SELFQ_HANDED>(g, pl, g.amax_in, st);
}

}  // namespace phyai
