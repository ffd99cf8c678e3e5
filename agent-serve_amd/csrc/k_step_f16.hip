// The step kernel's F16 and Q6_K builds (k_step.hpp), in a translation unit of their own so that
// they compile beside the others.
#include "k_step.hpp"

namespace tfk {

hipError_t launch_step_f16(const StepArgs& a, int n_wg, hipStream_t st) {
    using step_detail::launch_t;
    constexpr int F16 = TF_HIP_TYPE_F16;
    return a.hd <= 64 ? launch_t<F16, F16, 64>(a, n_wg, st) : launch_t<F16, F16, 128>(a, n_wg, st);
}

hipError_t launch_step_q6k(const StepArgs& a, int n_wg, hipStream_t st) {
    using step_detail::launch_t;
    constexpr int Q6 = TF_HIP_TYPE_Q6_K;
    return a.hd <= 64 ? launch_t<Q6, Q6, 64>(a, n_wg, st) : launch_t<Q6, Q6, 128>(a, n_wg, st);
}

}  // namespace tfk
