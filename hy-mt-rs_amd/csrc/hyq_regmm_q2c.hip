// Few-token batched products of Q2_0C weights (hyq_regmm_impl.hpp).
#include "hyq_regmm_impl.hpp"

namespace hyq {
template int launch_regmm_format<Q2_0C>(const regmm::Args &a, int tb, void *stream);
} // namespace hyq
