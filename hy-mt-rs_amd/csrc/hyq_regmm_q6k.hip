// Few-token batched products of Q6_K weights (hyq_regmm_impl.hpp).
#include "hyq_regmm_impl.hpp"

namespace hyq {
template int launch_regmm_format<Q6_K>(const regmm::Args &a, int tb, void *stream);
} // namespace hyq
