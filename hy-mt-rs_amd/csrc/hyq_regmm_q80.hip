// Few-token batched products of Q8_0 weights (hyq_regmm_impl.hpp).
#include "hyq_regmm_impl.hpp"

namespace hyq {
template int launch_regmm_format<Q8_0>(const regmm::Args &a, int tb, void *stream);
} // namespace hyq
