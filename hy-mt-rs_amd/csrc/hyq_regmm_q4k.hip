// Few-token batched products of Q4_K weights (hyq_regmm_impl.hpp).
#include "hyq_regmm_impl.hpp"

namespace hyq {
template int launch_regmm_format<Q4_K>(const regmm::Args &a, int tb, void *stream);
} // namespace hyq
