// Few-token batched products of STQ1_0 weights (hyq_regmm_impl.hpp).
#include "hyq_regmm_impl.hpp"

namespace hyq {
template int launch_regmm_format<STQ1_0>(const regmm::Args &a, int tb, void *stream);
} // namespace hyq
