// Score pass (select_kernel.hpp) for fp16 operands.
#include "select_kernel.hpp"

namespace asa {

hipError_t launch_select_f16(const SelectParams& p, hipStream_t s) { return launch_type<h16>(p, s); }

}  // namespace asa
