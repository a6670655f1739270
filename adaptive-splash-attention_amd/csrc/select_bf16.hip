// Score pass (select_kernel.hpp) for bf16 operands.
#include "select_kernel.hpp"

namespace asa {

hipError_t launch_select_bf16(const SelectParams& p, hipStream_t s) { return launch_type<u16>(p, s); }

}  // namespace asa
