// Score pass (select_kernel.hpp) for fp32 operands and for caller-given scores, and its LDS sizes.
#include "select_kernel.hpp"

namespace asa {

hipError_t launch_select_f32(const SelectParams& p, hipStream_t s) { return launch_type<float>(p, s); }

hipError_t launch_select_scores(const SelectParams& p, hipStream_t s) {
  return launch_r<float, 64, kGivenScores>(p, s);
}

size_t select_lds_bytes(const Dims& d, int dtype, bool from_scores, int cap) {
  (void)dtype;
  (void)from_scores;
  return size_t(sel_layout(d.k, cap, d.nKB).total);
}

int select_capacity(const Dims& d, int dtype, bool from_scores, size_t max_lds) {
  // k + 32 keys per row holds the candidates of random rows with room to
  // spare up to k = 42, and 1.75 k above (the floor's slack grows with k; at
  // k = 64 two blocks still share a compute unit, above it one runs either
  // way); less still works (overflow rounds), as long as it exceeds k.
  int cap = d.k + (d.k * 3 / 4 > 32 ? d.k * 3 / 4 : 32);
  if (cap > 256) cap = 256;
  while (cap > d.k && select_lds_bytes(d, dtype, from_scores, cap) > max_lds) cap -= 8;
  return cap > d.k ? cap : -1;
}

}  // namespace asa
